"""Which built files count as fresh (the host extension only beside the torch and the interpreter it was compiled for), and the
library without the extension."""
import sysconfig

import pytest
import torch

from semicat_amd import _lib, build, kernels


@pytest.fixture
def built():
    if build.is_stale():
        build.build()
    assert not build.is_stale()
    _lib.load()  # before anything is changed: loading builds what is stale


@pytest.mark.parametrize("change", [
    lambda m: m.setattr(torch, "__version__", torch.__version__ + "x"),
    lambda m: m.setattr(torch.version, "hip", "0.0"),
    lambda m: m.setattr(torch, "compiled_with_cxx11_abi", lambda now=torch.compiled_with_cxx11_abi(): not now),
    lambda m: m.setattr(sysconfig, "get_config_var", lambda name: "cpython-399"),
    lambda m: m.setattr(build, "HOST_FLAGS", build.HOST_FLAGS + ["-DX"]),
])
def test_extension_of_another_environment_is_stale(built, monkeypatch, change):
    library = build.source_id()
    change(monkeypatch)
    assert build.is_stale()
    assert build.source_id() == library  # the C library has no part of torch in it
    with pytest.raises(RuntimeError, match="another torch"):
        _lib._load_host(_lib.load())


def test_library_without_the_extension(built, monkeypatch):
    """The C library builds, loads and serves calls where the extension does not: one warning, then the general form."""
    monkeypatch.setattr(build, "host_is_stale", lambda: True)
    failing = []

    def fail(*a):
        failing.append(1)
        raise RuntimeError("the compiler failed")

    monkeypatch.setattr(build, "host_command", fail)
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(_lib, "_lib", None)
    assert _lib.load().sjvp_version() >= 1
    assert not failing  # nothing but a call asks for the extension
    with pytest.warns(RuntimeWarning, match="host extension"):
        assert _lib.host() is False
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    assert not kernels._on_gpu(torch.zeros(1)) and len(failing) == 1


def test_library_is_written_where_the_extension_fails(monkeypatch):
    done = []
    monkeypatch.setattr(build, "_run", lambda cmd, verbose: done.append(cmd[-1]))
    monkeypatch.setattr(build.os, "replace", lambda a, b: done.append(b))
    monkeypatch.setattr(build.os, "makedirs", lambda *a, **k: None)

    def no_torch():
        raise ModuleNotFoundError("torch")

    monkeypatch.setattr(build, "host_command", no_torch)
    with pytest.raises(ModuleNotFoundError):
        build.build()
    assert done[-1] == build.LIB_PATH
