"""Which built files count as fresh: the host extension only beside the torch and the interpreter it was compiled for."""
import sysconfig

import pytest
import torch

from semicat_amd import _lib, build


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
