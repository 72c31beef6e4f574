"""The fused element-wise calls report their own status: an error that another HIP call has left on the thread is neither
taken for theirs nor cleared."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def test_error_of_another_call():
    from semicat_amd import _lib
    lib = _lib.load()
    u = torch.randn(4096, device="cuda").bfloat16()
    x = torch.randn(2, 8, 64, device="cuda").bfloat16()
    y, z, gate = torch.empty_like(u), torch.empty_like(x), torch.ones(2, 64, device="cuda").bfloat16()
    p = _lib.AdaLn(x=x.data_ptr(), a=x.data_ptr(), gate=gate.data_ptr(), y=z.data_ptr(), B=2, S=8, W=64)
    p.mod_stride[0] = 64
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream().cuda_stream
    try:
        assert lib.hipSetDevice(1 << 20) != 0  # refused by the runtime, which remembers the error
        status = lib.sjvp_gelu(u.data_ptr(), None, None, None, y.data_ptr(), None, u.numel(), 0, stream)
        status_norm = lib.sjvp_adaln_fwd(ctypes.byref(p), 0, stream)
    finally:
        left = lib.hipGetLastError()
    assert (status, status_norm) == (_lib.SJVP_OK, _lib.SJVP_OK)
    assert left != 0
    torch.cuda.synchronize()
    assert (y.float() - F.gelu(u.float(), approximate="tanh")).abs().max() < 0.05
    assert torch.equal(z, x * 2)
