"""The library's multi-tensor cast against PyTorch's, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("widen", [False, True])
def test_same_bits_as_pytorch(half, widen):
    from semicat_amd import _lib
    src, dst = (half, torch.float32) if widen else (torch.float32, half)
    gen = torch.Generator("cuda").manual_seed(0)
    # ends of a thread's eight elements, of a workgroup's 8192 and none at all; more tensors than a launch takes
    sizes = [0, 1, 7, 8, 9, 8191, 8192, 8193, 20000, 3, 16384, 5, 64, 2, 1000, 12345, 77, 100001, 31]
    base = [torch.randn(n + 3, device="cuda", generator=gen) * 10.0 ** (i % 9 - 4) for i, n in enumerate(sizes)]
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 1e-45, 3.4e38, 65519.9, 65520.0, 1.00390625,
                            1.01171875, 6e-8, 2.9e-8], device="cuda")
    base.append(special.repeat(11))
    for off in (0, 1, 3):  # off the 16-byte boundaries
        x = [t.to(src)[off:off + n] for t, n in zip(base, sizes + [120])]
        x.insert(2, None)
        x.append(torch.randn(4, 6, 8, device="cuda", generator=gen).to(src).transpose(0, 1))
        x.append(torch.randn(5, device="cuda", generator=gen).to(dst))
        got = _lib.host().cast(x, dst)
        assert got[2] is None and got[-1] is x[-1]
        for t, y in zip(x, got):
            if t is None:
                continue
            ref = t.to(dst)
            assert y.dtype == dst and y.shape == ref.shape and y.stride() == ref.stride()
            assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y[~y.isnan()], ref[~ref.isnan()])
            assert torch.equal(y[~y.isnan()].signbit(), ref[~ref.isnan()].signbit())


def test_calls_that_are_left_to_pytorch():
    from semicat_amd import _lib
    cast = _lib.host().cast
    x = torch.randn(4, 6, device="cuda")
    assert cast([x[:, ::2]], torch.bfloat16) is None and cast([x[:1].expand(4, 6)], torch.bfloat16) is None
    assert cast([x.double()], torch.bfloat16) is None and cast([x.bfloat16()], torch.float16) is None
    assert cast([x, x.half()], torch.bfloat16) is None and cast([x.cpu()], torch.bfloat16) is None
    assert cast((x,), torch.bfloat16) is None and cast([x] * 65, torch.bfloat16) is None
    assert cast([], torch.bfloat16) == [] and cast([None], torch.bfloat16) == [None]


def test_status_of_the_entry_point():
    import ctypes
    from semicat_amd import _lib
    lib = _lib.load()
    one, none, count = (ctypes.c_void_p * 1)(16), (ctypes.c_void_p * 1)(), (ctypes.c_int64 * 1)(8)
    f32, bf16, fp16 = _lib.SJVP_FP32, _lib.SJVP_BF16, _lib.SJVP_FP16
    assert lib.sjvp_cast(1, None, one, count, f32, bf16, None) == _lib.SJVP_ERR_NULL
    assert lib.sjvp_cast(1, none, one, count, f32, bf16, None) == _lib.SJVP_ERR_NULL
    assert lib.sjvp_cast(0, one, one, count, f32, bf16, None) == lib.sjvp_cast(17, one, one, count, f32, bf16, None) != 0
    assert lib.sjvp_cast(1, one, one, (ctypes.c_int64 * 1)(-1), f32, bf16, None) != 0
    for a, b in ((f32, f32), (bf16, bf16), (bf16, fp16), (fp16, bf16), (7, f32), (f32, 7)):
        assert lib.sjvp_cast(1, one, one, count, a, b, None) != 0
    assert lib.sjvp_cast(1, none, none, (ctypes.c_int64 * 1)(0), f32, bf16, None) == 0
