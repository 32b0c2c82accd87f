"""GPU parity on both sides of the sizes where a call changes kernels: small-tile and default
four-step shapes, the one-pass forms of 2^15 (FP64: 2^14), for every order and direction.

The first, a middle and the last transform of each call against numpy's FP64 FFT in slot order,
within the bounds of the FFT path (FP32 2 log2N FLT_EPSILON, FP64 4 log2N DBL_EPSILON relative L2).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = [(15, 47), (15, 48), (15, 159), (15, 160), (15, 161), (16, 1024), (16, 1025), (17, 128), (17, 129), (17, 513),
       (18, 4), (18, 5), (18, 257), (19, 4), (19, 5), (19, 9), (20, 2), (20, 3), (20, 65)]
F64 = [(14, 95), (14, 96), (14, 97), (15, 32), (15, 33), (15, 513), (16, 2), (16, 3), (16, 257), (17, 3), (18, 1), (18, 2),
       (19, 8), (19, 9), (20, 4), (20, 5)]


@pytest.mark.parametrize("order", ["normal", "bit_reversed", "unordered"])
@pytest.mark.parametrize("dtype,lg,batch", [("float32", *c) for c in F32] + [("float64", *c) for c in F64])
def test_shape_limits(orc, order, dtype, lg, batch):
    import torch

    import packed_amd as pa

    if dtype == "float64" and order == "unordered":
        pytest.skip("no FP64 unordered order")
    n = 1 << lg
    src = pa.md_storage(n, batch, dtype=dtype)
    src.data.copy_(torch.randn(src.data.numel(), generator=torch.Generator("cuda").manual_seed(lg * 4096 + batch),
                               device="cuda", dtype=src.data.dtype))
    dst = pa.md_storage(n, batch, dtype=dtype)
    unit = pa.fft_unit(n, order=order, dtype=dtype)
    tol = 2 * lg * 2.0 ** -23 if dtype == "float32" else 4 * lg * 2.0 ** -52
    slots = orc.slot_freq(order, n)
    picks = sorted({0, batch // 2, batch - 1})
    unit(dst, src)
    for b in picks:
        want = np.fft.fft(src[b].to_complex())[slots]
        assert orc.rel_l2(dst[b].to_complex(), want) < tol, b
    unit.ifft(dst, src)
    for b in picks:
        spec = np.empty(n, np.complex128)
        spec[slots] = src[b].to_complex()
        assert orc.rel_l2(dst[b].to_complex(), np.fft.ifft(spec)) < tol, b
