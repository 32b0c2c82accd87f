"""GPU parity of transforms of interleaved data (pack 1 on both sides), whose single-pass kernels move an
element's two parts in one access: sizes on both sides of each kernel's range, bases that are aligned to
one value only, zero-extended sources, in place, both directions.

Against numpy's FP64 FFT within the bounds of the FFT path (FP32 2 log2N FLT_EPSILON, FP64 4 log2N
DBL_EPSILON relative L2); the words around the data keep their value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["normal", "bit_reversed"])
@pytest.mark.parametrize("dtype,lg,batch", [("float32", lg, b) for lg, b in
                                            ((9, 3), (10, 1), (10, 7), (11, 5), (12, 3), (13, 3), (14, 3), (15, 161),
                                             (15, 769), (16, 181))] +
                         [("float64", lg, b) for lg, b in ((9, 3), (10, 5), (11, 3), (12, 3), (13, 2), (14, 97))])
def test_interleaved(orc, dtype, lg, batch, order):
    import torch

    import packed_amd as pa

    n = 1 << lg
    rt = torch.float32 if dtype == "float32" else torch.float64
    dist = 2 * n + 5
    gen = torch.Generator("cuda").manual_seed(lg * 1000 + batch)
    src = torch.randn(batch * dist + 1, generator=gen, device="cuda", dtype=rt)
    tol = 2 * lg * 2.0 ** -23 if dtype == "float32" else 4 * lg * 2.0 ** -52
    unit = pa.fft_unit(n, order=order, dtype=dtype)
    slots = orc.slot_freq(order, n)
    step = src.element_size()

    def vec(t, b):
        x = t[1 + b * dist:1 + b * dist + 2 * n].cpu().numpy().astype(np.float64)
        return x[0::2] + 1j * x[1::2]

    for inverse, size, inplace in ((False, n, False), (True, n, False), (False, n - 3, False), (True, n, True)):
        work = src.clone()
        dst = work if inplace else torch.full_like(src, 7.0)
        unit.batch(dst.data_ptr() + step, work.data_ptr() + step, batch, 1, dist, 1, dist, inverse=inverse,
                   src_size=size)
        for b in sorted({0, batch // 2, batch - 1}):
            z = vec(src, b)
            if inverse:
                spec = np.empty(n, np.complex128)
                spec[slots] = z
                want = np.fft.ifft(spec)
            else:
                want = np.fft.fft(np.where(np.arange(n) < size, z, 0))[slots]
            assert orc.rel_l2(vec(dst, b), want) < tol, (inverse, size, b)
        keep = torch.ones_like(src, dtype=torch.bool)
        keep[1:].view(batch, dist)[:, :2 * n] = False
        assert bool((dst[keep] == (src[keep] if inplace else 7.0)).all())
