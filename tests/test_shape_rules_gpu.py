"""GPU parity on both sides of the sizes where a call changes kernels: small-tile and default
four-step shapes, the one-pass forms of 2^15 (FP64: 2^14), for every order and direction.

The first, a middle and the last transform of each call against numpy's FP64 FFT in slot order,
within the bounds of the FFT path (FP32 2 log2N FLT_EPSILON, FP64 4 log2N DBL_EPSILON relative L2).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = [(15, 47), (15, 48), (15, 159), (15, 160), (15, 161), (16, 1024), (16, 1025), (17, 128), (17, 129), (17, 513),
       (18, 4), (18, 5), (18, 257), (19, 4), (19, 5), (19, 9), (20, 2), (20, 3), (20, 4), (20, 5), (20, 65)]
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


@pytest.mark.parametrize("src_pack,dst_pack", [(1, 8), (8, 1), (64, 128), (128, 0), (0, 64), (8, 256), (8, None)])
@pytest.mark.parametrize("lg,rounds,rest", [(15, 3, 1), (16, 0, 180), (16, 1, 0), (16, 1, 1), (16, 1, 180)])
def test_whole_transforms_per_cu(orc, lg, rounds, rest, src_pack, dst_pack):
    """Natural-order 2^15 / 2^16 in one pass, one transform per CU and round: packs on both sides
    (0: the whole transform, None: in place; 256 is not taken), both directions, transforms spaced
    apart, guards between them untouched."""
    import torch

    import packed_amd as pa

    n = 1 << lg
    batch = rounds * torch.cuda.get_device_properties(0).multi_processor_count + rest
    src_pack = src_pack or n
    inplace, dst_pack = dst_pack is None, src_pack if dst_pack is None else dst_pack or n
    dist = 2 * n + 64
    src = torch.randn(batch * dist, generator=torch.Generator("cuda").manual_seed(lg + batch), device="cuda")
    keep = src.clone()
    tol = 2 * lg * 2.0 ** -23

    def vec(t, b, pack):
        x = t[b * dist:b * dist + 2 * n].cpu().numpy().astype(np.float64).reshape(n // pack, 2, pack)
        return (x[:, 0] + 1j * x[:, 1]).reshape(n)

    unit = pa.fft_unit(n)
    for inverse in (False, True):
        src.copy_(keep)
        dst = src if inplace else torch.full((batch * dist,), 7.0, device="cuda")
        unit.batch(dst.data_ptr(), src.data_ptr(), batch, dst_pack, dist, src_pack, dist, inverse=inverse)
        for b in sorted({0, batch // 2, max(batch - 1 - rest, 0), batch - 1}):
            z = vec(keep, b, src_pack)
            want = np.fft.ifft(z) if inverse else np.fft.fft(z)
            assert orc.rel_l2(vec(dst, b, dst_pack), want) < tol, (inverse, b)
        gaps = dst.view(batch, dist)[:, 2 * n:]
        assert bool((gaps == (keep.view(batch, dist)[:, 2 * n:] if inplace else 7.0)).all())


def _storages(n, batch, dtype, seed):
    import torch

    import packed_amd as pa

    src, dst = pa.md_storage(n, batch, dtype=dtype), pa.md_storage(n, batch, dtype=dtype)
    src.data.copy_(torch.randn(src.data.numel(), generator=torch.Generator("cuda").manual_seed(seed), device="cuda",
                               dtype=src.data.dtype))
    return src, dst


@pytest.mark.parametrize("dtype,lg,batch,order", [("float64", 14, 97, "normal"), ("float64", 14, 97, "bit_reversed"),
                                                  ("float32", 15, 161, "normal"), ("float32", 15, 161, "unordered")])
@pytest.mark.parametrize("inverse", [False, True])
def test_named_shape_is_the_one_that_runs(dtype, lg, batch, order, inverse):
    """A call that would run in one pass takes the four-step of a shape that was named (in place: the
    out-of-place form of 2^15 follows the one-pass switch): within the bounds of both, not bit for bit,
    and back to the first result with the automatic choice."""
    import torch

    import packed_amd as pa

    n = 1 << lg
    src, work = _storages(n, batch, dtype, lg + batch)
    unit = pa.fft_unit(n, order=order, dtype=dtype)
    outs = []
    for shape in (0, 7, 0):
        unit.set_shape(shape)
        work.data.copy_(src.data)
        unit.ifft(work) if inverse else unit(work)
        outs.append(work.data.clone())
    eps = 2.0 ** -23 if dtype == "float32" else 2.0 ** -52
    diff = float(torch.linalg.norm((outs[0] - outs[1]).double()) / torch.linalg.norm(outs[0].double()))
    assert 0 < diff < 4 * lg * eps
    assert torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("dtype,lg,batch,order", [("float64", 14, 701, "normal"), ("float32", 15, 800, "bit_reversed"),
                                                  ("float32", 16, 512, "normal")])
def test_row_cap_holds_for_whole_transforms(dtype, lg, batch, order):
    """The one-pass forms run under the caller's cap of row workgroups: 8 of them on 256 CUs take many
    times as long, with the same result bit for bit."""
    import torch

    import packed_amd as pa

    src, dst = _storages(1 << lg, batch, dtype, lg + batch)
    unit = pa.fft_unit(1 << lg, order=order, dtype=dtype)
    times, outs = [], []
    for cap in (0, 8):
        unit.set_grid(cap, cap)
        best = float("inf")
        for _ in range(3):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            unit(dst, src)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
        outs.append(dst.data.clone())
    assert torch.equal(outs[0], outs[1])
    assert times[1] > 4 * times[0], times


@pytest.mark.parametrize("dtype,lg,batch,order", [("float32", 15, 4, "normal"), ("float32", 15, 161, "unordered"),
                                                  ("float32", 15, 800, "normal"), ("float32", 16, 200, "normal"),
                                                  ("float64", 14, 97, "normal"), ("float64", 14, 97, "bit_reversed")])
@pytest.mark.parametrize("inverse", [False, True])
def test_one_pass_switch(dtype, lg, batch, order, inverse):
    """Every one-pass form (k_dif, one workgroup per transform, one per CU) against the four-step that the
    switch selects: within the bounds of both, not bit for bit, and on again as before."""
    import torch

    import packed_amd as pa

    n = 1 << lg
    src, dst = _storages(n, batch, dtype, lg + batch)
    unit = pa.fft_unit(n, order=order, dtype=dtype)
    outs = []
    for on in (None, False, True):
        if on is not None:
            unit.set_one_pass(on)
        unit.ifft(dst, src) if inverse else unit(dst, src)
        outs.append(dst.data.clone())
    eps = 2.0 ** -23 if dtype == "float32" else 2.0 ** -52
    diff = float(torch.linalg.norm((outs[0] - outs[1]).double()) / torch.linalg.norm(outs[0].double()))
    assert 0 < diff < 4 * lg * eps
    assert torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("dtype,lg,order", [("float32", 16, "bit_reversed"), ("float32", 17, "normal"),
                                            ("float32", 14, "normal"), ("float64", 15, "normal")])
def test_one_pass_switch_refused(dtype, lg, order):
    """Plans without a one-pass form refuse to turn it on."""
    import packed_amd as pa

    unit = pa.fft_unit(1 << lg, order=order, dtype=dtype)
    unit.set_one_pass(False)
    with pytest.raises(pa.PcxError):
        unit.set_one_pass(True)


@pytest.mark.parametrize("dtype,lg,other", [("float32", 15, 17), ("float32", 16, 17), ("float64", 14, 15)])
def test_one_pass_tables_cost_no_plan_time(dtype, lg, other):
    """Plans with tables of one-pass forms are made as fast as the next size's without (the quickest of
    many plans made in turn; the tables of a plan are filled by one launch)."""
    import time

    import torch

    import packed_amd as pa

    torch.zeros(1, device="cuda")
    times = {lg: [], other: []}
    for _ in range(200):
        for k in times:
            start = time.perf_counter()
            unit = pa.fft_unit(1 << k, dtype=dtype)
            times[k].append(time.perf_counter() - start)
            del unit
    a, b = min(times[lg]), min(times[other])
    assert a < 1.12 * b, (a, b)


@pytest.mark.parametrize("dtype,lg,batch,src_pack,dst_pack",
                         [("float32", lg, b, s, d) for lg, b in ((15, 161), (15, 769), (16, 256))
                          for s, d in ((1, 8), (8, 1), (2, 4))] +
                         [("float64", 14, 97, s, d) for s, d in ((1, 4), (4, 1), (2, 4))])
@pytest.mark.parametrize("inverse", [False, True])
def test_one_pass_in_place_between_small_packs(dtype, lg, batch, src_pack, dst_pack, inverse):
    """In place with two different packs of up to one register: a workgroup has read its whole
    transform before it writes, so the result is that of the out-of-place call bit for bit."""
    import torch

    import packed_amd as pa

    n = 1 << lg
    rt = torch.float32 if dtype == "float32" else torch.float64
    src = torch.randn(batch * 2 * n, generator=torch.Generator("cuda").manual_seed(lg), device="cuda", dtype=rt)
    dst = torch.zeros_like(src)
    unit = pa.fft_unit(n, dtype=dtype)
    for out in (dst, src):
        unit.batch(out.data_ptr(), src.data_ptr(), batch, dst_pack, 2 * n, src_pack, 2 * n, inverse=inverse)
    assert torch.equal(dst, src)
