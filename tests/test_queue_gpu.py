"""GPU parity of the uneven-batch work queue (pcx_queue_*): transforms of every power-of-two size
from 2 to 2^20, mixed directions, at arbitrary offsets, each checked against the FP64 oracle;
eager execution, hipGraph replays (with eager work between them) and the autotuned schedule."""
import numpy as np
import pytest

from helpers import fft_tol

pytestmark = pytest.mark.gpu


def _jobs(rng, sizes):
    jobs, off = [], 0
    for lg in sizes:
        inv = int(rng.integers(0, 2))
        n = 1 << lg
        off += int(rng.integers(0, 3)) * 8  # gaps between vectors
        jobs.append((lg, inv, off, off))
        off += 2 * n
    return jobs, off


def _fill(orc, jobs, total):
    buf = np.zeros(total, np.float32)
    data = []
    for k, (lg, inv, so, _) in enumerate(jobs):
        n = 1 << lg
        z = orc.gen_normal(0x5EED0004 + k, n)
        buf[so:so + n] = z.real
        buf[so + n:so + 2 * n] = z.imag
        data.append(z.astype(np.complex128))
    return buf, data


def _check(orc, jobs, data, out, normalized=True):
    worst = 0.0
    for (lg, inv, _, do), z in zip(jobs, data):
        n = 1 << lg
        got = out[do:do + n].astype(np.float64) + 1j * out[do + n:do + 2 * n]
        want = orc.fft64(z, inverse=bool(inv))
        if inv and normalized:
            want = want / n
        err = orc.rel_l2(got, want)
        assert err < fft_tol(n), (lg, inv, err)
        worst = max(worst, err / fft_tol(n))
    return worst


@pytest.fixture(scope="module")
def pa():
    import packed_amd

    return packed_amd


def _case(orc, seed):
    rng = np.random.default_rng(seed)
    sizes = [int(v) for v in rng.integers(1, 13, 200)] + list(range(1, 21)) + [13, 14, 15, 16, 16, 18]
    rng.shuffle(sizes)
    jobs, total = _jobs(rng, sizes)
    buf, data = _fill(orc, jobs, total)
    return jobs, total, buf, data


def test_queue_eager(orc, pa):
    import torch

    jobs, total, buf, data = _case(orc, 1)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    q = pa.fft_queue(jobs)
    q.exec(dst.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())
    f, b = q.work()
    assert b == sum(16 * (1 << lg) for lg, *_ in jobs)


def test_queue_in_place_unnormalized(orc, pa):
    import torch

    jobs, total, buf, data = _case(orc, 2)
    x = torch.from_numpy(buf).cuda()
    q = pa.fft_queue(jobs, normalized=False)
    q.exec(x.data_ptr(), x.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, x.cpu().numpy(), normalized=False)


def test_queue_graph_replays(orc, pa):
    """Captured pass replayed three times with eager work in between; every replay checked."""
    import torch

    jobs, total, buf, data = _case(orc, 3)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    q = pa.fft_queue(jobs)
    s = torch.cuda.Stream()
    q.capture(dst.data_ptr(), src.data_ptr(), s)
    for rep in range(3):
        dst.zero_()
        torch.cuda.synchronize()
        q.launch(s)
        s.synchronize()
        _check(orc, jobs, data, dst.cpu().numpy())
        junk = torch.randn(1 << 20, device="cuda") * 2  # eager work between replays
        torch.cuda.synchronize()
        del junk


def test_queue_autotune_and_cache(orc, pa, tmp_path):
    import torch

    jobs, total, buf, data = _case(orc, 4)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    cache = str(tmp_path / "tune.txt")
    q = pa.fft_queue(jobs)
    q.autotune(dst.data_ptr(), src.data_ptr(), cache)
    dst.zero_()
    q.exec(dst.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())
    text = open(cache).read()
    assert "queue_grid " in text
    q2 = pa.fft_queue(jobs)
    q2.autotune(dst.data_ptr(), src.data_ptr(), cache)  # reads the cache
    dst.zero_()
    q2.exec(dst.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())


def test_capture_then_autotune_then_capture(orc, pa):
    """Autotuning after a capture drops the captured graph (its kernels, grids and twiddle tables
    may all change); launching it fails until the queue is captured again, and the new graph
    gives the oracle's results.  Autotuning refuses dst == src (it overwrites dst many times)."""
    import torch

    from packed_amd import PcxError

    jobs, total, buf, data = _case(orc, 5)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    q = pa.fft_queue(jobs)
    s = torch.cuda.Stream()
    q.capture(dst.data_ptr(), src.data_ptr(), s)
    with pytest.raises(PcxError):
        q.autotune(src.data_ptr(), src.data_ptr())
    q.autotune(dst.data_ptr(), src.data_ptr())
    with pytest.raises(PcxError):
        q.launch(s)
    q.capture(dst.data_ptr(), src.data_ptr(), s)
    dst.zero_()
    torch.cuda.synchronize()
    q.launch(s)
    s.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())


def test_queue_above_persistent_range(orc, pa):
    """Sizes above 2^20 run as grouped launches after the persistent one, in the same pass."""
    import torch

    rng = np.random.default_rng(6)
    jobs, total = _jobs(rng, [21, 5, 16, 21, 20, 12])
    buf, data = _fill(orc, jobs, total)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    q = pa.fft_queue(jobs)
    q.exec(dst.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())


@pytest.mark.parametrize("extra", [1, 181])
def test_queue_many_of_one_large_size(orc, pa, extra):
    """More 2^16 transforms of each direction than the GPU has CUs, at scattered offsets: full
    rounds of one transform per CU with a short and a nearly full last one."""
    import torch

    n, count = 1 << 16, torch.cuda.get_device_properties(0).multi_processor_count + extra
    slots = np.random.default_rng(7).permutation(2 * count)
    jobs = [(16, k % 2, int(slots[k]) * 2 * n, (2 * count - 1 - k) * 2 * n) for k in range(2 * count)]
    src = torch.randn(4 * count * n, generator=torch.Generator("cuda").manual_seed(8), device="cuda")
    dst = torch.zeros_like(src)
    q = pa.fft_queue(jobs)
    q.exec(dst.data_ptr(), src.data_ptr())
    picks = [0, 1, count, 2 * count - extra - 2, 2 * count - 2, 2 * count - 1]
    part = [jobs[k] for k in picks]
    data = []
    for _, _, so, _ in part:
        x = src[so:so + 2 * n].cpu().numpy().astype(np.float64)
        data.append(x[:n] + 1j * x[n:])
    _check(orc, part, data, dst.cpu().numpy())


@pytest.mark.parametrize("graph_first", [False, True])
def test_replay_and_eager_pass_on_two_streams(orc, pa, graph_first):
    """An eager pass on one stream and a replay of the captured graph on another, with no
    synchronisation between them: both go through the queue's one intermediate, so the later waits."""
    import torch

    jobs, at = [], 0
    for lg, count in ((17, 24), (18, 12), (20, 5)):
        for k in range(count):
            jobs.append((lg, k % 2, at, at))
            at += 2 << lg
    gen = torch.Generator("cuda").manual_seed(9)
    srcs = [torch.randn(at, generator=gen, device="cuda") for _ in range(2)]
    dsts = [torch.zeros_like(s) for s in srcs]
    q = pa.fft_queue(jobs)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    q.capture(dsts[1].data_ptr(), srcs[1].data_ptr(), streams[1])
    torch.cuda.synchronize()

    def eager():
        q.exec(dsts[0].data_ptr(), srcs[0].data_ptr(), streams[0])

    def replay():
        q.launch(streams[1])

    for rep in range(4):
        for d in dsts:
            d.zero_()
        torch.cuda.synchronize()
        for call in ((replay, eager) if graph_first else (eager, replay)):
            call()
        torch.cuda.synchronize()
        for src, dst in zip(srcs, dsts):
            part = [jobs[k] for k in (0, 23, 24, 35, 36, 40)]
            data = []
            for lg, _, so, _ in part:
                x = src[so:so + (2 << lg)].cpu().numpy().astype(np.float64)
                data.append(x[:1 << lg] + 1j * x[1 << lg:])
            for (lg, inv, _, do), z in zip(part, data):
                y = dst[do:do + (2 << lg)].cpu().numpy().astype(np.float64)
                want = np.fft.ifft(z) if inv else np.fft.fft(z)
                assert orc.rel_l2(y[:1 << lg] + 1j * y[1 << lg:], want) < fft_tol(1 << lg), (rep, lg, inv)


def test_tuning_file_of_the_earlier_queue(orc, pa, tmp_path):
    """A file written when the persistent launch took sizes to 2^20: its classes above 2^14 are full-chip
    launches in any case, its workgroup count is cut to the launch's own, its shapes are taken."""
    import torch

    jobs, total, buf, data = _case(orc, 10)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    cache = tmp_path / "tune.txt"
    cache.write_text("grouped 9 0\ngrouped 15 0\ngrouped 15 1\ngrouped 18 1\ngrouped 20 0\ngrouped 20 1\nqueue_grid 4096\n"
                     "group 20 0 10 16 16 2048 2048\ngroup 20 1 10 16 16 1024 1024\ngroup 18 1 9 32 32 0 0\n"
                     "group 15 0 7 32 64 1024 1024\ngroup 15 1 7 64 128 0 0\n")
    text = cache.read_text()
    q = pa.fft_queue(jobs)
    q.autotune(dst.data_ptr(), src.data_ptr(), str(cache))
    q.exec(dst.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    _check(orc, jobs, data, dst.cpu().numpy())
    assert cache.read_text() == text


def test_queue_of_one_pass_transforms_needs_little_memory(pa):
    """1500 transforms of 2^16 run one per CU without an intermediate but for the last round: the queue
    holds one round's, not the 750 MiB of the whole list."""
    import torch

    n, count = 1 << 16, 1500
    jobs = [(16, 0, k * 2 * n, k * 2 * n) for k in range(count)]
    first = pa.fft_queue(jobs[:1])  # what the library itself holds
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    q = pa.fft_queue(jobs)
    torch.cuda.synchronize()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert free - torch.cuda.mem_get_info()[0] < (cus + 64) * 8 * n
    del first, q


def _many(seed, jobs, low, high):
    rng = np.random.default_rng(seed)
    return _jobs(rng, [int(v) for v in rng.integers(low, high + 1, jobs)])


@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("mixed", [0, 1])
def test_one_launch_over_mixed_sizes_or_launches_per_class(orc, pa, tmp_path, mixed, normalized):
    """Both forms of the sizes up to 2^18 (named by a tuning file), of every size from 2 on: eager, in
    place, and replayed with eager work between the replays; larger sizes run beside either."""
    import torch

    rng = np.random.default_rng(11)
    sizes = list(range(1, 20)) * 2 + [1, 3, 14, 15, 15, 15, 16, 16, 17, 18, 18] + [int(v) for v in rng.integers(5, 17, 60)]
    rng.shuffle(sizes)
    jobs, total = _jobs(rng, sizes)
    buf, data = _fill(orc, jobs, total)
    src = torch.from_numpy(buf).cuda()
    dst = torch.zeros_like(src)
    cache = tmp_path / "tune.txt"
    cache.write_text(f"queue_grid 512\nmixed {mixed}\n")
    q = pa.fft_queue(jobs, normalized=normalized)
    q.autotune(dst.data_ptr(), src.data_ptr(), str(cache))
    for rep in range(2):
        dst.zero_()
        q.exec(dst.data_ptr(), src.data_ptr())
        torch.cuda.synchronize()
        _check(orc, jobs, data, dst.cpu().numpy(), normalized)
    want = dst.clone()
    s = torch.cuda.Stream()
    q.capture(dst.data_ptr(), src.data_ptr(), s)
    for rep in range(3):
        dst.zero_()
        torch.cuda.synchronize()
        q.launch(s)
        s.synchronize()
        assert torch.equal(dst, want)
        torch.randn(1 << 20, device="cuda").mul_(2)
        torch.cuda.synchronize()
    q.exec(src.data_ptr(), src.data_ptr())
    torch.cuda.synchronize()
    for lg, _, _, do in jobs:  # (the gaps between the vectors are src's own)
        assert torch.equal(src[do:do + (2 << lg)], want[do:do + (2 << lg)])


@pytest.mark.parametrize("lines", [False, True])
@pytest.mark.parametrize("jobs,low,high", [(1400, 7, 16), (1000, 10, 17), (1000, 12, 18), (50, 4, 18), (400, 16, 16)])
def test_the_faster_of_the_two_forms_is_chosen(pa, tmp_path, jobs, low, high, lines):
    """Where the forms differ by a fifth and more: many classes of moderate count run as one launch, few
    transforms or one large class as launches per class.  The choice is within 10 % of the faster."""
    import torch

    todo, total = _many(jobs + high, jobs, low, high)
    if lines:  # every vector on whole 128-byte lines
        todo = [(lg, inv, (so + 31) // 32 * 32 + 32 * k, (do + 31) // 32 * 32 + 32 * k)
                for k, (lg, inv, so, do) in enumerate(todo)]
        total += 32 * jobs + 32
    src = torch.randn(total, device="cuda")
    dst = torch.zeros_like(src)
    times = []
    for mixed in (None, 0, 1):
        q = pa.fft_queue(todo)
        if mixed is not None:
            cache = tmp_path / f"{mixed}.txt"
            cache.write_text(f"queue_grid 512\nmixed {mixed}\n")
            q.autotune(dst.data_ptr(), src.data_ptr(), str(cache))
        best = float("inf")
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(3):
                q.exec(dst.data_ptr(), src.data_ptr())
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    assert times[0] < 1.1 * min(times[1:]), times
