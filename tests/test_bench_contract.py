"""CPU checks of bench.py's command-line contract that need no GPU: more than one GPU is refused
with a message (this build measures one GPU's share), before anything touches a device."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    res = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                         text=True, timeout=120)
    assert res.returncode != 0
    assert "one GPU" in res.stderr
    assert res.stdout.strip() == ""  # no JSON line


def test_help_lists_the_workload_switches():
    res = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--help"], capture_output=True, text=True,
                         timeout=120)
    assert res.returncode == 0
    for flag in ("--steps", "--warmup", "--gpus", "--config", "--dtype", "--precision"):
        assert flag in res.stdout


@pytest.mark.parametrize("log2n,batch,dtype,precision,want", [
    (16, 4096, "float32", "fp32", "k_tile, one transform per CU"),
    (16, 64, "float32", "fp32", "four-step"), (16, 180, "float32", "fp32", "k_tile, one"),
    (16, 257, "float32", "fp32", "k_tile for 256 transforms, then four-step column pass k_col + row pass k_row for 1 "),
    (16, 4096, "float32", "fp16x2", "four-step"), (16, 4096, "float64", "fp32", "four-step"),
    (15, 47, "float32", "fp32", "k_dif"), (15, 512, "float32", "fp32", "single pass k_row, one"),
    (15, 769, "float32", "fp32", "k_tile, one"), (12, 65536, "float32", "fp32", "single pass k_row ("),
    (14, 701, "float64", "fp32", "single pass k_row, one"), (14, 95, "float64", "fp32", "four-step"),
    (21, 4, "float32", "fp32", "three passes"), (21, 4, "float32", "bf16x3", "four-step")])
def test_roofline_names_the_kernels_that_run(log2n, batch, dtype, precision, want):
    """The kernels of a forward step on 256 CUs depend on the batch, not on the size alone, and the
    traffic summary that is quoted is that form's."""
    import bench

    assert bench.forward_kernels(log2n, batch, dtype, precision, 256).startswith(want)
    assert ("_tile_" in bench.traffic_profile(log2n, batch, dtype, 256)) == (
        precision == "fp32" and want.startswith("k_tile, one")) or precision != "fp32"
