"""The autotuner times the kernel that an untuned plan runs, so that tuning never ends with a slower one
for want of having tried it."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import glob, sys
import dtfft_amd as D
D.lib().dtfft_hip_set_cache_dir(sys.argv[1].encode())
n, lines, hm = (int(v) for v in sys.argv[3:])
D.FFTExecutor(2, D.FFTType.C2C, D.Precision.SINGLE, n * lines, n * lines, hm, [n, lines], effort=D.Effort[sys.argv[2]])
for f in glob.glob(sys.argv[1] + "/*.name"):
    if "kernel" in open(f).read():
        print("kernel", open(f).read())
"""


def kernels(path, effort, n, lines, hm):
    path.mkdir()
    out = subprocess.run([sys.executable, "-c", CHILD, str(path), effort, str(n), str(lines), str(hm)], cwd=ROOT,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stderr
    return {ln.split(" ", 1)[1].strip() for ln in out.stdout.splitlines() if ln.startswith("kernel ")}


@pytest.mark.parametrize("n,lines,hm", [
    (210, 64, 128),   # in-place columns by LDS-DMA: 15 14 on 16 threads
    (320, 64, 128),   # 8 8 5 on 32 threads
    (512, 64, 1024),  # 32-line tiles of the plain kernel
    (60, 210, 8),     # few lines: the plain kernel
])
def test_measure_times_the_default(n, lines, hm, tmp_path):
    print(f"case: columns of {n}, {lines} x {hm} lines", flush=True)
    untuned = kernels(tmp_path / "estimate", "ESTIMATE", n, lines, hm)
    timed = kernels(tmp_path / "measure", "MEASURE", n, lines, hm)
    assert untuned and untuned <= timed, untuned - timed
