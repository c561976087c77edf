"""R2R executors whose lines are spaced differently in and out (idist != odist).  In place, blocks of
one launch would write lines that other blocks have yet to read, so such stages hold the three
launches through the work buffer beside the one launch, and overlapping buffers take them.

Bars on the GPU: FP64 within 1e-12 relative L2 of the oracle, FP32 within 2e-6 (the R2R tests' own)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle.r2r as R

D = pytest.importorskip("dtfft_amd")
P = D.Precision
TOL = {P.DOUBLE: 1e-12, P.SINGLE: 2e-6}
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import glob, sys
import dtfft_amd as D
from dtfft_amd import _lib
_lib.lib().dtfft_hip_set_cache_dir(sys.argv[1].encode())
rank, n, idist, odist, kind = (int(v) for v in sys.argv[2:])
sizes = [n] if rank == 1 else [6, n]
D.FFTExecutor(rank, D.FFTType.R2R, D.Precision.DOUBLE, idist, odist, 5, sizes, r2r_kinds=[kind] * rank)
print(" ".join(sorted({k for f in glob.glob(sys.argv[1] + "/*.name") for k in ("r2r_pre", "r2r_post")
                       if k in open(f).read()})))
"""


@pytest.mark.parametrize("rank,n,idist,odist,three", [
    (1, 21, 21, 21, False), (1, 64, 64, 64, False),
    (1, 21, 21, 24, True), (1, 64, 70, 64, True),
    (2, 20, 120, 120, False), (2, 20, 120, 128, True), (2, 16, 128, 96, True),
])
@pytest.mark.parametrize("kind", [R.DCT_2, R.DST_4])
def test_three_launches_are_set_up(kind, rank, n, idist, odist, three, tmp_path):
    """Compile-only: the kernels of the three launches belong to the executor where spacings differ."""
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    out = subprocess.run([sys.executable, "-c", CHILD, str(tmp_path), *(str(v) for v in (rank, n, idist, odist, kind))],
                         env=dict(os.environ, DTFFT_HIP_COMPILE_ONLY="1"), cwd=ROOT, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    # the rank-2 slow axis is in place on lines spaced alike: one launch
    assert out.stdout.split() == (["r2r_post", "r2r_pre"] if three else [])


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def rdt(prec):
    return np.float64 if prec == P.DOUBLE else np.float32


def lines_at(buf, count, dist, shape):
    """`count` blocks of `shape`, `dist` elements apart in buf."""
    size = int(np.prod(shape))
    return np.stack([buf[i * dist:i * dist + size].reshape(shape) for i in range(count)])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", [16, 21, 64, 105])
@pytest.mark.parametrize("kind", [R.DCT_1, R.DCT_2, R.DST_3, R.DST_4])
@pytest.mark.parametrize("grow", [(0, 3), (7, 0), (2, 5)])
def test_rank1(kind, n, grow, prec):
    print(f"case: rank 1 kind {kind} n={n} spacing n + {grow} {prec.name}", flush=True)
    hm, idist, odist = 4099, n + grow[0], n + grow[1]
    x = np.random.default_rng(kind * 100 + n).standard_normal((hm, n)).astype(rdt(prec))
    ex = D.FFTExecutor(1, D.FFTType.R2R, prec, idist, odist, hm, [n], r2r_kinds=[kind])
    for sign, k, di, do in ((D.FFT_FORWARD, kind, idist, odist), (D.FFT_BACKWARD, R.INVERSE[kind], odist, idist)):
        want = R.r2r(x.astype(np.float64), k)
        h = np.zeros(hm * max(di, do), dtype=x.dtype)
        for i in range(hm):
            h[i * di:i * di + n] = x[i]
        a, b = D.DeviceArray.from_numpy(h), D.DeviceArray(h.nbytes)
        ex.execute(a, b, sign)
        assert rel(lines_at(b.download(h.shape, h.dtype), hm, do, (n,)).astype(np.float64), want) < TOL[prec]
        ex.execute(a, a, sign)  # in place
        assert rel(lines_at(a.download(h.shape, h.dtype), hm, do, (n,)).astype(np.float64), want) < TOL[prec]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n0,n1", [(12, 32), (9, 15)])
@pytest.mark.parametrize("grow", [(0, 24), (40, 0)])
def test_rank2(n0, n1, grow, prec):
    """Batches farther apart on one side."""
    print(f"case: rank 2 {n0}x{n1} spacing + {grow} {prec.name}", flush=True)
    hm, size, kinds = 257, n0 * n1, (R.DST_4, R.DCT_2)  # along n0, n1
    idist, odist = size + grow[0], size + grow[1]
    x = np.random.default_rng(n0 * n1).standard_normal((hm, n0, n1)).astype(rdt(prec))
    ex = D.FFTExecutor(2, D.FFTType.R2R, prec, idist, odist, hm, [n0, n1], r2r_kinds=list(kinds))
    for sign, ks, di, do in ((D.FFT_FORWARD, kinds, idist, odist),
                             (D.FFT_BACKWARD, [R.INVERSE[k] for k in kinds], odist, idist)):
        want = R.r2r(x.astype(np.float64), ks[1])
        want = np.swapaxes(R.r2r(np.swapaxes(want, 1, 2).copy(), ks[0]), 1, 2)
        h = np.zeros(hm * max(di, do), dtype=x.dtype)
        for i in range(hm):
            h[i * di:i * di + size] = x[i].reshape(-1)
        a, b = D.DeviceArray.from_numpy(h), D.DeviceArray(h.nbytes)
        ex.execute(a, b, sign)
        assert rel(lines_at(b.download(h.shape, h.dtype), hm, do, (n0, n1)).astype(np.float64), want) < TOL[prec]
        ex.execute(a, a, sign)  # in place
        assert rel(lines_at(a.download(h.shape, h.dtype), hm, do, (n0, n1)).astype(np.float64), want) < TOL[prec]
