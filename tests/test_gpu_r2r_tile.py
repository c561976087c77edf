"""GPU parity of the general R2R tile kernel and of the half-length forms against the FP64 oracle:
every kind at lengths around its forms' edges (odd, even, single-pass and prime work lengths, work
lengths without a schedule), rows and columns, partial tiles, and plans whose axes mix stages with
and without a column form.

Bars: FP64 within 1e-12 relative L2 of the oracle, FP32 within 2e-6 (the R2R tests' own)."""
import numpy as np
import pytest

import oracle.r2r as R

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")
P = D.Precision
TOL = {P.DOUBLE: 1e-12, P.SINGLE: 2e-6}


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def rdt(prec):
    return np.float64 if prec == P.DOUBLE else np.float32


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", [2, 3, 4, 6, 9, 10, 26, 33, 38, 75, 129, 134])
@pytest.mark.parametrize("kind", R.KINDS)
def test_rows_and_columns(kind, n, prec):
    """Rank 2: rows of n1 = n, then columns of n0 = n in place, 3 batches; 134 = 2 67 has work
    lengths (67, 133 = 7 19, 135) with and without a schedule."""
    print(f"case: kind {kind} n={n} {prec.name}", flush=True)
    hm, n0, n1 = 3, n, n
    x = np.random.default_rng(kind * 1000 + n).standard_normal((hm, n0, n1)).astype(rdt(prec))
    ex = D.FFTExecutor(2, D.FFTType.R2R, prec, n0 * n1, n0 * n1, hm, [n0, n1], r2r_kinds=[kind, kind])
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    ex.execute(a, b, D.FFT_FORWARD)
    want = R.r2r(x.astype(np.float64), kind)
    want = np.swapaxes(R.r2r(np.swapaxes(want, 1, 2).copy(), kind), 1, 2)
    assert rel(b.download(x.shape, x.dtype).astype(np.float64), want) < TOL[prec]
    ex.execute(b, a, D.FFT_BACKWARD)
    back = a.download(x.shape, x.dtype).astype(np.float64) / R.logical_size(kind, n) ** 2
    assert rel(back, x.astype(np.float64)) < 4 * TOL[prec]


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("dims,kinds", [
    ((33, 20, 15), (3, 6, 9)),      # every stage by the tile kernel, partial tiles
    ((48, 32, 64), (5, 5, 5)),      # Y lines in whole tile rows, X lines not
    ((20, 134, 18), (4, 10, 7)),    # Y without a column form: permute and rows
    ((134, 12, 10), (6, 5, 3)),     # X without one, backward
    ((16, 18, 134), (8, 4, 10)),    # Z without one
    ((134, 134, 6), (6, 10, 5)),    # only Z with one
    ((70, 41), (7, 4)), ((134, 30), (6, 8)), ((30, 134), (9, 6)),
])
def test_plans(dims, kinds, prec):
    print(f"case: plan {dims} {kinds} {prec.name}", flush=True)
    three = len(dims) == 3
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(tuple(reversed(dims))).astype(rdt(prec))
    run = R.execute_generic_r2r if three else R.execute_2d_r2r
    out_shape = (dims[1], dims[0], dims[2]) if three else (dims[0], dims[1])
    plan = D.PlanR2R(dims, kinds, prec, D.Effort.ESTIMATE, D.Executor.HIP)
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    plan.execute(a, b, D.Execute.FORWARD)
    assert rel(b.download(out_shape, x.dtype).astype(np.float64), run(x.astype(np.float64), kinds, True)) < TOL[prec]
    assert np.array_equal(a.download(x.shape, x.dtype), x)  # the forward keeps its input
    y = rng.standard_normal(out_shape).astype(rdt(prec))
    a.upload(y)
    plan.execute(a, b, D.Execute.BACKWARD)
    want = run(y.astype(np.float64), kinds, False)
    assert rel(b.download(x.shape, x.dtype).astype(np.float64), want) < TOL[prec]
    a.upload(x)
    plan.execute(a, a, D.Execute.FORWARD)  # in place
    assert rel(a.download(out_shape, x.dtype).astype(np.float64), run(x.astype(np.float64), kinds, True)) < TOL[prec]
