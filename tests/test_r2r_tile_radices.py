"""FP64 R2R work lengths with a prime above 13 stay off
r2r_tile_kernel, whose pass code has faulted a card with a radix-31 butterfly in FP64, in every kind
and on rows and columns; FP32 keeps it."""
import numpy as np
import pytest

import oracle.r2r as R

D = pytest.importorskip("dtfft_amd")
P = D.Precision
# (kind, n) -> work length 1023 = 31 11 3, 51 = 17 3 and 37
CASES = [(R.DCT_1, 1024), (R.DST_1, 1022), (R.DCT_2, 2046), (R.DCT_4, 2046), (R.DST_3, 51), (R.DCT_4, 102),
         (R.DCT_1, 38)]


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("kind,n", CASES)
def test_large_primes(kind, n, prec, capfd):
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    for dims, kinds in (((n, 64, 18), (kind, R.DCT_4, R.DCT_2)), ((64, n), (R.DCT_4, kind))):
        plan = D.PlanR2R(dims, kinds, prec, D.Effort.ESTIMATE, D.Executor.HIP)
        capfd.readouterr()
        plan.report()
        text = capfd.readouterr().out
        tiles = [ln for ln in text.splitlines() if "r2r_tile_kernel" in ln]
        scheds = [[int(v) for v in ln.split("sched<")[1].split(">")[0].split(",")[1:]] for ln in tiles]
        assert scheds
        assert any(max(s) > 16 for s in scheds) == (prec == P.SINGLE), text


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("m", [37, 51, 305, 1235])  # 305 = 61 5, 1235 = 19 13 5
@pytest.mark.parametrize("kind", [R.DCT_1, R.DCT_3, R.DST_2, R.DCT_4])
def test_parity(kind, m, prec):
    """Rows and (rank 2, in place) columns against the FP64 oracle: FP64 within 1e-12 relative L2,
    FP32 within 2e-6 (the R2R tests' own bars)."""
    n, hm, tol = (m + 1 if kind == R.DCT_1 else 2 * m), 37, {P.DOUBLE: 1e-12, P.SINGLE: 2e-6}[prec]
    print(f"case: kind {kind} n={n} {prec.name}", flush=True)
    x = np.random.default_rng(kind * 100 + n).standard_normal((hm, n)).astype(
        np.float64 if prec == P.DOUBLE else np.float32)
    want = R.r2r(x.astype(np.float64), kind)
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    D.FFTExecutor(1, D.FFTType.R2R, prec, n, n, hm, [n], r2r_kinds=[kind]).execute(a, b, D.FFT_FORWARD)
    got = b.download(x.shape, x.dtype).astype(np.float64)
    assert np.linalg.norm(got - want) < tol * np.linalg.norm(want)
    y = np.ascontiguousarray(x.T)  # DCT-4 along the rows of hm, then `kind` down the columns
    want = R.r2r(R.r2r(y.astype(np.float64), R.DCT_4).T.copy(), kind).T
    a.upload(y)
    D.FFTExecutor(2, D.FFTType.R2R, prec, n * hm, n * hm, 1, [n, hm], r2r_kinds=[kind, R.DCT_4]).execute(
        a, b, D.FFT_FORWARD)
    got = b.download(y.shape, y.dtype).astype(np.float64)
    assert np.linalg.norm(got - want) < tol * np.linalg.norm(want)
