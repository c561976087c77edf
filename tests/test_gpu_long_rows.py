"""GPU parity of the four-pass schedules of long rows (1024 to 4096 points, launches of many lines)
against numpy in FP64, forward and backward, plain and with a partial last tile.

Bars: FP64 within 1e-12 relative L2, FP32 within 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")
P = D.Precision
TOL = {P.DOUBLE: 1e-12, P.SINGLE: 1e-6}


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", [1024, 1050, 1280, 1536, 2000, 2048, 2560, 3072, 4000, 4096])
def test_rows(n, prec):
    print(f"case: rows n={n} {prec.name}", flush=True)
    ct = np.complex128 if prec == P.DOUBLE else np.complex64
    lines = 2051
    rng = np.random.default_rng(n)
    x = (rng.uniform(-1, 1, (lines, n)) + 1j * rng.uniform(-1, 1, (lines, n))).astype(ct)
    ex = D.FFTExecutor(1, D.FFTType.C2C, prec, n, n, lines, [n])
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    pick = np.r_[0:20, lines - 20:lines]
    for sign, f in ((D.FFT_FORWARD, np.fft.fft), (D.FFT_BACKWARD, lambda z: np.fft.ifft(z) * n)):
        ex.execute(a, b, sign)
        want = f(x[pick].astype(np.complex128))
        assert np.linalg.norm(b.download(x.shape, ct)[pick] - want) < TOL[prec] * np.linalg.norm(want), sign
