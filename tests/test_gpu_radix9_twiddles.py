"""FP32 radix-9 butterflies multiply by their inner twiddles as passes do: hi+lo pairs, one rounding.

An impulse x at point 3 m (m = 1, 2) of 27 = 9 3 meets exact sums only on its way to the outputs k
with k % 9 = 1, 2, and one twiddle product, w9^(m k).  A product by a hi+lo pair of a value with one
zero part rounds once (the pair is within 2^-48 of the twiddle), so those outputs are within half a
unit in the last place, and 1 % of it for what the pair and 64 bits leave out; a twiddle held in one float
is off by up to half a unit more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")


@pytest.mark.parametrize("part", [1.0, 1j])
@pytest.mark.parametrize("m", [1, 2])
def test_products_round_once(m, part):
    n, lines = 27, 4096
    v = np.random.default_rng(m).uniform(1, 2, lines).astype(np.float32)
    x = np.zeros((lines, n), dtype=np.complex64)
    x[:, 3 * m] = v * np.complex64(part)
    ex = D.FFTExecutor(1, D.FFTType.C2C, D.Precision.SINGLE, n, n, lines, [n])
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    ex.execute(a, b, D.FFT_FORWARD)
    y = b.download(x.shape, x.dtype)
    for k in (1, 2, 10, 11, 19, 20):
        want = v.astype(np.float64) * (part * np.exp(-2j * np.pi * m * k / 9))
        for got, exact in ((y[:, k].real, want.real), (y[:, k].imag, want.imag)):
            ulp = np.spacing(np.abs(exact).astype(np.float32)).astype(np.float64)
            assert np.max(np.abs(got.astype(np.float64) - exact) / ulp) < 0.505, k
