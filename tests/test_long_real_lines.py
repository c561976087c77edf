"""R2C and C2R of long lines, where one unit of the untangling pass per thread would take more than
the 1024 threads of a block: the half lengths 8918 = 2 13 7^3, 17496, 18432 and 19683 = 3^9."""
import re

import numpy as np
import pytest

D = pytest.importorskip("dtfft_amd")
P = D.Precision
CASES = [(17836, P.SINGLE), (17836, P.DOUBLE), (34992, P.SINGLE), (36864, P.SINGLE), (39366, P.SINGLE)]


@pytest.mark.parametrize("n,prec", CASES)
def test_block_sizes(n, prec, capfd):
    """Compile-only: rows both ways and the fused C2R keep to 1024 threads."""
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    plan = D.PlanR2C([n, 16], prec, D.Effort.ESTIMATE, D.Executor.HIP)
    capfd.readouterr()
    plan.report()
    text = capfd.readouterr().out
    blocks = [int(a) * int(b) for a, b in re.findall(r"fft_(?:r2c|c2r)_kernel<.*?>, (\d+), (\d+)", text)]
    assert len(blocks) >= 2 and max(blocks) <= 1024, text


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec", CASES)
def test_parity(n, prec):
    """Against 64 bits: FP64 within 1e-12 relative L2, FP32 within 1e-6."""
    print(f"case: R2C/C2R n={n} {prec.name}", flush=True)
    hm, nc, tol = 16, n // 2 + 1, {P.DOUBLE: 1e-12, P.SINGLE: 1e-6}[prec]
    rd, cd = (np.float64, np.complex128) if prec == P.DOUBLE else (np.float32, np.complex64)
    x = np.random.default_rng(n).standard_normal((hm, n)).astype(rd)
    want = np.fft.rfft(x.astype(np.float64))
    ex = D.FFTExecutor(1, D.FFTType.R2C, prec, n, nc, hm, [n], [n], [nc])
    a, b, c = D.DeviceArray.from_numpy(x), D.DeviceArray(want.astype(cd).nbytes), D.DeviceArray(x.nbytes)
    ex.execute(a, b, D.FFT_FORWARD)
    assert np.linalg.norm(b.download(want.shape, cd) - want) < tol * np.linalg.norm(want)
    ex.execute(b, c, D.FFT_BACKWARD)
    assert np.linalg.norm(c.download(x.shape, rd) / n - x) < 2 * tol * np.linalg.norm(x)
    plan = D.PlanR2C([n, hm], prec, D.Effort.ESTIMATE, D.Executor.HIP)
    a = D.DeviceArray.from_numpy(x, plan.alloc_bytes)
    b, c = D.DeviceArray(plan.alloc_bytes), D.DeviceArray(plan.alloc_bytes)
    plan.execute(a, b, D.Execute.FORWARD)
    want = np.fft.fft(want, axis=0).T
    assert np.linalg.norm(b.download((nc, hm), cd) - want) < tol * np.linalg.norm(want)
    plan.execute(b, c, D.Execute.BACKWARD)  # the fused C2R
    assert np.linalg.norm(c.download(x.shape, rd) / (n * hm) - x) < 2 * tol * np.linalg.norm(x)
