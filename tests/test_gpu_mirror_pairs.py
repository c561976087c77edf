"""GPU parity of the R2C / C2R kernels that untangle on mirror pairs in registers: pass counts one
to four, even and odd numbers of butterflies and radices of the pair pass, odd halves, partial tiles,
rows and columns, both precisions, against numpy in FP64.

Bars: FP64 within 1e-12 relative L2, FP32 within 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")
P = D.Precision
TOL = {P.DOUBLE: 1e-12, P.SINGLE: 1e-6}
LENGTHS = [4, 8, 10, 12, 18, 22, 26, 30, 34, 36, 42, 50, 64, 66, 84, 90, 110, 130, 154, 210, 256, 338, 420, 640, 1024, 2700, 4096]


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", LENGTHS)
def test_rows(n, prec):
    print(f"case: rows n={n} {prec.name}", flush=True)
    rt, ct = (np.float64, np.complex128) if prec == P.DOUBLE else (np.float32, np.complex64)
    lines, nc = 37, n // 2 + 1
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (lines, n)).astype(rt)
    ex = D.FFTExecutor(1, D.FFTType.R2C, prec, n, nc, lines, [n], [n], [nc])
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(lines * nc * np.dtype(ct).itemsize)
    ex.execute(a, b, D.FFT_FORWARD)
    want = np.fft.rfft(x.astype(np.float64))
    got = b.download((lines, nc), ct)
    assert np.linalg.norm(got - want) < TOL[prec] * np.linalg.norm(want)
    # any X: the imaginary parts of X_0 and X_M do not contribute
    z = (rng.uniform(-1, 1, (lines, nc)) + 1j * rng.uniform(-1, 1, (lines, nc))).astype(ct)
    b.upload(z)
    ex.execute(b, a, D.FFT_BACKWARD)
    zz = z.astype(np.complex128)
    zz[:, 0] = zz[:, 0].real
    zz[:, -1] = zz[:, -1].real
    want = np.fft.irfft(zz, n) * n
    assert np.linalg.norm(a.download((lines, n), rt) - want) < TOL[prec] * np.linalg.norm(want)


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("dims", [(12, 7, 9), (36, 25, 18), (210, 21, 13), (128, 40, 24), (640, 12, 10), (1024, 17, 3)])
def test_plan(dims, prec):
    print(f"case: 3D {dims} {prec.name}", flush=True)
    nx, ny, nz = dims
    rt = np.float64 if prec == P.DOUBLE else np.float32
    ct = np.complex128 if prec == P.DOUBLE else np.complex64
    x = np.random.default_rng(nx).uniform(-1, 1, (nz, ny, nx)).astype(rt)
    plan = D.PlanR2C(list(dims), prec, D.Effort.ESTIMATE, D.Executor.HIP)
    a, b = D.DeviceArray.from_numpy(x, plan.alloc_bytes), D.DeviceArray(plan.alloc_bytes)
    c = D.DeviceArray(plan.alloc_bytes)
    plan.execute(a, b, D.Execute.FORWARD)
    z = np.fft.fftn(np.fft.rfft(x.astype(np.float64), axis=2), axes=(0, 1)).transpose(1, 2, 0)
    got = b.download((ny, nx // 2 + 1, nz), ct)
    assert np.linalg.norm(got - z) < TOL[prec] * np.linalg.norm(z)
    plan.execute(b, c, D.Execute.BACKWARD)
    back = c.download(x.shape, rt) / x.size
    assert np.linalg.norm(back - x) < TOL[prec] * np.linalg.norm(x)
