"""GPU parity of the composite and large prime radices against the FP64 oracle: each radix alone
and in schedules of two and three passes, rows and columns, in both precisions, with few lines
(the smallest tiles) and many, partial tiles included.

Bars: FP64 within 1e-12 relative L2 of the oracle, FP32 within 1e-6."""
import numpy as np
import pytest

import oracle as O
import oracle.plan as OP

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")
P = D.Precision
TOL = {P.DOUBLE: 1e-12, P.SINGLE: 1e-6}


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def random_c(shape, prec, seed):
    rng = np.random.default_rng(seed)
    dt = np.complex128 if prec == P.DOUBLE else np.complex64
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(dt)


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", [6, 9, 10, 12, 13, 14, 15, 16, 17, 29, 36, 41, 61, 74, 81, 90, 105, 136, 148, 168, 210,
                               247, 323, 333, 444, 610, 945, 1147])
@pytest.mark.parametrize("lines", [3, 4099])
def test_rows(n, lines, prec):
    print(f"case: rows n={n} lines={lines} {prec.name}", flush=True)
    x = random_c((lines, n), prec, n + lines)
    ex = D.FFTExecutor(1, D.FFTType.C2C, prec, n, n, lines, [n])
    a, b = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes)
    pick = slice(None) if lines < 100 else np.r_[0:40, lines - 40:lines]
    for sign in (D.FFT_FORWARD, D.FFT_BACKWARD):
        want = O.fft_c2c(x[pick].astype(np.complex128), sign)
        ex.execute(a, b, sign)
        assert rel(b.download(x.shape, x.dtype)[pick].astype(np.complex128), want) < TOL[prec], sign
    ex.execute(a, a, D.FFT_BACKWARD)  # in place
    assert rel(a.download(x.shape, x.dtype)[pick].astype(np.complex128), want) < TOL[prec]


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("dims", [(12, 13, 15), (74, 31, 14), (45, 136, 29), (21, 34, 444), (84, 210, 105)])
def test_columns(dims, prec):
    """The fused transposes read and write columns of every one of these lengths, forward and
    backward (in place along Y in the backward)."""
    print(f"case: 3D {dims} {prec.name}", flush=True)
    nx, ny, nz = dims
    x = random_c((nz, ny, nx), prec, nx + ny + nz)
    plan = D.PlanC2C(dims, prec, D.Effort.ESTIMATE, D.Executor.HIP)
    a, b, c = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes), D.DeviceArray(x.nbytes)
    plan.execute(a, b, D.Execute.FORWARD)
    z = b.download((ny, nx, nz), x.dtype).astype(np.complex128)
    assert rel(z, OP.execute_generic(x.astype(np.complex128), True)) < TOL[prec]
    plan.execute(b, c, D.Execute.BACKWARD)
    back = c.download((nz, ny, nx), x.dtype).astype(np.complex128)
    assert rel(back, OP.execute_generic(z, False)) < TOL[prec]


@pytest.mark.parametrize("prec", [P.SINGLE, P.DOUBLE])
@pytest.mark.parametrize("n", [34, 74, 122, 210, 420, 888])
def test_real(n, prec):
    """Half-length transforms over the new radices: R2C and C2R rows and the fused C2R."""
    print(f"case: real {n} {prec.name}", flush=True)
    ny, nz, nc = 12, 10, n // 2 + 1
    rd, cd = (np.float32, np.complex64) if prec == P.SINGLE else (np.float64, np.complex128)
    x = np.random.default_rng(n).standard_normal((nz, ny, n)).astype(rd)
    plan = D.PlanR2C((n, ny, nz), prec, D.Effort.ESTIMATE, D.Executor.HIP)
    a = D.DeviceArray.from_numpy(x, plan.alloc_bytes)
    b, c = D.DeviceArray(plan.alloc_bytes), D.DeviceArray(plan.alloc_bytes)
    plan.execute(a, b, D.Execute.FORWARD)
    z = b.download((ny, nc, nz), cd).astype(np.complex128)
    assert rel(z, OP.execute_generic_r2c(x.astype(np.float64))) < TOL[prec]
    plan.execute(b, c, D.Execute.BACKWARD)
    back = c.download((nz, ny, n), rd).astype(np.float64)
    assert rel(back, OP.execute_generic_c2r(z, n)) < TOL[prec]
    ex = D.FFTExecutor(1, D.FFTType.R2C, prec, n, nc, ny * nz, [n], [n], [nc])
    ex.execute(a, b, D.FFT_FORWARD)
    h = b.download((nz, ny, nc), cd).astype(np.complex128)
    assert rel(h, O.fft_r2c(x.astype(np.float64).reshape(-1, n)).reshape(h.shape)) < TOL[prec]
    ex.execute(b, c, D.FFT_BACKWARD)
    assert rel(c.download((nz, ny, n), rd).astype(np.float64), x.astype(np.float64) * n) < 2 * TOL[prec]
