"""CPU check (no GPU): plans of lengths with a large prime radix compile in layouts that would
let a column stage run the LDS-DMA kernels, which hold radices up to 16 only (lines a multiple of
16, an axis a multiple of 8).  Plans of the same lengths are run against the oracle on a GPU."""
import numpy as np
import pytest

D = pytest.importorskip("dtfft_amd")
DIMS = [(16, 136, 32), (136, 16, 16), (48, 272, 16)]


@pytest.fixture(autouse=True)
def defaults():
    yield
    D.set_config()


@pytest.mark.parametrize("lds_dma", [1, 2, 3])
@pytest.mark.parametrize("dims", DIMS)
def test_plans_compile(dims, lds_dma):
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    D.set_config(enable_fused=True, lds_dma=lds_dma)
    D.PlanC2C(list(dims), D.Precision.SINGLE, D.Effort.ESTIMATE, D.Executor.HIP)
    D.PlanR2C([2 * dims[0] if dims[0] == 136 else dims[0], dims[1], dims[2]], D.Precision.SINGLE, D.Effort.ESTIMATE,
              D.Executor.HIP)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", DIMS)
def test_roundtrip(dims):
    """Backward of forward is n times the input: FP32 within 1e-6 relative L2."""
    print(f"case: 3D {dims}", flush=True)
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * ny)
    x = (rng.uniform(-1, 1, (nz, ny, nx)) + 1j * rng.uniform(-1, 1, (nz, ny, nx))).astype(np.complex64)
    plan = D.PlanC2C(list(dims), D.Precision.SINGLE, D.Effort.ESTIMATE, D.Executor.HIP)
    a, b, c = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes), D.DeviceArray(x.nbytes)
    plan.execute(a, b, D.Execute.FORWARD)
    z = b.download((ny, nx, nz), x.dtype).astype(np.complex128)
    want = np.fft.fftn(x.astype(np.complex128)).transpose(1, 2, 0)
    assert np.linalg.norm(z - want) < 1e-6 * np.linalg.norm(want)
    plan.execute(b, c, D.Execute.BACKWARD)
    back = c.download(x.shape, x.dtype).astype(np.complex128) / x.size
    assert np.linalg.norm(back - x) < 1e-6 * np.linalg.norm(x)
