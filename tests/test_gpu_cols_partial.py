"""GPU parity of the LDS-DMA column stages on tiles that are not full and lengths that are not a
multiple of 8, single plans and batched cycles, against numpy in FP64: FP32 within 1e-6 relative
L2.  The lines around the edges: 2 (one 16-byte piece), 14, 16, 18, and odd numbers, which keep
the plain kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = pytest.importorskip("dtfft_amd")


def random_c(shape, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


def forward(x):
    return np.fft.fftn(x.astype(np.complex128)).transpose(1, 2, 0)


@pytest.fixture(autouse=True)
def defaults():
    yield
    D.set_config()


@pytest.mark.parametrize("lds_dma", [1, 2, 3])
@pytest.mark.parametrize("dims", [(2, 24, 30), (14, 60, 18), (18, 105, 22), (50, 36, 84), (15, 64, 48), (16, 10, 130)])
def test_plan(dims, lds_dma):
    print(f"case: {dims} lds_dma={lds_dma}", flush=True)
    nx, ny, nz = dims
    x = random_c((nz, ny, nx), nx + 7 * ny)
    D.set_config(enable_fused=True, lds_dma=lds_dma)
    plan = D.PlanC2C(list(dims), D.Precision.SINGLE, D.Effort.ESTIMATE, D.Executor.HIP)
    a, b, c = D.DeviceArray.from_numpy(x), D.DeviceArray(x.nbytes), D.DeviceArray(x.nbytes)
    plan.execute(a, b, D.Execute.FORWARD)
    want = forward(x)
    assert np.linalg.norm(b.download((ny, nx, nz), x.dtype) - want) < 1e-6 * np.linalg.norm(want)
    plan.execute(b, c, D.Execute.BACKWARD)
    back = c.download(x.shape, x.dtype) / x.size
    assert np.linalg.norm(back - x) < 1e-6 * np.linalg.norm(x)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("grids", [[[14, 60, 18], [15, 60, 18], [18, 60, 105]], [[48, 64, 96], [50, 64, 96]]])
def test_cycle(grids, shift):
    """Groups split between the two kernels; shift 1: buffers 8 bytes off the 16-byte grid."""
    print(f"case: {grids} shift={shift}", flush=True)
    cy = D.Cycle(grids, D.Precision.SINGLE)
    xs = [random_c((g[2], g[1], g[0]), i) for i, g in enumerate(grids)]
    offs, total = cy.layout()
    host = np.zeros(total + shift, np.complex64)
    for x, o in zip(xs, offs):
        host[shift + o:shift + o + x.size] = x.reshape(-1)
    bufs = [D.DeviceArray.from_numpy(host) for _ in range(3)]
    ptr = [b.ptr + 8 * shift for b in bufs]
    cy.execute(ptr[0], ptr[1], ptr[2], D.Execute.FORWARD)
    z = bufs[1].download(host.shape, host.dtype)
    for x, o in zip(xs, offs):
        want = forward(x).reshape(-1)
        got = z[shift + o:shift + o + x.size]
        assert np.linalg.norm(got - want) < 1e-6 * np.linalg.norm(want)
    cy.execute(ptr[1], ptr[0], ptr[2], D.Execute.BACKWARD)
    z = bufs[0].download(host.shape, host.dtype)
    for x, o in zip(xs, offs):
        got = z[shift + o:shift + o + x.size] / x.size
        assert np.linalg.norm(got - x.reshape(-1)) < 1e-6 * np.linalg.norm(x)
