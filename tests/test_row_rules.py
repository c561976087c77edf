"""The default rules for long FP32 rows hold by what they say, not by length: the twiddle table is kept
in LDS where two blocks fit a CU with it, and rows whose schedule of fewest passes holds up to 16
points per thread keep it."""
import re

import numpy as np
import pytest

D = pytest.importorskip("dtfft_amd")
P = D.Precision


def rows_kernel(n, lines, capfd):
    """(radices, threads per line, lines per block, table in LDS) of a plan's X rows."""
    plan = D.PlanC2C([n, lines], P.SINGLE, D.Effort.ESTIMATE, D.Executor.HIP)
    capfd.readouterr()
    plan.report()
    line = next(ln for ln in capfd.readouterr().out.splitlines() if ln.split()[0] == "fft_x")
    m = re.search(r"sched<\d+((?:, \d+)+)>, (\d+), (\d+), false, false, \d+(, \d+, true)?", line)
    return [int(v) for v in m.group(1).split(",")[1:]], int(m.group(2)), int(m.group(3)), m.group(4) is not None


@pytest.mark.parametrize("n", [1024, 1280, 1792, 1920, 2048, 2560, 3072, 3200, 3600, 4000, 4096])
def test_rules(n, capfd):
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    radices, tpl, lpb, table = rows_kernel(n, 8192, capfd)
    lds = 8 * lpb * n + 16 * n  # the tile and a table of n - 1 entries with 16 bytes of slack
    assert table == (n > 1024 and 2 * lds <= 160 * 1024), (radices, tpl, lpb, table)
    fewest = {1024: True, 1280: False, 1792: True, 1920: True, 2048: True, 2560: False, 3072: False, 3200: True,
              3600: True, 4000: False, 4096: False}[n]  # 4000 = 10 10 8 5 either way; 4096: no table, no idle thread
    assert (max(radices) > 10) == fewest, (radices, tpl)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["rows", "unpack"])
@pytest.mark.parametrize("n", [1024, 1792, 1920, 2048, 3200, 3600, 4000, 4096])
def test_parity(n, form):
    """Many lines (the last tile partial), both signs: FP32 within 1e-6 relative L2 of 64 bits."""
    print(f"case: {form} n={n}", flush=True)
    peers, c, am = 4, 3, 1367
    lines = c * am
    rng = np.random.default_rng(n)
    x = (rng.uniform(-1, 1, (lines, n)) + 1j * rng.uniform(-1, 1, (lines, n))).astype(np.complex64)
    if form == "rows":
        ex, src = D.FFTExecutor(1, D.FFTType.C2C, P.SINGLE, n, n, lines, [n]), x
    else:
        from dtfft_amd import pencil
        _, recv, _, _ = pencil.forward_exchange(am * peers, n, c, peers, 1)
        ex = D.UnpackFFT((n, c, am), recv, P.SINGLE)
        src = np.concatenate([x[:, p * (n // peers):(p + 1) * (n // peers)].reshape(-1) for p in range(peers)])
    a, b = D.DeviceArray.from_numpy(src), D.DeviceArray(x.nbytes)
    pick = np.r_[0:20, lines - 20:lines]
    for sign, f in ((D.FFT_FORWARD, np.fft.fft), (D.FFT_BACKWARD, lambda z: np.fft.ifft(z) * n)):
        ex.execute(a, b, sign)
        want = f(x[pick].astype(np.complex128))
        assert np.linalg.norm(b.download(x.shape, x.dtype)[pick] - want) < 1e-6 * np.linalg.norm(want), sign
