"""Tuning of the batched cycle's column groups that load LDS directly: a set of grids of which some rows
allow it is tuned in two groups, what an untuned cycle runs is among the candidates, and a record of
such a kernel does not overrule lds_dma = 0."""
import os
import struct
import subprocess
import sys

import numpy as np
import pytest

import oracle.plan as OP

D = pytest.importorskip("dtfft_amd")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# nx, ny, nz; lines of an odd axis do not start on 16 bytes
GRIDS = [[64, 96, 48], [63, 96, 50], [48, 96, 105], [32, 96, 96]]

CHILD = """
import ast, glob, sys
import dtfft_amd as D
D.lib().dtfft_hip_set_cache_dir(sys.argv[1].encode())
D.set_config(lds_dma=int(sys.argv[3]))
D.Cycle(ast.literal_eval(sys.argv[4]), D.Precision.SINGLE, D.Effort[sys.argv[2]])
for f in glob.glob(sys.argv[1] + "/*.name"):
    if "kernel" in open(f).read():
        print("kernel", open(f).read())
"""


def kernels(path, effort, grids, lds_dma=1, **env):
    path.mkdir(exist_ok=True)
    out = subprocess.run([sys.executable, "-c", CHILD, str(path), effort, str(lds_dma), repr(grids)], cwd=ROOT,
                         env=dict(os.environ, **env), capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stderr
    return {ln.split(" ", 1)[1].strip() for ln in out.stdout.splitlines() if ln.startswith("kernel ")}


def column_key(grids):
    """The record key of the forward Y stage of grids with one ny, all of them in one group."""
    h, mask = 1469598103934665603, (1 << 64) - 1
    for nx, ny, nz in grids:
        # nx lines of nz batches; in: lines 1, batches nx ny, elements nx apart; out: ny nz, ny, 1
        for v in (nx, nz, 1, nx * ny, nx, ny * nz, ny, 1):
            for b in struct.pack("<q", v):
                h = ((h ^ b) * 1099511628211) & mask
    return f"cyc|{grids[0][1]}|f|10|{len(grids)}|{h:016x}"


def test_record_keeps_to_lds_dma(tmp_path):
    if D.device_arch().startswith("gfx950"):
        pytest.skip("a GPU is present; compile-only behaviour is exercised on CPU hosts")
    grids = [[64, 96, 48], [32, 96, 80]]
    for lds_dma, expected in ((1, True), (0, False)):
        path = tmp_path / str(lds_dma)
        path.mkdir()
        (path / "tuning.txt").write_text(f"{column_key(grids)}\t16 16 1 8,12 2\n")  # not the default schedule
        names = kernels(path, "ESTIMATE", grids, lds_dma, DTFFT_HIP_COMPILE_ONLY="1")
        assert any("batched_cols_dma_kernel" in k and "Li96ELi8ELi12E" in k for k in names) == expected, names
        assert any("batched_cols_dma_kernel" in k for k in names) == expected, names


@pytest.mark.gpu
def test_measure_times_the_default(tmp_path):
    untuned = kernels(tmp_path / "estimate", "ESTIMATE", GRIDS)
    timed = kernels(tmp_path / "measure", "MEASURE", GRIDS)
    assert any("batched_cols_dma_kernel" in k for k in untuned)
    assert untuned <= timed, untuned - timed


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [D.Precision.SINGLE, D.Precision.DOUBLE])
def test_tuned_mixed_set(prec, tmp_path):
    """Forward of every grid within 1e-6 (FP32) or 1e-12 (FP64) of the oracle, twice: tuned, then from
    the records."""
    tol, ct = (1e-6, np.complex64) if prec == D.Precision.SINGLE else (1e-12, np.complex128)
    L = D.lib()
    default_dir = os.environ.get("DTFFT_HIP_CACHE_DIR") or os.path.join(os.path.dirname(D._lib.LIB_PATH), "kcache")
    assert L.dtfft_hip_set_cache_dir(str(tmp_path).encode()) == 0
    try:
        for rnd in range(2):
            cy = D.Cycle(GRIDS, prec, D.Effort.MEASURE)
            offs, total = cy.layout()
            rng, buf, xs = np.random.default_rng(rnd), np.zeros(total, dtype=ct), []
            for (nx, ny, nz), o in zip(GRIDS, offs):
                x = (rng.uniform(-1, 1, (nz, ny, nx)) + 1j * rng.uniform(-1, 1, (nz, ny, nx))).astype(ct)
                buf[o:o + x.size] = x.reshape(-1)
                xs.append(x)
            a = D.DeviceArray.from_numpy(buf)
            b, aux = D.DeviceArray(buf.nbytes), D.DeviceArray(buf.nbytes)
            cy.execute(a, b, aux, D.Execute.FORWARD)
            out = b.download(total, ct)
            for (nx, ny, nz), o, x in zip(GRIDS, offs, xs):
                want = OP.execute_generic(x.astype(np.complex128), True)
                z = out[o:o + x.size].reshape(want.shape).astype(np.complex128)
                assert np.linalg.norm(z - want) < tol * np.linalg.norm(want), (nx, ny, nz)
    finally:
        L.dtfft_hip_set_cache_dir(default_dir.encode())
