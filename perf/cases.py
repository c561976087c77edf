"""Performance cases: the work that programs have this library do, through its public entry points.

A case is a dict of plain values.  ``family`` names the entry point:

* ``c2c`` / ``r2c`` / ``r2r`` -- a single-rank plan (PlanC2C / PlanR2C / PlanR2R, effort
  ESTIMATE, the default configuration).  ``way``: "both" runs forward (a -> b) and backward
  (b -> c) and returns b and c; "cycle" runs the same and returns c alone, for plans whose
  backward sequence uses its input as a work buffer; "forward" runs and returns the forward.
* ``cycle``   -- many uneven C2C grids, forward and backward, replayed as one hipGraph;
* ``share``   -- one GPU's share of a P-rank transpose: per-peer packs, loopback exchange,
  unpack and the FFT along the newly aligned axis;
* ``permute`` -- three permute kernels of the kernel plugin, once round the pencils.

Buffers are torch tensors on the GPU, allocated before the call as a program keeps them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import dtfft_amd as D

# Axis lengths of the uneven-grid workload (also the smooth lengths of the drawn shares).
UNEVEN = [48, 60, 64, 84, 96, 105, 128, 160, 192, 210, 256, 320, 384]
KINDS = {"DCT_1": 3, "DCT_2": 5, "DCT_3": 4, "DCT_4": 6, "DST_1": 7, "DST_2": 9, "DST_3": 8, "DST_4": 10}
INVERSE = {"DCT_2": "DCT_3", "DCT_3": "DCT_2", "DST_2": "DST_3", "DST_3": "DST_2"}


def listed():
    return [
        # a slice or image transformed by itself: launches and latency, the smallest call
        {"name": "c2c-2d-256-f64", "family": "c2c", "x": 256, "y": 256, "z": 0, "double": True, "way": "both"},
        # a small ragged 3D block (lengths with 3, 5 and 7, an odd axis)
        {"name": "c2c-3d-60x84x35-f32", "family": "c2c", "x": 60, "y": 84, "z": 35, "double": False, "way": "both"},
        # the headline benchmark: spectral solvers on a cube that fills a GPU's share
        {"name": "c2c-3d-512-f32", "family": "c2c", "x": 512, "y": 512, "z": 512, "double": False, "way": "both"},
        # a large double-precision box with uneven axes
        {"name": "c2c-3d-384x210x320-f64", "family": "c2c", "x": 384, "y": 210, "z": 320, "double": True,
         "way": "both"},
        # axes with a large prime factor (37), as the reference's own 333 x 444 test
        {"name": "c2c-3d-333x444x74-f32", "family": "c2c", "x": 333, "y": 444, "z": 74, "double": False,
         "way": "both"},
        # real fields of a turbulence or weather code, the R2C benchmark
        {"name": "r2c-3d-1024x512x256-f32", "family": "r2c", "x": 1024, "y": 512, "z": 256, "double": False,
         "way": "both"},
        # a mid-size ragged real box in double precision
        {"name": "r2c-3d-210x105x96-f64", "family": "r2c", "x": 210, "y": 105, "z": 96, "double": True,
         "way": "both"},
        # Neumann problems: DCT-2 forward, DCT-3 back, the R2R benchmark
        {"name": "r2r-3d-512-dct2-f32", "family": "r2r", "x": 512, "y": 512, "z": 512, "double": False,
         "kinds": "DCT_2,DCT_2,DCT_2", "way": "both"},
        # mixed boundary conditions on uneven axes (Chebyshev points along X) in double precision
        {"name": "r2r-3d-129x96x105-mixed-f64", "family": "r2r", "x": 129, "y": 96, "z": 105, "double": True,
         "kinds": "DCT_1,DCT_4,DST_2", "way": "cycle"},
        # many uneven grids at once (block-structured meshes), the batched benchmark
        {"name": "cycle-64-uneven-f32", "family": "cycle", "grids": 64, "grid_seed": 20250104, "double": False},
        # one GPU's share of a 2048^3 cube on a 4 x 4 process grid: the largest
        {"name": "share-2048x512x512-f32", "family": "share", "a": 2048, "b": 2048, "c": 512, "peers": 4, "me": 1,
         "double": False},
        # transposes alone, for callers who bring their own FFT
        {"name": "permute-512-c128", "family": "permute", "x": 512, "y": 512, "z": 512, "bytes": 16, "back": False},
    ]


# ---- drawn cases ------------------------------------------------------------------------
def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, lo, hi):
    """An axis length, spread over the logarithm of its range: more often a product of small
    primes, else whatever comes (odd numbers and large primes among them)."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.65:
        while not _smooth(n):
            n -= 1
    return max(lo, n)


def _dims(rng, most):
    """Two or three axis lengths with between 4096 and `most` points."""
    while True:
        if rng.random() < 0.3:
            d = [_length(rng, 32, 2048), _length(rng, 32, 2048), 0]
        else:
            d = [_length(rng, 12, 640) for _ in range(3)]
        if 4096 <= d[0] * d[1] * max(1, d[2]) <= most:
            return d


def draw(rng):
    family = rng.choice(["c2c"] * 4 + ["r2c"] * 2 + ["r2r"] * 2 + ["cycle", "share"] + ["permute"] * 2)
    dbl = rng.random() < 0.5
    if family == "c2c":
        x, y, z = _dims(rng, 1 << 27 if not dbl else 1 << 26)
        return {"family": family, "x": x, "y": y, "z": z, "double": dbl, "way": "both"}
    if family == "r2c":
        x, y, z = _dims(rng, 1 << 27)
        way = "both" if x % 2 == 0 else rng.choice(["forward", "cycle"])
        return {"family": family, "x": x, "y": y, "z": z, "double": dbl, "way": way}
    if family == "r2r":
        x, y, z = _dims(rng, 1 << 25)
        kinds = [rng.choice(sorted(KINDS))] * 3
        if rng.random() < 0.5:
            kinds = [rng.choice(sorted(KINDS)) for _ in range(3)]
        return {"family": family, "x": x, "y": y, "z": z, "double": dbl, "kinds": ",".join(kinds[:3 if z else 2]),
                "way": rng.choice(["forward", "cycle"])}
    if family == "cycle":
        return {"family": family, "grids": int(round(math.exp(rng.uniform(math.log(2), math.log(40))))),
                "grid_seed": rng.randrange(1 << 30), "double": False}
    if family == "share":
        while True:
            peers = rng.choice([2, 3, 4, 8])
            a, b, c = peers * _length(rng, 8, 256), peers * rng.choice(UNEVEN), _length(rng, 8, 512)
            if (1 << 14) <= a * (b // peers) * c <= 1 << 27:
                return {"family": family, "a": a, "b": b, "c": c, "peers": peers, "me": rng.randrange(peers),
                        "double": dbl}
    x, y, z = _dims(rng, 1 << 26)
    return {"family": family, "x": x, "y": y, "z": z, "bytes": rng.choice([4, 8, 16]), "back": rng.random() < 0.5}


# ---- inputs -----------------------------------------------------------------------------
def _gpu():
    return torch.device("cuda", torch.cuda.current_device())


def _extent(case):
    """Axis lengths, X (the contiguous one) first."""
    return [case["x"], case["y"]] + ([case["z"]] if case["z"] else [])


def _types(case):
    return (torch.float64, torch.complex128) if case["double"] else (torch.float32, torch.complex64)


def _uniform(n, dtype, seed):
    """n values in [-1, 1), both parts of complex ones."""
    gen = torch.Generator(device=_gpu()).manual_seed(int(seed))
    t = torch.empty(n, dtype=dtype, device=_gpu())
    (torch.view_as_real(t) if dtype.is_complex else t).uniform_(-1, 1, generator=gen)
    return t


def _grids(case):
    rng = np.random.default_rng(case["grid_seed"])
    return [[int(v) for v in rng.choice(UNEVEN, 3)] for _ in range(case["grids"])]


def _offsets(grids):
    """Element offset of each grid in the packed buffers, and their length."""
    offs, at = [], 0
    for g in grids:
        offs.append(at)
        at += (math.prod(g) + 63) // 64 * 64
    return offs, at


def _permuted_dims(dims, back):
    if len(dims) == 2:
        return [dims[1], dims[0]]
    return [dims[2], dims[0], dims[1]] if back else [dims[1], dims[2], dims[0]]


def _permute_type(case):
    return {4: torch.float32, 8: torch.complex64, 16: torch.complex128}[case["bytes"]]


def _input(case, seed):
    f = case["family"]
    if f == "permute":
        return _uniform(math.prod(_extent(case)), _permute_type(case), seed)
    real, cplx = _types(case)
    if f == "share":
        return _uniform(case["a"] * (case["b"] // case["peers"]) * case["c"], cplx, seed)
    if f == "cycle":
        return _uniform(_offsets(_grids(case))[1], cplx, seed)
    return _uniform(math.prod(_extent(case)), cplx if f == "c2c" else real, seed)


# ---- a pass -----------------------------------------------------------------------------
def prepare(case, seed):
    f = case["family"]
    x = _input(case, seed)
    s = {"family": f, "a": x}
    prec = D.Precision.DOUBLE if case.get("double") else D.Precision.SINGLE
    if f == "permute":
        dims, kind = _extent(case), D.KernelType.PERMUTE_BACKWARD if case["back"] else D.KernelType.PERMUTE_FORWARD
        s["kernels"], s["bufs"] = [], [x]
        for _ in range(len(dims)):
            s["kernels"].append(D.Kernel(kind, dims, case["bytes"]))
            s["bufs"].append(torch.empty_like(x))
            dims = _permuted_dims(dims, case["back"])
        s["out"] = s["bufs"][1:]
    elif f == "share":
        s["share"] = D.ExchangeShare(case["a"], case["b"], case["c"], case["peers"], case["me"], prec)
        s["send"], s["recv"], s["b"] = (torch.empty_like(x) for _ in range(3))
        s["out"] = [s["send"], s["b"]]
    elif f == "cycle":
        s["cycle"] = D.Cycle(_grids(case), prec)
        s["b"], s["c"], s["aux"] = (torch.zeros_like(x) for _ in range(3))
        s["out"] = [s["b"], s["c"]]
    else:
        dims = _extent(case)
        if f == "r2r":
            kinds = [KINDS[k] for k in case["kinds"].split(",")]
            plan = D.PlanR2R(dims, kinds, prec, D.Effort.ESTIMATE, D.Executor.HIP)
        else:
            plan = (D.PlanC2C if f == "c2c" else D.PlanR2C)(dims, prec, D.Effort.ESTIMATE, D.Executor.HIP)
        real, cplx = _types(case)
        item = x.element_size()
        n = (plan.alloc_bytes + item - 1) // item
        s["plan"], s["way"] = plan, case["way"]
        s["b"], s["c"], s["aux"] = (torch.empty(n, dtype=x.dtype, device=x.device) for _ in range(3))
        fwd = s["b"]
        if f == "r2c":  # nx / 2 + 1 complex values along X
            nc = (dims[0] // 2 + 1) * math.prod(dims[1:])
            fwd = torch.view_as_complex(s["b"][:2 * nc].view(nc, 2))
        else:
            fwd = fwd[:x.numel()]
        back = s["c"][:x.numel()]
        s["out"] = {"both": [fwd, back], "forward": [fwd], "cycle": [back]}[case["way"]]
    return s


def run(s):
    f = s["family"]
    if f == "permute":
        for k, src, dst in zip(s["kernels"], s["bufs"], s["bufs"][1:]):
            k.execute(src, dst)
    elif f == "share":
        s["share"].run(s["a"], s["send"], s["recv"], s["b"], D.FFT_FORWARD)
    elif f == "cycle":
        s["cycle"].execute_graph(s["a"], s["b"], s["aux"], s["c"])
    else:
        s["plan"].execute(s["a"], s["b"], D.Execute.FORWARD, s["aux"])
        if s["way"] != "forward":
            s["plan"].execute(s["b"], s["c"], D.Execute.BACKWARD, s["aux"])
    return s["out"]


def work(case):
    f = case["family"]
    if f == "permute":
        dims = _extent(case)
        return {"bytes": 2 * len(dims) * math.prod(dims) * case["bytes"], "flops": 0}
    es = 16 if case["double"] else 8  # bytes of a complex value
    if f == "share":
        n = case["a"] * (case["b"] // case["peers"]) * case["c"]
        # packed chunks written and read, the exchange, the pencil written
        return {"bytes": 6 * n * es, "flops": 5 * n * math.log2(case["b"])}
    if f == "cycle":
        sizes = [math.prod(g) for g in _grids(case)]
        return {"bytes": 4 * sum(sizes) * es, "flops": sum(10 * n * math.log2(n) for n in sizes)}
    dims = _extent(case)
    n = math.prod(dims)
    passes = 1 if case["way"] == "forward" else 2
    if f == "c2c":
        return {"bytes": passes * 2 * n * es, "flops": passes * 5 * n * math.log2(n)}
    spectrum = n // dims[0] * (dims[0] // 2 + 1) * es if f == "r2c" else n * es // 2
    return {"bytes": passes * (n * es // 2 + spectrum), "flops": passes * 2.5 * n * math.log2(n)}


# ---- the same in 64 bits ----------------------------------------------------------------
def _to_spectral_pencil(t):
    """(z, y, x) or (y, x) -> the layout of a plan's forward output: the last axis contiguous."""
    return (t.permute(1, 2, 0) if t.dim() == 3 else t.permute(1, 0)).contiguous().reshape(-1)


def _r2r_matrix(kind, n):
    """FFTW's unnormalised REDFT / RODFT as an n x n matrix in 64 bits."""
    j = torch.arange(n, dtype=torch.float64, device=_gpu())
    k = j[:, None]
    m = {"DCT_1": lambda: 2 * torch.cos(math.pi * k * j / (n - 1)),
         "DCT_2": lambda: 2 * torch.cos(math.pi * k * (2 * j + 1) / (2 * n)),
         "DCT_3": lambda: 2 * torch.cos(math.pi * (2 * k + 1) * j / (2 * n)),
         "DCT_4": lambda: 2 * torch.cos(math.pi * (2 * k + 1) * (2 * j + 1) / (4 * n)),
         "DST_1": lambda: 2 * torch.sin(math.pi * (k + 1) * (j + 1) / (n + 1)),
         "DST_2": lambda: 2 * torch.sin(math.pi * (k + 1) * (2 * j + 1) / (2 * n)),
         "DST_3": lambda: 2 * torch.sin(math.pi * (2 * k + 1) * (j + 1) / (2 * n)),
         "DST_4": lambda: 2 * torch.sin(math.pi * (2 * k + 1) * (2 * j + 1) / (4 * n))}[kind]()
    if kind == "DCT_1":  # the end points enter once
        m[:, 0] /= 2
        m[:, n - 1] /= 2
    elif kind == "DCT_3":
        m[:, 0] /= 2
    elif kind == "DST_3":
        m[:, n - 1] /= 2
    return m


def _r2r_logical(kind, n):
    return 2 * (n - 1) if kind == "DCT_1" else 2 * (n + 1) if kind == "DST_1" else 2 * n


def exact(case, seed):
    f = case["family"]
    x = _input(case, seed)
    if f == "permute":
        dims, t, out = _extent(case), x, []
        for _ in range(len(dims)):
            t = t.reshape(dims[::-1])
            if len(dims) == 2:
                t = t.permute(1, 0)
            else:  # (z, y, x) -> (x, z, y), or (y, x, z) the other way
                t = t.permute(1, 2, 0) if case["back"] else t.permute(2, 0, 1)
            t = t.contiguous().reshape(-1)
            out.append(t)
            dims = _permuted_dims(dims, case["back"])
        return out
    if f == "share":
        a, b, c, peers = case["a"], case["b"], case["c"], case["peers"]
        t = x.reshape(c, b // peers, peers, a // peers).permute(2, 3, 0, 1).contiguous()  # (peer, x, z, y)
        want = torch.empty(a // peers, c, b, dtype=torch.complex128, device=x.device)
        for i in range(a // peers):
            want[i] = torch.fft.fft(t[:, i].permute(1, 0, 2).reshape(c, b).to(torch.complex128), dim=-1)
        return [t.reshape(-1), want.reshape(-1)]
    if f == "cycle":
        grids = _grids(case)
        offs, total = _offsets(grids)
        fwd, back = (torch.zeros(total, dtype=torch.complex128, device=x.device) for _ in range(2))
        for g, o in zip(grids, offs):
            n = math.prod(g)
            t = x[o:o + n].to(torch.complex128)
            fwd[o:o + n] = _to_spectral_pencil(torch.fft.fftn(t.reshape(g[::-1])))
            back[o:o + n] = t * n
        return [fwd, back]
    dims = _extent(case)
    t = x.to(torch.float64 if f != "c2c" else torch.complex128).reshape(dims[::-1])
    fwd, scale = None, math.prod(dims)
    if f == "c2c":
        fwd = torch.fft.fftn(t)
    elif f == "r2c":
        fwd = torch.fft.rfftn(t)
    else:
        kinds = case["kinds"].split(",")
        scale = math.prod(_r2r_logical(k, n) for k, n in zip(kinds, dims))
        if case["way"] != "cycle":
            fwd = t
            for axis, (k, n) in enumerate(zip(kinds, dims)):
                at = len(dims) - 1 - axis
                m = _r2r_matrix(k, n)
                w = fwd.movedim(at, -1).contiguous()
                fwd = torch.mm(w.reshape(-1, n), m.t().contiguous()).reshape(w.shape).movedim(-1, at)
    out = []
    if case["way"] != "cycle":
        out.append(_to_spectral_pencil(fwd))
    if case["way"] != "forward":
        out.append((t * scale).reshape(-1))
    return out
