"""The work that users of the stencil engine have it do, as timed cases.

Four paths, each through its public entry point in pyan5d:
  forward   T steps on a device-resident grid (forward_device)
  host      the kernel_stencil drop-in on a host array: copies in, steps, out
  adjoint   forward + adjoint: loss, dL/du0 and dL/dcoefs (adjoint_device)
  batch     many independent 2D grids in one plan (Batch.run)

T is even everywhere, so the result sits in buffer 0 and a repeated pass goes
on from it, as a program that steps a simulation in chunks does.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "an5d-artifact_amd"))

import pyan5d  # noqa: E402

# stencil: (dimensions, radius, shape, divisor of its source)
STENCILS = {
    "star2d1r": (2, 1, "star", 0), "star2d2r": (2, 2, "star", 0), "star2d3r": (2, 3, "star", 0),
    "star2d4r": (2, 4, "star", 0), "box2d1r": (2, 1, "box", 0), "box2d2r": (2, 2, "box", 0),
    "box2d3r": (2, 3, "box", 0), "box2d4r": (2, 4, "box", 0), "j2d5pt": (2, 1, "star", 118),
    "j2d9pt": (2, 2, "star", 118), "j2d9pt-gol": (2, 1, "box", 118), "gradient2d": (2, 1, "star", 0),
    "star3d1r": (3, 1, "star", 0), "star3d2r": (3, 2, "star", 0), "star3d3r": (3, 3, "star", 0),
    "star3d4r": (3, 4, "star", 0), "box3d1r": (3, 1, "box", 0), "box3d2r": (3, 2, "box", 0),
    "box3d3r": (3, 3, "box", 0), "box3d4r": (3, 4, "box", 0), "j3d27pt": (3, 1, "box", 159),
}
BATCH_STENCILS = ("j2d5pt", "j2d9pt", "star2d2r")
# the largest listed pass: 1000 steps of the 7-point star on 512^3
MOST_FLOPS = 1000 * 512.0**3 * 13


def listed():
    return [
        # the smallest grid of the batch workload on its own: launches and latency count
        {"name": "j2d5pt f32 256x256", "path": "forward", "stencil": "j2d5pt", "dtype": "f32",
         "n0": 256, "n1": 256, "n2": 0, "T": 64, "mode": "exact", "pad": 0},
        # a small ragged box of a 3D simulation in double precision
        {"name": "star3d1r f64 100x90x110", "path": "forward", "stencil": "star3d1r", "dtype": "f64",
         "n0": 100, "n1": 90, "n2": 110, "T": 100, "mode": "exact", "pad": 0},
        # an ordinary rectangle with padded rows, FMA mode
        {"name": "j2d9pt-gol f32 fast 1000x3001", "path": "forward", "stencil": "j2d9pt-gol", "dtype": "f32",
         "n0": 1000, "n1": 3001, "n2": 0, "T": 256, "mode": "fast", "pad": 27},
        # the drop-in on host arrays at the size a workstation also runs on its CPU
        {"name": "kernel_stencil j2d5pt 4096x4096", "path": "host", "stencil": "j2d5pt", "dtype": "f32",
         "n0": 4096, "n1": 4096, "n2": 0, "T": 100},
        # the benchmark's headline
        {"name": "star3d1r f32 512^3", "path": "forward", "stencil": "star3d1r", "dtype": "f32",
         "n0": 512, "n1": 512, "n2": 512, "T": 1000, "mode": "exact", "pad": 0},
        # the high-order set of the benchmark: 2D box, 3D star, both at full size
        {"name": "box2d4r f64 16384x16384", "path": "forward", "stencil": "box2d4r", "dtype": "f64",
         "n0": 16384, "n1": 16384, "n2": 0, "T": 20, "mode": "exact", "pad": 0},
        {"name": "star3d4r f32 512^3", "path": "forward", "stencil": "star3d4r", "dtype": "f32",
         "n0": 512, "n1": 512, "n2": 512, "T": 100, "mode": "exact", "pad": 0},
        # 27 points with the source's division, odd extents, double precision
        {"name": "j3d27pt f64 257x300x411", "path": "forward", "stencil": "j3d27pt", "dtype": "f64",
         "n0": 257, "n1": 300, "n2": 411, "T": 60, "mode": "exact", "pad": 0},
        # a wide 3D box (125 points) at a middle size
        {"name": "box3d2r f32 256^3", "path": "forward", "stencil": "box3d2r", "dtype": "f32",
         "n0": 256, "n1": 256, "n2": 256, "T": 50, "mode": "exact", "pad": 0},
        # gradients of an inverse problem: a large one in single precision, a small one in double
        {"name": "adjoint j2d9pt f32 4096x4096", "path": "adjoint", "stencil": "j2d9pt", "dtype": "f32",
         "n0": 4096, "n1": 4096, "n2": 0, "T": 64},
        {"name": "adjoint star2d1r f64 300x500", "path": "adjoint", "stencil": "star2d1r", "dtype": "f64",
         "n0": 300, "n1": 500, "n2": 0, "T": 40},
        # the batched workload: sides 256 to 4096, 64 to 1024 steps
        {"name": "batch of 24", "path": "batch", "count": 24, "mix": 2024},
    ]


def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _flops_per_cell(name):
    dim, rad, shape, div = STENCILS[name]
    if name == "gradient2d":
        return 19
    taps = (2 * rad + 1) ** dim if shape == "box" else 2 * dim * rad + 1
    return 2 * taps - 1 + (1 if div else 0)


def draw(rng):
    path = rng.choice(["forward"] * 6 + ["adjoint", "adjoint", "host", "batch"])
    if path == "batch":
        return {"path": path, "count": rng.randint(8, 30), "mix": rng.randrange(1 << 30)}
    names = [s for s in STENCILS if path != "adjoint" or STENCILS[s][0] == 2 and s != "gradient2d"]
    if path == "host":
        # the sources' own literals: these three's amplify a field until it overflows
        names = [s for s in names if s not in ("star2d4r", "box3d2r", "box3d3r")]
    name = rng.choice(names)
    dim = STENCILS[name][0]
    case = {"path": path, "stencil": name, "dtype": rng.choice(["f32", "f64"]), "n0": 0, "n1": 0, "n2": 0}
    if dim == 2:
        side = _log_uniform(rng, 256, {"forward": 16384, "adjoint": 4096, "host": 4096}[path])
        case["n0"], case["n1"] = (int(side * f) for f in rng.choice([(1, 1), (1, 0.25), (0.25, 1), (0.7, 0.9)]))
    else:
        side = _log_uniform(rng, 64, 512 if path == "forward" else 256)
        case["n0"], case["n1"], case["n2"] = (int(side * rng.uniform(0.6, 1)) for _ in range(3))
    steps = _log_uniform(rng, 16, 1000)
    cells = case["n0"] * case["n1"] * max(1, case["n2"])
    most = MOST_FLOPS / (cells * _flops_per_cell(name))
    if path == "adjoint":
        # forward, states again and two products per tap; as many states as the listed largest case
        most = min(most / 4, 64 * 4096.0**2 / cells)
    if name == "gradient2d":
        most = min(most, 32)
    if path == "host":
        # the drop-in runs cubes with the source's own coefficients
        case["n1"] = case["n0"]
        case["n2"] = case["n0"] if dim == 3 else 0
        cells = float(case["n0"]) ** dim
        most = min(100, MOST_FLOPS / (cells * _flops_per_cell(name)))
    case["T"] = max(2, int(min(steps, most)) // 2 * 2)
    if path == "forward":
        # the FMA mode is for the stencils whose taps all add; these two subtract some
        case["mode"] = "exact" if name in ("box3d2r", "box3d3r") else rng.choice(["exact", "exact", "exact", "fast"])
        case["pad"] = rng.choice([0, 0, 0, rng.randint(1, 64)])
    return case


def _extents(c):
    return [c[k] for k in ("n0", "n1", "n2") if c[k]]


def _torch_dtype(c):
    return torch.float32 if c["dtype"] == "f32" else torch.float64


def _offsets(name):
    dim, rad, shape, _ = STENCILS[name]
    span = range(-rad, rad + 1)
    grid = [(a, b, d) for a in span for b in (span if dim == 3 else (0,)) for d in span]
    return [o for o in grid if shape == "box" or sum(x != 0 for x in o) <= 1]


def _weights(name, dtype):
    """{offset: coefficient} as the working precision holds them, and the
    divisor: the benchmark's coefficients for the two small stars, else
    uniform (0, 1] ones that sum to the source's divisor (or 1)."""
    offs = _offsets(name)
    div = float(STENCILS[name][3])
    if name == "j2d5pt":
        w = {(-1, 0, 0): 5.1, (0, 0, -1): 12.1, (0, 0, 0): 15.0, (0, 0, 1): 12.2, (1, 0, 0): 12.3}
    elif name == "star3d1r":
        w = {o: 0.4 if o == (0, 0, 0) else 0.1 for o in offs}
    else:
        v = 1.0 - np.random.default_rng(1000 + sorted(STENCILS).index(name)).random(len(offs))
        v *= (div or 1.0) / v.sum()
        w = dict(zip(offs, v))
    hold = np.float32 if dtype == torch.float32 else np.float64
    return {o: float(hold(x)) for o, x in w.items()}, div


def _coefs(name, dtype):
    """The library's coefficient array (its tap order, its signs) and divisor."""
    if name == "gradient2d":
        return np.array([1e-4, 0.01]), -1.0
    w, div = _weights(name, dtype)
    taps, _ = pyan5d.taps(name)
    return np.array([s * w[(a, b, d)] for s, a, b, d in taps.tolist()]), div


def _rand(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(shape, dtype=dtype, device="cuda", generator=g)


def _batch_work(case):
    """(stencil, extents, steps) of a batch: sides log-uniform in [256, 4096],
    half squares and half 1:4 rectangles, 64 to 1024 steps."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["count"]):
        name = BATCH_STENCILS[int(rng.integers(0, 3))]
        side = int(round(float(np.exp(rng.uniform(np.log(256), np.log(4096))))))
        n = [[side, side], [side, side], [max(1, side // 4), side], [side, max(1, side // 4)]][int(rng.integers(0, 4))]
        out.append((name, n, 2 * int(rng.integers(32, 513))))
    return out


def _start_grid(name, n, dtype, seed):
    r = STENCILS[name][1]
    return _rand([x + 2 * r for x in n], dtype, seed)


def _host_grid(case, seed):
    r = STENCILS[case["stencil"]][1]
    hold = np.float32 if case["dtype"] == "f32" else np.float64
    return np.random.default_rng(seed).random([x + 2 * r for x in _extents(case)], dtype=hold)


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        items = []
        for i, (name, n, T) in enumerate(_batch_work(case)):
            u = _start_grid(name, n, torch.float32, 1000 * seed + i)
            c, div = _coefs(name, torch.float32)
            items.append((name, n, T, torch.stack([u, u]), c, div))
        return {"path": path, "batch": pyan5d.Batch(items), "grids": [it[3] for it in items]}
    name, n = case["stencil"], _extents(case)
    state = {"path": path, "name": name, "n": n, "T": case["T"]}
    if path == "host":
        u = _host_grid(case, seed)
        state["A"] = np.stack([u, u])
        return state
    dtype = _torch_dtype(case)
    state["coefs"], state["div"] = _coefs(name, dtype)
    u = _start_grid(name, n, dtype, seed)
    if path == "forward":
        D = list(u.shape)
        t = torch.zeros([2] + D[:-1] + [D[-1] + case["pad"]], dtype=dtype, device="cuda")[..., :D[-1]]
        t.copy_(u.expand(2, *D))
        state["grid"] = t
        state["mode"] = pyan5d.FAST if case["mode"] == "fast" else pyan5d.EXACT
        return state
    state["u0"] = u
    state["target"] = _start_grid(name, n, dtype, seed + 500000)
    state["grad"] = torch.zeros_like(u)
    state["gcoef"] = torch.zeros(len(state["coefs"]), dtype=torch.float64, device="cuda")
    state["loss"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    state["ws"] = pyan5d.AdjointWorkspace(name, n, case["T"], np.float32 if dtype == torch.float32 else np.float64)
    return state


def run(state):
    path = state["path"]
    if path == "batch":
        state["batch"].run()
        return [t[0] for t in state["grids"]]
    name, n, T = state["name"], state["n"], state["T"]
    if path == "host":
        pyan5d.kernel_stencil(name, state["A"], n[0], T)
        return state["A"][0]
    if path == "forward":
        pyan5d.forward_device(name, state["grid"], n, T, coefs=state["coefs"], divisor=state["div"],
                              mode=state["mode"])
        return state["grid"][0]
    pyan5d.adjoint_device(name, state["u0"], state["target"], state["grad"], state["gcoef"], state["loss"], n, T,
                          state["ws"], coefs=state["coefs"], divisor=state["div"])
    return {"grad": state["grad"], "gcoef": state["gcoef"], "loss": state["loss"]}


def work(case):
    """One read and one write of every grid that goes in or comes out; the
    C expression's operations at every step (adjoint: those, and a
    multiply-add per tap each for the states, the coefficients and the
    transposed taps)."""
    if case["path"] == "batch":
        cells = [(float(np.prod(n)), T, name) for name, n, T in _batch_work(case)]
        return {"bytes": sum(8 * c for c, _, _ in cells), "flops": sum(c * T * _flops_per_cell(s) for c, T, s in cells)}
    size = 4 if case["dtype"] == "f32" else 8
    cells = float(np.prod(_extents(case)))
    flops = cells * case["T"] * _flops_per_cell(case["stencil"])
    if case["path"] == "adjoint":
        return {"bytes": 3 * size * cells, "flops": 3 * flops}
    return {"bytes": 2 * size * cells, "flops": flops}


# ---- 64-bit values ---------------------------------------------------------

def _slices(n, r, o):
    """The interior of a grid (extents n, halo r) moved by offset o."""
    o = (o[0], o[2]) if len(n) == 2 else o
    return tuple(slice(r + d, r + d + x) for d, x in zip(o, n))


def _step(u, out, n, r, w, div):
    acc = out[_slices(n, r, (0, 0, 0))]
    acc.zero_()
    for o, c in w.items():
        acc.add_(u[_slices(n, r, o)], alpha=c)
    if div:
        acc.div_(div)


def _forward64(u, n, T, r, w, div):
    a, b = u, u.clone()
    for _ in range(T):
        _step(a, b, n, r, w, div)
        a, b = b, a
    return a


def exact(case, seed):
    path = case["path"]
    if path == "batch":
        out = []
        for i, (name, n, T) in enumerate(_batch_work(case)):
            w, div = _weights(name, torch.float32)
            u = _start_grid(name, n, torch.float32, 1000 * seed + i).double()
            out.append(_forward64(u, n, T, STENCILS[name][1], w, div))
        return out
    name, n, T = case["stencil"], _extents(case), case["T"]
    if name == "gradient2d":
        return None  # its steep reciprocal root amplifies every rounding: no 64-bit value to hold it to
    r = STENCILS[name][1]
    if path == "host":
        if name != "j2d5pt":
            return None  # the other sources' literals are the library's own table
        w = {(-1, 0, 0): 5.1, (0, 0, -1): 12.1, (0, 0, 0): 15.0, (0, 0, 1): 12.2, (1, 0, 0): 5.2}
        w = {o: float(np.float32(c)) for o, c in w.items()}
        return _forward64(torch.from_numpy(_host_grid(case, seed)).cuda().double(), n, T, r, w, 118.0)
    dtype = _torch_dtype(case)
    w, div = _weights(name, dtype)
    u = _start_grid(name, n, dtype, seed).double()
    if path == "forward":
        return _forward64(u, n, T, r, w, div)
    # adjoint of 1/2 sum (u_T - target)^2 over the interior, halo fixed
    target = _start_grid(name, n, dtype, seed + 500000).double()
    mid = _slices(n, r, (0, 0, 0))
    states = [u]
    for _ in range(T):
        nxt = states[-1].clone()
        _step(states[-1], nxt, n, r, w, div)
        states.append(nxt)
    mu = torch.zeros_like(u)
    mu[mid] = states[-1][mid] - target[mid]
    loss = 0.5 * mu.square().sum().reshape(1)
    d = div or 1.0
    back = {tuple(-x for x in o): c for o, c in w.items()}
    signs = {(a, b, e): s for s, a, b, e in pyan5d.taps(name)[0].tolist()}
    order = list(signs)
    gc = {o: torch.zeros((), dtype=torch.float64, device="cuda") for o in order}
    for t in range(T - 1, -1, -1):
        for o in order:
            gc[o] += (mu[mid] * states[t][_slices(n, r, o)]).sum()
        lam = torch.zeros_like(mu)
        _step(mu, lam, n, r, back, div)
        mu = lam
        states.pop()
    return {"grad": mu, "gcoef": torch.stack([signs[o] * gc[o] / d for o in order]), "loss": loss}
