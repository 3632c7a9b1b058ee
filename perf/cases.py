"""The work that is timed: batched tridiagonal solves as programs that use this
library make them, through its Python entry points (the same C calls a C
program makes). Every call is stream-ordered (sync=False, the default) and
takes the library's own choice of kernel shape: nothing is tuned beforehand.

Kinds of case (the key "kind"):

  sweeps   the x, y and z solves of one right-hand side one after another, in
           place, on a small cube: the call pattern of an ADI code whose grid
           is small, where launches and host time count
  solve    one batched solve of a 2-D or 3-D grid along one direction, in
           place (d <- x) or incremental (u += x), FP64 or FP32, dense or
           inside a halo
  ragged   systems of uneven lengths stored back to back, in place
  mixed32  the FP64 solution of a batch stored in FP32, one refinement
  grad     a differentiable solve: forward, then the gradients of all four
           operands for an incoming gradient
  adi      a number of ADI heat-diffusion steps on a grid, with the
           coefficient arrays or matrix-free

Operands: solves that add into u, the FP32-stored and the differentiable ones
take a, c ~ U(-1, 1), b = 2 + |a| + |c| + U(0, 1), d ~ U(-1, 1). Solves in
place take an implicit diffusion step with zero-flux ends, a, c ~ -U(0, 1)
(0 at the ends of a system), b = 1 - a - c: its solution has the size of its
right-hand side, so that solving again and again in the same array neither
grows nor dies out. The ADI grids keep random values on their boundary.
"""
import math

import numpy as np
import torch

from tridsolver_amd import adi, api
from tridsolver_amd.autograd import trid_solve

DTYPE = {"f64": torch.float64, "f32": torch.float32}
AXIS = {"x": 0, "y": 1, "z": 2}

# The most that a drawn case may move (the grid of the largest listed solve,
# 512^3 points of five FP64 arrays).
MOST_BYTES = 40 * 512**3


def listed():
    return [
        # the smallest: a 64^3 FP64 cube, one solve along each direction
        {"name": "sweeps_64_f64", "kind": "sweeps", "nx": 64, "ny": 64, "nz": 64,
         "dtype": "f64"},
        # the largest single solves: 512^3 FP64 along the contiguous and the
        # slowest direction
        {"name": "solve_x_512_f64", "kind": "solve", "nx": 512, "ny": 512, "nz": 512,
         "dir": "x", "dtype": "f64", "inc": False, "halo": 0},
        {"name": "solve_z_512_f64", "kind": "solve", "nx": 512, "ny": 512, "nz": 512,
         "dir": "z", "dtype": "f64", "inc": False, "halo": 0},
        # an ordinary FP32 grid, not a power of two, adding the solution into
        # the field
        {"name": "solve_y_inc_f32", "kind": "solve", "nx": 400, "ny": 360, "nz": 300,
         "dir": "y", "dtype": "f32", "inc": True, "halo": 0},
        # a domain inside a halo (offset first point, padded pitches), long in z
        {"name": "solve_z_halo_f64", "kind": "solve", "nx": 190, "ny": 150, "nz": 700,
         "dir": "z", "dtype": "f64", "inc": False, "halo": 2},
        # a large 2-D grid along its slow direction: few long strided systems
        {"name": "solve_2d_y_f64", "kind": "solve", "nx": 4096, "ny": 4096, "nz": 1,
         "dir": "y", "dtype": "f64", "inc": False, "halo": 0},
        # 40,000 systems of 8 to 8192 rows, lengths log-uniform
        {"name": "ragged_40k_f64", "kind": "ragged", "systems": 40000, "min_len": 8,
         "max_len": 8192, "dtype": "f64"},
        # an ordinary ragged batch of short and middle-sized FP32 systems
        {"name": "ragged_6k_f32", "kind": "ragged", "systems": 6000, "min_len": 30,
         "max_len": 1500, "dtype": "f32"},
        # a large batch stored in FP32 and solved to FP64 accuracy
        {"name": "mixed32_z_384", "kind": "mixed32", "nx": 384, "ny": 384, "nz": 384,
         "dir": "z", "refinements": 1},
        # training through a solve: forward and all four gradients
        {"name": "grad_y_256_f64", "kind": "grad", "nx": 256, "ny": 256, "nz": 256,
         "dir": "y", "dtype": "f64"},
        # whole calls: 20 ADI steps with coefficient arrays, as the reference
        # app keeps them, and 10 matrix-free FP32 steps on an odd-sized grid
        {"name": "adi_256_f64", "kind": "adi", "nx": 256, "ny": 256, "nz": 256,
         "dtype": "f64", "matrix_free": False, "steps": 20},
        {"name": "adi_free_f32", "kind": "adi", "nx": 200, "ny": 168, "nz": 147,
         "dtype": "f32", "matrix_free": True, "steps": 10},
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        kind = rng.choice(("sweeps", "solve", "solve", "solve", "solve", "ragged", "ragged",
                           "mixed32", "grad", "adi"))
        case = {"kind": kind}
        if kind == "ragged":
            lo = size(8, 64)
            case.update(systems=size(300, 40000), min_len=lo, max_len=size(2 * lo, 8192),
                        dtype=rng.choice(("f64", "f32")))
        elif kind == "solve" and rng.random() < 0.25:
            case.update(nx=size(64, 8192), ny=size(64, 8192), nz=1, dir=rng.choice("xy"),
                        dtype=rng.choice(("f64", "f32")), inc=rng.random() < 0.3, halo=0)
        else:
            hi = {"sweeps": 96, "solve": 1024, "mixed32": 512, "grad": 300, "adi": 300}[kind]
            lo = {"sweeps": 16, "solve": 24, "mixed32": 48, "grad": 32, "adi": 32}[kind]
            case.update(nx=size(lo, hi), ny=size(lo, hi), nz=size(lo, hi))
            if kind != "adi":
                case["dir"] = rng.choice("xyz")
            if kind == "sweeps":
                del case["dir"]
            if kind == "mixed32":
                case["refinements"] = 1
            else:
                case["dtype"] = rng.choice(("f64", "f64", "f32"))
            if kind == "solve":
                case.update(inc=rng.random() < 0.3, halo=rng.choice((0, 0, 1, 2)))
            if kind == "adi":
                case.update(matrix_free=rng.random() < 0.5, steps=rng.choice((5, 10, 20)))
        if work(case)["bytes"] <= MOST_BYTES and _points(case) >= 4000:
            return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _lengths(case):
    """The lengths of a ragged batch: the quantiles of a log-uniform law, the
    same multiset for every seed (prepare shuffles it)."""
    n, lo, hi = case["systems"], case["min_len"], case["max_len"]
    q = (np.arange(n) + 0.5) / n
    return np.clip(np.floor(lo * (hi / lo) ** q + 0.5).astype(np.int64), lo, hi)


def _dims(case):
    d = [case["nx"], case["ny"], case["nz"]]
    return d[:2] if case["nz"] == 1 and case["kind"] == "solve" else d


def _points(case):
    if case["kind"] == "ragged":
        return int(_lengths(case).sum())
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Each input read once and each output written once; about nine
    operations a point for one solve."""
    n = _points(case)
    kind = case["kind"]
    real = 4 if case.get("dtype") == "f32" else 8
    if kind == "sweeps":
        return {"bytes": 5 * real * n, "flops": 27 * n}
    if kind == "solve":
        return {"bytes": (6 if case["inc"] else 5) * real * n, "flops": 9 * n}
    if kind == "ragged":
        return {"bytes": 5 * real * n + 8 * (case["systems"] + 1), "flops": 9 * n}
    if kind == "mixed32":
        return {"bytes": 24 * n, "flops": 30 * n}
    if kind == "grad":
        # forward a, b, c, d read, x written; backward a, b, c, x and the
        # incoming gradient read, four gradients written
        return {"bytes": 14 * real * n, "flops": 24 * n}
    # adi: per step u read and du written, du read and written, du and u read
    # and u written; the three coefficient arrays written once
    coef = 0 if case["matrix_free"] else 3
    return {"bytes": (7 * case["steps"] + coef) * real * n, "flops": 37 * n * case["steps"]}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.dtype = dtype

    def __call__(self, lo, hi, *shape):
        t = torch.empty(shape, dtype=self.dtype, device="cuda")
        return t.uniform_(lo, hi, generator=self.g)


def _dominant(rand, *shape):
    a, c = rand(-1, 1, *shape), rand(-1, 1, *shape)
    b = rand(2, 3, *shape).add_(a.abs()).add_(c.abs())
    return a, b, c


def _diffusion(rand, *shape):
    return rand(-1, 0, *shape), rand(-1, 0, *shape)


def _flux_free(a, c, first, last):
    """b = 1 - a - c with a 0 in every system's first row and c in its last."""
    a[first] = 0
    c[last] = 0
    return 1 - a - c


def _grid_inputs(case, seed):
    """The operands of a grid solve: (a, b, c, d, u or None, layout)."""
    rand = _Rand(seed, DTYPE[case.get("dtype", "f32")])
    dims = _dims(case)
    h = case.get("halo", 0)
    pads = [n + 2 * h for n in dims]
    shape = pads[::-1]
    offset, stride = 0, 1
    for p in pads:
        offset += h * stride
        stride *= p
    if case["kind"] == "solve" and not case["inc"]:
        a, c = _diffusion(rand, *shape)
        axis = len(dims) - 1 - AXIS[case["dir"]]
        first = [slice(None)] * len(dims)
        last = list(first)
        first[axis], last[axis] = h, h + dims[AXIS[case["dir"]]] - 1
        b = _flux_free(a, c, tuple(first), tuple(last))
    else:
        a, b, c = _dominant(rand, *shape)
    d = rand(-1, 1, *shape)
    u = rand(-1, 1, *shape) if case["kind"] == "solve" and case["inc"] else None
    return a, b, c, d, u, {"dims": dims, "pads": pads, "offset": offset}


def _sweep_inputs(case, seed):
    """One coefficient set for all three directions: zero flux at every face."""
    rand = _Rand(seed, DTYPE[case["dtype"]])
    shape = _dims(case)[::-1]
    a, c = _diffusion(rand, *shape)
    for axis in range(3):
        for end in (0, shape[axis] - 1):
            face = [slice(None)] * 3
            face[axis] = end
            a[tuple(face)] = 0
            c[tuple(face)] = 0
    return a, 1 - a - c, c, rand(-1, 1, *shape)


def _ragged_inputs(case, seed):
    rand = _Rand(seed, DTYPE[case["dtype"]])
    lengths = np.random.default_rng(seed).permutation(_lengths(case))
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)])).cuda()
    n = int(lengths.sum())
    a, c = _diffusion(rand, n)
    b = _flux_free(a, c, offsets[:-1], offsets[1:] - 1)
    return a, b, c, rand(-1, 1, n), offsets


def _adi_field(case, seed):
    rand = _Rand(seed, DTYPE[case["dtype"]])
    return rand(0, 1, case["nx"] * case["ny"] * case["nz"])


LAMBDA = 1.0


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sweeps":
        return dict(zip("abcd", _sweep_inputs(case, seed)), case=case)
    if kind == "ragged":
        return dict(zip(("a", "b", "c", "d", "offsets"), _ragged_inputs(case, seed)), case=case)
    if kind == "adi":
        u = _adi_field(case, seed)
        if case["matrix_free"]:
            return {"case": case, "u": u, "du": torch.empty_like(u)}
        return {"case": case, "u": u,
                "ws": adi.Workspace(case["nx"], case["ny"], case["nz"], u.dtype)}
    a, b, c, d, u, layout = _grid_inputs(case, seed)
    state = {"case": case, "a": a, "b": b, "c": c, "d": d, "u": u, "layout": layout,
             "solvedim": AXIS[case["dir"]]}
    if kind == "mixed32":
        state["x"] = torch.empty(d.shape, dtype=torch.float64, device="cuda")
    if kind == "grad":
        # the incoming gradient of x, and the operands as leaves
        state["w"] = _Rand(seed + 1, d.dtype)(-1, 1, *d.shape)
        for k in "abcd":
            state[k].requires_grad_(True)
    return state


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "sweeps":
        for sd in range(3):
            api.trid_strided_batch(s["a"], s["b"], s["c"], s["d"], solvedim=sd)
        return s["d"]
    if kind == "solve":
        return api.trid_strided_batch(s["a"], s["b"], s["c"], s["d"], u=s["u"],
                                      solvedim=s["solvedim"], **s["layout"])
    if kind == "ragged":
        return api.ragged_batch(s["a"], s["b"], s["c"], s["d"], s["offsets"],
                                max_len=case["max_len"])
    if kind == "mixed32":
        return api.mixed_f32_strided_batch(s["a"], s["b"], s["c"], s["d"], s["x"],
                                           solvedim=s["solvedim"],
                                           refinements=case["refinements"])
    if kind == "grad":
        x = trid_solve(s["a"], s["b"], s["c"], s["d"], s["solvedim"])
        return (x.detach(),) + torch.autograd.grad(x, [s[k] for k in "abcd"], s["w"])
    if case["matrix_free"]:
        adi.run_fused(LAMBDA, s["u"], s["du"], case["steps"],
                      (case["nx"], case["ny"], case["nz"]))
        return s["u"]
    ws = s["ws"]
    adi.run(LAMBDA, s["u"], ws, case["steps"])
    return s["u"], ws.a, ws.b, ws.c


# ---------------------------------------------------------------------------
# the same in 64 bits, by plain Thomas recurrences
# ---------------------------------------------------------------------------
def _thomas(a, b, c, d):
    """Solves along the first axis of [rows, systems] arrays: x."""
    n = d.shape[0]
    cp, x = [None] * n, d.clone()
    inv = 1 / b[0]
    x[0] *= inv
    for i in range(n):
        if i:
            inv = 1 / (b[i] - a[i] * cp[i - 1])
            x[i] = (x[i] - a[i] * x[i - 1]) * inv
        cp[i] = c[i] * inv if i + 1 < n else None
    for i in range(n - 2, -1, -1):
        x[i] -= cp[i] * x[i + 1]
    return x


def _along(axis, a, b, c, d):
    """_thomas along an axis of dense arrays, in FP64."""
    def rows(t):
        return t.detach().double().movedim(axis, 0).contiguous()

    ta, tb, tc, td = rows(a), rows(b), rows(c), rows(d)
    return _thomas(ta, tb, tc, td).movedim(0, axis).contiguous()


def _ragged_exact(a, b, c, d, offsets):
    """Row i of every system that has one, longest systems first."""
    a, b, c, x = (t.double() for t in (a, b, c, d))
    x = x.clone()
    lengths, order = (offsets[1:] - offsets[:-1]).sort(descending=True)
    start = offsets[:-1][order]
    host = lengths.cpu().numpy()
    alive = np.searchsorted(-host, -np.arange(int(host[0])), side="left")  # length > i
    cp = torch.zeros_like(x)
    for i in range(int(host[0])):
        at = start[:alive[i]] + i
        if i:
            ai = a[at]
            inv = 1 / (b[at] - ai * cp[at - 1])
            x[at] = (x[at] - ai * x[at - 1]) * inv
        else:
            inv = 1 / b[at]
            x[at] = x[at] * inv
        cp[at] = c[at] * inv
    for i in range(int(host[0]) - 2, -1, -1):
        at = start[:alive[i + 1]] + i  # rows that have a next one
        x[at] -= cp[at] * x[at + 1]
    return x


def _adi_exact(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    u = _adi_field(case, seed).double().view(nz, ny, nx)
    inner = torch.zeros_like(u, dtype=torch.bool)
    inner[1:-1, 1:-1, 1:-1] = True
    zero = torch.zeros_like(u)
    a = torch.where(inner, zero - 0.5 * LAMBDA, zero)
    b = torch.where(inner, zero + 1 + LAMBDA, zero + 1)
    for _ in range(case["steps"]):
        du = zero.clone()
        du[1:-1, 1:-1, 1:-1] = LAMBDA * (
            u[1:-1, 1:-1, :-2] + u[1:-1, 1:-1, 2:] + u[1:-1, :-2, 1:-1] + u[1:-1, 2:, 1:-1]
            + u[:-2, 1:-1, 1:-1] + u[2:, 1:-1, 1:-1] - 6 * u[1:-1, 1:-1, 1:-1])
        for axis in (2, 1, 0):
            du = _along(axis, a, b, a, du)
        u = u + du
    if case["matrix_free"]:
        return u.reshape(-1)
    return tuple(t.reshape(-1) for t in (u, a, b, a))


def exact(case, seed):
    kind = case["kind"]
    if kind == "adi":
        return _adi_exact(case, seed)
    if kind == "sweeps":
        a, b, c, x = _sweep_inputs(case, seed)
        for axis in (2, 1, 0):
            x = _along(axis, a, b, c, x)
        return x
    if kind == "ragged":
        return _ragged_exact(*_ragged_inputs(case, seed))
    a, b, c, d, u, layout = _grid_inputs(case, seed)
    axis = d.dim() - 1 - AXIS[case["dir"]]
    h = case.get("halo", 0)
    inside = tuple(slice(h, n - h) for n in d.shape)
    x = _along(axis, *(t[inside] for t in (a, b, c, d)))
    if kind == "mixed32":
        return x
    if kind == "solve":
        out = (u if case["inc"] else d).double()
        if case["inc"]:
            out[inside] += x
        else:
            out[inside] = x
        return out
    # grad: A^T lam = w, and the products with x
    w = _Rand(seed + 1, d.dtype)(-1, 1, *d.shape).double()
    n = d.shape[axis]

    def shifted(t, by):
        """Row i holds t's row i + by, 0 where there is none."""
        r = torch.zeros_like(t, dtype=torch.float64)
        lo, hi = max(0, -by), n - max(0, by)
        r.narrow(axis, lo, hi - lo).copy_(t.narrow(axis, lo + by, hi - lo))
        return r

    lam = _along(axis, shifted(c, -1), b, shifted(a, 1), w)
    return (x, -lam * shifted(x, -1), -lam * x, -lam * shifted(x, 1), lam)
