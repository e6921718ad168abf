"""Performance cases of the RBF-FD framework: the calls a program makes through the public entry
points (the C ABI of include/rbfx.h and the Python classes over it), with sizes from the
smallest derivative test to the million-node time step.

Kinds of work:
  step       RK4 steps of a time-dependent PDE (set the state, advance, read the state back)
  apply      derivative application: one operator to one field, or several fused
  weights    batched RBF-FD weight solves
  stencils   kd-tree stencil lists from the GPU search
  operators  building an operator set from stencils and weights, and its first application
  setup      the Stokes solver's set-up: the coupled system and its ILU(0) factor
  solve      Stokes GMRES steps with that preconditioner

Inputs are made from the seed: a jittered golden-angle spiral on the unit sphere, nearest
neighbour stencils, smooth fields. Where a case applies weights (it does not solve for them),
they are consistent finite-difference weights on those stencils: first derivatives and
Laplacians whose rows sum to zero, of the size RBF-FD weights have there.
"""
import math

import numpy as np
import torch

import rbffd_gpu_amd as R
from rbffd_gpu_amd.lib import DeviceView

# shape parameter eps = a sqrt(N) - b per stencil size, the reference's fits
EPS = {17: (0.026, 0.08), 31: (0.035, 0.1), 50: (0.044, 0.14), 75: (0.051, 0.15), 101: (0.058, 0.16)}
UNEVEN = "17,31,50,75,101"
# weights and fields in FP64; both FP32 with FP32 sums; both FP32 with FP64 sums
PRECISIONS = {"f64": (R.F64, R.F64, R.F64), "f32": (R.F32, R.F32, R.F32), "f32_sum64": (R.F32, R.F32, R.F64)}
TORCH_TYPE = {R.F64: torch.float64, R.F32: torch.float32}
STOKES_TYPES = [R.LSFC, R.XSFC, R.YSFC, R.ZSFC]


def listed():
    return [
        # a small interactive run: one field, a few thousand nodes; launches and latency decide
        {"name": "step_small", "kind": "step", "N": 4096, "n": 31, "ops": 3, "fields": 1, "precision": "f64", "steps": 20},
        # the cosine-bell advection: one field, wide stencils, three operators, FP64
        {"name": "step_bell", "kind": "step", "N": 163842, "n": 101, "ops": 3, "fields": 1, "precision": "f64", "steps": 5},
        # the fused shallow-water style step at full size, stored in FP32
        {"name": "step_fields_f32", "kind": "step", "N": 1000000, "n": 50, "ops": 4, "fields": 16, "precision": "f32",
         "steps": 4},
        # the same kind of step in FP64, at an odd size with the reference's common stencil
        {"name": "step_fields_f64", "kind": "step", "N": 262147, "n": 31, "ops": 4, "fields": 16, "precision": "f64",
         "steps": 4},
        # one derivative of one field at full size
        {"name": "apply_one", "kind": "apply", "N": 1000000, "n": 50, "ops": 1, "fields": 1, "precision": "f64"},
        # several derivatives of a handful of fields, all sizes odd
        {"name": "apply_odd", "kind": "apply", "N": 20011, "n": 33, "ops": 4, "fields": 5, "precision": "f32_sum64"},
        # weights of one small derivative test
        {"name": "weights_small", "kind": "weights", "N": 4096, "sizes": "31", "degree": 2},
        # weights of an uneven stencil set
        {"name": "weights_uneven", "kind": "weights", "N": 200000, "sizes": UNEVEN, "degree": 2},
        # stencil lists of the full-size node set
        {"name": "stencils_large", "kind": "stencils", "N": 1000000, "n": 50},
        # stencils and weights in hand: what a program pays until the first derivatives are there
        {"name": "operators_large", "kind": "operators", "N": 400009, "n": 50, "ops": 4, "fields": 16, "precision": "f32"},
        # steady Stokes flow: set-up, and one restart cycle of GMRES(50)
        {"name": "stokes_setup", "kind": "setup", "N": 40962, "n": 31},
        {"name": "stokes_solve", "kind": "solve", "N": 40962, "n": 31, "steps": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "apply", "apply", "weights", "weights", "stencils", "operators", "setup", "solve"])
    if kind == "step":
        fields = rng.choice([1, 1, 2, 3, 4, 8, 16, 16])
        n, ops = rng.choice([17, 31, 37, 50, 75, 101]), rng.choice([3, 4])
        top = min(1000000, int(5e7 / n))
        return {"kind": kind, "N": _log_int(rng, 4096, top), "n": n, "ops": ops, "fields": fields,
                "precision": rng.choice(sorted(PRECISIONS)), "steps": rng.choice([1, 2, 4])}
    if kind == "apply":
        n, ops = rng.choice([17, 31, 33, 50, 101]), rng.choice([1, 1, 2, 3, 4])
        top = min(1000000, int(5e7 / n))
        return {"kind": kind, "N": _log_int(rng, 4096, top), "n": n, "ops": ops, "fields": rng.choice([1, 1, 2, 4, 5, 8, 16]),
                "precision": rng.choice(sorted(PRECISIONS))}
    if kind == "weights":
        sizes = rng.choice(["17", "31", "31", "50", "75", "101", UNEVEN, UNEVEN])
        return {"kind": kind, "N": _log_int(rng, 4096, 100000), "sizes": sizes, "degree": rng.choice([0, 2, 2, 3])}
    if kind == "stencils":
        n = rng.choice([17, 31, 50, 75, 101])
        return {"kind": kind, "N": _log_int(rng, 4096, min(1000000, int(5e7 / n))), "n": n}
    if kind == "operators":
        return {"kind": kind, "N": _log_int(rng, 4096, 400000), "n": rng.choice([31, 37, 50]), "ops": rng.choice([3, 4]),
                "fields": 16, "precision": rng.choice(sorted(PRECISIONS))}
    n = rng.choice([17, 25, 31, 31, 33, 37])
    case = {"kind": kind, "N": _log_int(rng, 2562, 40962 if n <= 31 else 30000), "n": n}
    if kind == "solve":
        case["steps"] = rng.choice([20, 35, 50])
    return case


# ---- inputs ------------------------------------------------------------------------------------


def _nodes(N, seed, project=True):
    """Golden-angle spiral with a uniform jitter of up to 1e-3 (less where nodes are closer) per
    coordinate; numbered along a Morton curve."""
    rng = np.random.default_rng(seed)
    i = np.arange(N) + 0.5
    z = 1.0 - 2.0 * i / N
    phi = i * (math.pi * (3.0 - math.sqrt(5.0)))
    s = np.sqrt(1.0 - z * z)
    xyz = np.stack([s * np.cos(phi), s * np.sin(phi), z], axis=1)
    xyz += rng.uniform(-1.0, 1.0, xyz.shape) * min(1e-3, 0.25 * math.sqrt(4.0 * math.pi / N))
    if project:
        xyz /= np.linalg.norm(xyz, axis=1, keepdims=True)
    q = np.minimum(((xyz + 1.01) * (2**20 / 2.02)).astype(np.int64), 2**20 - 1)
    key = np.zeros(N, np.int64)
    for b in range(20):
        for d in range(3):
            key |= ((q[:, d] >> b) & 1) << (3 * b + d)
    return np.ascontiguousarray(xyz[np.argsort(key, kind="stable")])


def _neighbours(xyz, k):
    """The k nearest nodes of every node, nearest (the node itself) first: int64 (N, k) on the GPU."""
    x = torch.from_numpy(xyz).cuda()
    N = x.shape[0]
    out = torch.empty((N, k), dtype=torch.int64, device="cuda")
    if N <= 16384:
        for a in range(0, N, 4096):
            d = torch.zeros((min(4096, N - a), N), dtype=torch.float64, device="cuda")
            for c in range(3):
                d += (x[a : a + 4096, c, None] - x[None, :, c]) ** 2
            out[a : a + 4096] = torch.topk(d, k, largest=False).indices
        return out
    # cells of the stencil radius: the 27 cells around a node hold all its neighbours
    h = 1.25 * 2.0 * math.sqrt(k / N)
    G = int(2.2 / h) + 3
    c = ((x + 1.1) / h).long() + 1
    key = (c[:, 0] * G + c[:, 1]) * G + c[:, 2]
    by_cell = torch.argsort(key)
    count = torch.bincount(key, minlength=G**3)
    start = torch.cumsum(count, 0) - count
    near = torch.tensor([(a * G + b) * G + d for a in (-1, 0, 1) for b in (-1, 0, 1) for d in (-1, 0, 1)], device="cuda")
    slot = torch.arange(int(count.max()), device="cuda")
    for a in range(0, N, 32768):
        cell = key[a : a + 32768, None] + near
        # non-empty cells first: a surface meets about a third of them
        cell = torch.gather(cell, 1, torch.argsort((count[cell] == 0).to(torch.int8), dim=1, stable=True))
        cell = cell[:, : int((count[cell] > 0).sum(1).max())]
        have = (slot < count[cell][..., None]).flatten(1)
        cand = by_cell[(start[cell][..., None] + slot).clamp(max=N - 1)].flatten(1)
        d = torch.zeros(cand.shape, dtype=torch.float64, device="cuda")
        for e in range(3):
            d += (x[:, e][cand] - x[a : a + 32768, e, None]) ** 2
        d.masked_fill_(~have, math.inf)
        out[a : a + 32768] = torch.gather(cand, 1, torch.topk(d, k, largest=False).indices)
    return out


def _weights(xyz, idx, want):
    """Consistent weights on the stencils, FP64 (N, n) each: 'L' the surface Laplacian, 'x', 'y', 'z'
    the surface gradient's components; Gaussian-weighted, rows summing to zero."""
    x = torch.from_numpy(xyz).cuda()
    N, n = idx.shape
    d = torch.stack([x[:, e][idx] - x[:, e, None] for e in range(3)])
    r2 = (d * d).sum(0)
    g = torch.exp(-2.0 * r2 / r2.mean(1, keepdim=True))
    g[:, 0] = 0.0
    size = (g * r2).sum(1, keepdim=True)
    out = []
    for name in want:
        w = 4.0 * g / size if name == "L" else 2.0 * g * d["xyz".index(name)] / size
        w[:, 0] = -w[:, 1:].sum(1)
        out.append(w)
    return out


def _fields(xyz, F, seed):
    """F smooth fields (N, F): a few plane waves each."""
    g = torch.Generator().manual_seed(int(seed) + 1)
    x = torch.from_numpy(xyz).cuda()
    u = torch.zeros((x.shape[0], F), dtype=torch.float64, device="cuda")
    for _ in range(5):
        k = torch.randn((3, F), generator=g, dtype=torch.float64) * 4.0
        a, p = torch.randn(F, generator=g, dtype=torch.float64), torch.rand(F, generator=g, dtype=torch.float64) * 6.0
        phase = sum(x[:, e, None] * k[e].cuda() for e in range(3))
        u += a.cuda() * torch.cos(phase + p.cuda())
    return u


def _sphere_system(case, seed):
    """Nodes, stencils and operator weights of a case."""
    xyz = _nodes(case["N"], seed)
    idx = _neighbours(xyz, case["n"])
    if case["kind"] in ("setup", "solve"):
        want = "Lxyz"
    elif case["ops"] == 1:
        want = "x"
    else:
        want = "Lxyz"[: case["ops"]]
    return xyz, idx, _weights(xyz, idx, want)


def _pde(case, xyz, ws):
    """Solid-body rotation with a damping term: weights and coefficients per operator, and the time
    step. The damping operator comes scaled into its weights (as hyperviscosity weights do)."""
    spacing = math.sqrt(4.0 * math.pi / case["N"])
    ws = [ws[0] * (0.05 * spacing)] + ws[1:]
    axis = np.array([0.3, -0.2, 1.0])
    vel = np.cross(2.0 * math.pi * axis / np.linalg.norm(axis), xyz)
    coefs = [None] + [torch.from_numpy(np.ascontiguousarray(-vel[:, e])).cuda() for e in range(case["ops"] - 1)]
    return ws, coefs, 0.2 * spacing / (2.0 * math.pi)


def _sizes(case, seed):
    """Stencil sizes, as many of each choice, in an order of the seed; and the CSR offsets."""
    choices = np.array([int(s) for s in case["sizes"].split(",")])
    size = np.random.default_rng([seed, 7]).permutation(np.resize(choices, case["N"]))
    return size, np.concatenate([[0], np.cumsum(size)]).astype(np.int32)


def _weight_problem(case, seed):
    """Nodes, CSR stencils and shape parameters of a weights case."""
    xyz = _nodes(case["N"], seed, project=False)
    size, off = _sizes(case, seed)
    idx = _neighbours(xyz, int(size.max()))
    keep = torch.arange(idx.shape[1], device="cuda") < torch.from_numpy(size).cuda()[:, None]
    a, b = np.array([EPS[s] for s in size]).T
    return xyz, size, off, idx[keep].to(torch.int32), a * math.sqrt(case["N"]) - b


# ---- the framework's handles -------------------------------------------------------------------

_context = None


def _ctx():
    """One context (one stream) for the whole program."""
    global _context
    if _context is None:
        _context = R.Context(0)
    return _context


class _Base:
    def __init__(self, t):
        self.tensor, self.ctx, self.size = t, _ctx(), t.numel()
        self.dtype = np.dtype(str(t.dtype).replace("torch.", ""))
        self.ptr = R.lib.C.c_void_p(t.data_ptr())


def _view(t):
    """A GPU tensor as one of the framework's device arrays."""
    assert t.is_contiguous()
    return DeviceView(_Base(t), 0, tuple(t.shape))


class _State(dict):
    """What a program keeps between calls; its handles are closed with it."""

    def __del__(self):
        for h in reversed(self.get("handles", [])):
            h.close()


def _operators(idx, ws, precision, types=None):
    d_idx = _view(idx.to(torch.int32).contiguous())
    d_ws = [_view(w.contiguous()) for w in ws]
    torch.cuda.synchronize()
    return R.EllOperators(_ctx(), d_idx, d_ws, storage=PRECISIONS[precision][0], types=types)


def _tiles(case):
    """Rows and nodes per tile of the LDS staging, as the benchmark builds them: for 16 fields and
    three or more operators."""
    if case["fields"] != 16 or case["ops"] < 3:
        return None
    f64 = case["precision"] == "f64"
    return 128, (78 * 1024 if f64 else 48 * 1024) // (16 * (8 if f64 else 4))


def prepare(case, seed):
    kind = case["kind"]
    s = _State(case=case, handles=[])
    if kind == "stencils":
        s["xyz"] = _nodes(case["N"], seed, project=False)
        s["out"] = torch.empty((case["N"], case["n"]), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return s
    if kind == "weights":
        xyz, _, off, idx, eps = _weight_problem(case, seed)
        s["off"], s["xyz"], s["eps"] = (torch.from_numpy(v).cuda() for v in (off, xyz, eps))
        s["idx"] = idx
        s["out"] = torch.empty((4, idx.numel()), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        return s
    xyz, idx, ws = _sphere_system(case, seed)
    if kind == "operators":
        s["idx"], s["ws"] = _view(idx.to(torch.int32).contiguous()), [_view(w) for w in ws]
        s["order"] = _view(torch.arange(case["N"], dtype=torch.int32, device="cuda"))
        s["u"] = _fields(xyz, case["fields"], seed).to(TORCH_TYPE[PRECISIONS[case["precision"]][1]])
        s["out"] = torch.empty((case["ops"],) + tuple(s["u"].shape), dtype=s["u"].dtype, device="cuda")
        torch.cuda.synchronize()
        return s
    if kind in ("setup", "solve"):
        ops = _operators(idx, ws, "f64", STOKES_TYPES)
        s["ops"] = ops
        s["handles"].append(ops)
        if kind == "setup":
            s["out"] = torch.empty((case["N"], case["n"]), dtype=torch.float64, device="cuda")
        else:
            s["stokes"] = R.Stokes(_ctx(), ops)
            s["handles"].append(s["stokes"])
            s["b"] = _force(xyz, seed)
            s["x"] = torch.empty_like(s["b"])
        torch.cuda.synchronize()
        return s
    _, ft, acc = PRECISIONS[case["precision"]]
    if kind == "apply":
        ops = _operators(idx, ws, case["precision"])
        s["u"] = _fields(xyz, case["fields"], seed).to(TORCH_TYPE[ft])
        s["out"] = torch.empty((case["ops"],) + tuple(s["u"].shape), dtype=s["u"].dtype, device="cuda")
    else:
        ws, coefs, s["dt"] = _pde(case, xyz, ws)
        ops = _operators(idx, ws, case["precision"])
        s["u"] = _fields(xyz, case["fields"], seed)
        s["out"] = torch.empty_like(s["u"])
        s["coefs"] = coefs
    s["ops"] = ops
    s["handles"].append(ops)
    if _tiles(case):
        ops.build_local(*_tiles(case))
    if kind == "step":
        d_coefs = [None if c is None else _view(c) for c in s["coefs"]]
        s["rk"] = R.RK4(_ctx(), ops, case["fields"], field_storage=ft, accum=acc, coefs=d_coefs)
        s["handles"].append(s["rk"])
    torch.cuda.synchronize()
    return s


def _force(xyz, seed):
    """Right-hand side of the Stokes system: a smooth body force, no divergence, no constraints."""
    N = xyz.shape[0]
    b = torch.zeros(4 * N + 4, dtype=torch.float64, device="cuda")
    b[: 3 * N] = _fields(xyz, 3, seed).T.reshape(-1)
    return b


def run(s):
    case = s["case"]
    kind = case["kind"]
    ctx = _ctx()
    if kind == "step":
        s["rk"].set_state(_view(s["u"]))
        s["rk"].step(s["dt"], case["steps"])
        ctx.check(R.RBFX.rbfx_rk4_get_state(s["rk"].h, _view(s["out"]).ptr))
        return s["out"]
    if kind == "apply":
        _, ft, acc = PRECISIONS[case["precision"]]
        if case["ops"] == 1 and case["fields"] == 1:
            s["ops"].spmv(0, _view(s["u"]), _view(s["out"]), ft, acc)
        else:
            s["ops"].spmm(case["fields"], _view(s["u"]), _view(s["out"]), ft, acc)
        return s["out"]
    if kind == "weights":
        singular = R.lib.C.c_int32()
        ctx.check(R.RBFX.rbfx_weights(ctx.h, case["N"], s["off"].data_ptr(), s["idx"].data_ptr(), case["N"],
                                      s["xyz"].data_ptr(), s["eps"].data_ptr(), R.X | R.Y | R.Z | R.LAPL, 3, case["degree"],
                                      0, 1.0, R.SOLVE_F64_LU, s["out"].data_ptr(), None, R.lib.C.byref(singular)))
        return s["out"]
    if kind == "stencils":
        rows = R.lib.C.c_int32()
        ctx.check(R.RBFX.rbfx_knn_gpu_device(ctx.h, case["N"], s["xyz"].ctypes.data, case["n"], s["out"].data_ptr(),
                                             R.lib.C.byref(rows)))
        return s["out"]
    if kind == "operators":
        storage, ft, acc = PRECISIONS[case["precision"]]
        ops = R.EllOperators(ctx, s["idx"], s["ws"], storage=storage)
        ops.set_row_order(s["order"])
        ops.build_local(*_tiles(case))
        ops.spmm(case["fields"], _view(s["u"]), _view(s["out"]), ft, acc)
        ops.close()
        return s["out"]
    if kind == "setup":
        stokes = R.Stokes(ctx, s["ops"])
        ctx.check(R.RBFX.rbfx_stokes_factor(stokes.h, s["out"].data_ptr()))
        stokes.close()
        return s["out"]
    it, err = R.lib.C.c_int32(), R.lib.C.c_double()
    ctx.check(R.RBFX.rbfx_stokes_gmres(s["stokes"].h, s["b"].data_ptr(), s["x"].data_ptr(), 1e-12, case["steps"],
                                       case["steps"], R.F64, R.lib.C.byref(it), R.lib.C.byref(err)))
    return {"x": s["x"], "steps": it.value, "residual": err.value}


def work(case):
    """Bytes and operations a pass cannot do without: every input read once, every output written
    once (in a time step and in an iteration, once per stage and per iteration)."""
    kind, N = case["kind"], case["N"]
    if kind == "weights":
        size, _ = _sizes(case, 0)
        m = size + math.comb(case["degree"] + 3, 3)
        flops = float((2.0 / 3.0 * m**3 + 2.0 * 4 * m**2).sum())
        return {"bytes": float(size.sum()) * (4 + 4 * 8) + N * 32.0, "flops": flops}
    n = case["n"]
    if kind == "stencils":
        return {"bytes": N * (24.0 + 4.0 * n), "flops": 8.0 * N * n}
    if kind in ("setup", "solve"):
        # row by row: about half the entries are multipliers, each updates what its row shares
        if kind == "setup":
            return {"bytes": N * n * (4 + 8 + 8.0), "flops": N * (n / 2.0) * (n / 4.0) * 2.0}
        k = case["steps"]
        operator, factor, basis = N * n * (4 + 4 * 8.0), N * n * (4 + 8.0), 4.0 * N * 8
        return {"bytes": k * (operator + factor + 6 * basis) + basis * k * k, "flops": k * N * n * 26.0 + 8.0 * N * k * k * 2}
    ops, F = case["ops"], case["fields"]
    s_w = s_f = 8 if case["precision"] == "f64" else 4
    layout = N * n * (4.0 + ops * s_w)
    if kind == "step":
        # the state and the running sum stay FP64; each stage reads and writes a field
        return {"bytes": 2 * 8.0 * N * F + case["steps"] * (4 * (layout + 8.0 * N * (ops - 1)) + N * F * (7 * s_f + 80.0)),
                "flops": case["steps"] * 8.0 * N * n * ops * F}
    applied = N * F * s_f * (1.0 + ops)
    if kind == "apply":
        return {"bytes": layout + applied, "flops": 2.0 * N * n * ops * F}
    return {"bytes": N * n * (4.0 + ops * 8.0) + layout + applied, "flops": 2.0 * N * n * ops * F}


# ---- 64-bit results ----------------------------------------------------------------------------


def _applied(idx, ws, u):
    out = torch.empty((len(ws),) + tuple(u.shape), dtype=torch.float64, device="cuda")
    rows = max(1, 60000000 // (idx.shape[1] * u.shape[1]))
    for a in range(0, idx.shape[0], rows):
        near = u[idx[a : a + rows]]
        for o, w in enumerate(ws):
            out[o, a : a + rows] = (w[a : a + rows, :, None] * near).sum(1)
    return out


def _exact_weights(case, seed):
    xyz, size, off, idx, eps = _weight_problem(case, seed)
    x, idx, eps = torch.from_numpy(xyz), idx.cpu().long(), torch.from_numpy(eps)
    out = torch.empty((4, idx.numel()), dtype=torch.float64)
    for n in sorted(set(size.tolist())):
        deg = case["degree"]
        while deg > 0 and math.comb(deg + 3, 3) > n:
            deg -= 1
        powers = [(a, b, t - a - b) for t in range(deg + 1) for a in range(t, -1, -1) for b in range(t - a, -1, -1)]
        every = torch.from_numpy(np.nonzero(size == n)[0])
        for s in torch.split(every, 2000):
            at = torch.from_numpy(off)[s].long()[:, None] + torch.arange(n)
            p = x[idx[at]]
            d, e2 = p - p[:, :1], (eps[s] ** 2)[:, None]
            r2 = ((p[:, :, None] - p[:, None]) ** 2).sum(-1)
            m = n + len(powers)
            M = torch.zeros((len(s), m, m), dtype=torch.float64)
            M[:, :n, :n] = torch.exp(-e2[..., None] * r2)
            for q, pw in enumerate(powers):
                M[:, :n, n + q] = M[:, n + q, :n] = d[..., 0] ** pw[0] * d[..., 1] ** pw[1] * d[..., 2] ** pw[2]
            rhs = torch.zeros((len(s), m, 4), dtype=torch.float64)
            c2 = (d * d).sum(-1)
            phi = torch.exp(-e2 * c2)
            for e in range(3):
                rhs[:, :n, e] = 2.0 * e2 * d[..., e] * phi
            rhs[:, :n, 3] = e2 * (4.0 * e2 * c2 - 6.0) * phi
            for q, pw in enumerate(powers):
                for e in range(3):
                    rhs[:, n + q, e] = 1.0 if sum(pw) == 1 and pw[e] == 1 else 0.0
                rhs[:, n + q, 3] = 2.0 if sum(pw) == 2 and max(pw) == 2 else 0.0
            w = torch.linalg.solve(M, rhs)[:, :n]
            out[:, at.reshape(-1)] = w.permute(2, 0, 1).reshape(4, -1)
    return out


class _Ilu0:
    """ILU(0) of -L by rows, columns ascending, and the two sweeps by dependency levels."""

    def __init__(self, idx, lap):
        idx = idx.cpu().numpy()
        order = np.argsort(idx, axis=1)
        N, n = idx.shape
        self.col = col = np.take_along_axis(idx, order, 1)
        self.f = f = -np.take_along_axis(lap.cpu().numpy(), order, 1)
        self.diag = dg = (col == np.arange(N)[:, None]).argmax(1)
        place = np.full(N, -1)
        for r in range(N):
            w, c = f[r], col[r]
            place[c] = np.arange(n)
            for q in range(dg[r]):
                k = c[q]
                t = w[q] / f[k, dg[k]]
                w[q] = t
                at = place[col[k, dg[k] + 1 :]]
                hit = at >= 0
                w[at[hit]] -= t * f[k, dg[k] + 1 :][hit]
            place[c] = -1

    def levels(self):
        N, n = self.col.shape
        slot = np.arange(n)
        self.steps = []
        for lower in (True, False):
            side = slot < self.diag[:, None] if lower else slot > self.diag[:, None]
            lev = np.zeros(N, int)
            for r in range(N) if lower else range(N - 1, -1, -1):
                c = self.col[r, : self.diag[r]] if lower else self.col[r, self.diag[r] + 1 :]
                lev[r] = lev[c].max() + 1 if c.size else 0
            rows = np.split(np.argsort(lev, kind="stable"), np.cumsum(np.bincount(lev))[:-1])
            val = np.where(side, self.f, 0.0)
            div = np.ones(N) if lower else self.f[np.arange(N), self.diag]
            for r in rows:
                a, b = (0, self.diag[r].max()) if lower else (self.diag[r].min() + 1, n)
                self.steps.append((r, self.col[r, a:b], val[r, None, a:b], div[r][:, None]))
        return self

    def solve(self, v):
        """Both sweeps on the three velocity blocks of v."""
        N = self.col.shape[0]
        x = np.ascontiguousarray(v[: 3 * N].reshape(3, N).T)
        for r, c, val, div in self.steps:
            x[r] = (x[r] - (val @ x[c])[:, 0]) / div
        return np.concatenate([x.T.reshape(-1), v[3 * N :]])


def _exact_solve(case, seed):
    """GMRES(steps) from zero with left preconditioning: one cycle."""
    xyz, idx, ws = _sphere_system(case, seed)
    N, m = case["N"], case["steps"]
    ilu = _Ilu0(idx, ws[0]).levels()
    b = _force(xyz, seed).cpu().numpy()
    lap, dx, dy, dz = ws

    def operator(v):
        t = torch.from_numpy(v).cuda()
        D = _applied(idx, [lap, dx, dy, dz], t[: 4 * N].reshape(4, N).T.contiguous())
        lam = t[4 * N :]
        y = [-D[0, :, e] + D[e + 1, :, 3] + lam[e] for e in range(3)]
        y.append(D[1, :, 0] + D[2, :, 1] + D[3, :, 2] + lam[3])
        return torch.cat(y + [t[: 4 * N].reshape(4, N).sum(1)]).cpu().numpy()

    V = np.empty((m + 1, 4 * N + 4))
    H = np.zeros((m + 1, m))
    r = ilu.solve(b)
    beta = np.linalg.norm(r)
    V[0] = r / beta
    for k in range(m):
        w = ilu.solve(operator(V[k]))
        for _ in range(2):
            h = V[: k + 1] @ w
            w = w - h @ V[: k + 1]
            H[: k + 1, k] += h
        H[k + 1, k] = np.linalg.norm(w)
        V[k + 1] = w / H[k + 1, k]
    g = np.zeros(m + 1)
    g[0] = beta
    y, _, _, _ = np.linalg.lstsq(H, g, rcond=None)
    return {"x": torch.from_numpy(y @ V[:m]), "steps": None,
            "residual": float(np.linalg.norm(g - H @ y) / np.linalg.norm(b))}


def exact(case, seed):
    kind = case["kind"]
    if kind == "stencils":
        return None
    if kind == "weights":
        # dense solves on the host
        return _exact_weights(case, seed) if case["N"] <= 20000 else None
    if kind == "solve":
        return _exact_solve(case, seed)
    xyz, idx, ws = _sphere_system(case, seed)
    if kind == "setup":
        return torch.from_numpy(_Ilu0(idx, ws[0]).f)
    if kind in ("apply", "operators"):
        return _applied(idx, ws, _fields(xyz, case["fields"], seed))
    ws, coefs, dt = _pde(case, xyz, ws)
    u = _fields(xyz, case["fields"], seed)

    def rhs(v):
        D = _applied(idx, ws, v)
        return sum(D[o] if c is None else c[:, None] * D[o] for o, c in enumerate(coefs))

    for _ in range(case["steps"]):
        k1 = rhs(u)
        k2 = rhs(u + 0.5 * dt * k1)
        k3 = rhs(u + 0.5 * dt * k2)
        k4 = rhs(u + dt * k3)
        u = u + dt / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)
    return u
