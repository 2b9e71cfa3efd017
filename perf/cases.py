"""The work that programs on this framework have it do, as timed cases.

Each case is a dict of plain values; its "kind" names what a program calls:

  solve     GMG.solve_device: BiCGStab preconditioned by a multigrid cycle, from x = 0
  batch     Batch.solve_device: many independent 2D problems solved together
  variable  GMG.solve_device with the variable-coefficient operator and the Krylov patch smoother
  cycle     GMG.vcycle_device: one multigrid cycle, as the preconditioner of a caller's own iteration
  sweep     DftPlan.apply, then smooth: two smoothing sweeps from u = 0 with the direct patch solver
  krylov    GhostFiller.patch_bicgstab_smooth: two sweeps from u = 0 with the Krylov patch solver
  operator  GhostFiller.star_apply and residual
  transfer  LevelLink.restrict and interpolate
  vector    the vector algebra of one Krylov step: copies, updates, a dot product and a norm

A mesh is a uniform forest of 2^base patches a side, or one whose leaves near a few points are
refined up to level "top"; "mesh" seeds the points.  Vectors are torch tensors in the
framework's padded layout; their ghost cells are scratch space, so results are returned as the
interior cells, except that of a call which fills ghost cells for its caller.
"""
import functools
import math

import numpy as np
import torch

from thunderegg_amd import mesh as M
from thunderegg_amd import runtime as R
from thunderegg_amd import solver as S

FILLERS = {"linear": R.BILINEAR, "quadratic": R.BIQUADRATIC, "trilinear": R.TRILINEAR}
TOL = 1e-10  # of the outer solves, relative to the right-hand side


def listed():
    return [
        # the benchmark's workload: a whole solve on a uniform 3D mesh that fills the card, FP32 cycle
        dict(name="solve_3d_uniform", kind="solve", dim=3, n=16, base=5, top=5, mesh=0, filler="trilinear",
             precision="f32", pre=2, post=2, levels=5),
        # a whole solve on a mesh refined over six levels, as adaptive codes run every time step
        dict(name="solve_2d_adaptive", kind="solve", dim=2, n=16, base=4, top=9, mesh=2, filler="quadratic",
             precision="f32", pre=1, post=1, levels=99),
        # many small problems at once (patch sizes 8, 16 and 32 mixed), each from 16 to about 1000 patches
        dict(name="batch_2d", kind="batch", count=48, mesh=5, precision="f32"),
        # a heterogeneous medium: beta over three decades, Krylov smoother (the direct one does not converge there)
        dict(name="variable_2d", kind="variable", dim=2, n=32, base=4, top=6, mesh=4, filler="linear",
             precision="f32"),
        # one cycle on a locally refined 3D mesh, the preconditioner of a caller's own outer iteration
        dict(name="cycle_3d_refined", kind="cycle", dim=3, n=16, base=2, top=5, mesh=3, filler="trilinear",
             precision="f32", pre=2, post=2, type="V"),
        # the smallest call: one FP64 cycle on 16 patches, where latency and launches count
        dict(name="cycle_2d_small", kind="cycle", dim=2, n=16, base=2, top=2, mesh=0, filler="linear",
             precision="f64", pre=1, post=1, type="V"),
        # the direct patch solver on small 3D patches (deep refinement is done with small patches)
        dict(name="sweep_3d_n8", kind="sweep", dim=3, n=8, base=4, top=4, mesh=0, filler="trilinear",
             precision="f32"),
        # the Krylov patch solver at the reference's own default tolerance, few large patches, FP64
        dict(name="krylov_2d", kind="krylov", dim=2, n=32, base=3, top=3, mesh=0, filler="linear",
             precision="f64", variable=False, tol=1e-12),
        # the operator and the residual of a caller's own iteration, refined 2D mesh, FP64
        dict(name="operator_2d", kind="operator", dim=2, n=16, base=4, top=9, mesh=2, filler="quadratic",
             precision="f64", neumann=False),
        # the same on a refined 3D mesh in FP32, as a level of a caller's own FP32 cycle
        dict(name="operator_3d", kind="operator", dim=3, n=16, base=2, top=5, mesh=3, filler="trilinear",
             precision="f32", neumann=False),
        # the transfers between the two finest levels of a refined 3D mesh
        dict(name="transfer_3d", kind="transfer", dim=3, n=16, base=2, top=5, mesh=3, precision="f64"),
        # the vector algebra of a caller's own Krylov method, 16.8 M cells in FP64
        dict(name="vector_3d", kind="vector", dim=3, n=16, base=4, top=4, mesh=0, precision="f64"),
    ]


def draw(rng):
    kind = rng.choice(["solve", "solve", "batch", "variable", "cycle", "cycle", "sweep", "sweep", "krylov", "operator",
                       "operator", "transfer", "vector"])
    prec = rng.choice(["f32", "f64"])
    seed = rng.randrange(1, 1000)
    if kind == "batch":
        return dict(kind=kind, count=int(round(math.exp(rng.uniform(math.log(6), math.log(48))))), mesh=seed,
                    precision=prec)
    dim = 2 if kind == "variable" else rng.choice([2, 3])
    refined = rng.random() < 0.5 or kind in ("variable", "transfer")
    if dim == 2:
        even = refined or kind == "solve"  # odd sizes are for uniform meshes
        n = rng.choice([8, 12, 16, 16, 20, 32] if even else [7, 8, 10, 13, 16, 16, 24, 32])
        base = rng.randrange(2, 5) if refined else rng.randrange(2, 7)
        top = base + rng.randrange(1, 5) if refined else base
    else:
        n = rng.choice([6, 8, 10, 12, 16, 16])  # the trilinear filler takes even sizes
        base = rng.randrange(1, 3) if refined else rng.randrange(1, 5)
        top = base + rng.randrange(1, 4 if base == 1 else 3) if refined else base
    filler = "trilinear" if dim == 3 else rng.choice(["linear", "quadratic"])
    c = dict(kind=kind, dim=dim, n=n, base=base, top=top, mesh=seed, precision=prec)
    if kind in ("transfer", "vector"):
        return c
    c["filler"] = filler
    if kind == "variable":
        c.update(n=rng.choice([8, 16, 32]), filler="linear", base=rng.randrange(2, 5))
        c["top"] = c["base"] + rng.randrange(1, 3)
    elif kind == "solve":
        c.update(pre=rng.randrange(1, 3), post=rng.randrange(1, 3), levels=99)
    elif kind == "cycle":
        c.update(pre=rng.randrange(1, 3), post=rng.randrange(1, 3), type=rng.choice(["V", "V", "W", "F"]))
    elif kind == "krylov":
        c.update(variable=rng.random() < 0.5, tol=1e-12 if prec == "f64" else 1e-5)
    elif kind == "operator":
        c.update(neumann=rng.random() < 0.25)
    return c


# ---------------------------------------------------------------------------- meshes


@functools.lru_cache(maxsize=64)
def _forest(dim, n, base, top, seed, radius=None):
    """The patch tables of every level, finest first."""
    f = S.Forest(dim, base)
    if top > base:
        pts = np.random.default_rng(seed).uniform(0.0, 1.0, size=(8 if dim == 2 else 4, dim))
        radius = radius or (0.05 if dim == 2 else 0.1)
        for level in range(base, top):
            lo, size = f.leaf_boxes()
            lv, _ = f.leaves()
            q = np.clip(pts[:, None, :], lo[None], (lo + size[:, None])[None])
            near = (((q - pts[:, None, :]) ** 2).sum(axis=2) <= radius * radius).any(axis=0)
            f.refine((near & (lv == level)).astype(np.uint8))
        f.balance()
    return f.build_domains((n,) * dim)


def _levels(c):
    lv = _forest(c["dim"], c["n"], c["base"], c["top"], c["mesh"])
    return lv[: c.get("levels", 99)]


def _problems(c):
    """The problems of a batch: (cells a side, patch tables), sizes and depths spread as in use."""
    out = []
    for k in range(c["count"]):
        r = np.random.default_rng(1000 * c["mesh"] + k)
        n, top = int(r.choice([8, 16, 32])), int(r.integers(3, 8))
        out.append((n, _forest(2, n, 2, top, 1000 * c["mesh"] + k, float(r.uniform(0.01, 0.06)))))
    return out


# --------------------------------------------------------------------------- vectors


class _Vec(R.DeviceArray):
    """A torch tensor handed to the framework where it is."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()
        self.shape, self.dtype = tuple(t.shape), np.dtype(np.float64 if t.dtype == torch.float64 else np.float32)
        self.nbytes = t.numel() * t.element_size()

    def free(self):
        self.ptr = None


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _ftype(c):
    return torch.float64 if c["precision"] == "f64" else torch.float32


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


def _shape(lv, dim, n):
    return M.padded_shape(len(lv), dim, (n,) * dim)


def _rand(shape, g, dtype=torch.float64):
    return torch.randn(shape, generator=g, device=_dev(), dtype=torch.float64).to(dtype)


def _centers(lv, dim, n):
    """Cell-centre coordinates along each axis, (patches, n + 2), ghost cells included."""
    i = torch.arange(-1, n + 1, dtype=torch.float64, device=_dev()) + 0.5
    s, h = (torch.from_numpy(np.ascontiguousarray(lv[k][:, :dim])).to(_dev()) for k in ("starts", "spacings"))
    return [s[:, a, None] + h[:, a, None] * i for a in range(dim)]


def _outer(ax):
    """The product of one factor an axis, in the vector layout."""
    if len(ax) == 2:
        return (ax[1][:, :, None] * ax[0][:, None, :])[:, None]
    return (ax[2][:, :, None, None] * ax[1][:, None, :, None] * ax[0][:, None, None, :])[:, None]


def _rhs(lv, dim, n, g):
    """A right-hand side as these solvers meet it: a few Gaussian sources over a smooth field with noise."""
    X = _centers(lv, dim, n)
    f = _outer([torch.sin(2 * math.pi * x) for x in X]) * (-4.0 * dim * math.pi**2)
    for _ in range(4):
        r = torch.rand(dim + 2, generator=g, device=_dev(), dtype=torch.float64)
        w = 0.005 + 0.045 * r[dim]
        e = _outer([torch.exp(-((x - r[a]) ** 2) / (2 * w * w)) for a, x in enumerate(X)])
        f += (r[dim + 1] - 0.5) * 200.0 * e
    f += 1e-3 * _rand(f.shape, g)
    return f


def _beta(lv, n, seed):
    """exp of a random field of 24 Fourier modes, scaled to three decades."""
    r = np.random.default_rng(seed)
    k, ph = r.integers(-8, 9, size=(24, 2)), r.uniform(0, 2 * np.pi, 24)
    am = r.normal(size=24) / np.maximum(1.0, np.hypot(k[:, 0], k[:, 1]))
    t = np.linspace(0.0, 1.0, 129)
    G = sum(a * np.cos(2 * np.pi * (p * t[:, None] + q * t[None, :]) + w) for a, (p, q), w in zip(am, k, ph))
    am = am * math.log(1e3) / (G.max() - G.min())
    X, Y = _centers(lv, 2, n)
    f = torch.zeros((len(lv), n + 2, n + 2), dtype=torch.float64, device=_dev())
    for a, (p, q), w in zip(am, k, ph):
        f += float(a) * torch.cos(2 * math.pi * (int(p) * X[:, None, :] + int(q) * Y[:, :, None]) + float(w))
    return torch.exp(f)[:, None].contiguous()


def _inner(t, dim):
    return t[..., 1:-1, 1:-1] if dim == 2 else t[..., 1:-1, 1:-1, 1:-1]


def _inputs(c, seed):
    """The case's input tensors, from the seed alone."""
    g, kind = _gen(seed), c["kind"]
    if kind == "batch":
        return [_rhs(lv[0], 2, n, g) for n, lv in _problems(c)]
    lv, dim, n, ty = _levels(c), c["dim"], c["n"], _ftype(c)
    shape = _shape(lv[0], dim, n)
    if kind in ("solve", "variable", "cycle"):
        return [_rhs(lv[0], dim, n, g)]  # the outer vectors are FP64 at either precision of the cycle
    if kind == "transfer":
        return [_rand(shape, g, ty)]
    if kind == "vector":
        return [_rand(shape, g, ty) for _ in range(3)]
    if kind == "operator":
        return [_rand(shape, g, ty), _rhs(lv[0], dim, n, g).to(ty)]
    return [_rhs(lv[0], dim, n, g).to(ty)]


# ------------------------------------------------------------------ the measured calls


def prepare(case, seed):
    c, kind = case, case["kind"]
    ins = [_Vec(t) for t in _inputs(c, seed)]
    prec = R.F64 if c["precision"] == "f64" else R.F32
    st = dict(case=c, ins=ins)
    if kind == "batch":
        probs = _problems(c)
        st["batch"] = S.Batch([((n, n), lv) for n, lv in probs], filler_kind=R.BIQUADRATIC, precision=prec)
        st["xs"] = [_Vec(torch.zeros_like(b.t)) for b in ins]
        torch.cuda.synchronize()
        return st
    lv, dim, n = _levels(c), c["dim"], c["n"]
    ns, like = (n,) * dim, ins[0].t
    if kind in ("solve", "variable", "cycle"):
        o = dict(filler_kind=FILLERS[c["filler"]], precision=prec)
        if kind == "variable":
            o.update(smoother=1, op_kind=1, inner_max_it=50, inner_tol=1e-8,
                     coeffs=[_beta(x, n, c["mesh"]).cpu().numpy() for x in lv])
        else:
            o.update(pre_sweeps=c["pre"], post_sweeps=c["post"], cycle_type=c.get("type", "V"))
        st["gmg"] = S.GMG(dim, ns, lv, **o)
        st["x"] = _Vec(torch.zeros_like(like))
    else:
        st["dom"] = dom = R.Domain(dim, ns, lv[0])
        st["out"] = [_Vec(torch.zeros_like(like)) for _ in range(2)]
        if kind == "transfer":
            st["coarse"] = R.Domain(dim, ns, lv[1])
            st["link"] = R.LevelLink(dom, st["coarse"])
            st["fc"] = _Vec(torch.zeros(_shape(lv[1], dim, n), dtype=like.dtype, device=like.device))
        if kind in ("sweep", "krylov", "operator"):
            st["gf"] = R.GhostFiller(dom, FILLERS[c["filler"]], R.FACES)
        if kind == "sweep":
            st["plan"] = R.DftPlan(st["gf"])
        if kind == "krylov":
            st["beta"] = None
            if c["variable"]:
                st["beta"] = _Vec(_beta(lv[0], n, c["mesh"]).to(like.dtype)) if dim == 2 else _Vec(
                    torch.exp(0.5 * _rand(like.shape, _gen(c["mesh"]))).to(like.dtype))
                st["gf"].fill_ghost(st["beta"])
    torch.cuda.synchronize()
    return st


def run(state):
    c, kind, ins = state["case"], state["case"]["kind"], state["ins"]
    if kind == "batch":
        for x in state["xs"]:
            x.zero()
        state["batch"].solve_device(ins, state["xs"], tol=TOL, precond=2)
        return [_inner(x.t, 2) for x in state["xs"]]
    dim = c["dim"]
    if kind in ("solve", "variable"):
        state["x"].zero()
        state["gmg"].solve_device(ins[0], state["x"], tol=TOL, precond=2)
        return _inner(state["x"].t, dim)
    if kind == "cycle":
        state["gmg"].vcycle_device(ins[0], state["x"])
        return _inner(state["x"].t, dim)
    a, b = state["out"]
    if kind == "sweep":
        state["plan"].apply(ins[0], a)
        state["plan"].smooth(ins[0], a)
        return _inner(a.t, dim)
    if kind == "krylov":
        a.zero()
        for _ in range(2):
            state["gf"].patch_bicgstab_smooth(ins[0], a, op_kind=int(c["variable"]), coeffs=state["beta"],
                                              max_it=1000, tol=c["tol"])
        return _inner(a.t, dim)
    if kind == "operator":
        u, f = ins
        state["gf"].star_apply(u, a, neumann=c["neumann"])
        state["gf"].residual(f, u, b, neumann=c["neumann"])
        return [_inner(a.t, dim), _inner(b.t, dim), u.t]  # u's ghost cells are filled for the caller
    if kind == "transfer":
        state["link"].restrict(ins[0], state["fc"])
        a.zero()
        state["link"].interpolate(state["fc"], a)
        return [_inner(state["fc"].t, dim), _inner(a.t, dim)]
    r, ap, p = ins
    L, h, dt = R.lib(), state["dom"].h, R.F64 if c["precision"] == "f64" else R.F32
    R.check(L.te_vec_copy(h, dt, a.ptr, r.ptr, 1, None))
    R.check(L.te_vec_add_scaled(h, dt, a.ptr, -0.375, ap.ptr, 1, None))
    R.check(L.te_vec_copy(h, dt, b.ptr, p.ptr, 1, None))
    R.check(L.te_vec_scale_then_add(h, dt, b.ptr, 0.625, a.ptr, 1, None))
    return [_inner(a.t, dim), _inner(b.t, dim), state["dom"].dot(a, b), state["dom"].two_norm(a)]


# ------------------------------------------------------------------- what a pass needs


def work(case):
    """Bytes and operations that a pass cannot do without: each step of the method reads its
    operands and writes its results once (a solve: its usual number of iterations)."""
    c, kind = case, case["kind"]
    if kind == "batch":
        w = [_cycle_work(lv, 2, n, c["precision"], 1, 1) for n, lv in _problems(c)]
        cells = sum(len(lv[0]) * n * n for n, lv in _problems(c))
        return dict(bytes=7 * (2 * sum(b for b, _ in w) + 96 * cells), flops=7 * (2 * sum(f for _, f in w) + 60 * cells))
    lv, dim, n = _levels(c), c["dim"], c["n"]
    cells, s = len(lv[0]) * n**dim, 8 if c["precision"] == "f64" else 4
    if kind in ("solve", "cycle", "variable"):
        b, f = _cycle_work(lv, dim, n, c["precision"], c.get("pre", 1), c.get("post", 1))
        if kind == "cycle":
            return dict(bytes=b, flops=f)
        if kind == "variable":  # about 40 inner iterations a sweep, two operators each
            f += sum(len(x) for x in lv) * n * n * 2 * 40 * 60
        return dict(bytes=8 * (2 * b + 96 * cells), flops=8 * (2 * f + 60 * cells))
    if kind == "sweep":
        return dict(bytes=4 * s * cells, flops=2 * 4 * dim * n * cells)
    if kind == "krylov":
        return dict(bytes=5 * s * cells, flops=2 * 60 * 60 * cells)
    if kind == "operator":
        return dict(bytes=5 * s * cells, flops=2 * (3 * dim + 1) * cells)
    if kind == "transfer":
        return dict(bytes=2 * s * (cells + len(lv[1]) * n**dim), flops=2 * cells)
    return dict(bytes=13 * s * cells, flops=8 * cells)


def _cycle_work(lv, dim, n, precision, pre, post):
    s = 8 if precision == "f64" else 4
    cells = sum(len(x) for x in lv) * n**dim
    return s * cells * (3 * (pre + post) + 2), cells * ((pre + post) * 4 * dim * n + 10)


def tolerance(case):
    """About four times the largest differences from 64-bit results that the ranges showed."""
    kind, f64 = case["kind"], case["precision"] == "f64"
    if kind in ("solve", "batch", "variable"):
        rel = 1e-9  # stops at a residual of 1e-10: one iteration more or less changes what is left
    elif kind == "krylov":
        rel = 1e-10 if f64 else 2e-4  # each patch stops at its own residual tolerance
    elif kind == "cycle":
        rel = 4e-13 if f64 else 2e-6
    else:
        rel = 1e-14 if f64 else 1e-6
    return {"rel": rel, "max": 100 * rel}


# ------------------------------------------------------- the same in plain torch, 64 bits


class _Level:
    """One level's patches; vectors are (patches, [z,] y, x) interior cells."""

    def __init__(self, lv, dim, n, filler, beta=None, neumann=False):
        self.P, self.dim, self.n, self.filler, self.neumann = len(lv), dim, n, filler, neumann
        t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(_dev())  # noqa: E731
        at = np.full(int(lv["id"].max()) + 2, -1, dtype=np.int64)
        at[lv["id"]] = np.arange(len(lv))
        self.ih2 = t(1.0 / lv["spacings"][:, :dim] ** 2)
        self.side = []
        for s in range(2 * dim):
            k = M.side_slot(dim, s)
            ty, orth, ids = lv["nbr_type"][:, k], lv["nbr_orth"][:, k], lv["nbr_ids"][:, k]
            pick = lambda m: t(np.flatnonzero(m))  # noqa: E731
            nb = lambda m, w: t(at[ids[m][:, :w]])  # noqa: E731
            self.side.append(dict(
                has=t(ty >= 0), normal=(pick(ty == 0), nb(ty == 0, 1)[:, 0]),
                coarse=[(pick((ty == 1) & (orth == o)), nb((ty == 1) & (orth == o), 1)[:, 0], o)
                        for o in range(1 << (dim - 1))],
                fine=(pick(ty == 2), nb(ty == 2, 1 << (dim - 1)))))
        self.parent = lv["parent_id"].astype(np.int64)
        self.orth = lv["orth_on_parent"].astype(np.int64)
        self.at = at
        # one axis of the patch operator with every side at zero, diagonalised
        T = torch.diag(torch.full((n,), -2.0, dtype=torch.float64)) + torch.diag(torch.ones(n - 1, dtype=torch.float64), 1) \
            + torch.diag(torch.ones(n - 1, dtype=torch.float64), -1)
        T[0, 0] = T[-1, -1] = -3.0
        w, Q = torch.linalg.eigh(T)
        self.w, self.Q = w.to(_dev()), Q.to(_dev())
        self._weights()
        self.beta = None
        if beta is not None:
            b = self.pad(_inner(beta[:, 0], dim), beta[:, 0])
            self.beta = [(b[self._sl(a, 1, n + 1)], b[self._sl(a, 0, n)], b[self._sl(a, 2, n + 2)]) for a in range(dim)]

    def _sl(self, axis, lo, hi):
        ix = [slice(None)] + [slice(1, -1)] * self.dim
        ix[self.dim - axis] = slice(lo, hi)
        return tuple(ix)

    def _weights(self):
        n, z = self.n, lambda *s: torch.zeros(s, dtype=torch.float64)  # noqa: E731
        par, own, inn, up, down = z(2, n, n), z(2, n, n), 0.0, z(2 * n, n), z(n, 2 * n)
        self.fine_inner = 0.0
        i = torch.arange(n)
        if self.filler == "quadratic":
            own[0] = 2.0 / 3 * torch.eye(n, dtype=torch.float64)
            inn = -1.0 / 5
            for k in range(2 * n):
                m = k // 2
                if k == 0 or k == 2 * n - 1:
                    q, wt = (0, 1, 2), (3 / 4, -3 / 10, 1 / 12)
                elif k == 1 or k == 2 * n - 2:
                    q, wt = (0, 1, 2), (7 / 20, 7 / 30, -1 / 20)
                else:
                    q, wt = (m - 1, m, m + 1), ((1 / 12, 1 / 2, -1 / 20) if k % 2 == 0 else (-1 / 20, 1 / 2, 1 / 12))
                for a, b in zip(q, wt):
                    up[k, a if 1 < k < 2 * n - 2 or k < 2 else n - 1 - a] = b
            for k in range(n):
                if k in (0, n - 1):
                    for a, b in zip((0, 1, 2), (-1 / 10, 1 / 15, -1 / 30)):
                        own[1, k, a if k == 0 else n - 1 - a] = b
                else:
                    own[1, k, k - 1] = own[1, k, k + 1] = -1 / 30
            for k in range(2 * n):
                down[k // 2, k] = 1 / 3
            self.fine_inner = 1 / 5
        else:
            own[0] = 2.0 / 3 * torch.eye(n, dtype=torch.float64)
            own[1] = -1.0 / 3 * torch.eye(n, dtype=torch.float64)
            for k in range(2 * n):
                up[k, k // 2] = down[k // 2, k] = 2 / 3
        self.swap = []
        for off in (0, n):  # the other cell of the pair a coarse cell faces
            self.swap.append(torch.where((i + off) % 2 == 0, i + 1, i - 1).clamp(0, n - 1).to(_dev()))
        self.own, self.inn, self.up, self.down = own.to(_dev()), inn, up.to(_dev()), down.to(_dev())

    def _face(self, u, s, depth):
        a, n = s >> 1, self.n
        return u.select(self.dim - a, n - 1 - depth if s & 1 else depth)

    def ghosts(self, u, s):
        """The ghost values over side s (zero where no patch lies across)."""
        d, n = self.side[s], self.n
        own, opp = self._face(u, s, 0), self._face(u, s ^ 1, 0)
        G = torch.zeros_like(own)
        i, q = d["normal"]
        G[i] = opp[q]
        for i, q, o in d["coarse"]:
            if not len(i):
                continue
            if self.dim == 3:
                oi, oj = n * (o & 1), n * (o >> 1)
                x, pi, pj = own[i], self.swap[o & 1], self.swap[o >> 1]
                k = torch.arange(n, device=u.device)
                G[i] = (5 * x - x[:, :, pi] - x[:, pj] - x[:, pj][:, :, pi]) / 6 \
                    + 2 / 3 * opp[q][:, (k + oj) // 2][:, :, (k + oi) // 2]
            else:
                v = own[i] @ self.own[0].T + opp[q] @ self.up[o * n:(o + 1) * n].T
                if self.filler == "quadratic":
                    v += self.inn * self._face(u, s, 1)[i]
                else:
                    v -= own[i][:, self.swap[o]] / 3
                G[i] = v
        i, q = d["fine"]
        if len(i):
            if self.dim == 3:
                F = opp[q].reshape(-1, 2, 2, n, n).permute(0, 1, 3, 2, 4).reshape(-1, n, 2, n, 2).sum(dim=(2, 4))
                G[i] = (F - own[i]) / 3
            else:
                v = own[i] @ self.own[1].T + opp[q].reshape(-1, 2 * n) @ self.down.T
                if self.fine_inner:
                    e = self._face(u, s ^ 1, 1)[q].reshape(-1, n, 2).sum(dim=2)
                    v += self.fine_inner * e
                G[i] = v
        return G

    def pad(self, u, like=None):
        """u with its side ghosts; those over physical sides from `like`, else by the boundary condition."""
        n, D = self.n, self.dim
        v = like.clone() if like is not None else torch.zeros((self.P,) + (n + 2,) * D, dtype=u.dtype, device=u.device)
        v[(slice(None),) + (slice(1, -1),) * D] = u
        for s in range(2 * D):
            ix = list((slice(None),) + (slice(1, -1),) * D)
            ix[D - (s >> 1)] = n + 1 if s & 1 else 0
            own = self._face(u, s, 0)
            phys = v[tuple(ix)] if like is not None else (own if self.neumann else -own)
            has = self.side[s]["has"].reshape((-1,) + (1,) * (D - 1))
            v[tuple(ix)] = torch.where(has, self.ghosts(u, s), phys)
        return v

    def _h(self, a):
        return self.ih2[:, a].reshape((-1,) + (1,) * self.dim)

    def _star(self, v):
        n, out = self.n, 0
        for a in range(self.dim):
            m, lo, hi = (v[self._sl(a, k, n + k)] for k in (1, 0, 2))
            if self.beta is None:
                out = out + (hi - 2 * m + lo) * self._h(a)
            else:
                bm, bl, bh = self.beta[a]
                out = out + ((bh + bm) * (hi - m) - (bl + bm) * (m - lo)) * (self._h(a) / 2)
        return out

    def apply(self, u):
        return self._star(self.pad(u))

    def _patch_rhs(self, f, u):
        f = f.clone()
        for s in range(2 * self.dim):
            a = s >> 1
            has = self.side[s]["has"].reshape((-1,) + (1,) * (self.dim - 1))
            t = (self.ghosts(u, s) + self._face(u, s, 0)) * self.ih2[:, a].reshape((-1,) + (1,) * (self.dim - 1))
            if self.beta is not None:
                bm, bl, bh = self.beta[a]
                t = t * (self._face(bm, s, 0) + self._face(bh if s & 1 else bl, s, 0)) / 2
            self._face(f, s, 0).sub_(torch.where(has, t, torch.zeros_like(t)))
        return f

    def _alone(self, x):
        """The patch operator with zero on every side."""
        v = torch.nn.functional.pad(x, (1, 1) * self.dim)
        for s in range(2 * self.dim):
            ix = list((slice(None),) + (slice(1, -1),) * self.dim)
            ix[self.dim - (s >> 1)] = self.n + 1 if s & 1 else 0
            v[tuple(ix)] = -self._face(x, s, 0)
        return self._star(v)

    def _direct(self, f):
        for back in (0, 1):
            for a in range(self.dim):
                t = f.movedim(self.dim - a, -1)
                f = (t @ (self.Q.T if back else self.Q)).movedim(-1, self.dim - a)
            if not back:
                e = 0
                for a in range(self.dim):
                    sh = [1] * (self.dim + 1)
                    sh[self.dim - a] = self.n
                    e = e + self.w.reshape(sh) * self._h(a)
                f = f / e
        return f.contiguous()

    def smooth(self, f, u):
        f = self._patch_rhs(f, u)
        if self.beta is None:
            return self._direct(f)
        return self._krylov(f)

    def _krylov(self, f, tol=1e-13):
        """Conjugate gradients on every patch at once."""
        dims = tuple(range(1, self.dim + 1))
        dot = lambda a, b: (a * b).sum(dim=dims, keepdim=True)  # noqa: E731
        x, r = torch.zeros_like(f), -f
        p, rr = r.clone(), dot(r, r)
        stop = tol * tol * rr.max()
        for it in range(20 * self.n):
            if it % 16 == 0 and bool((rr <= stop).all()):
                break
            q = -self._alone(p)
            al = rr / dot(p, q).clamp_min(1e-300)
            x += al * p
            r -= al * q
            new = dot(r, r)
            p = r + (new / rr.clamp_min(1e-300)) * p
            rr = new
        return x

    def links(self, coarse):
        return [(o, torch.from_numpy(np.flatnonzero(self.orth == o)).to(_dev()),
                 torch.from_numpy(coarse.at[self.parent[self.orth == o]]).to(_dev())) for o in range(-1, 1 << self.dim)]

    def _over(self, o):
        """The coarse cell over each cell of a child with orthant o."""
        k, n = torch.arange(self.n, device=_dev()), self.n
        axes = [(k + (n if (o >> a) & 1 else 0)) // 2 for a in reversed(range(self.dim))]
        return functools.reduce(lambda a, b: a[..., None] * n + b, axes).reshape(-1)

    def restrict(self, r, coarse):
        f = torch.zeros((coarse.P,) + r.shape[1:], dtype=r.dtype, device=r.device)
        for o, i, q in self.links(coarse):
            if not len(i):
                continue
            if o < 0:
                f[q] += r[i]
                continue
            flat = self._over(o)
            f.view(coarse.P, -1).index_put_((q[:, None], flat[None, :]), r[i].reshape(len(i), -1) / (1 << self.dim),
                                            accumulate=True)
        return f

    def interpolate(self, uc, u, coarse):
        u = u.clone()
        for o, i, q in self.links(coarse):
            if not len(i):
                continue
            flat = self._over(o)
            v = uc[q].reshape(len(q), -1)
            u[i] += (v if o < 0 else v[:, flat]).reshape(u[i].shape)
        return u


def _cycle(L, k, f, u, c, only_v=False):
    pre, post, ty = c.get("pre", 1), c.get("post", 1), c.get("type", "V")
    if k == len(L) - 1:
        return L[k].smooth(f, u)
    for _ in range(pre):
        u = L[k].smooth(f, u)
    uc = torch.zeros((L[k + 1].P,) + f.shape[1:], dtype=f.dtype, device=f.device)
    uc = _cycle(L, k + 1, L[k].restrict(f - L[k].apply(u), L[k + 1]), uc, c)
    u = L[k].interpolate(uc, u, L[k + 1])
    if ty != "V" and not only_v:
        u = L[k].smooth(f, u)
        uc = _cycle(L, k + 1, L[k].restrict(f - L[k].apply(u), L[k + 1]), uc, c, ty == "F")
        u = L[k].interpolate(uc, u, L[k + 1])
    for _ in range(post):
        u = L[k].smooth(f, u)
    return u


def _solve(L, b, c, tol=1e-13):
    """BiCGStab with the 64-bit cycle, to rounding; keeps the best x."""
    pc = lambda v: _cycle(L, 0, v, torch.zeros_like(v), c)  # noqa: E731
    dot = lambda a, q: float((a * q).sum())  # noqa: E731
    x, bn, best = torch.zeros_like(b), math.sqrt(dot(b, b)), None
    for _ in range(3):  # from the true residual again, until that is at rounding
        r = b - L[0].apply(x)
        rn = math.sqrt(dot(r, r)) / bn
        if best is None or rn < best[0]:
            best = (rn, x)
        if rn < tol:
            break
        x, r0, p, rho = x.clone(), r.clone(), r.clone(), dot(r, r)
        for _ in range(60):
            mp = pc(p)
            ap = L[0].apply(mp)
            al = rho / dot(r0, ap)
            s = r - al * ap
            ms = pc(s)
            t = L[0].apply(ms)
            om = dot(t, s) / dot(t, t)
            x += al * mp + om * ms
            r = s - om * t
            if math.sqrt(dot(r, r)) / bn < tol:
                break
            new = dot(r0, r)
            p = r + (new * al / (rho * om)) * (p - om * ap)
            rho = new
    r = b - L[0].apply(x)
    return x if math.sqrt(dot(r, r)) / bn < best[0] else best[1]


def _exact_solution(lv, dim, n, filler, b, c, beta=None):
    L = [_Level(x, dim, n, filler, beta[k] if beta else None) for k, x in enumerate(lv)]
    return _solve(L, _inner(b[:, 0], dim).clone(), c)[:, None]


def exact(case, seed):
    c, kind = case, case["kind"]
    ins = [t.double() for t in _inputs(c, seed)]
    if kind == "batch":
        return [_exact_solution(lv, 2, n, "quadratic", b, c) for (n, lv), b in zip(_problems(c), ins)]
    lv, dim, n = _levels(c), c["dim"], c["n"]
    if kind in ("solve", "variable"):
        beta = [_beta(x, n, c["mesh"]) for x in lv] if kind == "variable" else None
        return _exact_solution(lv, dim, n, c["filler"], ins[0], c, beta)
    if kind == "cycle":
        L = [_Level(x, dim, n, c["filler"]) for x in lv]
        f = _inner(ins[0][:, 0], dim).clone()
        return _cycle(L, 0, f, torch.zeros_like(f), c)[:, None]
    if kind == "vector":
        r, ap, p = (_inner(t, dim) for t in ins)
        w = r - 0.375 * ap
        q = 0.625 * p + w
        return [w, q, float((w * q).sum()), float((w * w).sum().sqrt())]
    beta = None
    if kind == "krylov" and c["variable"]:
        beta = _beta(lv[0], n, c["mesh"]) if dim == 2 else torch.exp(0.5 * _rand(ins[0].shape, _gen(c["mesh"])))
        beta = beta.to(_ftype(c)).double()
    L = _Level(lv[0], dim, n, c.get("filler", "linear"), beta, c.get("neumann", False))
    if kind == "transfer":
        C = _Level(lv[1], dim, n, "linear")
        fc = L.restrict(_inner(ins[0][:, 0], dim).contiguous(), C)
        return [fc[:, None], L.interpolate(fc, torch.zeros_like(_inner(ins[0][:, 0], dim)), C)[:, None]]
    f = _inner(ins[-1][:, 0], dim).contiguous()
    if kind == "operator":
        u = _inner(ins[0][:, 0], dim).contiguous()
        au = L.apply(u)
        return [au[:, None], (f - au)[:, None], L.pad(u, ins[0][:, 0])[:, None]]
    u = torch.zeros_like(f)
    for _ in range(2):
        u = L.smooth(f, u)
    return u[:, None]
