"""GPU parity of the single-level kernels against the oracle, through the C ABI.

FP64: max-norm relative difference <= 1e-12 (the hot path's FP64 parity bar).
FP32: the oracle runs on the float-rounded inputs in FP64; max-norm relative
difference <= 2e-6 (a few float ulps accumulated over the stencil / transforms).
"""
import ctypes as C

import numpy as np
import pytest

from helpers import MESH_2D, MESH_3D, face_ghost_mask, load, random_field, relerr
from oracle import oracle as O
from thunderegg_amd import mesh
from thunderegg_amd import runtime as R
from thunderegg_amd import solver

pytestmark = pytest.mark.gpu

TOL64 = 1e-12
TOL32 = 2e-6


def _cases_2d():
    for name in MESH_2D:
        for ns in [(8, 8), (16, 16), (10, 6)]:
            yield name, ns


def _dev(dim, ns, lv):
    return R.Domain(dim, ns, lv)


def _print_case(*a):
    print("case:", *a, flush=True)


@pytest.mark.parametrize("name,ns", list(_cases_2d()))
@pytest.mark.parametrize("kind", [R.BILINEAR, R.BIQUADRATIC])
@pytest.mark.parametrize("fill_type", [R.FACES, R.CORNERS])
def test_ghost_fill_2d(name, ns, kind, fill_type):
    _print_case("ghost2d", name, ns, kind, fill_type)
    dim, levels = load(name, ns)
    lv = levels[0]
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, kind, fill_type)
    for dtype, tol in [(R.F64, TOL64), (R.F32, TOL32)]:
        for ncomp in (1, 2):
            u0 = random_field(od.shape(ncomp), 11 + ncomp, R.np_dtype(dtype))
            ref = u0.astype(np.float64)
            O.fill_ghost(od, ref, kind=kind, fill_type=fill_type)
            du = R.DeviceArray.from_host(u0)
            g.fill_ghost(du)
            got = du.get()
            assert relerr(got, ref) <= tol, (dtype, ncomp)
            # interior cells are untouched
            assert np.array_equal(mesh.interior(got, dim), mesh.interior(u0, dim))


@pytest.mark.parametrize("name", MESH_3D)
@pytest.mark.parametrize("ns", [(4, 4, 4), (6, 4, 8)])
@pytest.mark.parametrize("fill_type", [R.FACES, R.EDGES, R.CORNERS])
def test_ghost_fill_3d(name, ns, fill_type):
    _print_case("ghost3d", name, ns, fill_type)
    dim, levels = load(name, ns)
    lv = levels[0]
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, R.TRILINEAR, fill_type)
    for dtype, tol in [(R.F64, TOL64), (R.F32, TOL32)]:
        u0 = random_field(od.shape(1), 5, R.np_dtype(dtype))
        ref = u0.astype(np.float64)
        O.fill_ghost(od, ref, kind=2, fill_type=fill_type)
        du = R.DeviceArray.from_host(u0)
        g.fill_ghost(du)
        got = du.get()
        assert relerr(got, ref) <= tol
        assert face_ghost_mask(lv, dim, ns, fill_type).sum() > 0


@pytest.mark.parametrize("name,ns", [(n, s) for n, s in _cases_2d() if s != (10, 6)] +
                         [(n, (4, 4, 4)) for n in MESH_3D])
@pytest.mark.parametrize("neumann", [False, True])
def test_star_apply(name, ns, neumann):
    _print_case("star", name, ns, neumann)
    dim, levels = load(name, ns)
    lv = levels[0]
    kind = R.TRILINEAR if dim == 3 else R.BILINEAR
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, kind, R.FACES)
    for dtype, tol in [(R.F64, TOL64), (R.F32, 5e-6)]:
        u0 = random_field(od.shape(1), 3, R.np_dtype(dtype))
        ref = O.poisson_apply(od, u0.astype(np.float64), kind=kind, neumann=neumann)
        du = R.DeviceArray.from_host(u0)
        df = dd.vector(1, dtype)
        g.star_apply(du, df, neumann=neumann)
        got = df.get()
        assert relerr(got, ref) <= tol, dtype
        # residual r = f - A u
        f0 = random_field(od.shape(1), 4, R.np_dtype(dtype))
        dfin = R.DeviceArray.from_host(f0)
        dr = dd.vector(1, dtype)
        g.residual(dfin, du, dr, op_kind=0, neumann=neumann)
        rref = np.zeros_like(ref)
        mesh.interior(rref, dim)[...] = mesh.interior(f0.astype(np.float64) - ref, dim)
        assert relerr(dr.get(), rref) <= tol


@pytest.mark.parametrize("ns,kind,fill_type", [
    ((7, 5), R.BILINEAR, R.FACES), ((4, 32), R.BIQUADRATIC, R.CORNERS), ((34, 6), R.BILINEAR, R.CORNERS),
    ((2, 2, 2), R.TRILINEAR, R.FACES), ((6, 4, 8), R.TRILINEAR, R.EDGES), ((16, 16, 16), R.TRILINEAR, R.CORNERS)])
@pytest.mark.parametrize("off", [0, 1])
def test_star_with_fill_is_fill_then_star(ns, kind, fill_type, off):
    """The operator's launch that fills u's ghosts first: the bits of the ghost fill followed by
    the operator on the filled ghosts, in u and in the result, for two components, single
    values instead of pairs (odd rows, vectors one value off) and both residual operands."""
    dim = len(ns)
    name = "2d_uniform_2x2_mpi1.json" if ns[0] % 2 else (
        "2d_uniform_8x8_refined_cross_mpi1.json" if dim == 2 else "3d_mid_refine_4x4x4_mpi1.json")
    lv = load(name, ns)[1][0]
    dd, L = R.Domain(dim, ns, lv), R.lib()
    g = R.GhostFiller(dd, kind, fill_type)
    shape = mesh.padded_shape(len(lv), dim, ns, 2)
    n = int(np.prod(shape))
    for dtype in (R.F64, R.F32):
        t = R.np_dtype(dtype)
        u0, f0 = random_field((n + off,), 81, t), random_field((n + off,), 82, t)
        for neumann in (0, 1):
            u1, u2, f = (R.DeviceArray.from_host(v) for v in (u0, u0, f0))
            a1, a2, r1 = (R.DeviceArray.from_host(np.full(n + off, 7, t)) for _ in range(3))
            p = [d.ptr + off * t().itemsize for d in (u1, u2, f, a1, a2, r1)]
            R.check(L.te_ghost_fill(g.h, dtype, p[0], 2, None))
            R.check(L.te_star_apply_patches(g.h, dtype, neumann, p[0], p[3], 2, None))
            R.check(L.te_star_apply(g.h, dtype, neumann, p[1], p[4], 2, None))
            assert np.array_equal(u1.get(), u2.get()) and np.array_equal(a1.get(), a2.get())
            u2.upload(u0)
            R.check(L.te_residual(g.h, dtype, 0, neumann, None, p[2], p[1], p[5], 2, None))
            assert np.array_equal(u1.get(), u2.get())
            want = f0.astype(np.float64)[off:].reshape(shape) - a1.get().astype(np.float64)[off:].reshape(shape)
            got = r1.get()[off:].reshape(shape)
            eps = np.finfo(t).eps * (np.abs(a1.get()).max() + np.abs(f0).max())
            assert np.abs(mesh.interior(got, dim) - mesh.interior(want, dim)).max() <= 2 * eps
            mesh.interior(got, dim)[...] = 0
            assert not got.any()  # ghost cells of the output are zero


@pytest.mark.parametrize("name,ns", [("2d_uniform_2x2_refined_nw_mpi1.json", (8, 8)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (16, 16)),
                                     ("3d_refined_bnw_2x2x2_mpi1.json", (4, 4, 4))])
def test_varpoisson_apply(name, ns):
    _print_case("varpoisson", name, ns)
    dim, levels = load(name, ns)
    lv = levels[0]
    kind = R.TRILINEAR if dim == 3 else R.BILINEAR
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, kind, R.FACES)
    X = mesh.cell_centers(lv, dim, ns)
    beta = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]))[:, None]
    O.fill_ghost(od, beta, kind=kind)
    for dtype, tol in [(R.F64, TOL64), (R.F32, 5e-6)]:
        u0 = random_field(od.shape(1), 8, R.np_dtype(dtype))
        b = beta.astype(R.np_dtype(dtype))
        ref = O.varpoisson_apply(od, b.astype(np.float64), u0.astype(np.float64), kind=kind)
        du = R.DeviceArray.from_host(u0)
        dc = R.DeviceArray.from_host(b)
        df = dd.vector(1, dtype)
        g.varstar_apply(dc, du, df)
        assert relerr(df.get(), ref) <= tol


@pytest.mark.parametrize("name,ns", [("2d_uniform_2x2_refined_nw_mpi1.json", (8, 8)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (16, 16)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (6, 10)),
                                     ("3d_mid_refine_4x4x4_mpi1.json", (4, 4, 4)),
                                     ("3d_refined_bnw_2x2x2_mpi1.json", (6, 4, 4))])
def test_restrict_interpolate(name, ns):
    _print_case("transfer", name, ns)
    dim, levels = load(name, ns)
    of, oc = O.Domain(dim, ns, levels[0]), O.Domain(dim, ns, levels[1])
    of.link_parents(oc)
    df, dc = _dev(dim, ns, levels[0]), _dev(dim, ns, levels[1])
    link = R.LevelLink(df, dc)
    assert np.array_equal(link.parents(), [of.parent_local(p) for p in range(of.np)])
    for dtype, tol in [(R.F64, TOL64), (R.F32, TOL32)]:
        for ncomp in (1, 2):
            fv = random_field(of.shape(ncomp), 21, R.np_dtype(dtype))
            cref = O.restrict(of, oc, fv.astype(np.float64))
            dfv = R.DeviceArray.from_host(fv)
            dcv = R.DeviceArray.from_host(random_field(oc.shape(ncomp), 1, R.np_dtype(dtype)))
            link.restrict(dfv, dcv)
            assert relerr(dcv.get(), cref) <= tol
            cv = random_field(oc.shape(ncomp), 22, R.np_dtype(dtype))
            fref = fv.astype(np.float64).copy()
            O.interpolate(oc, of, cv.astype(np.float64), fref)
            dcv.upload(cv)
            link.interpolate(dcv, dfv)
            assert relerr(dfv.get(), fref) <= tol


@pytest.mark.parametrize("ns", [(2, 2), (4, 10), (16, 16), (5, 7), (2, 4, 6), (16, 16, 16), (6, 3, 5)])
@pytest.mark.parametrize("ncomp", [1, 3])
def test_transfer_shapes(ns, ncomp):
    """Restriction and interpolation between the two finest levels of a mesh with copied and
    with refined children: FP64 has the oracle's bits (dividing by 2^D is exact and the sums run in
    its order), FP32 stays within the roundings of its at most 8 additions.  Odd sizes
    interpolate value by value (their restriction adds two children into a cell, in the oracle
    in no fixed order)."""
    dim = len(ns)
    name = "2d_uniform_8x8_refined_cross_mpi1.json" if dim == 2 else "3d_mid_refine_4x4x4_mpi1.json"
    lv = load(name, ns)[1][:2]
    of, oc = (O.Domain(dim, ns, v) for v in lv)
    of.link_parents(oc)
    link = R.LevelLink(*(R.Domain(dim, ns, v) for v in lv))
    f0, c0 = random_field(of.shape(ncomp), 91), random_field(oc.shape(ncomp), 92)
    for t in (np.float64, np.float32):
        f, c = f0.astype(t).astype(np.float64), c0.astype(t).astype(np.float64)
        cref, fref = O.restrict(of, oc, f), f.copy()
        O.interpolate(oc, of, c, fref)
        df, dc, dr = (R.DeviceArray.from_host(v.astype(t)) for v in (f, c, c))
        link.restrict(df, dr)
        link.interpolate(dc, df)
        even = all(v % 2 == 0 for v in ns)
        if t == np.float64:
            assert np.array_equal(df.get(), fref) and (not even or np.array_equal(dr.get(), cref))
        assert relerr(df.get(), fref) <= 2.0**-24 and (not even or relerr(dr.get(), cref) <= 8 * 2.0**-24)


@pytest.mark.parametrize("name,ns", [("2d_uniform_2x2_mpi1.json", (8, 8)),
                                     ("2d_uniform_2x2_refined_nw_mpi1.json", (16, 16)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (32, 32)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (10, 6)),
                                     ("3d_uniform_2x2x2_mpi1.json", (8, 8, 8)),
                                     ("3d_refined_bnw_2x2x2_mpi1.json", (16, 16, 16))])
@pytest.mark.parametrize("neumann_mask", [0, 0b0101])
def test_dft_smooth(name, ns, neumann_mask):
    _print_case("dft", name, ns, neumann_mask)
    dim, levels = load(name, ns)
    lv = levels[0]
    kind = R.TRILINEAR if dim == 3 else R.BIQUADRATIC
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, kind, R.FACES)
    plan = R.DftPlan(g, neumann_mask=neumann_mask)
    for dtype, tol in [(R.F64, TOL64), (R.F32, 2e-5)]:
        f0 = random_field(od.shape(1), 31, R.np_dtype(dtype))
        u0 = random_field(od.shape(1), 32, R.np_dtype(dtype))
        uref = u0.astype(np.float64)
        O.dft_smooth(od, f0.astype(np.float64), uref, kind=kind, neumann_mask=neumann_mask)
        du = R.DeviceArray.from_host(u0)
        plan.smooth(R.DeviceArray.from_host(f0), du)
        got = du.get()
        assert relerr(mesh.interior(got, dim), mesh.interior(uref, dim)) <= tol, dtype


@pytest.mark.parametrize("name", ["3d_refined_bnw_2x2x2_mpi1.json", "3d_mid_refine_4x4x4_mpi1.json"])
@pytest.mark.parametrize("op_kind", [0, 1])
@pytest.mark.parametrize("neumann_mask", [0, 0b100101])
def test_dft3_mfma_matches_generic(name, op_kind, neumann_mask, monkeypatch):
    """The 3D matrix-core patch solve (16^3 cells) against the generic kernel and the oracle:
    Dirichlet and mixed Neumann transform types, Poisson and VarPoisson interface terms, the
    smoothing sweep and the zero-u apply."""
    _print_case("dft3-mfma", name, op_kind, neumann_mask)
    ns = (16, 16, 16)
    dim, levels = load(name, ns)
    lv = levels[0]
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, R.TRILINEAR, R.FACES)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(lv, dim, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]) + 0.5 * X[..., 2])[:, None].copy()
        O.fill_ghost(od, coeffs, kind=R.TRILINEAR)
    dc = R.DeviceArray.from_host(coeffs) if coeffs is not None else None
    plan_mfma = R.DftPlan(g, neumann_mask=neumann_mask, op_kind=op_kind, coeffs=dc)
    monkeypatch.setenv("TE_DFT_VALU", "1")
    plan_valu = R.DftPlan(g, neumann_mask=neumann_mask, op_kind=op_kind, coeffs=dc)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        f0 = random_field(od.shape(1), 71, R.np_dtype(dtype))
        u0 = random_field(od.shape(1), 72, R.np_dtype(dtype))
        uref = u0.astype(np.float64)
        O.dft_smooth(od, f0.astype(np.float64), uref, kind=R.TRILINEAR, neumann_mask=neumann_mask, op_kind=op_kind,
                     coeffs=coeffs)
        outs = []
        for plan in (plan_mfma, plan_valu):
            du = R.DeviceArray.from_host(u0)
            plan.smooth(R.DeviceArray.from_host(f0), du)
            outs.append(mesh.interior(du.get(), dim))
        assert relerr(outs[0], mesh.interior(uref, dim)) <= tol, dtype
        assert relerr(outs[0], outs[1]) <= tol, dtype
        du = R.DeviceArray.from_host(u0)
        plan_mfma.apply(R.DeviceArray.from_host(f0), du)
        uz = np.zeros_like(uref)
        O.dft_smooth(od, f0.astype(np.float64), uz, kind=R.TRILINEAR, neumann_mask=neumann_mask, op_kind=op_kind,
                     coeffs=coeffs)
        assert relerr(mesh.interior(du.get(), dim), mesh.interior(uz, dim)) <= tol, dtype


@pytest.mark.parametrize("name", ["3d_uniform_2x2x2_mpi1.json", "3d_refined_bnw_2x2x2_mpi1.json"])
@pytest.mark.parametrize("n", [8, 16])
@pytest.mark.parametrize("op_kind", [0, 1])
@pytest.mark.parametrize("neumann_mask", [0, 0b100101, 0b111111])
def test_dft3_tiles(name, n, op_kind, neumann_mask):
    """The 3D matrix-core patch solves (8^3: a patch per wave, 8 and 15 patches on workgroups of
    four; 16^3) against the oracle: transform types per patch, interface terms, and apply's
    zeroed ghosts, also on vectors off the wide stores' grid."""
    ns = (n,) * 3
    dim, levels = load(name, ns)
    lv = levels[0]
    od, dd = O.Domain(dim, ns, lv), _dev(dim, ns, lv)
    g = R.GhostFiller(dd, R.TRILINEAR, R.FACES)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(lv, dim, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]) + 0.5 * X[..., 2])[:, None].copy()
        O.fill_ghost(od, coeffs, kind=R.TRILINEAR)
    dc = R.DeviceArray.from_host(coeffs) if coeffs is not None else None
    plan = R.DftPlan(g, neumann_mask=neumann_mask, op_kind=op_kind, coeffs=dc)
    args = dict(kind=R.TRILINEAR, neumann_mask=neumann_mask, op_kind=op_kind, coeffs=coeffs)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        t = R.np_dtype(dtype)
        f0, u0 = random_field(od.shape(1), 73, t), random_field(od.shape(1), 74, t)
        uref, uz = u0.astype(np.float64), np.zeros(od.shape(1))
        O.dft_smooth(od, f0.astype(np.float64), uref, **args)
        O.dft_smooth(od, f0.astype(np.float64), uz, **args)
        df, du = R.DeviceArray.from_host(f0), R.DeviceArray.from_host(u0)
        plan.smooth(df, du)
        assert relerr(mesh.interior(du.get(), dim), mesh.interior(uref, dim)) <= tol, dtype
        for off in (0, 1):
            big = R.DeviceArray.from_host(np.full(u0.size + off, 7, t))
            R.check(R.lib().te_dft_apply(plan.h, dtype, df.ptr, big.ptr + off * t().itemsize, None))
            got = big.get()[off:].reshape(u0.shape)
            assert relerr(mesh.interior(got, dim), mesh.interior(uz, dim)) <= tol, dtype
            mesh.interior(got, dim)[...] = 0
            assert not got.any()


@pytest.mark.parametrize("ns", [(16, 16), (32, 32)])
@pytest.mark.parametrize("op_kind", [0, 1])
def test_dft_mfma_matches_generic(ns, op_kind, monkeypatch):
    """The matrix-core patch solve (2D, n = 16/32, Dirichlet) against the generic kernel
    and against the oracle."""
    _print_case("dft-mfma", ns, op_kind)
    dim, levels = load("2d_uniform_8x8_refined_cross_mpi1.json", ns)
    lv = levels[0]
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    g = R.GhostFiller(dd, R.BIQUADRATIC, R.FACES)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(lv, dim, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]))[:, None].copy()
        O.fill_ghost(od, coeffs, kind=R.BIQUADRATIC)
    dc = R.DeviceArray.from_host(coeffs) if coeffs is not None else None
    plan_mfma = R.DftPlan(g, op_kind=op_kind, coeffs=dc)
    monkeypatch.setenv("TE_DFT_VALU", "1")
    plan_valu = R.DftPlan(g, op_kind=op_kind, coeffs=dc)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        f0 = random_field(od.shape(1), 51, R.np_dtype(dtype))
        u0 = random_field(od.shape(1), 52, R.np_dtype(dtype))
        uref = u0.astype(np.float64)
        O.dft_smooth(od, f0.astype(np.float64), uref, kind=R.BIQUADRATIC, op_kind=op_kind, coeffs=coeffs)
        outs = []
        for plan in (plan_mfma, plan_valu):
            du = R.DeviceArray.from_host(u0)
            plan.smooth(R.DeviceArray.from_host(f0), du)
            outs.append(mesh.interior(du.get(), dim))
        assert relerr(outs[0], mesh.interior(uref, dim)) <= tol, dtype
        assert relerr(outs[0], outs[1]) <= tol, dtype
        # apply (u := 0 first): the zero-u variant of the kernel
        du = R.DeviceArray.from_host(u0)
        plan_mfma.apply(R.DeviceArray.from_host(f0), du)
        uz = np.zeros_like(uref)
        O.dft_smooth(od, f0.astype(np.float64), uz, kind=R.BIQUADRATIC, op_kind=op_kind, coeffs=coeffs)
        assert relerr(mesh.interior(du.get(), dim), mesh.interior(uz, dim)) <= tol


@pytest.mark.parametrize("name,ns", [("2d_uniform_8x8_refined_cross_mpi1.json", (16, 16)),
                                     ("2d_uniform_2x2_refined_nw_mpi1.json", (32, 32)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (8, 8)),
                                     ("2d_uniform_2x2_refined_nw_mpi1.json", (10, 6))])
@pytest.mark.parametrize("kind", [R.BILINEAR, R.BIQUADRATIC])
@pytest.mark.parametrize("op_kind", [0, 1])
def test_fused_vcycle_launches(name, ns, kind, op_kind):
    """te_dft_apply_mixed, te_dft_smooth_interp and te_residual_restrict against the oracle's
    unfused sequences (PatchSolver::apply; interpolate then smooth; residual then restrict),
    FP64 and FP32 arithmetic, including the mixed-precision input / output types; 16 x 16 and
    32 x 32 on the matrix cores, 8 x 8 and 10 x 6 in the generic patch-solve kernel."""
    _print_case("fused", name, ns, kind, op_kind)
    dim, levels = load(name, ns)
    fl, cl = levels[0], levels[1]
    fo, co = O.Domain(dim, ns, fl), O.Domain(dim, ns, cl)
    fo.link_parents(co)
    fd, cd = _dev(dim, ns, fl), _dev(dim, ns, cl)
    link = R.LevelLink(fd, cd)
    g = R.GhostFiller(fd, kind, R.FACES)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(fl, dim, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]))[:, None].copy()
        O.fill_ghost(fo, coeffs, kind=kind)
    f0 = random_field(fo.shape(1), 61)
    u0 = random_field(fo.shape(1), 62)
    uc0 = random_field(co.shape(1), 63)
    # oracle references, FP64
    ua = np.zeros_like(f0)
    O.dft_smooth(fo, f0.copy(), ua, kind=kind, op_kind=op_kind, coeffs=coeffs)
    ui = u0.copy()
    O.interpolate(co, fo, uc0, ui)
    O.dft_smooth(fo, f0.copy(), ui, kind=kind, op_kind=op_kind, coeffs=coeffs)
    if op_kind == 0:
        r = f0 - O.poisson_apply(fo, u0.copy(), kind=kind)
    else:
        r = f0 - O.varpoisson_apply(fo, coeffs, u0.copy(), kind=kind)
    fcr = O.restrict(fo, co, r)
    for dt, tol in [(R.F64, TOL64), (R.F32, 2e-5)]:
        npd = R.np_dtype(dt)
        dc = R.DeviceArray.from_host(coeffs, npd) if coeffs is not None else None
        dc64 = R.DeviceArray.from_host(coeffs) if coeffs is not None else None
        plan = R.DftPlan(g, op_kind=op_kind, coeffs=dc64)
        for tf, to in [(dt, dt), (R.F64, dt), (R.F64, R.F64)]:
            f = R.DeviceArray.from_host(f0, R.np_dtype(tf))
            out = R.DeviceArray(fo.shape(1), R.np_dtype(to))
            plan.apply_mixed(dt, f, out)
            assert relerr(mesh.interior(out.get(), dim), mesh.interior(ua, dim)) <= tol, (dt, tf, to)
            u = R.DeviceArray.from_host(u0, npd)
            for tc in ([R.F64, R.F32] if dt == R.F32 else [R.F64]):
                uc = R.DeviceArray.from_host(uc0, R.np_dtype(tc))
                out = R.DeviceArray(fo.shape(1), R.np_dtype(to))
                plan.smooth_interp(link, f, u, uc, out)
                assert relerr(mesh.interior(out.get(), dim), mesh.interior(ui, dim)) <= tol, (dt, tf, to, tc)
                fc = R.DeviceArray(co.shape(1), R.np_dtype(tc))
                fc.upload(np.zeros(co.shape(1)))
                link.residual_restrict(g, f, u, fc, op_kind=op_kind, coeffs=dc)
                assert relerr(mesh.interior(fc.get(), dim), mesh.interior(fcr, dim)) <= tol, (dt, tf, tc)
            # u and uc are inputs only
            assert np.array_equal(u.get(), u0.astype(npd))


@pytest.mark.parametrize("ns,base", [((5, 4), 1), ((16, 16), 0), ((16, 3), 3), ((2, 2), 0), ((6, 4, 8), 1), ((7, 5, 3), 1),
                                     ((16, 16, 16), 2)])
@pytest.mark.parametrize("dtype", [R.F64, R.F32])
@pytest.mark.parametrize("off", [0, 1])
def test_vector_kernels_shapes(ns, base, dtype, off):
    """Rows of odd and even length, one patch to several workgroups, and vectors that start one
    value off the paired accesses' grid: every update and reduction against numpy, the ghost
    cells untouched.  Sums of n terms agree to n ulp of the sum of magnitudes."""
    dim, t = len(ns), R.np_dtype(dtype)
    lv = solver.uniform_levels(dim, base, ns)[0]
    dd, L = R.Domain(dim, ns, lv), R.lib()
    shape = mesh.padded_shape(len(lv), dim, ns, 2)
    n = int(np.prod(shape))
    h = [random_field((n + off,), 61 + k, t) for k in range(3)]
    dev = [R.DeviceArray.from_host(v) for v in h]
    x, a, b = (d.ptr + off * t().itemsize for d in dev)
    xv, av, bv = (v[off:].reshape(shape).copy() for v in h)

    def check(op, want, *args):
        R.check(getattr(L, op)(dd.h, dtype, x, *args, 2, None))
        got = dev[0].get()
        if off:
            assert got[0] == h[0][0]
        got = got[off:].reshape(shape)
        if op == "te_vec_set_with_ghost":
            xv[...] = want
        else:
            mesh.interior(xv, dim)[...] = mesh.interior(np.broadcast_to(want, shape), dim)
        assert np.allclose(got, xv, rtol=4 * np.finfo(t).eps, atol=8 * np.finfo(t).eps), op
        xv[...] = got

    check("te_vec_add_scaled", xv + t(0.3) * av, 0.3, a)
    check("te_vec_add_scaled2", xv + (t(0.3) * av + t(-1.7) * bv), 0.3, a, -1.7, b)
    check("te_vec_scale_then_add", t(0.9) * xv + av, 0.9, a)
    check("te_vec_scale_then_add_scaled", t(0.9) * xv + t(0.2) * av, 0.9, 0.2, a)
    check("te_vec_scale_then_add_scaled2", t(0.9) * xv + t(0.2) * av + t(0.7) * bv, 0.9, 0.2, a, 0.7, b)
    check("te_vec_add", xv + av, a)
    check("te_vec_scale", xv * t(1.1), 1.1)
    check("te_vec_shift", xv + t(0.25), 0.25)
    X, A = mesh.interior(xv, dim).astype(np.float64), mesh.interior(av, dim).astype(np.float64)
    out = C.c_double()
    bound = X.size * np.finfo(np.float64).eps
    R.check(L.te_vec_dot(dd.h, dtype, x, a, 2, C.byref(out), None))
    assert abs(out.value - (X * A).sum()) <= bound * np.abs(X * A).sum()
    R.check(L.te_vec_two_norm(dd.h, dtype, x, 2, C.byref(out), None))
    assert abs(out.value - np.sqrt((X * X).sum())) <= bound * out.value
    R.check(L.te_vec_inf_norm(dd.h, dtype, x, 2, C.byref(out), None))
    assert out.value == max(0.0, X.max())  # Vector::infNorm takes the largest value, not magnitude
    vol = np.prod(lv["spacings"][:, :dim], axis=1).reshape((-1,) + (1,) * (dim + 1))
    R.check(L.te_vec_integrate(dd.h, dtype, x, 2, C.byref(out), None))
    assert abs(out.value - (X * vol).sum()) <= bound * np.abs(X * vol).sum()
    check("te_vec_copy", av, a)
    check("te_vec_set", t(-2.5), -2.5)
    check("te_vec_set_with_ghost", t(1.5), 1.5)


@pytest.mark.parametrize("dtype", [R.F64, R.F32])
def test_vector_algebra(dtype):
    _print_case("vector", dtype)
    dim, levels = load("2d_uniform_8x8_refined_cross_mpi1.json", (16, 16))
    lv = levels[0]
    od = O.Domain(dim, (16, 16), lv)
    dd = _dev(dim, (16, 16), lv)
    nt = R.np_dtype(dtype)
    tol = TOL64 if dtype == R.F64 else 1e-6
    a = random_field(od.shape(2), 1, nt)
    b = random_field(od.shape(2), 2, nt)
    da, db = R.DeviceArray.from_host(a), R.DeviceArray.from_host(b)
    ia, ib = mesh.interior(a, 2).astype(np.float64), mesh.interior(b, 2).astype(np.float64)
    assert abs(dd.dot(da, db) - (ia * ib).sum()) <= tol * np.abs(ia * ib).sum()
    assert abs(dd.two_norm(da) - np.sqrt((ia * ia).sum())) <= tol * np.sqrt((ia * ia).sum())
    assert dd.inf_norm(da) == pytest.approx(max(ia.max(), 0.0), rel=1e-15)
    neg = R.DeviceArray.from_host(-np.abs(a))
    assert dd.inf_norm(neg) == 0.0  # Vector::infNorm is max(0, max v)
    L = R.lib()
    x = da
    R.check(L.te_vec_add_scaled2(dd.h, dtype, x.ptr, 0.5, db.ptr, -2.0, db.ptr, 2, None))
    exp = a.astype(np.float64).copy()
    mesh.interior(exp, 2)[...] += ib * 0.5 + ib * -2.0
    assert relerr(x.get(), exp) <= tol
    R.check(L.te_vec_scale_then_add(dd.h, dtype, x.ptr, 3.0, db.ptr, 2, None))
    mesh.interior(exp, 2)[...] = mesh.interior(exp, 2) * 3.0 + ib
    assert relerr(x.get(), exp) <= tol
    R.check(L.te_vec_set_with_ghost(dd.h, dtype, x.ptr, 1.5, 2, None))
    assert np.all(x.get() == 1.5)
    R.check(L.te_vec_set(dd.h, dtype, x.ptr, 0.0, 2, None))
    got = x.get()
    assert np.all(mesh.interior(got, 2) == 0.0) and got.max() == 1.5


@pytest.mark.parametrize("name,dim,ns", [("2d_uniform_2x2_refined_nw_mpi1.json", 2, (10, 6)),
                                         ("2d_uniform_8x8_refined_cross_mpi1.json", 2, (16, 16)),
                                         ("3d_refined_bnw_2x2x2_mpi1.json", 3, (4, 6, 8))])
def test_boundary_data_rhs(name, dim, ns):
    """te_star_add_dirichlet_bc (Poisson and VarPoisson forms) and te_star_add_neumann_bc
    against the oracle on the same sampled boundary data (FP64 <= 1e-14, FP32 storage
    <= 1e-6), and the reference's linear-exactness identity on the device operator: for a
    linear g, A g (physical ghosts -g_b, or +g_b with Neumann) equals the boundary terms."""
    from thunderegg_amd import domain_tools as DT

    _print_case("boundary data", name, ns)
    _, levels = load(name, ns)
    lv = levels[0]
    od = O.Domain(dim, ns, lv)
    dd = _dev(dim, ns, lv)
    pts = DT.boundary_points(lv, dim, ns)
    assert len(pts) == dd.boundary_length()
    rng = np.random.default_rng(3)
    g = rng.standard_normal(len(pts))
    cval = rng.uniform(0.5, 2.0, len(pts))
    dg, dc = R.DeviceArray.from_host(g), R.DeviceArray.from_host(cval)
    for dtype, tol in [(R.F64, 1e-14), (R.F32, 1e-6)]:
        f0 = random_field(od.shape(1), 21, R.np_dtype(dtype))
        for form in ("dirichlet", "varpoisson", "neumann"):
            ref = f0.astype(np.float64)
            df = R.DeviceArray.from_host(f0)
            if form == "dirichlet":
                O.add_bc(od, ref, g)
                dd.add_dirichlet_bc(df, dg)
            elif form == "varpoisson":
                O.add_bc(od, ref, g, c=cval)
                dd.add_dirichlet_bc(df, dg, dc)
            else:
                O.add_bc(od, ref, g, neumann=True)
                dd.add_neumann_bc(df, dg)
            assert relerr(df.get(), ref) <= tol, (dtype, form)
    # linear exactness through the device operator
    kind = R.TRILINEAR if dim == 3 else R.BILINEAR
    coef = [5.0, 13.0, 7.0][:dim]
    Xg = mesh.cell_centers(lv, dim, ns, with_ghost=True)
    gv = (1 + sum(coef[a] * Xg[..., a] for a in range(dim)))[:, None].copy()
    filler = R.GhostFiller(dd, kind, R.FACES)
    for neumann in (False, True):
        du = R.DeviceArray.from_host(gv)
        df = R.DeviceArray(dd.shape(1), np.float64)
        filler.star_apply(du, df, neumann=neumann)
        fe = R.DeviceArray.from_host(np.zeros_like(gv))
        if neumann:
            DT.add_neumann_bc(dd, fe, [(lambda c, k=k: np.full_like(c[0], coef[k])) for k in range(dim)])
        else:
            DT.add_dirichlet_bc(dd, fe, lambda c: 1 + sum(coef[a] * c[a] for a in range(dim)))
        a, b = mesh.interior(df.get(), dim), mesh.interior(fe.get(), dim)
        assert np.abs(a - b).max() <= 1e-9 * np.abs(b).max(), neumann


@pytest.mark.parametrize("name,ns", [("2d_uniform_4x4_mpi1.json", (10, 2)), ("2d_uniform_2x2_refined_nw_mpi1.json", (4, 4)),
                                     ("2d_uniform_8x8_refined_cross_mpi1.json", (8, 8)),
                                     ("3d_refined_bnw_2x2x2_mpi1.json", (4, 4, 4)),
                                     ("3d_mid_refine_4x4x4_mpi1.json", (2, 4, 6))])
@pytest.mark.parametrize("ncomp", [1, 2])
def test_restrict_extrapolate(name, ns, ncomp):
    """LinearRestrictor with extrapolate_boundary_ghosts (te_restrict_extrapolate) against the
    oracle, every cell of the coarse vector including its ghosts, FP64 bit-exact (the same
    terms summed in the same order) and FP32 to rounding; without the flag the ghosts stay 0."""
    print("case: restrict_extrapolate", name, ns, ncomp, flush=True)
    dim, levels = load(name, ns)
    of, oc = O.Domain(dim, ns, levels[0]), O.Domain(dim, ns, levels[1])
    of.link_parents(oc)
    df, dc = R.Domain(dim, ns, levels[0]), R.Domain(dim, ns, levels[1])
    link = R.LevelLink(df, dc)
    fv = random_field(of.shape(ncomp), 17)
    ref = O.restrict(of, oc, fv, extrapolate=True)
    assert np.any(ref[..., 0, 1:-1]) if dim == 2 else np.any(ref[..., 0, 1:-1, 1:-1])
    dfv = R.DeviceArray.from_host(fv)
    dcv = R.DeviceArray(oc.shape(ncomp), np.float64)
    link.restrict_extrapolate(dfv, dcv)
    assert np.array_equal(dcv.get(), ref)
    d32 = R.DeviceArray.from_host(fv.astype(np.float32))
    c32 = R.DeviceArray(oc.shape(ncomp), np.float32)
    link.restrict_extrapolate(d32, c32)
    assert np.max(np.abs(c32.get() - ref)) <= 1e-5 * np.max(np.abs(ref))
    link.restrict(dfv, dcv)
    assert np.array_equal(dcv.get(), O.restrict(of, oc, fv))


@pytest.mark.parametrize("level", [0, 1, 2])
@pytest.mark.parametrize("op_kind", [0, 1])
@pytest.mark.parametrize("kind", [R.BILINEAR, R.BIQUADRATIC])
def test_dft32_pair(level, op_kind, kind):
    """The 32^2 patch solve on 1, 4 and 7 patches (fewer than the launch's eight groups and one
    more; refined at the largest): ghosts read from u in place, and the zero-u apply."""
    ns = (32, 32)
    lv = solver.uniform_levels(2, level, ns)[0] if level < 2 else load("2d_uniform_2x2_refined_nw_mpi1.json", ns)[1][0]
    od, dd = O.Domain(2, ns, lv), _dev(2, ns, lv)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(lv, 2, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]))[:, None].copy()
        O.fill_ghost(od, coeffs, kind=kind)
    plan = R.DftPlan(R.GhostFiller(dd, kind, R.FACES), op_kind=op_kind,
                     coeffs=R.DeviceArray.from_host(coeffs) if op_kind else None)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        t = R.np_dtype(dtype)
        f0, u0 = random_field(od.shape(1), 33, t), random_field(od.shape(1), 34, t)
        for zero in (False, True):
            uref = np.zeros(od.shape(1)) if zero else u0.astype(np.float64)
            O.dft_smooth(od, f0.astype(np.float64), uref, kind=kind, op_kind=op_kind, coeffs=coeffs)
            du = R.DeviceArray.from_host(u0)
            (plan.apply if zero else plan.smooth)(R.DeviceArray.from_host(f0), du)
            assert relerr(mesh.interior(du.get(), 2), mesh.interior(uref, 2)) <= tol, (dtype, zero)


@pytest.mark.parametrize("op_kind", [0, 1])
@pytest.mark.parametrize("kind", [R.BILINEAR, R.BIQUADRATIC])
def test_dft32_levels_past_the_card(op_kind, kind):
    """The 32^2 patch solve on a refined level of more patches than the card holds workgroups for
    (each then walks several in FP64): from zero, in place on filled ghosts, and on u plus the coarser
    level's correction, against the oracle."""
    _print_case("dft32-loop", op_kind, kind)
    ns = (32, 32)
    forest = solver.Forest(2, 6)
    forest.refine((np.arange(4096) % 41 == 0).astype(np.uint8))
    forest.balance()
    lv = forest.build_domains(ns)[:2]
    assert len(lv[0]) > 4096 and all((lv[0]["nbr_type"][:, 4:] == k).any() for k in (-1, 0, 1, 2))
    (od, oc), (dd, dc) = ([cls(2, ns, v) for v in lv] for cls in (O.Domain, R.Domain))
    od.link_parents(oc)
    link, g = R.LevelLink(dd, dc), R.GhostFiller(dd, kind, R.FACES)
    coeffs = np.exp(0.3 * random_field(od.shape(1), 38)) if op_kind else None
    if op_kind:
        O.fill_ghost(od, coeffs, kind=kind)
    plan = R.DftPlan(g, op_kind=op_kind, coeffs=R.DeviceArray.from_host(coeffs) if op_kind else None)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        t = R.np_dtype(dtype)
        f0, u0 = random_field(od.shape(1), 33, t), random_field(od.shape(1), 34, t)
        c0 = random_field(oc.shape(1), 35, t)
        df, dout = R.DeviceArray.from_host(f0), R.DeviceArray.from_host(np.zeros_like(u0))
        for mode in ("apply", "smooth", "interp"):
            uref = np.zeros(od.shape(1)) if mode == "apply" else u0.astype(np.float64)
            if mode == "interp":
                O.interpolate(oc, od, c0.astype(np.float64), uref)
            O.dft_smooth(od, f0.astype(np.float64), uref, kind=kind, op_kind=op_kind, coeffs=coeffs)
            du = R.DeviceArray.from_host(u0)
            if mode == "interp":
                plan.smooth_interp(link, df, du, R.DeviceArray.from_host(c0), dout)
            else:
                getattr(plan, mode)(df, du)
            got = (dout if mode == "interp" else du).get()
            assert relerr(mesh.interior(got, 2), mesh.interior(uref, 2)) <= tol, (dtype, mode)


@pytest.mark.parametrize("ns", [(4, 8), (8, 8), (10, 6), (20, 24), (32, 32), (40, 12)])
@pytest.mark.parametrize("kind", [R.BILINEAR, R.BIQUADRATIC])
@pytest.mark.parametrize("neumann", [False, True])
def test_residual_restrict_sizes(ns, kind, neumann):
    """Residual and restriction in one launch over the even sizes (a workgroup of 64 to 256
    threads a patch) against the oracle's operator and restriction."""
    lv = load("2d_uniform_8x8_refined_cross_mpi1.json", ns)[1][:2]
    of, oc = (O.Domain(2, ns, v) for v in lv)
    of.link_parents(oc)
    df, dc = (R.Domain(2, ns, v) for v in lv)
    link, g = R.LevelLink(df, dc), R.GhostFiller(df, kind, R.FACES)
    for dtype, tol in [(R.F64, TOL64), (R.F32, TOL32)]:
        t = R.np_dtype(dtype)
        f0, u0 = random_field(of.shape(1), 51, t), random_field(of.shape(1), 52, t)
        au = O.poisson_apply(of, u0.astype(np.float64), kind=kind, neumann=neumann)
        want = O.restrict(of, oc, f0.astype(np.float64) - au)
        fc = R.DeviceArray.from_host(np.zeros(oc.shape(1), t))
        link.residual_restrict(g, R.DeviceArray.from_host(f0), R.DeviceArray.from_host(u0), fc, neumann=neumann)
        assert relerr(mesh.interior(fc.get(), 2), mesh.interior(want, 2)) <= tol, dtype


@pytest.mark.parametrize("ns", [(7, 7), (5, 9), (8, 8), (10, 12), (24, 24), (40, 6), (50, 50), (6, 6, 6), (4, 6, 8), (12, 12, 12),
                                (16, 14, 18)])
@pytest.mark.parametrize("neumann_mask", [0, 0b0110])
@pytest.mark.parametrize("op_kind", [0, 1])
def test_dft_generic_sizes(ns, neumann_mask, op_kind):
    """The generic patch solve over odd, even, mixed and large sizes (padded and unpadded LDS, one
    matrix for all axes or one per axis and patch, several patches a workgroup): sweep and
    apply with its zeroed ghosts, in place and on vectors one value off, against the oracle."""
    dim = len(ns)
    odd = any(v % 2 for v in ns)
    name = ("2d_uniform_4x4_mpi1.json" if odd else "2d_uniform_2x2_refined_nw_mpi1.json") if dim == 2 else (
        "3d_refined_bnw_2x2x2_mpi1.json")
    lv = load(name, ns)[1][0]
    kind = R.TRILINEAR if dim == 3 else R.BIQUADRATIC
    od, dd = O.Domain(dim, ns, lv), _dev(dim, ns, lv)
    coeffs = None
    if op_kind == 1:
        X = mesh.cell_centers(lv, dim, ns)
        coeffs = np.exp(np.sin(3 * X[..., 0]) * np.cos(2 * X[..., 1]))[:, None].copy()
        O.fill_ghost(od, coeffs, kind=kind)
    plan = R.DftPlan(R.GhostFiller(dd, kind, R.FACES), neumann_mask=neumann_mask, op_kind=op_kind,
                     coeffs=R.DeviceArray.from_host(coeffs) if op_kind else None)
    args = dict(kind=kind, neumann_mask=neumann_mask, op_kind=op_kind, coeffs=coeffs)
    for dtype, tol in [(R.F64, 1e-12), (R.F32, 2e-5)]:
        t = R.np_dtype(dtype)
        f0, u0 = random_field(od.shape(1), 35, t), random_field(od.shape(1), 36, t)
        uref, uz = u0.astype(np.float64), np.zeros(od.shape(1))
        O.dft_smooth(od, f0.astype(np.float64), uref, **args)
        O.dft_smooth(od, f0.astype(np.float64), uz, **args)
        df, du = R.DeviceArray.from_host(f0), R.DeviceArray.from_host(u0)
        plan.smooth(df, du)
        assert relerr(mesh.interior(du.get(), dim), mesh.interior(uref, dim)) <= tol, dtype
        big = R.DeviceArray.from_host(np.full(u0.size + 1, 7, t))
        R.check(R.lib().te_dft_apply(plan.h, dtype, df.ptr, big.ptr + t().itemsize, None))
        got = big.get()[1:].reshape(u0.shape)
        assert relerr(mesh.interior(got, dim), mesh.interior(uz, dim)) <= tol, dtype
        mesh.interior(got, dim)[...] = 0
        assert not got.any()


@pytest.mark.parametrize("n", [8, 16])
@pytest.mark.parametrize("off", [0, 1])
def test_star3_tile(n, off):
    """The LDS operator of large 3D levels (more patches than CUs, 8^3 and 16^3; refined, so that
    every face type occurs) against the ghost fill followed by the operator: the bits of u, and
    the result but for contracted products (a few roundings of its largest term)."""
    ns = (n,) * 3
    forest = solver.Forest(3, 2)
    forest.refine((np.arange(64) % 3 != 0).astype(np.uint8))
    forest.balance()
    lv = forest.build_domains(ns)[0]
    assert len(lv) > 256 and len(lv) % 8 != 0 and all((lv["nbr_type"][:, 20:] == k).any() for k in (-1, 0, 1, 2))
    dd, L = R.Domain(3, ns, lv), R.lib()
    g = R.GhostFiller(dd, R.TRILINEAR, R.FACES)
    shape = mesh.padded_shape(len(lv), 3, ns, 2)
    size = int(np.prod(shape))
    ih2 = 1.0 / lv["spacings"].min() ** 2
    for dtype in (R.F64, R.F32):
        t = R.np_dtype(dtype)
        u0, f0 = random_field((size + off,), 83, t), random_field((size + off,), 84, t)
        cf = R.DeviceArray.from_host(np.exp(random_field(mesh.padded_shape(len(lv), 3, ns), 85, t)).astype(t))
        beta = float(np.abs(cf.get()).max())
        for op, neumann in ((0, 0), (0, 1), (1, 0)):
            u1, u2, f = (R.DeviceArray.from_host(v) for v in (u0, u0, f0))
            a1, a2, r1 = (R.DeviceArray.from_host(np.full(size + off, 7, t)) for _ in range(3))
            p = [d.ptr + off * t().itemsize for d in (u1, u2, f, a1, a2, r1)]
            R.check(L.te_ghost_fill(g.h, dtype, p[0], 2, None))
            if op == 0:
                R.check(L.te_star_apply_patches(g.h, dtype, neumann, p[0], p[3], 2, None))
                R.check(L.te_star_apply(g.h, dtype, neumann, p[1], p[4], 2, None))
            else:
                R.check(L.te_varstar_apply(g.h, dtype, cf.ptr, p[1], p[4], 2, None))
            assert np.array_equal(u1.get(), u2.get())
            tol = 8 * np.finfo(t).eps * 12 * ih2 * float(np.abs(u0).max()) * (beta if op else 1.0)
            got = a2.get()[off:].reshape(shape)
            if op == 0:
                assert np.abs(got - a1.get()[off:].reshape(shape)).max() <= tol
            else:
                U = u1.get()[off:].reshape(shape).astype(np.float64)
                B = cf.get().astype(np.float64)[:, :1]
                M, C0 = mesh.interior(U, 3), mesh.interior(B, 3)
                want = np.zeros(M.shape)
                for a in range(3):
                    h2 = (1.0 / lv["spacings"][:, a] ** 2).reshape(-1, 1, 1, 1, 1)
                    ax = 4 - a
                    sl = [slice(None), slice(None)] + [slice(1, -1)] * 3
                    sl_l, sl_u = list(sl), list(sl)
                    sl_l[ax], sl_u[ax] = slice(0, -2), slice(2, None)
                    UL, UU = U[tuple(sl_l)].copy(), U[tuple(sl_u)].copy()
                    first, last = [slice(None)] * 5, [slice(None)] * 5
                    first[ax], last[ax] = 0, -1
                    pl, pu = lv["nbr_type"][:, 20 + 2 * a] < 0, lv["nbr_type"][:, 21 + 2 * a] < 0
                    UL[tuple(first)][pl] = -M[tuple(first)][pl]
                    UU[tuple(last)][pu] = -M[tuple(last)][pu]
                    CL, CU = B[tuple(sl_l)], B[tuple(sl_u)]
                    want += ((CU + C0) * (UU - M) - (CL + C0) * (M - UL)) * (0.5 * h2)
                assert np.abs(mesh.interior(got, 3) - want).max() <= tol
            u2.upload(u0)
            R.check(L.te_residual(g.h, dtype, op, neumann, cf.ptr if op else None, p[2], p[1], p[5], 2, None))
            assert np.array_equal(u1.get(), u2.get())
            want = f0.astype(np.float64)[off:].reshape(shape) - got.astype(np.float64)
            r = r1.get()[off:].reshape(shape)
            assert np.abs(mesh.interior(r, 3) - mesh.interior(want, 3)).max() <= tol + np.finfo(t).eps * float(np.abs(f0).max())
            for v in (r, got):
                mesh.interior(v, 3)[...] = 0
                assert not v.any()  # ghost cells of the output are zero


@pytest.mark.parametrize("ns", [(32, 32), (64, 64), (33, 70), (256, 128), (1024, 6), (6, 1024), (16, 16, 16), (32, 32, 32),
                                (40, 24, 6), (128, 2, 2), (4, 4, 128), (2, 64, 64), (64, 64, 2)])
def test_patches_of_many_cells(ns):
    """Few patches of many cells, each shared by several wavefronts or workgroups (runs of rows, of
    slices, of a patch's values, of its faces' cells; faces in a launch of their own): ghost fill,
    operators, residual, restriction and interpolation against the oracle."""
    _print_case("many-cells", ns)
    dim, odd = len(ns), any(v % 2 for v in ns)
    name = "3d_refined_bnw_2x2x2_mpi1.json" if dim == 3 else "2d_uniform_2x2_mpi1.json" if odd else "2d_uniform_2x2_refined_nw_mpi1.json"
    lv = load(name, ns)[1][:2]
    kind = R.TRILINEAR if dim == 3 else R.BILINEAR
    of, oc = (O.Domain(dim, ns, v) for v in lv)
    of.link_parents(oc)
    df, dc = (R.Domain(dim, ns, v) for v in lv)
    link, g = R.LevelLink(df, dc), R.GhostFiller(df, kind, R.FACES)
    beta = np.exp(0.3 * random_field(of.shape(1), 70))
    O.fill_ghost(of, beta, kind=kind)
    for dtype, t64, t32 in ((R.F64, TOL64, None), (R.F32, None, 5e-6)):
        t, tol = R.np_dtype(dtype), t64 or t32
        u0, f0, c0 = (random_field(o.shape(2), s, t).astype(np.float64) for o, s in ((of, 71), (of, 72), (oc, 73)))
        filled = u0.copy()
        O.fill_ghost(of, filled, kind=kind)
        du = R.DeviceArray.from_host(u0.astype(t))
        g.fill_ghost(du)
        assert relerr(du.get(), filled) <= tol
        b = beta.astype(t).astype(np.float64)
        for op, neumann in ((0, False), (0, True), (1, False)):
            dcf = R.DeviceArray.from_host(b.astype(t)) if op else None
            du.upload(u0)
            dr, da = (R.DeviceArray.from_host(np.full(u0.shape, 7, t)) for _ in range(2))
            g.residual(R.DeviceArray.from_host(f0.astype(t)), du, dr, op_kind=op, neumann=neumann, coeffs=dcf)
            assert relerr(du.get(), filled) <= tol
            du.upload(u0)
            g.varstar_apply(dcf, du, da) if op else g.star_apply(du, da, neumann=neumann)
            assert relerr(du.get(), filled) <= tol
            for c in range(2):
                one = np.ascontiguousarray(u0[:, c:c + 1])
                want = O.varpoisson_apply(of, b, one, kind=kind) if op else O.poisson_apply(of, one, kind=kind, neumann=neumann)
                assert relerr(da.get()[:, c:c + 1], want) <= tol
                r = np.zeros(want.shape)
                mesh.interior(r, dim)[...] = mesh.interior(f0[:, c:c + 1] - want, dim)
                assert relerr(dr.get()[:, c:c + 1], r) <= tol
        fref = f0.copy()
        O.interpolate(oc, of, c0, fref)
        dfv, dcv = R.DeviceArray.from_host(f0.astype(t)), R.DeviceArray.from_host(c0.astype(t))
        link.interpolate(dcv, dfv)
        assert relerr(dfv.get(), fref) <= (TOL64 if t64 else TOL32)
        if not odd:
            dfv.upload(f0)
            link.restrict(dfv, dcv)
            assert relerr(dcv.get(), O.restrict(of, oc, f0)) <= (TOL64 if t64 else TOL32)


@pytest.mark.parametrize("ns", [(2, 2, 2), (2, 2, 8), (4, 2, 4), (4, 4, 6), (8, 8, 8), (4, 16, 6), (12, 6, 10), (16, 16, 2)])
@pytest.mark.parametrize("big", [False, True])
def test_ghost_fill_3d_forms(ns, big):
    """Every form of the 3D face fill (faces of at most 16 cells, of at most 64, of more; few
    patches and many, every neighbour type): FP64 and FP32 against the oracle, two components."""
    _print_case("ghost3d-forms", ns, big)
    if big:
        forest = solver.Forest(3, 3)
        forest.refine((np.arange(512) % 5 == 0).astype(np.uint8))
        forest.balance()
        lv = forest.build_domains(ns)[0]
        assert len(lv) * 6 > 4096 and all((lv["nbr_type"][:, 20:] == k).any() for k in (-1, 0, 1, 2))
    else:
        lv = load("3d_refined_bnw_2x2x2_mpi1.json", ns)[1][0]
    od, dd = O.Domain(3, ns, lv), R.Domain(3, ns, lv)
    g = R.GhostFiller(dd, R.TRILINEAR, R.FACES)
    for dtype, tol in ((R.F64, TOL64), (R.F32, TOL32)):
        u0 = random_field(od.shape(2), 74, R.np_dtype(dtype))
        ref = u0.astype(np.float64)
        O.fill_ghost(od, ref, kind=R.TRILINEAR)
        du, df = R.DeviceArray.from_host(u0), R.DeviceArray(dd.shape(2), R.np_dtype(dtype))
        g.fill_ghost(du)
        got = du.get()
        assert relerr(got, ref) <= tol
        du.upload(u0)
        g.star_apply(du, df)  # the operator's own fill
        assert np.array_equal(du.get(), got)


@pytest.mark.parametrize("ns,level,ncomp,dtype", [
    ((16, 16, 16), 5, 3, R.F64), ((16, 16, 16), 5, 8, R.F32), ((12, 12, 12), 5, 8, R.F64), ((64, 64), 7, 8, R.F64)])
def test_vectors_past_4_gib(ns, level, ncomp, dtype):
    """Vectors of several components whose bytes pass 2^32: the ghost fill, the operator and the
    residual of every component have the bits of the same calls on that component alone.  Only the
    last patches and those 4 GiB before them (where an offset cut to 32 bits would land) hold data."""
    _print_case("past-4-gib", ns, level, ncomp, dtype)
    dim, L, t = len(ns), R.lib(), R.np_dtype(dtype)
    lv = solver.uniform_levels(dim, level, ns)[0]
    dd = R.Domain(dim, ns, lv)
    g = R.GhostFiller(dd, R.TRILINEAR if dim == 3 else R.BILINEAR, R.FACES)
    np_, cs, sz, k = len(lv), int(np.prod([n + 2 for n in ns])), t().itemsize, 64
    ps = cs * ncomp
    assert (np_ - k) * ps * sz > 1 << 32
    back = (np_ - k) - (((1 << 32) // sz + ps - 1) // ps)
    blocks = [(back, k + 2), (np_ - k, k)]

    def fresh(nc, data):
        d = R.DeviceArray(dd.shape(nc), t)
        d.zero()
        for (p, n), v in zip(blocks, data):
            v = np.ascontiguousarray(v)
            R.check(L.te_memcpy_h2d(d.ptr + p * cs * nc * sz, v.ctypes.data, v.nbytes))
        return d

    def got(d, nc):
        out = []
        for p, n in blocks:
            v = np.empty((n,) + dd.shape(nc)[1:], t)
            R.check(L.te_memcpy_d2h(v.ctypes.data, d.ptr + p * cs * nc * sz, v.nbytes))
            out.append(v)
        return out

    u0, f0 = ([random_field((n,) + dd.shape(ncomp)[1:], s + i, t) for i, (p, n) in enumerate(blocks)] for s in (91, 95))
    f = fresh(ncomp, f0)
    out = R.DeviceArray(dd.shape(ncomp), t)
    results = []
    for call in ("fill", "apply", "residual"):
        u = fresh(ncomp, u0)
        if call == "fill":
            g.fill_ghost(u)
        elif call == "apply":
            g.star_apply(u, out)
        else:
            g.residual(f, u, out)
        results.append((got(u, ncomp), None if call == "fill" else got(out, ncomp),
                        None if call == "fill" else dd.two_norm(out)))
        u.free()
    f.free()
    out.free()
    squares = [0.0, 0.0]
    out = R.DeviceArray(dd.shape(1), t)
    for c in range(ncomp):
        f = fresh(1, [v[:, c:c + 1] for v in f0])
        for i, call in enumerate(("fill", "apply", "residual")):
            u = fresh(1, [v[:, c:c + 1] for v in u0])
            if call == "fill":
                g.fill_ghost(u)
            elif call == "apply":
                g.star_apply(u, out)
            else:
                g.residual(f, u, out)
            for want, have in zip(got(u, 1), results[i][0]):
                assert np.array_equal(want[:, 0], have[:, c]), (call, c)
            if call != "fill":
                for want, have in zip(got(out, 1), results[i][1]):
                    assert np.array_equal(want[:, 0], have[:, c]), (call, c)
                squares[i - 1] += dd.two_norm(out) ** 2
            u.free()
        f.free()
    for i in (0, 1):  # and nothing was written elsewhere: the whole results' norms agree
        assert abs(results[i + 1][2] - np.sqrt(squares[i])) <= 1e-12 * results[i + 1][2]
