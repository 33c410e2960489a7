"""The marched variable-coefficient sweep where it is chosen (FP64 from level 8 on few cells, FP32 from level 7), Jacobi cycles with odd
numbers of steps, and the matrix-core coefficient integrals with 32-row blocks.

FP64: 1e-13 relative l-infinity, as the other parity tests. FP32: 8e-6 for one sweep (34 roundings of at most twice the largest
result each, twice that for its sum), plus 2e-5 from the coefficient where it is evaluated in FP32."""
import functools

import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu
MODES = ol.random_field(33, modes=8, kmax=3)


def rel_inf(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def rnd(n, seed, f32=False):
    v = np.random.default_rng(seed).uniform(-1.0, 1.0, n)
    return v.astype(np.float32).astype(np.float64) if f32 else v


@functools.lru_cache(maxsize=None)
def oracle_product(name, L):
    """Operator with 8 modes times a vector of FP32 values, and its inverse diagonal."""
    om = ol.Mesh(name)
    oop = ol.DivKGradOperator(om, L, L, ("fourier", 1.3, MODES))
    ox, od = ol.Function(om, L, L), ol.Function(om, L, L)
    x0 = rnd(om.ndofs(L), 30, True)
    ox.set(L, x0)
    oop.apply(ox, od, L, ol.ALL, False)
    return x0, od.get(L), oop.inv_diag(L)


@pytest.mark.parametrize("name,L,dtype,planes", [("tet_1el.msh", 8, "F64", None), ("tet_1el.msh", 8, "F64", 24), ("tet_1el.msh", 8, "F32", 24),
                                                 ("three_tets_with_two_joint_faces.msh", 7, "F32", None),
                                                 ("three_tets_with_two_joint_faces.msh", 7, "F32", 24)])
def test_marched_sweep_against_the_oracle(hyg, monkeypatch, name, L, dtype, planes):
    """Rows of several 62-point windows and every kind of point, in segments of 4 planes (what the rule gives on few cells) and of 24 (what
    it gives on many)."""
    if planes:
        monkeypatch.setenv("HYG_ZCHUNK", str(planes))
    else:
        monkeypatch.delenv("HYG_ZCHUNK", raising=False)
    dt = getattr(hyg, dtype)
    tol = 1e-13 if dtype == "F64" else 2.8e-5
    x0, Ax, dinv = oracle_product(name, L)
    gm = hyg.Mesh(name)
    n = gm.ndofs(L)
    b0, d0 = rnd(n, 31, True), rnd(n, 32, True)
    op = hyg.P1DivKGradOperator(gm, L, L, 1.3, MODES)
    op.store_local_matrices()
    bnd = gm.boundary(L)
    x, b, d = (hyg.Function(gm, L, L, dt) for _ in range(3))
    x.upload(L, x0)
    b.upload(L, b0)
    for flag in (hyg.INNER, hyg.ALL):
        on = ~bnd if flag == hyg.INNER else np.ones(n, dtype=bool)
        for what, ref in (("apply", Ax), ("add", d0 + Ax), ("residual", b0 - Ax), ("jacobi", x0 + 0.7 * dinv * (b0 - Ax))):
            print(name, L, dtype, planes, flag, what, flush=True)
            d.upload(L, d0)
            if what in ("apply", "add"):
                op.apply(x, d, L, flag, hyg.ADD if what == "add" else hyg.REPLACE)
            elif what == "residual":
                op.residual(d, b, x, L, flag)
            else:
                op.smooth_jac(d, b, x, 0.7, L, flag)
            assert rel_inf(d.download(L), np.where(on, ref, d0)) <= tol, (what, flag)


@pytest.mark.parametrize("batched", [False, True])
def test_chebyshev_steps_of_the_march(hyg, batched):
    """A Chebyshev sweep writes two vectors. FP32 marches at level 7, FP64 takes a thread per point there: six sweeps on each of eight
    levels, 34 roundings of at most twice the iterate each, set the iterates 8 * 6 * 34 * 2 * 2^-24 = 2e-4 apart at most."""
    L, name = 7, "three_tets_with_two_joint_faces.msh"
    mesh = hyg.Mesh(name)
    n = mesh.ndofs(L)
    b0 = rnd(n, 3, True)
    b0[mesh.boundary(L)] = 0.0
    out = {}
    for dtype in ("F64", "F32"):
        dt = getattr(hyg, dtype)
        op = hyg.P1DivKGradOperator(mesh, 0, L, 1.3, MODES)
        op.store_local_matrices()
        g = hyg.GMG(op, 0, L, dt, pre=1, post=1, smoother="cheb", cheb_order=3, cheb_bounds=(0.57, 2.28))
        x, b = hyg.Function(mesh, 0, L, dt), hyg.Function(mesh, 0, L, dt)
        b.upload(L, b0)
        if batched:
            hyg.Batch([g], [x], [b]).vcycle()
        else:
            g.vcycle(x, b, L)
        out[dtype] = x.download(L)
    assert np.abs(out["F64"]).max() > 0
    assert rel_inf(out["F32"], out["F64"]) <= 2e-4


@pytest.mark.parametrize("kind", ["const", "divkgrad"])
@pytest.mark.parametrize("pre,post", [(1, 3), (3, 2), (0, 1), (1, 0)])
def test_jacobi_cycles_with_odd_numbers_of_steps(hyg, hip_stream, kind, pre, post):
    """The steps alternate between the iterate and a second vector; values outside the flag (here not 0) hold in both."""
    L, name = 3, "cube_kuhn_6el.msh"
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    if kind == "const":
        op, oop = hyg.P1ConstantOperator(gm, 0, L), ol.Operator(om, 0, L)
    else:
        op, oop = hyg.P1DivKGradOperator(gm, 0, L, 1.0, MODES), ol.DivKGradOperator(om, 0, L, ("fourier", 1.0, MODES))
    x0, b0 = rnd(n, 1), rnd(n, 2)
    kw = dict(pre=pre, post=post, smoother="jacobi")
    ox, ob = ol.Function(om, 0, L), ol.Function(om, 0, L)
    ox.set(L, x0)
    ob.set(L, b0)
    ol.gmg(oop, ox, ob, 0, L, 2, **kw)
    ref = ox.get(L)
    g = hyg.GMG(op, 0, L, **kw)
    x, b = hyg.Function(gm, 0, L), hyg.Function(gm, 0, L)
    b.upload(L, b0)
    for graph in (False, True):
        x.upload(L, x0)
        for _ in range(2):
            if graph:
                g.vcycle_graph(x, b, L, 20, hip_stream)
            else:
                g.vcycle(x, b, L)
        assert rel_inf(x.download(L), ref) <= 1e-10, graph


def test_fp32_coefficient_integrals_of_the_matrix_cores_in_32_row_blocks(hyg):
    """32 modes at level 7: FP32 by matrix products in blocks of 32 rows, FP64 with a thread per anchor. FP32 phase factors are products of
    three rounded ones (4 * 2^-24 each) over a total amplitude of 0.5 sqrt(2 * 32) = 4: 4 * 6 * 2^-24 on log k at most, next to
    the 34 roundings of the sweep."""
    L, name = 7, "cube_kuhn_6el.msh"
    mesh = hyg.Mesh(name)
    n = mesh.ndofs(L)
    modes = ol.random_field(33, modes=32, kmax=8, std=0.5)
    op = hyg.P1DivKGradOperator(mesh, L, L, 1.3, modes)
    v = rnd(n, 4, True)
    out = {}
    for dtype in ("F64", "F32"):
        dt = getattr(hyg, dtype)
        x, y = hyg.Function(mesh, L, L, dt), hyg.Function(mesh, L, L, dt)
        x.upload(L, v)
        op.apply(x, y, L, hyg.ALL)
        out[dtype] = y.download(L)
    assert rel_inf(out["F32"], out["F64"]) <= 8e-6 + 4 * 6 * 2.0 ** -24 * 2


@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("nmodes,name,L", [(2, "cube_kuhn_6el.msh", 3), (3, "cube_kuhn_6el.msh", 3), (8, "cube_kuhn_6el.msh", 3),
                                           (9, "cube_kuhn_6el.msh", 2), (9, "cube_kuhn_6el.msh", 3), (13, "cube_kuhn_6el.msh", 3),
                                           (33, "cube_24el.msh", 3), (64, "cube_24el.msh", 2), (25, "cube_24el.msh", 4),
                                           (24, "cube_24el.msh", 4), (33, "cube_24el.msh", 4), (64, "tet_1el.msh", 0)])
def test_coefficient_integrals_on_both_sides_of_the_rule(hyg, nmodes, name, L, dtype):
    """By matrix products on few anchors (3 to 8, 13 to 64 modes up to level 3, 25 to 32 modes at level 4), else with a thread per anchor; the
    constant matrix is read in the same order by both."""
    dt = getattr(hyg, dtype)
    modes = ol.random_field(5, modes=nmodes, kmax=3)
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    x0 = rnd(n, 40, True)
    op = hyg.P1DivKGradOperator(gm, L, L, 1.3, modes)
    oop = ol.DivKGradOperator(om, L, L, ("fourier", 1.3, modes))
    x, y = hyg.Function(gm, L, L, dt), hyg.Function(gm, L, L, dt)
    ox, od = ol.Function(om, L, L), ol.Function(om, L, L)
    x.upload(L, x0)
    ox.set(L, x0)
    op.apply(x, y, L, hyg.ALL)
    oop.apply(ox, od, L, ol.ALL, False)
    assert rel_inf(y.download(L), od.get(L)) <= (1e-13 if dtype == "F64" else 2.8e-5)
