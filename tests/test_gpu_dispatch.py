"""Rules that choose between kernels, at the sizes on both sides of their lines, against the CPU oracle.

FP64: 1e-13 relative l-infinity, as the other parity tests. FP32: a stencil value is a sum of at most 30 products of FP32
weights and values (a face point: 15 per cell), so its error is below (30 + 4) 2^-24 sum |w x|; sum |w x| is at most
twice the centre weight times max |x|, which the largest result reaches up to a factor of two: 34 * 4 * 2^-24 = 8e-6.
"""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu
TOL = {8: 1e-13, 4: 8e-6}


def rel_inf(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def rnd(n, seed, f32):
    v = np.random.default_rng(seed).uniform(-1.0, 1.0, n)
    return v.astype(np.float32).astype(np.float64) if f32 else v


@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("name,L", [("three_tets_with_two_joint_faces.msh", 6), ("three_tets_with_two_joint_faces.msh", 7),
                                    ("cube_kuhn_6el.msh", 1), ("cube_kuhn_6el.msh", 7)])
def test_face_points_in_the_sweep_and_from_one_sided_sums(hyg, name, L, dtype):
    """Up to level 6 the sweep gathers face points itself, above it the cells leave one-sided sums."""
    dt = getattr(hyg, dtype)
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    x0, b0, d0 = (rnd(n, 20 + k, dt == hyg.F32) for k in range(3))
    op, oop = hyg.P1ConstantOperator(gm, L, L), ol.Operator(om, L, L)
    ox, ob = ol.Function(om, L, L), ol.Function(om, L, L)
    ox.set(L, x0)
    ob.set(L, b0)
    od = ol.Function(om, L, L)
    oop.apply(ox, od, L, ol.ALL, False)
    Ax = od.get(L)
    inv = hyg.Function(gm, L, L)
    op.inverse_diagonal(inv, L)
    dinv = inv.download(L)
    bnd = gm.boundary(L)
    for flag in (hyg.INNER, hyg.ALL):
        on = ~bnd if flag == hyg.INNER else np.ones(n, dtype=bool)
        x, b, d = (hyg.Function(gm, L, L, dt) for _ in range(3))
        x.upload(L, x0)
        b.upload(L, b0)
        for what, ref in (("apply", Ax), ("add", d0 + Ax), ("residual", b0 - Ax), ("jacobi", x0 + 0.7 * dinv * (b0 - Ax))):
            print(name, L, dtype, flag, what, flush=True)
            d.upload(L, d0)
            if what in ("apply", "add"):
                op.apply(x, d, L, flag, hyg.ADD if what == "add" else hyg.REPLACE)
            elif what == "residual":
                op.residual(d, b, x, L, flag)
            else:
                op.smooth_jac(d, b, x, 0.7, L, flag)
            assert rel_inf(d.download(L), np.where(on, ref, d0)) <= TOL[dt], (what, flag)


# 8 modes of wavenumber <= 3: FP32 phases up to 2 pi 3 sqrt(3) |x| ~ 60 are off by 60 * 2^-24, which moves a cosine of total
# amplitude 0.5 sqrt(2 * 8) and so log k by 8e-6 at most; with the 34 roundings of the sum this stays below 2e-5
@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("name,L", [("three_tets_with_two_joint_faces.msh", 0), ("three_tets_with_two_joint_faces.msh", 1),
                                    ("pyramid_tilted_4el.msh", 6), ("three_tets_with_two_joint_faces.msh", 7)])
def test_variable_coefficient_sweep(hyg, name, L, dtype):
    """The sweep with a thread per point and, for FP32 at level 7, the march in segments of 4 planes: every kind of point. The inverse
    diagonal is the library's own here (against the oracle: test_gpu_divkgrad.py, test_gpu_march.py)."""
    dt = getattr(hyg, dtype)
    modes = ol.random_field(33, modes=8, kmax=3)
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    x0, b0, d0 = (rnd(n, 30 + k, dt == hyg.F32) for k in range(3))
    op = hyg.P1DivKGradOperator(gm, L, L, 1.3, modes)
    op.store_local_matrices()
    oop = ol.DivKGradOperator(om, L, L, ("fourier", 1.3, modes))
    ox, od = ol.Function(om, L, L), ol.Function(om, L, L)
    ox.set(L, x0)
    oop.apply(ox, od, L, ol.ALL, False)
    Ax = od.get(L)
    inv = hyg.Function(gm, L, L)
    op.inverse_diagonal(inv, L)
    dinv = inv.download(L)
    bnd = gm.boundary(L)
    for flag in (hyg.INNER, hyg.ALL):
        on = ~bnd if flag == hyg.INNER else np.ones(n, dtype=bool)
        x, b, d = (hyg.Function(gm, L, L, dt) for _ in range(3))
        x.upload(L, x0)
        b.upload(L, b0)
        for what, ref in (("apply", Ax), ("add", d0 + Ax), ("residual", b0 - Ax), ("jacobi", x0 + 0.7 * dinv * (b0 - Ax))):
            print(name, L, dtype, flag, what, flush=True)
            d.upload(L, d0)
            if what in ("apply", "add"):
                op.apply(x, d, L, flag, hyg.ADD if what == "add" else hyg.REPLACE)
            elif what == "residual":
                op.residual(d, b, x, L, flag)
            else:
                op.smooth_jac(d, b, x, 0.7, L, flag)
            assert rel_inf(d.download(L), np.where(on, ref, d0)) <= (1e-13 if dt == hyg.F64 else 2e-5), (what, flag)


def test_points_do_not_see_values_that_are_not_their_neighbours(hyg):
    """An infinite value stays within the stencil of its point (which neighbours of weight 0 do not see: test_gpu_nonfinite.py)."""
    L, name = 6, "tet_1el.msh"
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    modes = ol.random_field(33, modes=8, kmax=3)
    op = hyg.P1DivKGradOperator(gm, L, L, 1.3, modes)
    op.store_local_matrices()
    xyz, _ = gm.coords(L)
    rng = np.random.default_rng(8)
    x, y = hyg.Function(gm, L, L), hyg.Function(gm, L, L)
    for k in rng.choice(n, 12, replace=False):
        v = rng.uniform(-1.0, 1.0, n)
        v[k] = np.inf
        x.upload(L, v)
        op.apply(x, y, L, hyg.ALL)
        bad = ~np.isfinite(y.download(L))
        assert bad[k]
        # neighbours lie within one lattice step in every local coordinate
        assert np.abs(xyz[bad] - xyz[k]).max() <= 2.0 * np.abs(xyz).max() / (1 << L) + 1e-12


@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("nmodes,L", [(0, 1), (1, 3), (8, 5), (9, 2), (32, 6), (33, 4), (64, 5)])
def test_coefficient_integrals_of_every_variant(hyg, nmodes, L, dtype):
    """The matrix product behind k by the number of modes (tables padded to 8, 32 or 64) and the length of rows; which of the two kernels
    forms it: test_gpu_march.py."""
    dt = getattr(hyg, dtype)
    name = "pyramid_tilted_4el.msh"
    modes = ol.random_field(5, modes=nmodes, kmax=3) if nmodes else []
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L)
    x0 = rnd(n, 40, dt == hyg.F32)
    op = hyg.P1DivKGradOperator(gm, L, L, 1.3, modes)
    oop = ol.DivKGradOperator(om, L, L, ("fourier", 1.3, modes if nmodes else np.zeros((0, 5))))
    x, y = hyg.Function(gm, L, L, dt), hyg.Function(gm, L, L, dt)
    ox, od = ol.Function(om, L, L), ol.Function(om, L, L)
    x.upload(L, x0)
    ox.set(L, x0)
    print(nmodes, L, dtype, flush=True)
    op.apply(x, y, L, hyg.ALL)
    oop.apply(ox, od, L, ol.ALL, False)
    # FP32: rounding of up to 2 * 64 terms of total size sqrt(2 * 64) * 0.5 in log k, 6e-6, and 34 roundings of the sum
    assert rel_inf(y.download(L), od.get(L)) <= (1e-13 if dt == hyg.F64 else 2e-5)


@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("name,L", [("tet_1el.msh", 0), ("tet_1el.msh", 1), ("three_tets_with_two_joint_faces.msh", 2),
                                    ("pyramid_tilted_4el.msh", 4)])
def test_variable_p2_every_kind_of_point(hyg, name, L, stored):
    """Vertex, edge-midpoint, face and cell-edge points by the moments of k, one and several components, both value types."""
    gm, om = hyg.Mesh(name), ol.Mesh(name)
    n = gm.ndofs(L + 1)
    op = hyg.P2DivKGradOperator(gm, L, L, kind=0, k0=1.2, alpha=0.7, beta=0.3, seed=11)
    if stored:
        op.store_local_matrices()
    oop = ol.P2DivKGradOperator(om, L, L, kind=0, k0=1.2, alpha=0.7, beta=0.3, seed=11)
    # FP32: at most 24 micro-cells of 10 products, 240 + 24 roundings of terms of at most a few times the largest result
    for dt, tol in ((hyg.F64, 1e-13), (hyg.F32, 264 * 4 * 2.0 ** -24)):
        xs = [hyg.Function(gm, L, L, dt, space="p2") for _ in range(3)]
        ys = [hyg.Function(gm, L, L, dt, space="p2") for _ in range(3)]
        ref = []
        for k in range(3):
            v = rnd(n, 50 + k, dt == hyg.F32)
            xs[k].upload(L, v)
            ox, oy = ol.Function(om, L + 1, L + 1), ol.Function(om, L + 1, L + 1)
            ox.set(L + 1, v)
            oop.apply(ox, oy, L + 1, ol.ALL, False)
            ref.append(oy.get(L + 1))
        for comps in (1, 2, 3):
            print(name, L, stored, dt, comps, flush=True)
            for y in ys:
                y.interpolate(0.0, L)
            hyg.apply_vector(op, xs[:comps], ys[:comps], L, hyg.ALL)
            for k in range(comps):
                assert rel_inf(ys[k].download(L), ref[k]) <= tol, (comps, k)
