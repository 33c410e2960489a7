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
