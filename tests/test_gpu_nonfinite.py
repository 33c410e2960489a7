"""Infinite values: they reach the points whose stencil holds them with a weight that is not 0, and no other. Which weights are 0 is
read off the operator applied to unit vectors."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu


def points(n, seed, k):
    return np.random.default_rng(seed).choice(n, k, replace=False)


def check_apply(apply, x, y, n, L, k, own=None):
    """Column k of the operator from a unit vector, then the same vector with an infinite entry: infinities of the weights' signs where
    the weight is not 0, finite and equal to the product without it elsewhere. own: the value expected at the point itself."""
    e = np.zeros(n)
    e[k] = 1.0
    x.upload(L, e)
    apply(x, y)
    col = y.download(L)
    v = np.random.default_rng(5).uniform(-1.0, 1.0, n)
    v[k] = 0.0
    x.upload(L, v)
    apply(x, y)
    rest = y.download(L)
    v[k] = np.inf
    x.upload(L, v)
    apply(x, y)
    got = y.download(L)
    others = np.arange(n) != k
    touched = others & (col != 0.0)
    assert touched.any()
    assert (got[touched] == np.copysign(np.inf, col[touched])).all()
    same = others & (col == 0.0)
    assert np.isfinite(got[same]).all()
    assert np.abs(got[same] - rest[same]).max() <= 1e-5 * np.abs(rest).max()
    assert not np.isfinite(got[k])
    if own is not None:
        assert got[k] == own


@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("name,L", [("cube_kuhn_6el.msh", 3), ("cube_kuhn_6el.msh", 7), ("tet_1el.msh", 8)])
def test_variable_coefficient_operator(hyg, name, L, dtype):
    """The edges of these cells are orthogonal in part, so a third of the stencil weights are 0. FP32 at level 7 and both types at level 8
    march (planes whose sums are not finite are done again point by point), the others take a thread per point."""
    dt = getattr(hyg, dtype)
    mesh = hyg.Mesh(name)
    op = hyg.P1DivKGradOperator(mesh, L, L, 1.3, ol.random_field(33, modes=8, kmax=3))
    op.store_local_matrices()
    n = mesh.ndofs(L)
    x, y = hyg.Function(mesh, L, L, dt), hyg.Function(mesh, L, L, dt)
    xyz, _ = mesh.coords(L)
    # random points, and points on an inner macro-face (x = y) and on the outer faces
    inner = np.flatnonzero((np.abs(xyz[:, 0] - xyz[:, 1]) < 1e-12) & (xyz[:, 2] > 0.1) & (xyz[:, 2] < 0.8))
    face = np.flatnonzero(np.abs(xyz[:, 2] - xyz[:, 2].min()) < 1e-12)
    for k in [*points(n, 3, 3), *inner[len(inner) // 3:][:1], face[len(face) // 2]]:
        print(name, L, dtype, int(k), flush=True)
        check_apply(lambda a, b: op.apply(a, b, L, hyg.ALL), x, y, n, L, int(k))


@pytest.mark.parametrize("dtype", ["F64", "F32"])
def test_variable_coefficient_residual_and_jacobi_with_infinite_values(hyg, dtype):
    """The planes of the march that are done again read their right-hand side and store both ways: against the same sweep whose
    infinite value is replaced by 0, at the points that do not see it; adding results adds them once."""
    dt, L = getattr(hyg, dtype), 8
    mesh = hyg.Mesh("tet_1el.msh")
    op = hyg.P1DivKGradOperator(mesh, L, L, 1.3, ol.random_field(33, modes=8, kmax=3))
    op.store_local_matrices()
    n = mesh.ndofs(L)
    x, y, b = (hyg.Function(mesh, L, L, dt) for _ in range(3))
    rng = np.random.default_rng(4)
    v, rhs, old = (rng.uniform(-1.0, 1.0, n) for _ in range(3))
    ks = points(n, 9, 5)
    calls = {"residual": lambda: op.residual(y, b, x, L, hyg.ALL), "jacobi": lambda: op.smooth_jac(y, b, x, 0.7, L, hyg.ALL),
             "add": lambda: op.apply(x, y, L, hyg.ALL, hyg.ADD)}
    b.upload(L, rhs)
    for what, call in calls.items():
        res = []
        for value in (0.0, np.inf):
            v[ks] = value
            x.upload(L, v)
            y.upload(L, old)
            call()
            res.append(y.download(L))
        fine = np.isfinite(res[1])
        assert not fine[ks].any() and (~fine).sum() <= 15 * len(ks), what
        assert np.abs(res[1][fine] - res[0][fine]).max() <= 1e-5 * np.abs(res[0]).max(), what


@pytest.mark.parametrize("dtype", ["F64", "F32"])
def test_constant_operator_and_restriction_at_the_point_itself(hyg, dtype):
    """Lanes of face, edge and vertex points have no neighbours outside a cell; the point's own infinite value stays infinite."""
    dt, L = getattr(hyg, dtype), 3
    mesh = hyg.Mesh("cube_kuhn_6el.msh")
    n, nc = mesh.ndofs(L), mesh.ndofs(L - 1)
    op = hyg.P1ConstantOperator(mesh, L, L)
    x, y = hyg.Function(mesh, L, L, dt), hyg.Function(mesh, L, L, dt)
    r = hyg.Function(mesh, L - 1, L, dt)
    xyz, _ = mesh.coords(L)
    cxyz, _ = mesh.coords(L - 1)
    for k in points(n, 6, 60):
        v = np.zeros(n)
        v[k] = np.inf
        x.upload(L, v)
        op.apply(x, y, L, hyg.ALL)
        assert y.download(L)[k] == np.inf
        r.upload(L, v)
        r.restrict(L, hyg.ALL)
        c = np.flatnonzero(np.abs(cxyz - xyz[k]).max(axis=1) < 1e-12)
        if len(c):
            assert r.download(L - 1)[c[0]] == np.inf
    assert nc < n


@pytest.mark.parametrize("dtype", ["F64", "F32"])
@pytest.mark.parametrize("stored", [False, True])
def test_variable_p2_operator_at_the_point_itself(hyg, stored, dtype):
    """A point on a cell face has stencil nodes outside the cell, of weight 0; its own infinite value stays infinite."""
    dt, L = getattr(hyg, dtype), 2
    mesh = hyg.Mesh("three_tets_with_two_joint_faces.msh")
    n = mesh.ndofs(L + 1)
    op = hyg.P2DivKGradOperator(mesh, L, L, kind=1)
    if stored:
        op.store_local_matrices()
    x, y = (hyg.Function(mesh, L, L, dt, space="p2") for _ in range(2))
    lost = []
    for k in range(n):
        v = np.zeros(n)
        v[k] = np.inf
        x.upload(L, v)
        op.apply(x, y, L, hyg.ALL)
        if y.download(L)[k] != np.inf:
            lost.append(k)
    assert not lost
