"""The conjugate gradient at the edges of its budget and of the host's chunks of eight iterations:
iterates, iteration counts and residuals of the same algorithm in numpy on the context's own matrix. Both sides are FP64
and differ by summation order: 1e-16 per operation, amplified by at most the condition number of these systems (below
1e6) over the few dozen iterations, hence 1e-9."""
import numpy as np
import pytest

from spg_amd import native, scenes

pytestmark = pytest.mark.gpu


def _reference(A, b, tol, budget):
    d = A.diagonal()
    inv = np.where(d != 0, 1.0 / np.where(d != 0, d, 1.0), 1.0)
    x, r = np.zeros_like(b), b.copy()
    limit = max(tol * tol * (b @ b), np.finfo(float).tiny)
    p, it, rr = inv * r, 0, b @ b
    rz = r @ p
    if rr < limit:
        return x, 0, 0.0 if rr == 0 else 1.0
    while it < budget:
        q = A @ p
        alpha = rz / (p @ q)
        x, r = x + alpha * p, r - alpha * q
        rr = r @ r
        if rr < limit:
            break
        z = inv * r
        old, rz = rz, r @ z
        p, it = z + rz / old * p, it + 1
    return x, it, np.sqrt(rr / (b @ b))


@pytest.fixture(scope="module", params=["cloth", "cube", "one particle"])
def system(request):
    s = {"cloth": lambda: scenes.cloth(21, young=1e3, pin="top_row", noise=1e-3),
         "cube": lambda: scenes.cube(5, young=1e4),
         "one particle": lambda: scenes.Scene(x=np.ones((1, 3)), x0=np.ones((1, 3)), m=np.array([2.0]),
                                              energies=[("anchor", np.array([[0]], np.int32), np.array([[1, 1, 1.5, 30.0]]))])}[request.param]()
    import scipy.sparse as sp
    ctx = native.ImplicitContext([s.vbd_object()], "baraff_witkin")
    h = scenes.DT
    A = (sp.diags(np.repeat(s.m, 3)) - h * h * ctx.stiffness()).tocsr()
    b = h * ctx.system_force(s.gravity) + 1e-3 * np.random.default_rng(4).standard_normal(3 * s.n)
    return ctx, A, b, h


@pytest.mark.parametrize("budget", [0, 1, 2, 7, 8, 9, 16, 17, 300])
@pytest.mark.parametrize("tol", [1e-3, 1e-6, 1e-10])
def test_iterates_and_counts(system, budget, tol):
    ctx, A, b, h = system
    x, it, err = ctx.cg_solve(1.0, -h * h, b, tol=tol, max_iters=budget)
    ex, eit, eerr = _reference(A, b, tol, budget)
    assert it == eit
    assert np.linalg.norm(x - ex) <= 1e-9 * max(np.linalg.norm(ex), 1e-300)
    assert err == pytest.approx(eerr, rel=1e-5, abs=1e-14)


def test_zero_right_hand_side(system):
    ctx, A, b, h = system
    x, it, err = ctx.cg_solve(1.0, -h * h, np.zeros_like(b))
    assert it == 0 and err == 0 and not x.any()


@pytest.fixture(scope="module")
def large_system():
    """A cloth whose matrix and vectors the caches do not hold: an iteration takes three kernels instead of two. beta is such
    that no row of beta K sums to more than 0.9 of the mass: by Gershgorin the eigenvalues of M + beta K lie between 0.1 and
    1.9 of the mass, the condition number is below 19, and 1e-9 is far above what the summation order can do."""
    import scipy.sparse as sp
    s = scenes.cloth(520, young=1e3, pin="top_row", noise=1e-4)
    ctx = native.ImplicitContext([s.vbd_object()], "baraff_witkin")
    assert ctx.spmv_bytes() + 48 * ctx.num_dofs() > 201326592
    K = ctx.stiffness()
    beta = -0.9 * s.m[0] / abs(K).sum(axis=1).max()
    A = (sp.diags(np.repeat(s.m, 3)) + beta * K).tocsr()
    b = scenes.DT * ctx.system_force(s.gravity) + 1e-3 * np.random.default_rng(4).standard_normal(3 * s.n)
    return ctx, A, b, beta


@pytest.mark.parametrize("budget,tol", [(0, 1e-6), (1, 1e-6), (2, 1e-6), (7, 1e-9), (8, 1e-9), (9, 1e-9), (17, 1e-12), (300, 1e-2),
                                        (300, 1e-3), (300, 1e-4), (300, 1e-8), (300, 10.0)])
def test_iterates_and_counts_of_a_large_system(large_system, budget, tol):
    ctx, A, b, beta = large_system
    x, it, err = ctx.cg_solve(1.0, beta, b, tol=tol, max_iters=budget)
    ex, eit, eerr = _reference(A, b, tol, budget)
    assert it == eit
    assert np.linalg.norm(x - ex) <= 1e-9 * max(np.linalg.norm(ex), 1e-300)
    assert err == pytest.approx(eerr, rel=1e-5, abs=1e-14)
