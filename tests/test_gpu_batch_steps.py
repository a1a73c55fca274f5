"""The batched CG keeps a few directions and adds their steps to X together: X
after k iterations, for every k around a full set of directions, against the CG
iterates of an FP64 restatement; systems that freeze at different iterations."""
import numpy as np
import pytest

from test_gpu_batch import A, laplace7  # noqa: F401

pytestmark = pytest.mark.gpu


def cg_iterates(M, b, k):
    x, r = np.zeros_like(b), b.copy()
    p, rz = r.copy(), r @ r
    out = []
    for _ in range(k):
        ap = M @ p
        alpha = rz / (p @ ap)
        x = x + alpha * p
        r = r - alpha * ap
        rr = r @ r
        p, rz = r + rr / rz * p, rr
        out.append(x)
    return out


@pytest.mark.parametrize("nrhs", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_iterates_at_every_slot(A, nrhs, precision):  # noqa: F811
    """9 iterations are far from converged (sides 7 to 19). Ten CG steps at a condition
    number below 1e3 carry rounding of the recurrences to x with a factor below
    1e3: 1e3 * 2^-53 in FP64 and 1e3 * 2^-24 in FP32, relative."""
    rng = np.random.default_rng(nrhs * 10 + precision)
    sides = np.array([[7, 11, 19], [16, 5, 13], [9, 17, 8]])
    coef = rng.uniform(0.5, 2.0, (3, 3))
    B = A.Batch(*sides.T, *coef.T, nrhs)
    b = rng.standard_normal((B.nrows, nrhs))
    rhs = A.Vector.from_numpy(b.ravel())
    want = np.zeros((9, B.nrows, nrhs))
    for s in range(3):
        r0, r1 = int(B.row0[s]), int(B.row0[s + 1])
        M = laplace7(*map(int, sides[s]), *map(float, coef[s]))
        for j in range(nrhs):
            want[:, r0:r1, j] = cg_iterates(M, b[r0:r1, j], 9)
    for k in range(1, 10):
        X = A.Vector(B.nrows * nrhs, fill=7.0)
        # precision 2 limits each refinement step; k iterations bring every residual below
        # 0.999 of b, so that there is one step
        rc, its, _, _ = B.solve(rhs, X, 0.999 if precision == 2 else 1e-12, k, precision)
        got = X.numpy().reshape(B.nrows, nrhs)
        assert np.all(np.asarray(its) == k)
        bound = 1e3 * 2.0 ** (-53 if precision == 0 else -24)
        assert np.max(np.abs(got - want[k - 1])) <= bound * np.max(np.abs(want[k - 1]))


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_systems_freeze_apart(A, precision):  # noqa: F811
    """Sides 1 to 24: systems stop after 1 to about 60 iterations, a right-hand side of
    zeros at once and an eigenvector after one; every instance reaches the tolerance
    and its neighbours' X stay theirs."""
    rng = np.random.default_rng(precision)
    nx, ny, nz = np.array([1, 24, 3, 9, 2, 17]), np.array([1, 20, 2, 9, 1, 5]), np.array([1, 22, 4, 9, 3, 6])
    c = rng.uniform(0.5, 2.0, (3, 6))
    B = A.Batch(nx, ny, nz, *c, 8)
    b = rng.standard_normal((B.nrows, 8))
    b[:, 3] = 0.0
    r0, r1 = int(B.row0[3]), int(B.row0[4])
    w = np.sin(np.pi * np.arange(1, 10) / 10)
    b[r0:r1, 5] = np.einsum("i,j,k->ijk", w, w, w).ravel()
    X = A.Vector(B.nrows * 8, fill=3.0)
    rc, its, rel, _ = B.solve(A.Vector.from_numpy(b.ravel()), X, 1e-9, 1000, precision)
    assert rc == A.SUCCESS and np.max(rel) <= 1e-9
    got = X.numpy().reshape(-1, 8)
    assert np.all(got[:, 3] == 0.0)
    for s in range(6):
        q0, q1 = int(B.row0[s]), int(B.row0[s + 1])
        M = laplace7(int(nx[s]), int(ny[s]), int(nz[s]), *map(float, c[:, s]))
        res = np.linalg.norm(b[q0:q1] - M @ got[q0:q1], axis=0)
        # the solver's own residual differs by the rounding of one product
        assert np.all(res <= 1.1e-9 * np.linalg.norm(b[q0:q1], axis=0))
