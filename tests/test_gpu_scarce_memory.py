"""Memory that layouts and solvers can do without, refused (ALP_HIP_OPTIONAL_BYTES): what
already runs keeps its arrays and its captured iterations, and every call still
gives its result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import alp_amd
    alp_amd.init(0)
    return alp_amd


def spd(n, offsets, rng, shuffle=False):
    """A symmetric diagonally dominant matrix with entries at the offsets (of both signs),
    the columns of a row in a random order with shuffle (no diagonal form then)."""
    off, idx, val = [0], [], []
    weight = {d: rng.uniform(0.1, 1.0, n) for d in offsets if d > 0}
    for r in range(n):
        row = [(r + d, -(weight[d][r] if d > 0 else weight[-d][r + d])) for d in offsets if d and 0 <= r + d < n]
        row.append((r, 1.0 - sum(v for _, v in row)))
        if shuffle:
            rng.shuffle(row)
        idx += [int(c) for c, _ in row]
        val += [float(v) for _, v in row]
        off.append(len(idx))
    return np.array(off, np.uint64), np.array(idx, np.uint32), np.array(val)


def make(A, kind, rng, flags=0):
    if kind == "runs":  # 27 points, a value per entry
        s = 12
        return A.Matrix.conductance27(s, s, s, A.Vector.from_numpy(rng.uniform(0.5, 2.0, 13 * s ** 3)), 1.0, flags)
    if kind == "constant":
        return A.Matrix.stencil27(12, 12, 12, flags=flags)
    n = 2000
    off, idx, val = spd(n, [-40, -1, 1, 40], rng, kind == "sliced")
    return A.Matrix.from_crs(n, n, off, idx, val, flags=flags)


KINDS = ["runs", "diagonal", "sliced", "constant"]


@pytest.mark.parametrize("kind", KINDS)
def test_fp32_copy_refused_between_two_solves(A, kind, monkeypatch):
    """An FP64 solve, a mixed solve that gets no memory for the layout's FP32 values, and
    the FP64 solve again on its captured iterations: the same bits, and the layout holds
    what it held (beside the FP32 copy of the CRS values)."""
    rng = np.random.default_rng(1)
    M = make(A, kind, rng)
    assert M.form() == getattr(A, "FORM_" + kind.upper())
    b, x = A.Vector.from_numpy(rng.standard_normal(M.nrows)), A.Vector(M.nrows)

    def solve(precision, tol, limit):
        x.set(0.0)
        return A.cg(M, b, x, limit, tol, precision)[0], x.numpy()

    first = solve(0, 1e-300, 20)[1]
    held, form = M.device_bytes(), (M.form(), M.layout(), M.get_kernel())
    monkeypatch.setenv("ALP_HIP_OPTIONAL_BYTES", "0")
    mixed = [solve(p, 1e-10, 1000) for p in (1, 3)]
    monkeypatch.delenv("ALP_HIP_OPTIONAL_BYTES")
    assert M.device_bytes() == held + 4 * M.nnz
    assert (M.form(), M.layout(), M.get_kernel()) == form
    assert np.array_equal(solve(0, 1e-300, 20)[1], first)
    rc, want = solve(0, 1e-12, 1000)
    assert rc == A.SUCCESS
    # residuals below 1e-10 of b on matrices of condition number below 1e3
    for rc, got in mixed:
        assert rc == A.SUCCESS
        assert np.linalg.norm(got - want) <= 1e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("kind", KINDS)
def test_layouts_refused_at_build(A, kind, monkeypatch):
    """With no memory for any layout the products run on the CRS."""
    full = make(A, kind, np.random.default_rng(2))
    monkeypatch.setenv("ALP_HIP_OPTIONAL_BYTES", "0")
    bare = make(A, kind, np.random.default_rng(2))
    monkeypatch.delenv("ALP_HIP_OPTIONAL_BYTES")
    assert bare.form() == A.FORM_CRS and bare.device_bytes() < full.device_bytes()
    rng = np.random.default_rng(3)
    x = rng.standard_normal(full.nrows)
    got = []
    for M in (full, bare):
        y = A.Vector(M.nrows, fill=0.0)
        assert A.mxv(y, M, A.Vector.from_numpy(x)) == A.SUCCESS
        got.append(y.numpy())
    # two orders of at most 27 products
    assert np.max(np.abs(got[0] - got[1])) <= 28 * 2.0 ** -53 * 60 * np.max(np.abs(x))


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


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("precision", [0, 1, 3])
def test_cg_iterates_at_every_slot(A, precision, transpose, monkeypatch):
    """x after 1 to 9 and 15 to 18 iterations, with four directions between the updates of
    x and, where those are refused, with one: the same bits, and the iterates of an FP64
    restatement. Rounding reaches x with a factor below 1e3 (the condition number)."""
    import scipy.sparse as sp
    rng = np.random.default_rng(4)
    n = 1999
    off, idx, val = spd(n, [-40, -7, -1, 1, 7, 40], rng)
    S = sp.csr_matrix((val, idx.astype(np.int64), off.astype(np.int64)), shape=(n, n))
    b = rng.standard_normal(n)
    want = cg_iterates(S.T if transpose else S, b, 18)
    four, one = (A.Matrix.from_crs(n, n, off, idx, val, flags=A.MAT_WITH_F32 | A.MAT_WITH_CCS) for _ in range(2))
    rhs = A.Vector.from_numpy(b)
    bound = 1e3 * 2.0 ** (-53 if precision == 0 else -24)
    for k in list(range(1, 10)) + [15, 16, 17, 18]:
        got = []
        for M in (four, one):
            if M is one:
                monkeypatch.setenv("ALP_HIP_OPTIONAL_BYTES", "0")
            else:
                monkeypatch.delenv("ALP_HIP_OPTIONAL_BYTES", raising=False)
            x = A.Vector(n, fill=0.0)
            rc, it, _ = A.cg(M, rhs, x, k, 1e-300, precision, transpose=transpose)
            assert it == k
            got.append(x.numpy())
        assert np.array_equal(got[0], got[1]), k
        assert np.max(np.abs(got[0] - want[k - 1])) <= bound * np.max(np.abs(want[k - 1])), k


@pytest.mark.parametrize("kind", ["runs", "diagonal"])
@pytest.mark.parametrize("precision", [0, 1, 3])
def test_one_direction_equals_four(A, kind, precision, monkeypatch):
    """Whole solves, whose reliable updates restart from whichever direction a segment ended
    on, and again on the captured iterations after the refusal is over."""
    four, one = (make(A, kind, np.random.default_rng(6), A.MAT_WITH_F32) for _ in range(2))
    ends = set()
    for t in range(7):
        b = A.Vector.from_numpy(np.random.default_rng(t).standard_normal(four.nrows))
        got = []
        for M in (four, one):
            if M is one and t < 6:
                monkeypatch.setenv("ALP_HIP_OPTIONAL_BYTES", "0")
            else:
                monkeypatch.delenv("ALP_HIP_OPTIONAL_BYTES", raising=False)
            x = A.Vector(M.nrows, fill=0.0)
            rc, it, res = A.cg(M, b, x, 2000, 10.0 ** -(6 + t % 6), precision)
            assert rc == A.SUCCESS
            got.append((it, res, x.numpy()))
        assert got[0][:2] == got[1][:2]
        assert np.array_equal(got[0][2], got[1][2])
        ends.add(got[0][0] % 4)
    assert len(ends) > 1  # not all on one slot
