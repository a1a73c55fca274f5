"""The constant form (one template of offsets and values for all rows): every product
and solve on it must equal the forms that keep values bit for bit, and matrices
that only nearly fit must keep those forms. ALP_HIP_CONST_DIA=0 builds without it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import alp_amd
    alp_amd.init(0)
    return alp_amd


def banded(n, m, offs, vals, drop=None):
    """Rows r of an n x m matrix with entries (r + d, v) for the offsets in the given
    order that land in [0, m); drop(r, q) leaves entry q of row r out."""
    R = np.repeat(np.arange(n, dtype=np.int64), len(offs))
    C = R + np.tile(np.asarray(offs, np.int64), n)
    V = np.tile(np.asarray(vals), n)
    keep = (C >= 0) & (C < m)
    if drop is not None:
        keep &= ~drop
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(R[keep], minlength=n), out=off[1:])
    return off, C[keep].astype(np.uint32), V[keep]


def both(A, monkeypatch, build):
    monkeypatch.setenv("ALP_HIP_CONST_DIA", "0")
    plain = build()
    monkeypatch.delenv("ALP_HIP_CONST_DIA")
    return build(), plain


def products(A, M, x, y0, ring, mask):
    out = []
    for descr, mk in ((0, None), (A.OVERWRITE, None), (0, mask), (A.INVERT_MASK, mask), (A.OVERWRITE, mask)):
        y = A.Vector.from_numpy(y0)
        assert A.mxv(y, M, A.Vector.from_numpy(x), ring=ring, descr=descr,
                     mask=None if mk is None else A.Vector.from_numpy(mk)) == A.SUCCESS
        out.append(y.numpy())
    return out


# widths around the compile-time ones (7 and 27) and the largest; one slice, a last
# slice of one (short) row, of 31 rows and of one full row; wider and narrower than
# long, with NaN and infinities at entries of x
@pytest.mark.parametrize("w", [1, 2, 6, 7, 8, 9, 26, 27, 28, 32])
@pytest.mark.parametrize("n,m", [(64, 64), (129, 400), (223, 215), (257, 1000), (1000, 1000), (3001, 2950)])
def test_const_products_equal_kept_values(A, w, n, m, monkeypatch):
    rng = np.random.default_rng(1000 * w + n)
    reach = min(45, max((w + 1) // 2, n // 16))
    offs = rng.permutation(rng.choice(np.arange(-reach, reach + 1), size=w, replace=False))
    vals = rng.standard_normal(w)
    drop = rng.random((n, w)) < (0.0 if n == 64 else 0.02 if n < 1000 else 0.1)
    drop[n // 2] = False  # a row with the whole list
    if n == 129:
        drop[-1] = True
        drop[-1, rng.integers(0, w)] = False
    off, idx, val = banded(n, m, offs, vals, drop.ravel())
    x, y0 = rng.standard_normal(m), rng.standard_normal(n)
    if n == 1000:
        x[17], x[400], x[999] = np.nan, np.inf, -np.inf
    mask = (rng.random(n) < 0.5).astype(np.uint8)
    F, P = both(A, monkeypatch, lambda: A.Matrix.from_crs(n, m, off, idx, val, flags=A.MAT_WITH_F32))
    F32, P32 = both(A, monkeypatch, lambda: A.Matrix.from_crs(n, m, off, idx, val.astype(np.float32)))
    x32, y32 = x.astype(np.float32), y0.astype(np.float32)
    for c, p, ring, xv, yv in ((F, P, A.PLUS_TIMES_F64, x, y0), (F, P, A.MIN_PLUS_F64, x, y0),
                               (F, P, A.PLUS_TIMES_F32, x32, y32), (F32, P32, A.PLUS_TIMES_F32, x32, y32),
                               (F, P, A.PLUS_PATTERN_F64, x, y0)):
        # kernel 4 folds each row in storage order whatever the default is
        for k in (c, p):
            k.set_kernel(4)
        assert c.form() == A.FORM_CONSTANT and p.form() in (A.FORM_SLICED, A.FORM_DIAGONAL)
        for a, b in zip(products(A, c, xv, yv, ring, mask), products(A, p, xv, yv, ring, mask)):
            assert np.array_equal(a, b, equal_nan=True), (w, n, ring)


@pytest.mark.parametrize("sides", [(4, 4, 4), (8, 8, 8), (65, 3, 5), (33, 17, 9), (64, 12, 10), (130, 20, 3)])
def test_const_stencil_takes_the_form(A, sides, monkeypatch):
    """27-point stencils, also where slices straddle lines and planes, hold fewer bytes
    than with values; products are the same bits through mxv and the transposed vxm."""
    C, P = both(A, monkeypatch, lambda: A.Matrix.stencil27(*sides, flags=A.MAT_WITH_CCS | A.MAT_WITH_F32))
    assert C.form(0) == C.form(1) == (A.FORM_CRS if sides == (4, 4, 4) else A.FORM_CONSTANT)  # padding of 4^3: 1.7
    if P.layout()[0]:
        assert C.device_bytes() < P.device_bytes()
        P.set_kernel(4)
        C.set_kernel(4)
    rng = np.random.default_rng(7)
    x = A.Vector.from_numpy(rng.standard_normal(C.nrows))
    for f in (lambda M, y: A.mxv(y, M, x), lambda M, y: A.vxm(y, x, M), lambda M, y: A.mxv(y, M, x, descr=A.TRANSPOSE_MATRIX)):
        got = []
        for M in (C, P):
            y = A.Vector(C.nrows, fill=0.5)
            assert f(M, y) == A.SUCCESS
            got.append(y.numpy())
        assert np.array_equal(got[0], got[1])


def in_runs(n, layout, f32):
    """Whether rows in runs of three with a value per entry take 27 values each: unless
    the slices stream much less."""
    slices, entries, diagonal = layout
    limit = (1.2 if f32 else 1.085) * (1 if diagonal else 2 if f32 else 1.5)
    return slices > 0 and 27 * n <= limit * entries


# boxes with fills from 1.03 to 1.7; (64, 12, 10) takes the form in FP32 alone
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("sides", [(4, 4, 4), (65, 3, 5), (33, 17, 13), (64, 12, 10), (130, 20, 3), (16, 16, 16),
                                   (17, 19, 23), (65, 13, 21)])
def test_run_values_equal_kept_values(A, sides, flip, monkeypatch):
    """27-point patterns with a value per entry take the template's offsets and keep their
    values slot by slot: the same bits as the sliced ELL's fold in every ring and mask
    mode, rows in descending and ascending order, with NaN and infinities in the matrix
    and in x (also where a row lacks the neighbour), and after a change of precision."""
    rng = np.random.default_rng(sum(sides))
    off, idx, _ = A.Matrix.stencil27(*sides).download(0)
    n = off.size - 1
    val = rng.standard_normal(idx.size)
    x, y0 = rng.standard_normal(n), rng.standard_normal(n)
    if flip:  # rows in ascending order
        order = np.concatenate([np.arange(int(off[r + 1]) - 1, int(off[r]) - 1, -1) for r in range(n)])
        idx, val = idx[order], val[order]
    else:
        val[rng.integers(0, val.size, 3)] = [np.nan, np.inf, -np.inf]
        x[rng.integers(0, n, 3)] = [np.nan, np.inf, -np.inf]
    mask = (rng.random(n) < 0.5).astype(np.uint8)
    F, P = both(A, monkeypatch, lambda: A.Matrix.from_crs(n, n, off, idx, val, flags=A.MAT_WITH_F32))
    F32, P32 = both(A, monkeypatch, lambda: A.Matrix.from_crs(n, n, off, idx, val.astype(np.float32)))
    x32, y32 = x.astype(np.float32), y0.astype(np.float32)
    for c, p, ring, xv, yv in ((F, P, A.PLUS_TIMES_F64, x, y0), (F, P, A.MIN_PLUS_F64, x, y0),
                               (F, P, A.PLUS_TIMES_F32, x32, y32), (F32, P32, A.PLUS_TIMES_F32, x32, y32),
                               (F, P, A.PLUS_PATTERN_F64, x, y0)):
        for k in (c, p):
            if k.layout()[0]:
                k.set_kernel(4)
        assert (c.form() == A.FORM_RUNS) == in_runs(n, c.layout(), c is F32)
        for a, b in zip(products(A, c, xv, yv, ring, mask), products(A, p, xv, yv, ring, mask)):
            assert np.array_equal(a, b, equal_nan=True), ring
    # the FP32 copy made by a mixed solve instead of at build time
    if not flip:
        return
    D = A.Matrix.from_crs(n, n, off, idx, val)
    b, s = A.Vector.from_numpy(y0), A.Vector(n, fill=0.0)
    A.cg(D, b, s, 1, 1e-10, 1)
    for a, b in zip(products(A, D, x32, y32, A.PLUS_TIMES_F32, mask), products(A, F, x32, y32, A.PLUS_TIMES_F32, mask)):
        assert np.array_equal(a, b)


# both sides of the lines between one row per lane and several (98304 rows with FP64
# sums, 524288 with FP32 ones), wider and narrower than long
@pytest.mark.parametrize("n,m,f32", [(257, 300, False), (98303, 98290, False), (98305, 98400, False),
                                     (524287, 524280, True), (524291, 524400, True)])
@pytest.mark.parametrize("uniform", [True, False])
def test_runs_at_each_row_count_per_lane(A, n, m, f32, uniform, monkeypatch):
    """Nine runs of three offsets, constant and with a value per entry, on non-square
    matrices: the bits of the kept values, also with NaN and infinities in x where a row
    lacks the neighbour."""
    rng = np.random.default_rng(n + uniform)
    up = (n + m) % 2 == 0
    base = np.array([-21, -17, -8, -4, 0, 4, 9, 13, 20])
    offs = (base[:, None] + np.arange(-1, 2)[None, :]).ravel()
    offs = offs if up else offs[::-1]
    drop = rng.random((n, 27)) < 0.02
    drop[n // 2] = False
    off, idx, val = banded(n, m, offs, rng.standard_normal(27), drop.ravel())
    if not uniform:
        val = rng.standard_normal(val.size)
    dt = np.float32 if f32 else np.float64
    x, y0 = rng.standard_normal(m).astype(dt), rng.standard_normal(n).astype(dt)
    x[rng.integers(0, m, 3)] = [np.nan, np.inf, -np.inf]
    x[0], x[m - 1] = np.nan, np.inf
    mask = (rng.random(n) < 0.5).astype(np.uint8)
    C, P = both(A, monkeypatch, lambda: A.Matrix.from_crs(n, m, off, idx, val.astype(dt)))
    C.set_kernel(4)
    P.set_kernel(4)
    assert C.form() == (A.FORM_CONSTANT if uniform else A.FORM_RUNS) and P.form() != C.form()
    ring = A.PLUS_TIMES_F32 if f32 else A.PLUS_TIMES_F64
    for a, b in zip(products(A, C, x, y0, ring, mask), products(A, P, x, y0, ring, mask)):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("sides", [(46, 46, 46), (48, 46, 46)])
@pytest.mark.parametrize("constant", [True, False])
def test_solves_at_each_row_count_per_lane(A, sides, constant, monkeypatch):
    """The product with its dot on both sides of 98304 rows: five iterations differ from
    those on kept values by the order of the dot's partial sums alone (a relative 2^-53
    or, in FP32 directions, 2^-24 per operation on systems of condition number below 1e3)."""
    n = int(np.prod(sides))
    rng = np.random.default_rng(n)
    theta = A.Vector.from_numpy(rng.uniform(0.5, 2.0, 13 * n))
    build = (lambda: A.Matrix.stencil27(*sides)) if constant else (lambda: A.Matrix.conductance27(*sides, theta, 1.0))
    C, P = both(A, monkeypatch, build)
    assert C.form() == (A.FORM_CONSTANT if constant else A.FORM_RUNS) and P.form() == A.FORM_DIAGONAL
    b = A.Vector.from_numpy(rng.standard_normal(n))
    for precision, bound in ((0, 1e3 * 2.0 ** -53), (1, 1e3 * 2.0 ** -24), (3, 1e3 * 2.0 ** -24)):
        got = []
        for M in (C, P):
            x = A.Vector(n, fill=0.0)
            A.cg(M, b, x, 5, 1e-300, precision)
            got.append(x.numpy())
        assert np.linalg.norm(got[0] - got[1]) <= bound * np.linalg.norm(got[1])


@pytest.mark.parametrize("part,f32,runs", [(1.0, False, True), (0.875, False, False), (0.875, True, True), (0.6, True, False)])
def test_sparse_domains_keep_their_slices(A, part, f32, runs):
    """27-point rows in the lower part of a box and identity rows above it: one list of 27
    offsets fits all, but rows above would stream 27 values for one."""
    s = 24
    off, idx, _ = A.Matrix.stencil27(s, s, s).download(0)
    n = off.size - 1
    row = np.repeat(np.arange(n), np.diff(off).astype(int))
    keep = (row < int(part * s) * s * s) | (idx == row)
    noff = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(row[keep], minlength=n), out=noff[1:])
    rng = np.random.default_rng(5)
    val = rng.standard_normal(int(keep.sum())).astype(np.float32 if f32 else np.float64)
    M = A.Matrix.from_crs(n, n, noff, idx[keep], val)
    assert in_runs(n, M.layout(), f32) == runs and M.form() == (A.FORM_RUNS if runs else A.FORM_DIAGONAL)
    assert M.device_bytes() <= 2.5 * (12 if not f32 else 8) * int(noff[-1]) + 100 * n


def test_const_near_misses_keep_their_values(A, monkeypatch):
    """One value off by an ulp, one row in another order, one column stored twice: not
    one template, so the bytes held and the results are those without the form."""
    rng = np.random.default_rng(3)
    n, offs = 2000, [-40, -1, 0, 1, 40]
    off, idx, val = banded(n, n, offs, [-1.0, -1.0, 4.0, -1.0, -1.0])
    x = rng.standard_normal(n)

    def variant(k):
        i, v = idx.copy(), val.copy()
        a = int(off[n // 2])
        if k == 0:
            v[a + 2] = np.nextafter(4.0, 5.0)
        elif k == 1:
            i[a], i[a + 1] = i[a + 1], i[a]
        else:
            i[a + 1] = i[a]
        return A.Matrix.from_crs(n, n, off, i, v)

    for k in range(3):
        C, P = both(A, monkeypatch, lambda: variant(k))
        assert C.form() == P.form() != A.FORM_CONSTANT
        assert C.device_bytes() == P.device_bytes(), k
        got = []
        for M in (C, P):
            M.set_kernel(4)
            y = A.Vector(n, fill=0.0)
            assert A.mxv(y, M, A.Vector.from_numpy(x)) == A.SUCCESS
            got.append(y.numpy())
        assert np.array_equal(got[0], got[1]), k


@pytest.mark.parametrize("sizes,levels,pre,post,const", [
    ((16, 16, 16), 2, 1, 1, 3), ((24, 16, 40), 1, 2, 2, 2), ((12, 20, 28), 1, 1, 1, 2),
    ((32, 16, 16), 2, 0, 1, 3), ((16, 32, 16), 2, 1, 0, 3), ((8, 12, 10), 0, 1, 1, 1),
    # a coarsest level of one workgroup's most rows, and of more
    ((16, 16, 28), 0, 1, 1, 1), ((16, 18, 26), 0, 1, 1, 1),
    ((4, 4, 4), 1, 1, 1, 1),  # 2^3 has no inner row
    ((9, 11, 7), 0, 1, 1, 0)])
def test_const_hpcg_equals_kept_values(A, sizes, levels, pre, post, const, monkeypatch):
    """V-cycle and solves on levels in constant form (whose steps on one colour, and
    transfers, run in one launch) equal the sliced layouts' bit for bit; odd sides
    (whose colours do not share offsets) keep those layouts."""
    C, P = both(A, monkeypatch, lambda: A.Hpcg(*sizes, max_levels=levels, colours=0, presmooth=pre, postsmooth=post))
    assert (C.constant_levels(), P.constant_levels()) == (const, 0)
    rng = np.random.default_rng(11)
    r = A.Vector.from_numpy(rng.standard_normal(C.n))
    z = [A.Vector(C.n, fill=0.0) for _ in range(2)]
    C.vcycle(r, z[0])
    P.vcycle(r, z[1])
    assert np.array_equal(z[0].numpy(), z[1].numpy())
    for precision in (0, 1, 2, 3):
        got = []
        for H in (C, P):
            x = A.Vector(C.n, fill=0.0)
            got.append((H.solve(r, x, 60, 1e-9, precision), x.numpy()))
        assert got[0][0] == got[1][0], precision
        assert np.array_equal(got[0][1], got[1][1]), precision
