"""CSR-stream on skewed rows: rows longer than a thread group folds go to a list that
whole wavefronts take. Whole-number data makes every fold order exact, so each variant
must equal the brute force in every ring and mask mode."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import alp_amd
    alp_amd.init(0)
    return alp_amd


def rows_of(lengths, ncols, rng):
    off = np.zeros(len(lengths) + 1, np.uint64)
    np.cumsum(lengths, out=off[1:])
    idx = np.concatenate([rng.choice(ncols, n, replace=False) for n in lengths] + [np.zeros(0, np.int64)])
    return off, idx.astype(np.uint32)


# lengths around the wavefront limit of one, two and four threads per row, around a
# wavefront's and the fold's steps, around a tile (2048, 4096) and past the chunk limit
LENGTHS = {
    "limits": [0, 1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 0, 511, 513] * 9,
    "one_per_tile": ([3] * 240 + [1300]) * 3 + [2, 0, 1],
    "tile_edges": [5] * 100 + [2047, 2048, 2049, 4095, 4096, 4097] + [1] * 30 + [5000],
    "many": [40] * 700 + [7] * 500,
}


@pytest.mark.parametrize("tile", [8, 16])
@pytest.mark.parametrize("variant", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_skewed_rows_exact(A, name, variant, tile):
    rng = np.random.default_rng(len(name) + variant)
    lengths, ncols = LENGTHS[name], 6000
    n = len(lengths)
    off, idx = rows_of(lengths, ncols, rng)
    val = rng.integers(-9, 10, idx.size).astype(np.float64)
    x, y0 = rng.integers(-9, 10, ncols).astype(np.float64), rng.integers(-9, 10, n).astype(np.float64)
    mask = (rng.random(n) < 0.6).astype(np.uint8)
    row = np.repeat(np.arange(n), lengths)
    prod = np.bincount(row, val * x[idx], minlength=n)
    low = np.full(n, np.inf)
    np.minimum.at(low, row, val + x[idx])
    empty = np.asarray(lengths) == 0
    bx = (rng.random(ncols) < 0.002).astype(np.uint8)
    lor = np.zeros(n, np.uint8)
    np.maximum.at(lor, row, bx[idx])
    M = A.Matrix.from_crs(n, ncols, off, idx, val)
    M32 = A.Matrix.from_crs(n, ncols, off, idx, val.astype(np.float32))
    for mat, ring, xv, yv, fresh, folded in (
            (M, A.PLUS_TIMES_F64, x, y0, prod, y0 + prod), (M, A.MIN_PLUS_F64, x, y0, low, np.minimum(y0, low)),
            (M32, A.PLUS_TIMES_F32, x.astype(np.float32), y0.astype(np.float32), prod, y0 + prod),
            (M, A.LOR_LAND_BOOL, bx, (y0 > 0).astype(np.uint8), lor, np.maximum(lor, y0 > 0))):
        mat.set_kernel(2, tile, variant)
        for descr, mk in ((0, None), (A.OVERWRITE, None), (0, mask), (A.INVERT_MASK, mask)):
            y = A.Vector.from_numpy(yv)
            assert A.mxv(y, mat, A.Vector.from_numpy(xv), ring=ring, descr=descr,
                         mask=None if mk is None else A.Vector.from_numpy(mk)) == A.SUCCESS
            want = fresh if descr == A.OVERWRITE else np.where(empty, yv, folded)
            if mk is not None:
                want = np.where((mk != 0) != bool(descr & A.INVERT_MASK), want, yv)
            assert np.array_equal(y.numpy().astype(np.float64), want.astype(np.float64)), (ring, descr)


@pytest.mark.parametrize("rows,mean,sigma", [(30011, 40, 0.2), (30011, 40, 1.2), (9001, 20, 0.0)])
def test_default_kernel_of_unstructured_matrices(A, rows, mean, sigma):
    """The default choice on both sides of its nonzero count, plain and transposed."""
    rng = np.random.default_rng(rows + mean)
    lengths = np.clip(np.round(mean * np.exp(sigma * rng.standard_normal(rows))), 1, 3000).astype(np.int64)
    off, idx = rows_of(lengths, rows, rng)
    val = rng.integers(-9, 10, idx.size).astype(np.float64)
    x = rng.integers(-9, 10, rows).astype(np.float64)
    M = A.Matrix.from_crs(rows, rows, off, idx, val, flags=A.MAT_WITH_CCS)
    row = np.repeat(np.arange(rows), lengths)
    y, z = A.Vector(rows, fill=1.0), A.Vector(rows, fill=1.0)
    assert A.mxv(y, M, A.Vector.from_numpy(x)) == A.SUCCESS
    assert A.vxm(z, A.Vector.from_numpy(x), M) == A.SUCCESS
    assert np.array_equal(y.numpy(), 1.0 + np.bincount(row, val * x[idx], minlength=rows))
    assert np.array_equal(z.numpy(), 1.0 + np.bincount(idx, val * x[row], minlength=rows))


@pytest.mark.parametrize("sigma", [0.2, 1.4])
def test_masked_products_read_the_rows_of_the_mask(A, sigma):
    """Above the nonzero count from which row segments are the default, a masked product
    on evenly long rows runs on CSR-vector, which reads the mask's rows alone: the bits of
    that kernel's fold. Skewed rows keep row segments, masked or not."""
    rng = np.random.default_rng(17)
    rows = 60011
    lengths = np.clip(np.round(20 * np.exp(sigma * rng.standard_normal(rows))), 1, 3000).astype(np.int64)
    off = np.zeros(rows + 1, np.uint64)
    np.cumsum(lengths, out=off[1:])
    idx = rng.integers(0, rows, int(off[-1])).astype(np.uint32)
    M = A.Matrix.from_crs(rows, rows, off, idx, rng.standard_normal(idx.size))
    x, y0 = A.Vector.from_numpy(rng.standard_normal(rows)), rng.standard_normal(rows)
    assert M.get_kernel()[::2] == (2, 64)
    for mask in (None, (rng.random(rows) < 0.02).astype(np.uint8)):
        got = {}
        for kernel in ((0, 0, 0), (1, 0, 0), (2, 0, 64)):
            M.set_kernel(*kernel)
            y = A.Vector.from_numpy(y0)
            assert A.mxv(y, M, x, mask=None if mask is None else A.Vector.from_numpy(mask)) == A.SUCCESS
            got[kernel[0]] = y.numpy()
        assert not np.array_equal(got[1], got[2])
        assert np.array_equal(got[0], got[1 if mask is not None and sigma < 1 else 2])
