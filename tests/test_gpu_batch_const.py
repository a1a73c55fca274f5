"""Batches whose systems each have one (offset, value) template, against the products
over CRS (ALP_HIP_BATCH_DIA=0) bit for bit and an FP64 CPU product: every number of
right-hand sides, systems from one row up, wide templates, empty rows, and systems that
break the form by one value, one column or one entry too many."""
import numpy as np
import pytest

from test_gpu_batch import A  # noqa: F401

pytestmark = pytest.mark.gpu


def banded(n, offsets, rng, drop=0.3):
    """Rows of one template with random entries missing; the diagonal stays, and the middle
    row has the whole template."""
    off, idx, val = [0], [], []
    values = rng.uniform(0.1, 1.0, len(offsets)) * rng.choice([-1, 1], len(offsets))
    for r in range(n):
        for d, v in zip(offsets, values):
            if 0 <= r + d < n and (d == 0 or r == n // 2 or rng.random() > drop):
                idx.append(r + d)
                val.append(v if d else 40.0)
        off.append(len(idx))
    return np.array(off, np.uint64), np.array(idx, np.uint32), np.array(val)


def break_one(system, how, rng):
    off, idx, val = (a.copy() for a in system)
    if how == "value":
        val[val.size // 2] *= 1.5
    elif how == "column":
        r = int(off.size) // 2
        k = int(off[r])
        idx[k] = (idx[k] + 2) % (off.size - 1)
    return off, idx, val


@pytest.mark.parametrize("nrhs", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("breaks", ["none", "value", "column"])
def test_products_and_solves_equal_crs(A, monkeypatch, nrhs, breaks):  # noqa: F811
    rng = np.random.default_rng(nrhs)
    wide = sorted(set(rng.integers(-60, 61, 34).tolist()) | {0})[:32]
    if 0 not in wide:
        wide = sorted(wide[:31] + [0])
    systems = [banded(1, [0], rng), banded(700, [-20, -1, 0, 1, 20], rng), banded(257, wide, rng),
               banded(63, [-7, 0, 7], rng, 0.0), banded(256, [0], rng), banded(713, [-300, -1, 0, 1, 300], rng)]
    if breaks != "none":
        systems[1] = break_one(systems[1], breaks, rng)
    C = A.Batch.from_crs(systems, nrhs)
    monkeypatch.setenv("ALP_HIP_BATCH_DIA", "0")
    P = A.Batch.from_crs(systems, nrhs)
    monkeypatch.delenv("ALP_HIP_BATCH_DIA")
    assert (C.constant(), P.constant()) == (breaks == "none", False)
    x = rng.standard_normal((C.nrows, nrhs))
    X = A.Vector.from_numpy(x.ravel())
    Yc, Yp = A.Vector(C.nrows * nrhs), A.Vector(C.nrows * nrhs)
    C.spmm(X, Yc)
    P.spmm(X, Yp)
    assert np.array_equal(Yc.numpy(), Yp.numpy())
    got = Yc.numpy().reshape(C.nrows, nrhs)
    for s, (off, idx, val) in enumerate(systems):
        r0 = int(C.row0[s])
        for r in range(off.size - 1):
            k = slice(int(off[r]), int(off[r + 1]))
            want = val[k] @ x[r0 + idx[k].astype(int)]
            size = np.abs(val[k]) @ np.abs(x[r0 + idx[k].astype(int)])
            # at most 32 products and sums, each within 2^-53 of its terms' size
            assert np.all(np.abs(got[r0 + r] - want) <= 33 * 2.0 ** -53 * size)
    for precision in (0, 1, 2):
        Sc, Sp = A.Vector(C.nrows * nrhs, fill=0.0), A.Vector(C.nrows * nrhs, fill=0.0)
        ic, ip = C.solve(X, Sc, 1e-6, 7, precision)[1], P.solve(X, Sp, 1e-6, 7, precision)[1]
        assert np.array_equal(ic, ip)
        assert np.array_equal(Sc.numpy(), Sp.numpy(), equal_nan=True)


def test_infinities_reach_only_their_rows(A):  # noqa: F811
    """An infinity or NaN in one system's X reaches the rows that store its column, and
    no neighbouring system."""
    rng = np.random.default_rng(5)
    systems = [banded(130, [-9, -1, 0, 1, 9], rng) for _ in range(3)]
    B = A.Batch.from_crs(systems, 8)
    assert B.constant()
    x = rng.standard_normal((B.nrows, 8))
    x[130, 2] = np.inf
    x[259, 5] = np.nan
    Y = A.Vector(B.nrows * 8)
    B.spmm(A.Vector.from_numpy(x.ravel()), Y)
    bad = ~np.isfinite(Y.numpy().reshape(-1, 8))
    want = np.zeros_like(bad)
    off, idx, _ = systems[1]
    for r in range(130):
        cols = idx[int(off[r]):int(off[r + 1])]
        want[130 + r, 2] = 0 in cols
        want[130 + r, 5] = 129 in cols
    assert np.array_equal(bad, want)


def test_no_memory_for_the_form(A, monkeypatch):  # noqa: F811
    """Without memory for the templates and masks a batch keeps its other forms."""
    rng = np.random.default_rng(9)
    systems = [banded(300, [-17, -1, 0, 1, 17], rng, 0.1), banded(190, [-3, 0, 3], rng, 0.1)]
    C = A.Batch.from_crs(systems, 4)
    monkeypatch.setenv("ALP_HIP_OPTIONAL_BYTES", "0")
    P = A.Batch.from_crs(systems, 4)
    monkeypatch.delenv("ALP_HIP_OPTIONAL_BYTES")
    assert (C.constant(), P.constant()) == (True, False)
    x = A.Vector.from_numpy(rng.standard_normal(C.nrows * 4))
    got = []
    for B in (C, P):
        y = A.Vector(B.nrows * 4)
        B.spmm(x, y)
        got.append(y.numpy())
    assert np.array_equal(got[0], got[1])
