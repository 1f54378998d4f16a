"""The sliced layouts of a matrix's FP64 and FP32 copies, worked out on the
host: every copy is stored with the steps its slices read, whichever way the
two plans are cut (the finest FP64 matrix of an aggressive hierarchy by row
block, the FP32 copy every 64 rows), and no copy stores more than its bound.
No device call is made here."""
import numpy as np
import pytest

from fem_amd import lina


def rows_with(lengths, seed=0):
    """CSR with the given row lengths (the diagonal and random columns)"""
    rng = np.random.default_rng(seed)
    n = len(lengths)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.empty(rp[-1], np.int32)
    for m in np.unique(lengths):
        rows = np.flatnonzero(lengths == m)
        start = rng.integers(0, n, len(rows))
        step = n // m
        c = np.sort((start[:, None] + step * np.arange(m)) % n, axis=1)
        col[(rp[rows][:, None] + np.arange(m)).ravel()] = c.ravel()
    return rp, col


def check_layout(rp, heads, lanes, steps):
    n, m = len(rp) - 1, np.diff(rp)
    if len(heads) == 0:
        return
    row0, row1, step0, count = heads.T.astype(np.int64)
    assert row0[0] == 0 and row1[-1] == n and np.all(row0[1:] == row1[:-1]) and np.all(row1 - row0 <= 64 // lanes)
    # an access is 64 (step0 + j) + lane, j < count: within the stored steps
    assert np.all(step0 >= 0) and np.all(step0 + count <= steps)
    assert np.all(step0[1:] == step0[:-1] + count[:-1]) and step0[-1] + count[-1] == steps
    real = row1 > row0  # a block's spare slices hold no rows
    assert np.all(np.maximum.reduceat(m, row0[real]) <= lanes * count[real])


def lengths_of(kind, seed):
    """blocks of up to 256 rows, a few of them shorter: as many slices by block
    (four a block) as by 64 rows, of other rows"""
    rng = np.random.default_rng(seed)
    if kind == "short":  # row blocks of 256 entries: 256 one-entry rows
        m = np.ones(256 * 24 - 30, np.int64)
        m[rng.integers(0, 4000, 6)] = rng.integers(2, 6, 6)
    elif kind == "patch":  # denser rows across what would be a slice's end
        m = np.ones(256 * 20 - 50, np.int64)
        first = 256 * rng.integers(1, 8) + rng.integers(50, 64)
        m[first:first + 12] = 4
    else:  # P1 mesh rows in blocks of 2,048 entries, two patches of longer rows
        m = np.full(256 * 2500 - 63, 7)
        for first in rng.integers(0, 400_000, 2):
            m[first - first % 256 + 100:first - first % 256 + 120] = 21
    return m


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("kind", ["short", "patch", "mesh"])
def test_copies_of_a_finest_matrix_are_stored_as_they_are_read(kind, seed):
    m = lengths_of(kind, seed)
    rp, ci = rows_with(m, seed)
    cut = []
    for precision in ("fp64", "mixed"):
        heads, lanes, steps = lina.slice_layout(rp, ci, free32=False, partials=True, precision=precision)
        assert lanes == 1 and len(heads) > 0
        check_layout(rp, heads, lanes, steps)
        cut.append(heads)
    # the FP64 copy is cut by row block here, some blocks shorter than 256 rows,
    # and the FP32 copy every 64 rows
    assert np.diff(cut[0][::4, 0]).min() < 256 and np.all(np.diff(cut[1][:, 0]) == 64)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1000])
@pytest.mark.parametrize("mean", [1, 7, 24, 25, 60, 200])
@pytest.mark.parametrize("free32,partials", [(True, True), (True, False), (False, True), (False, False)])
def test_layouts_over_row_counts_and_lengths(n, mean, free32, partials):
    rng = np.random.default_rng(31 * n + mean)
    m = np.clip(rng.integers((mean + 1) // 2, mean + 2, n), 1, n)
    rp, ci = rows_with(m, n)
    for precision in ("fp64", "mixed"):
        check_layout(rp, *lina.slice_layout(rp, ci, free32, partials, precision))


@pytest.mark.parametrize("free32", [True, False])
@pytest.mark.parametrize("clique,sliced", [(8, True), (700, False)])
def test_small_colours_of_long_rows_do_not_fill_memory(clique, sliced, free32):
    """a clique's rows have a colour each: a slice of one row stores 64 / lanes
    times the row"""
    n = 200_000
    m = np.full(n, 7)
    m[:clique] = clique
    rp, ci = rows_with(m, clique)
    colours = np.arange(n) % 4
    colours[:clique] = np.arange(clique)
    for precision in ("fp64", "mixed"):
        heads, lanes, steps = lina.slice_layout(rp, ci, free32, precision=precision, colours=colours)
        assert (len(heads) > 0) == sliced
        assert 64 * steps <= 4 * len(ci) + 2 ** 20
        check_layout(np.append(0, np.cumsum(m[np.argsort(colours, kind="stable")])), heads, lanes, steps)


@pytest.mark.parametrize("n,mean,longest,sliced", [
    (1200, 90, 90, True), (1200, 90, 800, False), (8000, 80, 3200, False), (9400, 104, 1000, True),
    (40_000, 7, 40, True), (40_000, 7, 300, False), (3000, 16, 16, True)])
def test_a_few_long_rows_take_row_blocks(n, mean, longest, sliced):
    """a slice runs its longest row's steps one after another"""
    m = np.full(n, mean)
    m[n // 3] = longest
    rp, ci = rows_with(m, n)
    for precision in ("fp64", "mixed"):
        assert (len(lina.slice_layout(rp, ci, precision=precision)[0]) > 0) == sliced


@pytest.mark.parametrize("n,mean,sliced64", [(70_000, 95, False), (18_000, 95, True), (120_000, 53, True)])
def test_large_fp64_matrices_of_long_rows_take_row_blocks(n, mean, sliced64):
    rp, ci = rows_with(np.full(n, mean), n)
    assert (len(lina.slice_layout(rp, ci, precision="fp64")[0]) > 0) == sliced64
    assert len(lina.slice_layout(rp, ci, precision="mixed")[0]) > 0


@pytest.mark.parametrize("n,sliced", [(100_000, True), (1_000_000, False)])
def test_large_padding_takes_row_blocks(n, sliced):
    """prolongation-like rows of 2 to 8 entries: 1.6 entries read for one"""
    m = np.random.default_rng(n).integers(2, 9, n)
    rp, ci = rows_with(m, 1)
    for precision in ("fp64", "mixed"):
        heads, lanes, _ = lina.slice_layout(rp, ci, precision=precision)
        assert (len(heads) > 0) == sliced
