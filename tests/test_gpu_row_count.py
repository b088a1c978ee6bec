"""The counting form of the sketch (64 items at a time while a row needs no
eviction) at its edges, tables bit for bit against the oracle: candidates that
occur more often than a count's bits allow, tables filled to their last free
entries, capacities past a table's entries, rows that begin with nearly only
new candidates, on both chunk tiers and on both forms of the global path (the
chunk sizes say which: PATHS); and rows of as many entries as the ways to put
out a row's list meet at, counted and not."""

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def csr(n, rows):
    """CSR of {row: columns}."""
    lens = np.zeros(n, np.int64)
    for r, c in rows.items():
        lens[r] = len(c)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    ind = np.concatenate([np.sort(rows[r]) for r in sorted(rows)]) if rows else np.zeros(0)
    return ptr.astype(np.int32), ind.astype(np.int32)


def band(n, width=9):
    """Rows of the `width` columns from their own on: neighbours share all but
    one, so the matrix is counted."""
    return {r: (r + np.arange(width)) % n for r in range(n)}


def twins(n, shared, seed):
    """Three rows holding the same `shared` columns (each pair meets `shared`
    times) and one of every eighth row a few columns of them, in a band."""
    rng = np.random.default_rng(seed)
    cols = rng.choice(n, shared, replace=False)
    rows = band(n)
    rows.update({r: cols for r in (1, 5, 130)})
    for r in range(8, n, 8):
        rows[r] = np.union1d(rows[r], rng.choice(cols, rng.integers(1, 6), replace=False))
    return csr(n, rows)


def groups(n, distinct, per_row, seed, scatter=False):
    """Blocks of `distinct` + 1 rows drawing `per_row` of 40 columns of their
    own: rows of about `distinct` candidates (exactly, with more than 20 of 40),
    each met several times.  scatter: the rows of each 1024 in random order, so
    that neighbours share few columns and nothing is counted."""
    rng = np.random.default_rng(seed)
    rows = {}
    at = np.arange(n)
    if scatter:
        for c in range(0, n, 1024):
            at[c:c + 1024] = rng.permutation(at[c:c + 1024])
    for r in range(n):
        b = r // (distinct + 1)
        own = (b * 40 + np.arange(40)) % n
        rows[int(at[r])] = rng.choice(own, per_row, replace=False)
    return csr(n, rows)


def repeats(n, seed):
    """Rows that hold one column 300 times (90,000 meetings of a pair), in a
    band with some random columns."""
    rng = np.random.default_rng(seed)
    rows = band(n)
    for r in range(0, n, 3):
        rows[r] = np.union1d(rows[r], rng.choice(n, 3, replace=False))
    for r in (3, 6, 300):
        rows[r] = np.concatenate([rows[r], np.full(300, 77)])
    return csr(n, rows)


def is_counted(ptr, ind):
    """The classification's sample: of the first 16 nonzeros of 64 rows, an
    eighth or more are among the first 16 of the row after."""
    n = ptr.size - 1
    shared = seen = 0
    for place in range(64):
        r = (2 * place + 1) * (n - 1) // 128
        mine = ind[ptr[r]:ptr[r + 1]][:16]
        shared += np.isin(mine, ind[ptr[r + 1]:ptr[r + 2]][:16]).sum()
        seen += mine.size
    return 8 * shared >= seen


def path(ptr, chunk):
    """Where the first chunk of a matrix that is not symmetric is sketched."""
    rows = min(chunk, ptr.size - 1)
    nnz = int(ptr[rows])
    if chunk > 4096:
        return "wide"
    if chunk <= 1024 and nnz <= 16384:
        return "tier 1"
    return "tier 2" if nnz <= 32768 else "narrow"


# Where the chunk sizes put the first chunk, which holds the rows that matter.
PATHS = {256: "tier 1", 1024: "tier 1", 3000: "tier 2", 4096: "narrow", 5000: "wide"}


CASES = {
    "repeats": lambda: repeats(5000, 8),
    # counts of 880 and 1500: below and past what ten bits take with a batch to go
    "twins880": lambda: twins(5000, 880, 1),
    "twins1500": lambda: twins(5000, 1500, 2),
    # 60 and 64 candidates (capacity 64), 100 and 119..122 (tier 1's table ends at 119)
    "groups60": lambda: groups(4500, 60, 12, 3),
    "groups64": lambda: groups(4500, 64, 12, 4),
    "groups100": lambda: groups(4500, 100, 10, 5),
    "groups120": lambda: groups(4500, 120, 10, 6),
    "groups127": lambda: groups(4500, 127, 12, 7),
    # chunks of 1024 rows past tier 1's nonzeros
    "groups90_long": lambda: groups(4500, 90, 24, 9),
    "groups127_long": lambda: groups(4500, 127, 36, 10),
    # up to 4 entries are merged, up to 128 sorted (past four cells)
    "groups4": lambda: groups(3100, 4, 21, 11),
    "groups5": lambda: groups(3100, 5, 21, 12),
    "groups128": lambda: groups(3100, 128, 21, 13),
    "groups129": lambda: groups(3100, 129, 21, 14),
    "scattered4": lambda: groups(3100, 4, 21, 15, scatter=True),
    "scattered5": lambda: groups(3100, 5, 21, 16, scatter=True),
    "scattered128": lambda: groups(3100, 128, 21, 17, scatter=True),
    "scattered129": lambda: groups(3100, 129, 21, 18, scatter=True),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("k,ovs", [(16, 2.0), (16, 4.0), (32, 4.0), (80, 4.0)])
@pytest.mark.parametrize("chunk", sorted(PATHS))
def test_counted_rows(name, k, ovs, chunk):
    from chunkedgreedy_amd import sporder

    ptr, ind = CASES[name]()
    assert is_counted(ptr, ind) == (not name.startswith("scattered"))
    if name in ("repeats", "twins880", "twins1500"):
        assert path(ptr, chunk) == PATHS[chunk]
    print(f"[row_count] {name} k={k} ovs={ovs} chunk={chunk}", flush=True)
    want_i, want_w = oracle.unpack_table(
        oracle.chunk_similarity_top_k(ptr, ind, k, chunk, ovs, is_symmetric=False))
    gi, gw = sporder.chunk_similarity_top_k(
        torch.from_numpy(ptr).to("cuda:0"), torch.from_numpy(ind).to("cuda:0"), k=k,
        oversampling=ovs, chunk_size=chunk)
    assert np.array_equal(gi.cpu().numpy(), want_i)
    assert np.array_equal(gw.cpu().numpy().view(np.uint32), want_w.view(np.uint32))
