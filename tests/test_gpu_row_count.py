"""The counting form of the sketch (64 items at a time while a row needs no
eviction) at its edges, tables bit for bit against the oracle: candidates that
occur more often than a count's bits allow, tables filled to their last free
entries, capacities past a table's entries, rows that begin with nearly only
new candidates, each on the chunk tiers and on both forms of the global path."""

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


def twins(n, shared, seed):
    """Three rows holding the same `shared` columns (each pair meets `shared`
    times) and one of every eighth row a few columns of them."""
    rng = np.random.default_rng(seed)
    cols = rng.choice(n, shared, replace=False)
    rows = {r: cols for r in (1, 5, 130)}
    for r in range(8, n, 8):
        rows[r] = rng.choice(cols, rng.integers(1, 6), replace=False)
    return csr(n, rows)


def groups(n, distinct, per_row, seed):
    """Blocks of `distinct` + 1 rows drawing `per_row` of 40 columns of their
    own: rows of about `distinct` candidates, each met several times."""
    rng = np.random.default_rng(seed)
    rows = {}
    for r in range(n):
        b = r // (distinct + 1)
        own = (b * 40 + np.arange(40)) % n
        rows[r] = rng.choice(own, per_row, replace=False)
    return csr(n, rows)


def repeats(n, seed):
    """Rows that hold one column 300 times: 90,000 meetings of a pair."""
    rng = np.random.default_rng(seed)
    rows = {r: rng.choice(n, 9, replace=False) for r in range(0, n, 3)}
    for r in (3, 6, 300):
        rows[r] = np.concatenate([rows[r], np.full(300, 77)])
    return csr(n, rows)


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
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("k,ovs", [(16, 2.0), (16, 4.0), (32, 4.0), (80, 4.0)])
@pytest.mark.parametrize("chunk", [256, 1024, 3000, 5000])
def test_counted_rows(name, k, ovs, chunk):
    from chunkedgreedy_amd import sporder

    ptr, ind = CASES[name]()
    print(f"[row_count] {name} k={k} ovs={ovs} chunk={chunk}", flush=True)
    want_i, want_w = oracle.unpack_table(
        oracle.chunk_similarity_top_k(ptr, ind, k, chunk, ovs, is_symmetric=False))
    gi, gw = sporder.chunk_similarity_top_k(
        torch.from_numpy(ptr).to("cuda:0"), torch.from_numpy(ind).to("cuda:0"), k=k,
        oversampling=ovs, chunk_size=chunk)
    assert np.array_equal(gi.cpu().numpy(), want_i)
    assert np.array_equal(gw.cpu().numpy().view(np.uint32), want_w.view(np.uint32))
