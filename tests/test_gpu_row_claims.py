"""Rows of the global sketch are claimed one at a time: tables of more rows
than the device has waves, bit for bit against the oracle, and neighbouring
long rows that run beside each other."""

import time

import numpy as np
import pytest
import torch

import oracle
from chunkedgreedy_amd import synth

pytestmark = pytest.mark.gpu


def on_gpu(ptr, ind):
    return [torch.from_numpy(np.ascontiguousarray(a, np.int32)).to("cuda:0") for a in (ptr, ind)]


# One chunk of 2^17 + 1 and of 150,001 rows (several runs of rows per counter, a
# last run that is cut), rows fewer than one run per counter, and listed chunks.
@pytest.mark.parametrize("n,chunk", [(131_073, 131_073), (150_001, 150_001), (100, 100),
                                     (17, 17), (60_001, 5_000)])
def test_claimed_rows(sporder, n, chunk):
    print(f"[row_claims] n={n} chunk={chunk}", flush=True)
    ptr, ind = synth.band(n, 2)[:2]
    want_i, want_w = oracle.unpack_table(
        oracle.chunk_similarity_top_k(ptr, ind, 16, chunk, 2.0, is_symmetric=True))
    gi, gw = sporder.chunk_similarity_top_k(*on_gpu(ptr, ind), k=16, oversampling=2.0,
                                            chunk_size=chunk, is_symmetric=True)
    assert np.array_equal(gi.cpu().numpy(), want_i)
    assert np.array_equal(gw.cpu().numpy().view(np.uint32), want_w.view(np.uint32))


def long_rows(n, at, seed=3):
    """n rows of 4 nonzeros; the rows `at` hold 20,000 more."""
    rng = np.random.default_rng(seed)
    rows = np.concatenate([np.repeat(np.arange(n), 4), np.repeat(at, 20_000)])
    keys = np.unique(rows * n + rng.integers(0, n, rows.size))
    ptr = np.concatenate([[0], np.cumsum(np.bincount(keys // n, minlength=n))])
    return ptr, keys % n


def test_neighbouring_long_rows(sporder):
    """16 long rows (some 100,000 items each, one after the other in their
    wave) at the front and spread over 300,000 rows: the same work, and each
    long row in a wave of its own.  Two of them in one wave would double the
    time that the longest takes."""
    n = 300_000
    took = {}
    for name, at in (("spread", np.arange(16) * (n // 16) + 5), ("front", np.arange(16))):
        ptr, ind = on_gpu(*long_rows(n, at))
        times = []
        for _ in range(5):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            sporder.chunk_greedy(ptr, ind, is_symmetric=False, k=16, oversampling=2.0)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        took[name] = min(times)
        print(f"[row_claims] long rows {name}: {took[name] * 1e3:.2f} ms", flush=True)
    assert took["front"] < 1.5 * took["spread"]
