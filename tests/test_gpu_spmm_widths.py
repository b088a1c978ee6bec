"""The SpMM at widths that are not a multiple of 4 and on operands that start
4, 8 or 12 bytes past a 16-byte boundary, bit for bit against the oracle, with
guard words around the result: the last lane of a row moves back to columns
N-4..N-1, rows narrower than 4 take a lane per column."""

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"
N_ROWS = 1111


def from_lengths(n, lens, seed):
    """Rows of the given lengths, columns drawn with repetition when a row is
    longer than n."""
    rng = np.random.default_rng(seed)
    ind = np.concatenate([np.sort(rng.choice(n, k, replace=k > n)) for k in lens])
    ptr = np.concatenate([[0], np.cumsum(lens)])
    val = rng.uniform(-1, 1, ind.size).astype(np.float32)
    return ptr.astype(np.int32), ind.astype(np.int32), val


def mixed(n, most, seed=21):
    """Rows of 0..most nonzeros, and five around and past the 512-nonzero
    segments (511, 512, 513, 1025, 1100)."""
    lens = np.random.default_rng(seed).integers(0, most + 1, n)
    lens[[5, 64, 300, 777, n - 1]] = [511, 512, 513, 1025, 1100]
    lens[[0, 63, 128]] = 0
    return from_lengths(n, lens, seed)


def mostly_long():
    """Neighbouring rows past a segment, and rows of 20,000 and 70,000
    nonzeros: more segments than a workgroup has row groups."""
    rng = np.random.default_rng(22)
    lens = rng.integers(0, 30, 700)
    lens[200:300] = rng.integers(500, 1400, 100)
    lens[[3, 250]] = [20_000, 70_000]
    return from_lengths(700, lens, 22)


def many_rows():
    """2^19 and some rows of 0..4 nonzeros, and the long rows of `mixed`."""
    n = (1 << 19) + 77
    lens = np.random.default_rng(23).integers(0, 5, n)
    lens[[5, 64, 300, 777, n - 1]] = [511, 512, 513, 1025, 1100]
    rows = np.repeat(np.arange(n), lens)
    rng = np.random.default_rng(24)
    ind = rng.integers(0, n, rows.size)
    ind = ind[np.lexsort((ind, rows))]
    return (np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), ind.astype(np.int32),
            rng.uniform(-1, 1, ind.size).astype(np.float32))


# One launch (ragged widths up to 2^19 nonzeros, 2^18 past 128 columns), the
# launches of a larger matrix, and one launch with more segments than groups.
MATRICES = {"small": lambda: mixed(N_ROWS, 80), "large": lambda: mixed(4 * N_ROWS, 260),
            "long": mostly_long}


@pytest.fixture(scope="module", params=sorted(MATRICES))
def matrix(request):
    m = MATRICES[request.param]()
    assert (m[1].size > 1 << 19) == (request.param == "large")
    assert m[1].size > 1 << 19 or m[1].size <= 1 << 18
    return m


@pytest.fixture(scope="module")
def rows_to_claim():
    """More rows than have a group of their own: claimed up to 32 columns."""
    return many_rows()


def shifted(a, words):
    """(buffer, view): a copy of `a` on the GPU that starts `words` floats
    after an aligned start, 16 words of -7 on both sides."""
    buf = torch.full((a.size + 32 + words,), -7.0, device=DEV)
    view = buf[16 + words:16 + words + a.size].view(a.shape)
    view.copy_(torch.from_numpy(a))
    return buf, view


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 7, 13, 16, 17, 31, 33, 47, 64, 67, 127, 130, 259])
@pytest.mark.parametrize("words", [0, 1, 2, 3])
def test_spmm_widths_and_alignments(matrix, N, words):
    check_all_calls(matrix, N, words)


@pytest.mark.parametrize("N,words", [(1, 0), (2, 3), (3, 1), (4, 1), (5, 0), (7, 2), (13, 0),
                                     (16, 3), (31, 0), (32, 2)])
def test_spmm_claimed_rows(rows_to_claim, N, words):
    check_all_calls(rows_to_claim, N, words)


def check_all_calls(matrix, N, words):
    from chunkedgreedy_amd import sporder

    ptr, ind, val = matrix
    rng = np.random.default_rng(N)
    n = ptr.size - 1
    Bh = rng.standard_normal((n, N)).astype(np.float32)
    rs, cs = (rng.uniform(0.05, 2.0, n).astype(np.float32) for _ in range(2))
    want = oracle.spmm_csr(ptr, ind, val, Bh)
    p, i, v = (torch.from_numpy(x).to(DEV) for x in (ptr, ind, val))
    _, B = shifted(Bh, words)
    buf, out = shifted(np.zeros_like(Bh), words)
    plan = sporder.spmm_plan(p, i)

    def check(what, ref):
        got = out.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), what
        assert torch.all(buf[:16 + words] == -7.0) and torch.all(buf[-16:] == -7.0), what
        out.zero_()

    print(f"[spmm_widths] N={N} words={words}", flush=True)
    sporder.spmm_csr(p, i, v, B, out=out)
    check("row_split", want)
    sporder.spmm_csr(p, i, v, B, out=out, plan=plan)
    check("plan", want)
    sporder.spmm_csr_noalloc(p, i, v, B, out=out)
    check("noalloc", want)
    sporder.spmm_csr_scaled(p, i, v, B, row_scale=torch.from_numpy(rs).to(DEV),
                            col_scale=torch.from_numpy(cs).to(DEV), out=out)
    check("scaled", rs[:, None] * oracle.spmm_csr(ptr, ind, val, cs[:, None] * Bh))
    sporder.spmm_csr(p, i, v, B, out=out, algo="merge_path")
    scale = np.abs(want).max()
    # A cut row adds its pieces in any order: rows of up to 1100 terms.
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * scale
    assert torch.all(buf[:16 + words] == -7.0) and torch.all(buf[-16:] == -7.0)
