"""What a ragged SpMM call launches, from the kernels that ran: few rows are
spread over the chip, and small calls are not mostly launches."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def kernels(call):
    """Names of the library's kernels that `call` runs, in order."""
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU,
                                            torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if "sporder_hip" in e.name]


def case(n, deg, N, seed=5):
    """A uniform matrix on the GPU (ptr, ind, val), B and an output."""
    rng = np.random.default_rng(seed)
    keys = np.unique(np.repeat(np.arange(n), deg) * n + rng.integers(0, n, n * deg))
    ptr = np.concatenate([[0], np.cumsum(np.bincount(keys // n, minlength=n))])
    p, i = (torch.from_numpy(a.astype(np.int32)).to("cuda:0") for a in (ptr, keys % n))
    v = torch.ones(i.numel(), device="cuda:0")
    return p, i, v, torch.ones((n, N), device="cuda:0"), torch.empty((n, N), device="cuda:0")


@pytest.mark.parametrize("N", [1, 3, 7, 30])
def test_few_rows_have_groups_of_their_own(sporder, N):
    """300,000 rows, 64 to a wave, would fill little more than half of the chip."""
    print(f"[spmm_launches] own groups N={N}", flush=True)
    p, i, v, B, out = case(300_000, 3, N)
    names = kernels(lambda: sporder.spmm_csr(p, i, v, B, out=out))
    assert any("spmm_rowsplit_v4<8" in k for k in names)
    assert not any("spmm_rows_dyn" in k for k in names)


@pytest.mark.parametrize("N", [2, 7, 47, 150])
@pytest.mark.parametrize("how", ["row_split", "scaled"])
def test_small_calls_are_one_launch(sporder, how, N):
    print(f"[spmm_launches] {how} N={N}", flush=True)
    p, i, v, B, out = case(2_000, 8, N)
    scale = torch.ones(2_000, device="cuda:0")
    calls = {"row_split": lambda: sporder.spmm_csr(p, i, v, B, out=out),
             "scaled": lambda: sporder.spmm_csr_scaled(p, i, v, B, row_scale=scale, out=out)}
    names = kernels(calls[how])
    assert len(names) == 1 and "spmm_rows_small" in names[0]


@pytest.mark.parametrize("N", [1, 47])
def test_many_empty_rows_are_not_small(sporder, N):
    """400,000 rows of one nonzero."""
    print(f"[spmm_launches] empty rows N={N}", flush=True)
    p, i, v, B, out = case(400_000, 1, N)
    names = kernels(lambda: sporder.spmm_csr(p, i, v, B, out=out))
    assert not any("spmm_rows_small" in k for k in names)


@pytest.mark.parametrize("n,deg,N,most", [(2_000, 8, 30, 1), (2_000, 8, 47, 1),
                                          (70_000, 10, 3, 4), (70_000, 10, 47, 4)])
def test_noalloc_counts_only_what_may_not_fit(sporder, n, deg, N, most):
    """The long rows of an input that cannot outgrow the static scratch are not
    counted, which would be a kernel, a readback and a synchronize."""
    print(f"[spmm_launches] noalloc n={n} N={N}", flush=True)
    p, i, v, B, out = case(n, deg, N)
    names = kernels(lambda: sporder.spmm_csr_noalloc(p, i, v, B, out=out))
    assert len(names) <= most and not any("count_long" in k for k in names)


@pytest.mark.parametrize("N", [5, 47, 101])
@pytest.mark.parametrize("n,deg,kernel", [(2_000, 8, "spmm_merge_path"),
                                          (40_000, 8, "spmm_merge_v4")])
def test_merge_spans_of_ragged_widths(sporder, n, deg, kernel, N):
    """A wave per span up to 2^18 nonzeros, row groups (8 lanes or more) past
    that: a few long walks in row groups took up to three times as long."""
    print(f"[spmm_launches] merge n={n} N={N}", flush=True)
    p, i, v, B, out = case(n, deg, N)
    names = kernels(lambda: sporder.spmm_csr(p, i, v, B, out=out, algo="merge_path"))
    assert any(kernel in k for k in names)
    assert not any(f"spmm_merge_v4<{g}," in k for k in names for g in (1, 2, 4))
