"""Where chunks are not classified (one chunk, or chunks of more than 4096
rows) a sample of the rows decides whether the sketch counts: the form that
does the work, from the kernels' names and times, and the table bit for bit
against the oracle either way."""

import numpy as np
import pytest
import torch

import oracle
from chunkedgreedy_amd import synth

pytestmark = pytest.mark.gpu


def uniform(n, deg, seed):
    rng = np.random.default_rng(seed)
    keys = np.unique(np.repeat(np.arange(n), deg) * n + rng.integers(0, n, n * deg))
    return np.concatenate([[0], np.cumsum(np.bincount(keys // n, minlength=n))]), keys % n


# Power-law rows evict all along; rows of a geometric graph and of scrambled
# blocks meet few others; rows of 3 nonzeros never hold more than the capacity.
CASES = {
    "power": (lambda: synth.chung_lu(20_000, 2.1, 16, 31)[:2], False),
    "rgg": (lambda: synth.rgg(20_000, 13, 32)[:2], True),
    "scrambled_blocks": (lambda: synth.planted(20_480, 320, 14, 33)[:2], True),
    "short_rows": (lambda: uniform(20_000, 3, 34), True),
    "long_uniform": (lambda: uniform(20_000, 24, 35), False),
}


def sketch_times(call):
    """{counting: microseconds} of the sketch kernels that `call` launches."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU,
                                            torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    times = {}
    for e in prof.events():
        if "ovf_sketch_kernel<" in e.name:
            counting = e.name.split("ovf_sketch_kernel<")[1].split(">")[0].split(",")[2].strip()
            times[counting == "true"] = times.get(counting == "true", 0.0) + e.device_time
    return times


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("chunk", [20_480, 6_000])
def test_form_and_table(sporder, name, chunk):
    print(f"[count_choice] {name} chunk={chunk}", flush=True)
    make, counted = CASES[name]
    ptr, ind = make()
    dptr, dind = (torch.from_numpy(np.ascontiguousarray(a, np.int32)).to("cuda:0")
                  for a in (ptr, ind))
    k, ovs = 16, 4.0

    def call():
        return sporder.chunk_similarity_top_k(dptr, dind, k=k, oversampling=ovs, chunk_size=chunk)

    gi, gw = call()
    want_i, want_w = oracle.unpack_table(
        oracle.chunk_similarity_top_k(ptr, ind, k, chunk, ovs, is_symmetric=False))
    assert np.array_equal(gi.cpu().numpy(), want_i)
    assert np.array_equal(gw.cpu().numpy().view(np.uint32), want_w.view(np.uint32))
    if chunk >= 20_480:
        times = sketch_times(call)
        print(f"[count_choice] {name}: {times}", flush=True)
        assert max(times, key=times.get) == counted
