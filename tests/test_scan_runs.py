"""The lists that cut a prompt's sequences into runs of rows for the state scan
(ops.scan_run_rows, ops.build_scan_runs) and the memory that a call takes."""
import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.models.llama import RaggedMeta

BATCHES = [[4000], [4000] + [20] * 100, [20] * 50 + [4000] + [20] * 50,
           [301, 640, 900, 1200, 1500, 1900], [7000] + [8] * 250,
           [300, 257, 31]]


def _starts(news):
    return [sum(news[:i]) for i in range(len(news))]


@pytest.mark.parametrize("news", BATCHES)
@pytest.mark.parametrize("size", [64, 128, 576])
def test_runs_hold_every_row_once(news, size):
    starts = _starts(news)
    runs, cut = ops.build_scan_runs(starts, news, size, "cpu")
    seen = []
    for i, (first, n, s, run0) in enumerate(runs.tolist()):
        assert 1 <= n <= size and run0 <= i and int(runs[run0, 2]) == s
        assert first == starts[s] + (i - run0) * size
        assert (news[s] > size) == (i < cut)
        seen += range(first, first + n)
    assert sorted(seen) == list(range(sum(news)))


@pytest.mark.parametrize("longest,others", [(500, [1] * 255), (500, [1] * 511),
                                            (1900, [1] * 85)])
def test_no_runs_where_no_chunk_kernel_runs(longest, others):
    """One long prompt among so many single rows that there are fewer than
    SCAN_CHUNK_ROWS rows a sequence: the scan walks row by row."""
    assert ops.scan_run_rows([longest] + others, 64, 64) == 0


@pytest.mark.parametrize("news", BATCHES)
@pytest.mark.parametrize("heads,vdim", [(64, 64), (16, 128)])
def test_places_only_for_what_is_cut(news, heads, vdim):
    z = torch.zeros(1, dtype=torch.int32)
    rg = RaggedMeta(z, z, z, z, _starts(news), [0] * len(news), news, max(news))
    got = rg.scan_runs(heads, 128, vdim, torch.bfloat16)
    rows = ops.scan_run_rows(news, heads, vdim)
    if not rows:
        assert not got
        return
    long = [n for n in news if n > rows]
    assert got["cut"] == sum(-(-n // rows) for n in long)
    # a longest sequence gives up to 8 runs, and all rows are fewer than 256 /
    # groups times it
    assert got["cut"] <= 4096 // (heads * -(-vdim // 64))
    assert got["runs"].shape == (got["cut"] + len(news) - len(long), 4)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("news,most", [([600] + [30] * 40, 7),
                                       ([600] + [1] * 255, 0)])
def test_memory_of_a_call(news, most):
    """Two states of all heads for every run of a cut sequence, no more."""
    H, N, P = 4, 64, 64
    T, S = sum(news), len(news)
    starts = _starts(news)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    src = torch.randn(T, H * P + 2 * H * N, device="cuda").bfloat16()
    y = torch.empty(T, H * P, device="cuda")
    state = torch.zeros(S, H, N, P, device="cuda")
    decay = torch.full((H,), 0.9, device="cuda")
    lists = (i32(starts), i32(news), i32(list(range(S))),
             i32([j for n in news for j in range(n)]))
    runs, cut = ops.build_scan_runs(starts, news, 96, "cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.state_scan(y, src, 0, H * P, H * (P + N), None, 0, H, H, N, P, False,
                   None, None, None, decay, state, *lists, runs=runs, cut=cut)
    took = torch.cuda.max_memory_allocated() - before
    assert took <= most * (2 * H * N * P * 4 + 4 * H) + 3 * 512
