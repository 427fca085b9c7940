"""The first of the largest words of a row, at vocabularies that end inside a round of
loads, and the copy of it in pinned memory."""
import pytest
import torch

from gpustack_amd import ops

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("V", [1, 4, 9, 4095, 4099, 8 * 1024 * 8, 8 * 1024 * 8 + 8,
                               4 * 1024 * 8 + 5, 151936])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_first_of_the_largest(V, dtype):
    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn(7, V, generator=g, device="cuda").to(dtype)
    x[1] = -2.0
    x[2, -1] = 99.0
    x[3, V // 2:] = 50.0
    x[4] = float("nan")                   # no number: the first word
    x[5] = float("nan")
    x[5, V // 3] = -1e30
    x[6, max(V - 9, 0):] = float("inf")
    want = [int((r == r.nan_to_num(nan=-float("inf"), posinf=float("inf")).max())
                .nonzero()[0, 0]) if bool((r == r).any()) else 0
            for r in x.float()]
    for host in (None, torch.full((9,), -5, dtype=torch.long, pin_memory=True)):
        out = torch.full((7,), -3, dtype=torch.long, device="cuda")
        ops.greedy_sample_into(out, x, None if host is None else host[:7])
        torch.cuda.synchronize()
        assert out.tolist() == want
        if host is not None:
            assert host.tolist() == want + [-5, -5]


@pytest.mark.parametrize("V", [40000, 40005, 69637])
def test_more_rows_than_the_chip_has(V):
    """257 rows: fp32 words one at a time above 40000, else four."""
    x = torch.zeros(257, V, device="cuda")
    at = [(i * 7919) % V for i in range(257)]
    for i, j in enumerate(at):
        x[i, j:] = 1.0
    x[5, V - 1] = 2.0
    out = torch.full((257,), -3, dtype=torch.long, device="cuda")
    ops.greedy_sample_into(out, x)
    assert out.tolist() == at[:5] + [V - 1] + at[6:]


def test_words_in_ordinary_memory_are_refused():
    out = torch.zeros(2, dtype=torch.long, device="cuda")
    for dtype in (torch.bfloat16, torch.float32):
        x = torch.zeros(2, 16, dtype=dtype, device="cuda")
        for host in (torch.zeros(2, dtype=torch.long),
                     torch.zeros(1, dtype=torch.long, pin_memory=True),
                     torch.zeros(2, dtype=torch.int32, pin_memory=True)):
            with pytest.raises(RuntimeError, match="pinned"):
                ops.greedy_sample_into(out, x, host)
