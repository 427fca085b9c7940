"""Single rows of a scan whose state rows lanes bring eight at a time: numbers of rows
that end inside the eight, several tokens of a sequence, fresh and kept states."""
import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.ops import torch_ref

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("N,P", [(56, 128), (64, 128), (72, 128), (136, 128),
                                 (31, 256), (5, 64), (129, 64)])
def test_state_rows(N, P):
    H, dev = 2, "cuda"
    news, hists, slots = [1, 1, 3, 2], [7, 0, 0, 4], [2, 0, 4, 1]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    first = [sum(news[:i]) for i in range(len(news))]
    T = sum(news)
    pos = i32([h + j for h, n in zip(hists, news) for j in range(n)])
    g = torch.Generator(device=dev).manual_seed(N + P)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    st0 = rnd(6, H, N, P)
    decay = torch.tensor([0.9, 0.99], device=dev)
    res = []
    for impl, kw in ((ops, {"single": True}), (torch_ref, {})):
        y, st = torch.zeros(T, H * P, device=dev), st0.clone()
        impl.state_scan(y, src, 0, H * P, H * (P + N), None, 0, H, H, N, P, True,
                        None, None, None, decay, st, i32(first), i32(news),
                        i32(slots), pos, **kw)
        res.append((y, st))
    # fp32 sums of up to N products, in another order
    for a, b in zip(*res):
        assert float((a - b).abs().max()) <= N * 2.0 ** -23 * float(b.abs().max())
    assert torch.equal(res[0][1][3], st0[3]) and torch.equal(res[0][1][5], st0[5])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,P", [(40, 64), (64, 64), (72, 64), (56, 128), (72, 128)])
@pytest.mark.parametrize("H", [64, 63])
def test_many_states(N, P, H, dtype):
    """16 and 17 sequences of 63 and 64 heads, 1008 and 1088 workgroups: state rows of a
    lane one by one, four and eight in flight; the last sequence of three tokens."""
    S, dev = 17 if H == 64 else 16, "cuda"
    news = [1] * (S - 1) + [3]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    first, hists = list(range(S)), [i % 2 * 5 for i in range(S)]
    T = sum(news)
    pos = i32([h + j for h, n in zip(hists, news) for j in range(n)])
    g = torch.Generator(device=dev).manual_seed(H)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    src, st0 = rnd(T, H * (P + 2 * N)).to(dtype), rnd(S, H, N, P)
    decay = torch.linspace(0.8, 0.99, H, device=dev)
    res = []
    for impl, kw in ((ops, {"single": True}), (torch_ref, {})):
        y, st = torch.zeros(T, H * P, device=dev), st0.clone()
        impl.state_scan(y, src, 0, H * P, H * (P + N), None, 0, H, H, N, P, False,
                        None, None, None, decay, st, i32(first), i32(news),
                        i32(list(range(S))), pos, **kw)
        res.append((y, st))
    for a, b in zip(*res):        # fp32 sums of up to N products, in another order
        assert float((a - b).abs().max()) <= N * 2.0 ** -23 * float(b.abs().max())
