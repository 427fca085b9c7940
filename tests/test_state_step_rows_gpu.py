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
