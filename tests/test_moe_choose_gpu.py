"""The choice of the experts and the sort of the assignments in one launch, against the
two launches and a plain top k."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("T", [1, 7, 8, 16])
@pytest.mark.parametrize("E,k,parts,renorm", [
    (1, 1, 1, True), (20, 20, 8, False), (64, 6, 8, True), (65, 64, 2, True),
    (128, 8, 8, True), (200, 1, 4, False), (256, 64, 4, True)])
def test_choose(T, E, k, parts, renorm):
    from gpustack_amd import ops

    hip = ops._load_hip()
    g = torch.Generator(device="cuda").manual_seed(T * E + k)
    logits = torch.randn(parts, T, E, generator=g, device="cuda")
    if E > 64:
        logits[:, T // 2] = 0.0                # equals: the lowest index first
        logits[0, 0, E - 1] = float("inf")     # no number among the weights
    pair = lambda: (torch.full((T, k), -1, dtype=torch.int32, device="cuda"),
                    torch.full((T, k), -1.0, device="cuda"))
    (experts, weights), (want, want_w) = pair(), pair()
    got = hip.moe_choose(experts, weights, logits, renorm)
    hip.moe_topk(want, want_w, logits, renorm)
    assert torch.equal(experts, want)
    assert torch.equal(weights.view(torch.int32), want_w.view(torch.int32))
    order, s_tok, counts, offs, tiles, n = got
    lists = hip.moe_sort(want.view(-1), E, k)
    for i in (2, 3, 5):
        assert torch.equal(got[i], lists[i])
    assert torch.equal(tiles[:int(n)], lists[4][:int(n)])
    assert torch.equal(order.sort().values.long(),
                       torch.arange(T * k, device="cuda"))
    assert torch.equal(s_tok, order // k)
    by = experts.view(-1)[order.long()]
    assert torch.equal(by, by.sort().values)
    assert torch.equal(counts.long(), torch.bincount(want.view(-1), minlength=E))


@pytest.mark.parametrize("T,E,k", [(17, 64, 4), (0, 64, 4), (4, 257, 4), (4, 8, 9)])
def test_refused(T, E, k):
    from gpustack_amd import ops

    experts = torch.zeros(T, k, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError):
        ops._load_hip().moe_choose(experts, torch.zeros(T, k, device="cuda"),
                                   torch.zeros(T, E, device="cuda"), True)


def test_rule():
    from gpustack_amd import ops

    takes = lambda E: [T for T in range(40) if ops.choose_sorts(T, E)]
    assert takes(64) == list(range(1, 17)) and takes(257) == []
    assert takes(65) == takes(256) == list(range(1, 9))
