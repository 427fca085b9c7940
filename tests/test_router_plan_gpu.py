"""The router's product in the tiles and parts of its plan, on both sides of each of the
plan's lines, and the choice on its parts."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("E,T,plan", [
    (32, 1, (32, 8)), (20, 9000, (32, 8)), (36, 2500, (32, 8)),
    (64, 2501, (64, 4)), (64, 12001, (64, 2)), (68, 1400, (32, 8)),
    (128, 1401, (32, 4)), (128, 2501, (64, 2)), (100, 6001, (128, 2)),
    (132, 2500, (32, 4)), (256, 2501, (128, 4)), (256, 6001, (128, 2)),
    (256, 12001, (128, 1)), (260, 64, (64, 2)), (512, 2049, (128, 2))])
def test_plan(E, T, plan):
    from gpustack_amd import ops

    H, k = 1024, 4
    assert ops.router_plan(T, E, H) == plan
    g = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    w = (torch.randn(E, H, generator=g, device="cuda") / H ** 0.5).bfloat16()
    hip = ops._load_hip()
    parts = hip.rows_tile_parts(x, w, *plan)
    assert parts.shape == (plan[1], T, E)
    experts = torch.full((T, k), -1, dtype=torch.int32, device="cuda")
    weights = torch.empty(T, k, device="cuda")
    hip.moe_topk(experts, weights, parts, True)
    logits = x.double() @ w.double().T
    # fp32 sums of exact products: at most 2^-18 of the terms' absolute sum, which is
    # 1024 terms of size |x| |w|
    eps = float((x.double().abs() @ w.double().abs().T).max()) * 2.0 ** -18
    assert float((parts.double().sum(0) - logits).abs().max()) <= eps
    got = logits.gather(1, experts.long())
    best = logits.topk(k, 1).values
    assert float((got - best).abs().max()) <= 2 * eps
    want = got.softmax(1)
    assert bool(((weights.double() - want).abs()
                 <= want * (4 * eps + 2.0 ** -18) + 2.0 ** -30).all())
