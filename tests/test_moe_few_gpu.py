"""Expert products 16 rows at a time straight from memory, against the tiles and the
products in 64 bits."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("E,T,k,H,I", [
    (1, 1, 1, 64, 64), (5, 7, 3, 128, 192), (8, 16, 2, 512, 640), (8, 17, 2, 576, 512),
    (3, 131, 2, 768, 832), (4, 300, 2, 1536, 320), (16, 9, 4, 1600, 1600),
    (64, 40, 6, 2048, 768), (2, 3, 2, 4160, 2048)])
def test_products(E, T, k, H, I):
    from gpustack_amd import ops

    hip = ops._load_hip()
    g = torch.Generator(device="cuda").manual_seed(T * E + H)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = rand(T, H).bfloat16()
    gate_up = (rand(E, 2 * I, H) / H ** 0.5).bfloat16()
    down = (rand(E, H, I) / I ** 0.5).bfloat16()
    experts = rand(T, E).argsort(1)[:, :k].int().contiguous()
    flat_w = torch.rand(T * k, generator=g, device="cuda")
    order, s_tok, counts, offs, tiles, n = hip.moe_sort(experts.view(-1), E, k)
    act = torch.full((T * k, I), float("nan"), device="cuda").bfloat16()
    hip.moe_few(False, act, x, gate_up, s_tok, tiles, n, offs, counts)
    by = experts.view(-1)[order.long()].long()
    for lo in range(0, T * k, 32):
        hi = min(lo + 32, T * k)
        rows, e = s_tok[lo:hi].long(), by[lo:hi]
        xs = x[rows].double()
        both = (gate_up[e].double() * xs[:, None]).sum(2)
        size = (gate_up[e].double() * xs[:, None]).abs().sum(2)
        gate, up = both[:, :I], both[:, I:]
        want = torch.nn.functional.silu(gate) * up
        # the fp32 sums of H terms in at most 8 parts of a chain each, one rounding to
        # bf16; the activation's slope is at most 1.1
        err = 2.0 ** -18 * (1.1 * size[:, :I] * up.abs() + gate.abs() * size[:, I:])
        assert bool(((act[lo:hi].double() - want).abs()
                     <= err + want.abs() * 2.0 ** -8 + 1e-30).all())
    out = torch.full((T * k, H), float("nan"), device="cuda").bfloat16()
    hip.moe_few(True, out, act, down, order, tiles, n, offs, counts, flat_w)
    for lo in range(0, T * k, 32):
        hi = min(lo + 32, T * k)
        at, e = order[lo:hi].long(), by[lo:hi]
        terms = down[e].double() * act[lo:hi].double()[:, None]
        want = terms.sum(2) * flat_w[at].double()[:, None]
        err = terms.abs().sum(2) * flat_w[at].double()[:, None] * 2.0 ** -18
        assert bool(((out[at].double() - want).abs()
                     <= err + want.abs() * 2.0 ** -8 + 1e-30).all())


def test_replays():
    """In a graph, on other rows' routing at each replay."""
    from gpustack_amd import ops

    hip = ops._load_hip()
    E, T, k, H, I = 32, 12, 4, 256, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, w = rand(T, H).bfloat16(), (rand(E, 2 * I, H) / 16).bfloat16()
    experts = torch.zeros(T, k, dtype=torch.int32, device="cuda")
    act, want = (torch.empty(T * k, I, device="cuda").bfloat16() for _ in range(2))

    def step(few, out):
        order, s_tok, counts, offs, tiles, n = hip.moe_sort(experts.view(-1), E, k)
        product = hip.moe_few if few else hip.moe_tile
        product(False, out, x, w, s_tok, tiles, n, offs, counts)
        return order

    step(True, act)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        place = step(True, act)
    for _ in range(4):
        experts.copy_(rand(T, E).argsort(1)[:, :k].int())
        x.copy_(rand(T, H))
        graph.replay()
        other = step(False, want)
        a, b = torch.empty_like(act), torch.empty_like(act)
        a[place.long()], b[other.long()] = act, want
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -7 * float(
            b.float().abs().max())


@pytest.mark.parametrize("rows,E,K,down,wins", [
    (512, 128, 2048, False, True), (513, 128, 2048, False, False),
    (512, 128, 768, True, True), (513, 128, 768, True, False),
    (512, 128, 512, True, True), (256, 128, 640, True, True), (257, 128, 640, True, False),
    (257, 128, 704, True, False), (513, 128, 704, False, False),
    (96, 128, 832, True, True), (97, 128, 3072, True, False),
    (16, 16, 3136, True, True), (17, 16, 6400, True, False),
    (0, 8, 14336, False, False)])
def test_rule(rows, E, K, down, wins):
    from gpustack_amd import ops

    assert ops.moe_few_wins(rows, E, K, down) is wins


@pytest.mark.parametrize("I", [512, 768, 3200])
def test_down_without_a_list(I):
    """moe_down_scale: workgroups for every expert or of the list, with a bias too."""
    from gpustack_amd import ops

    hip = ops._load_hip()
    E, T, k, H = 6, 60, 2, 192
    g = torch.Generator(device="cuda").manual_seed(I)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    act, w = rand(T * k, I).bfloat16(), (rand(E, H, I) / I ** 0.5).bfloat16()
    bias = rand(E, H).bfloat16()
    experts = rand(T, E - 1).argsort(1)[:, :k].int().contiguous()  # one has no rows
    flat_w = torch.rand(T * k, generator=g, device="cuda")
    order, _, counts, offs, tiles, n = hip.moe_sort(experts.view(-1), E, k)
    at = order.long()
    e = experts.view(-1)[at].long()
    terms = w[e].double() * act.double()[:, None]
    for b, lists in ((None, {}), (bias, {}), (bias, dict(tiles=tiles, ntiles=n))):
        out = torch.full((T * k, H), float("nan"), device="cuda").bfloat16()
        hip.moe_down_scale(out, act, w, offs, counts, order, flat_w, bias=b, **lists)
        sums = terms.sum(2) + (0 if b is None else b[e].double())
        size = terms.abs().sum(2) + (0 if b is None else b[e].double().abs())
        scale = flat_w[at].double()[:, None]
        assert bool(((out[at].double() - sums * scale).abs() <= scale * (
            size * 2.0 ** -18 + sums.abs() * 2.0 ** -8) + 1e-30).all())


@pytest.mark.parametrize("N,K", [(40, 128), (64, 96)])
def test_refused(N, K):
    from gpustack_amd import ops

    hip = ops._load_hip()
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError):
        hip.moe_few(True, torch.empty(1, N, device="cuda").bfloat16(),
                    torch.zeros(1, K, device="cuda").bfloat16(),
                    torch.zeros(1, N, K, device="cuda").bfloat16(), i32(0),
                    i32(0, 0), i32(1), i32(0), i32(1), torch.ones(1, device="cuda"))
