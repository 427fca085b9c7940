"""Expert products of prompts: tile edges (128 rows, 64 / 128 columns), empty
and overfull experts, both activations; softmax routing, the expert sort and
the sum over a row's experts."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _hip():
    from gpustack_amd import ops

    return ops._load_hip()


def _experts(counts, k, g):
    """Assignments [T, k] whose expert e has counts[e] rows."""
    flat = torch.repeat_interleave(
        torch.arange(len(counts)), torch.tensor(counts)).cuda()
    assert flat.numel() % k == 0
    return flat[torch.randperm(flat.numel(), generator=g, device="cuda")] \
        .int().view(-1, k)


@pytest.mark.parametrize("ext", [False, True])
@pytest.mark.parametrize("counts,k,H,I", [
    ([1, 0, 0, 1], 2, 128, 128),
    ([127, 0, 128, 129], 4, 256, 128),
    ([0, 0, 600, 0, 8], 8, 384, 256),
    ([33] * 16, 2, 2048, 768)])
def test_tiles(ext, counts, k, H, I):
    hip = _hip()
    E, TK = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(TK)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    experts = _experts(counts, k, g)
    T = experts.shape[0]
    x = rnd(T, H).bfloat16()
    gu = (rnd(E, 2 * I, H) * H ** -0.5).bfloat16()
    dn = (rnd(E, H, I) * I ** -0.5).bfloat16()
    gub, dnb = (rnd(E, 2 * I).bfloat16(), rnd(E, H).bfloat16()) if ext \
        else (None, None)
    fw = torch.rand(TK, generator=g, device="cuda")
    order, s_tok, cnt, offs, tiles, n = hip.moe_sort(experts.view(-1), E, k)
    act = torch.full((TK, I), 9.0, device="cuda").bfloat16()
    con = torch.full((TK, H), 9.0, device="cuda").bfloat16()
    hip.moe_tile(False, act, x, gu, s_tok, tiles, n, offs, cnt, bias=gub,
                 act_mode=int(ext))
    hip.moe_tile(True, con, act, dn, order, tiles, n, offs, cnt, fw, bias=dnb)
    out = torch.empty_like(x)
    hip.moe_sum(out, con, k)

    assert cnt.tolist() == counts
    assert n.item() == sum((c + 127) // 128 for c in counts)
    flat = experts.view(-1).long()
    o = order.long()
    assert torch.equal(o.sort().values, torch.arange(TK, device="cuda"))
    assert torch.equal(flat[o].sort().values, flat[o])
    assert torch.equal(s_tok.long(), o // k)
    e = flat[o]
    # 8 significant bits: a rounding moves a value by at most 2^-8 of itself;
    # fp32 sums of K unit-variance products of size K^-1/2 add under 1e-4
    close = lambda a, r: bool(((a.double() - r).abs()
                               <= r.abs() * 2.0 ** -8 + 2e-4).all())
    h = torch.empty(TK, 2 * I, dtype=torch.float64, device="cuda")
    y = torch.empty(TK, H, dtype=torch.float64, device="cuda")
    for i in range(E):
        r = (e == i).nonzero().flatten()
        h[r] = x[s_tok[r].long()].double() @ gu[i].double().T
        y[r] = act[r].double() @ dn[i].double().T
        if ext:
            h[r] += gub[i].double()
            y[r] += dnb[i].double()
    a, b = h[:, :I], h[:, I:]
    if ext:
        a, b = a.clamp(max=7), b.clamp(-7, 7)
        ref = (b + 1) * a * torch.sigmoid(1.702 * a)
    else:
        ref = torch.nn.functional.silu(a) * b
    # the activation multiplies fp32 errors of both halves by at most ~10
    assert bool(((act.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + 2e-3).all())
    assert close(con[o], y * fw[o].double()[:, None])
    assert close(out, con.double().view(T, k, H).sum(1))


@pytest.mark.parametrize("renorm", [False, True])
@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (5, 64, 6), (130, 128, 8),
                                   (7, 100, 1), (3, 384, 8), (4, 1000, 32)])
def test_softmax_routing(renorm, T, E, k):
    g = torch.Generator(device="cuda").manual_seed(T * E)
    logits = torch.randn(T, E, generator=g, device="cuda") * 3
    logits[0, : k + 1] = 20.0          # equals: the lowest indices win
    ex = torch.empty(T, k, dtype=torch.int32, device="cuda")
    w = torch.empty(T, k, device="cuda")
    _hip().moe_topk(ex, w, logits, renorm)
    assert ex[0].tolist() == list(range(k))
    top, at = torch.topk(logits.double(), k, -1)
    assert torch.equal(ex[1:].long(), at[1:])
    ref = top.softmax(-1) if renorm else \
        logits.double().softmax(-1).gather(1, ex.long())
    torch.testing.assert_close(w.double(), ref, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("renorm", [False, True])
@pytest.mark.parametrize("E,k", [(8, 2), (100, 4), (1000, 32)])
def test_routing_of_logits_that_are_not_finite(renorm, E, k):
    """As top-k and softmax have it: a row with a NaN or infinite logit has no
    weights, one of minus infinity none for that expert; experts in range."""
    inf, nan = float("inf"), float("nan")
    logits = torch.randn(7, E, device="cuda")
    logits[0, 3], logits[1, E - 1], logits[2, 5] = nan, inf, -inf
    logits[3], logits[4], logits[5, 1:] = nan, -inf, -inf
    ex = torch.full((7, k), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros(7, k, device="cuda")
    _hip().moe_topk(ex, w, logits, renorm)
    if renorm:
        ref = torch.topk(logits, k, -1).values.softmax(-1)
    else:
        ref = torch.topk(logits.softmax(-1), k, -1).values
    assert bool(((ex >= 0) & (ex < E)).all())
    torch.testing.assert_close(w, ref, rtol=1e-5, atol=1e-7, equal_nan=True)


@pytest.mark.parametrize("TK,E", [(65536, 4096), (4096, 128), (4097, 128),
                                  (32544, 128), (8192, 1025), (5000, 1)])
def test_sort_of_a_long_list(TK, E):
    g = torch.Generator(device="cuda").manual_seed(TK)
    ex = torch.randint(0, max(1, E - 60), (TK,), generator=g,
                       device="cuda").int()
    order, s_tok, cnt, offs, tiles, n = _hip().moe_sort(ex, E, 8)
    ref = torch.bincount(ex.long(), minlength=E)
    assert torch.equal(cnt.long(), ref)
    assert torch.equal(offs.long(), ref.cumsum(0) - ref)
    o = order.long()
    assert torch.equal(o.sort().values, torch.arange(TK, device="cuda"))
    assert torch.equal(ex[o].sort().values, ex[o])
    assert torch.equal(s_tok.long(), o // 8)
    want = [(e, r) for e, c in enumerate(ref.tolist())
            for r in range(0, c, 128)]
    assert n.item() == len(want)
    assert [tuple(t) for t in tiles[:len(want)].tolist()] == want


@pytest.mark.parametrize("T,E,H,k", [(1, 1, 128, 1), (15, 16, 256, 2),
                                     (17, 7, 2048, 4), (4068, 13, 4096, 13),
                                     (64, 64, 2176, 64), (100, 128, 2048, 8),
                                     (4100, 36, 1024, 8), (129, 500, 512, 4)])
@pytest.mark.parametrize("renorm", [True, False])
def test_route(T, E, H, k, renorm):
    g = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    w = (torch.randn(E, H, generator=g, device="cuda") / H ** 0.5).bfloat16()
    experts = torch.full((T, k), -1, dtype=torch.int32, device="cuda")
    weights = torch.empty(T, k, device="cuda")
    if E > 16:                        # 32, 64, 128 columns in turn
        _hip().moe_topk(experts, weights, _hip().rows_tile_parts(
            x, w, 32 << (T + k) % 3, 1 + T % 4), renorm)
    else:
        _hip().moe_route(experts, weights, x, w, renorm)
    logits = x.double() @ w.double().T
    # fp32 sums of exact products: at most 2^-18 of the terms' absolute sum
    eps = float((x.double().abs() @ w.double().abs().T).max()) * 2.0 ** -18
    got = logits.gather(1, experts.long())
    best = logits.sort(1, descending=True).values[:, :k]
    assert bool(((got - best).abs() <= 2 * eps).all())
    assert bool((experts.long().sort(1).values.diff(dim=1) > 0).all())
    p = torch.softmax(got if renorm else logits, 1)
    want = p if renorm else p.gather(1, experts.long())
    # a logit off by eps moves a weight by 2 eps of itself; fp32 exp and sum
    assert bool(((weights.double() - want).abs()
                 <= want * (4 * eps + 2.0 ** -18) + 2.0 ** -30).all())


def _moe(E, k, H, I, seed=0):
    import dataclasses

    from gpustack_amd.engine import EngineConfig
    from gpustack_amd.models.llama import MoEMLP
    from gpustack_amd.parallel import Communicator

    spec = dataclasses.replace(
        EngineConfig(model="qwen3-30b-a3b", device="cpu").spec,
        num_experts=E, num_experts_per_tok=k, hidden_size=H,
        moe_intermediate_size=I)
    m = MoEMLP(spec, 1, Communicator(), torch.bfloat16).cuda()
    g = torch.Generator(device="cuda").manual_seed(seed)
    for p in m.parameters():
        p.data.copy_(torch.randn(p.shape, generator=g, device="cuda")
                     * p.shape[-1] ** -0.5)
    return m, g


def _moe_reference(m, x):
    """The layer in float64: routing, experts, weighted sum."""
    x = x.double()
    top, ex = torch.topk(x @ m.router_w.double().T, m.top_k, -1)
    top = top.softmax(-1)
    out = torch.zeros_like(x)
    for e in range(m.e):
        t, j = (ex == e).nonzero(as_tuple=True)
        gu = x[t] @ m.gate_up_w[e].double().T
        h = torch.nn.functional.silu(gu[:, :m.i]) * gu[:, m.i:]
        out.index_add_(0, t, (h @ m.down_w[e].double().T) * top[t, j, None])
    return out


@pytest.mark.parametrize("k", [64, 65, 128])
def test_more_experts_a_row_than_lanes(k):
    m, g = _moe(128, k, 256, 128)
    x = torch.randn(9, 256, generator=g, device="cuda").bfloat16()
    ref = _moe_reference(m, x)
    # bf16 activations and contributions: 2^-8 of each, of about equal size
    assert float((m(x).double() - ref).norm() / ref.norm()) < 2.0 ** -7


@pytest.mark.parametrize("T", [3, 130])
def test_rows_at_any_address(T):
    m, g = _moe(4, 2, 256, 128)
    flat = torch.randn(T * 256 + 1, generator=g, device="cuda").bfloat16()
    x = flat[1:].view(T, 256)
    assert x.data_ptr() % 16
    ref = _moe_reference(m, x)
    # as above
    assert float((m(x).double() - ref).norm() / ref.norm()) < 2.0 ** -7


@pytest.mark.parametrize("T,loop,wide", [(12000, True, False), (11900, False, False),
                                         (12000, False, True)])
def test_long_prompts_of_few_large_experts(monkeypatch, T, loop, wide):
    """Both sides of the line between the tiles of 128 rows and the library's loop, and
    tiles of up to 320 rows, which have none."""
    from gpustack_amd import ops

    m, g = _moe(4, 2, 2048, 8192)
    if not wide:
        monkeypatch.setattr(ops, "moe_wide_wins", lambda *a: False)
    x = torch.randn(T, 2048, generator=g, device="cuda").bfloat16()
    taken = []
    for name in ("_fused_dispatch", "_loop_dispatch"):
        real = getattr(m, name)
        monkeypatch.setattr(m, name, lambda *a, r=real, n=name:
                            (taken.append(n), r(*a))[1])
    out = m(x)
    assert taken == ["_loop_dispatch" if loop else "_fused_dispatch"]
    part = torch.cat([torch.arange(64), torch.arange(T - 64, T)]).cuda()
    ref = _moe_reference(m, x[part])
    # as above, with one more rounding of the activation's operands
    assert float((out[part].double() - ref).norm() / ref.norm()) < 2.0 ** -6
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing",
                        lambda: True)
    assert not m._library_wins(T)


@pytest.mark.parametrize("E,T,H,I,tiles", [
    (8, 32, 256, 3200, False), (8, 33, 256, 3200, True),
    (8, 8, 256, 3072, True), (40, 4, 4096, 3200, False),
    (40, 5, 4096, 3200, True)])
def test_down_product_of_few_rows(monkeypatch, E, T, H, I, tiles):
    """Both sides of the lines between its two forms."""
    m, g = _moe(E, 2, H, I)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    hip, taken = _hip(), []
    real = hip.moe_down_scale
    monkeypatch.setattr(hip, "moe_down_scale",
                        lambda *a, **k: (taken.append(1), real(*a, **k)))
    out = m(x)
    assert (not taken) == tiles
    ref = _moe_reference(m, x)
    # as above
    assert float((out.double() - ref).norm() / ref.norm()) < 2.0 ** -7


@pytest.mark.parametrize("K", [64, 128, 192, 320])
@pytest.mark.parametrize("far", [False, True])
def test_steps_and_far_rows(K, far):
    """One to five steps of the K loop; rows of a source whose last lie past
    what 32 bits of byte offset reach (only the first product's are gathered
    from anywhere)."""
    hip = _hip()
    counts = [0, 33, 1, 130, 64]
    E, TK, N = len(counts), sum(counts), 128
    g = torch.Generator(device="cuda").manual_seed(K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    ex = _experts(counts, 1, g).view(-1)
    order, s_tok, cnt, offs, tiles, n = hip.moe_sort(ex, E, 1)
    T = TK + (2 ** 31 // K if far else 0)
    x = torch.empty(T, K, dtype=torch.bfloat16, device="cuda")
    x[-TK:] = rnd(TK, K)
    gu = (rnd(E, 2 * N, K) * K ** -0.5).bfloat16()
    act = torch.full((TK, N), 9.0, device="cuda").bfloat16()
    hip.moe_tile(False, act, x, gu, s_tok + (T - TK), tiles, n, offs, cnt)
    rows = x[-TK:].double()[s_tok.long()]
    e = ex.long()[order.long()]
    h = torch.stack([gu[int(i)].double() @ r for i, r in zip(e, rows)])
    ref = torch.nn.functional.silu(h[:, :N]) * h[:, N:]
    # bf16 result; fp32 sums of K products of size K^-1/2 under 1e-4
    assert bool(((act.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + 2e-4).all())
