"""Expert products in tiles of up to 320 rows: heights of a tile (64 rows a step), parts
of an expert, empty experts, columns that end inside a tile, more tiles than workgroups;
and the rule that takes them."""
import pytest
import torch

from gpustack_amd import ops
from test_wide_tiles_gpu import check_large, large_pairs

needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(),
                               reason="needs a GPU")


def _run(counts, k, H, I, weights=True):
    hip = ops._load_hip()
    E, TK = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(TK + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).cuda()
    flat = flat[torch.randperm(TK, generator=g, device="cuda")].int()
    x = rnd(TK // k, H).bfloat16()
    gu = (rnd(E, 2 * I, H) * H ** -0.5).bfloat16()
    dn = (rnd(E, H, I) * I ** -0.5).bfloat16()
    fw = torch.rand(TK, generator=g, device="cuda")
    order, s_tok, cnt, offs, _, _, s_w = hip.moe_sort(flat, E, k, weights=fw)
    assert torch.equal(s_w, fw[order.long()])
    # one row more on each side, which keeps what it holds
    act = torch.full((TK + 2, I), 9.0, device="cuda").bfloat16()
    con = torch.full((TK + 2, H), 9.0, device="cuda").bfloat16()
    hip.moe_wide(False, act[1:-1], x, gu, s_tok, offs, cnt)
    hip.moe_wide(True, con[1:-1], act[1:-1], dn, order, offs, cnt, s_w)
    for t in (act, con):
        assert bool((t[0] == 9).all()) and bool((t[-1] == 9).all())
    act, con = act[1:-1], con[1:-1]
    o = order.long()
    e = flat.long()[o]
    ref = torch.empty(TK, I, dtype=torch.float64, device="cuda")
    y = torch.empty(TK, H, dtype=torch.float64, device="cuda")
    for i in range(E):
        r = (e == i).nonzero().flatten()
        h = x[s_tok[r].long()].double() @ gu[i].double().T.contiguous()
        ref[r] = torch.nn.functional.silu(h[:, :I]) * h[:, I:]
        y[r] = act[r].double() @ dn[i].double().T.contiguous()
    y *= fw[o].double()[:, None]
    # 8 significant bits; fp32 sums of K unit-variance products of size K^-1/2 are off
    # by under 1e-4, which the activation multiplies by at most ~10
    assert bool(((act.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + 2e-3).all())
    assert bool(((con[o].double() - y).abs()
                 <= y.abs() * 2.0 ** -8 + 2e-4).all())


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("counts,k,H,I", [
    ([1, 0, 0, 1], 2, 192, 192),
    ([63, 0, 64, 65], 1, 256, 320),       # heights 2, 2, 4; columns end inside
    ([128, 129, 192, 193, 256, 257], 5, 320, 256),
    ([319, 320, 321, 0, 640, 641, 7], 8, 384, 256),
    ([1999], 1, 192, 448),
    ([3] * 255 + [300], 3, 2048, 192),    # 256 experts, eight tiles a workgroup
    ([0] * 100 + [97] * 30, 2, 2048, 768)])
def test_tiles(counts, k, H, I):
    _run(counts, k, H, I)


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("rows", [64, 320])
def test_gate_and_up_beyond_fp32(rows):
    hip = ops._load_hip()
    g, u, ref = large_pairs()
    I, H = -(-len(g) // 8) * 8, 192
    x = torch.zeros(rows, H, dtype=torch.bfloat16)
    x[:, 0] = 1
    w = torch.zeros(1, 2 * I, H, dtype=torch.bfloat16)
    w[0, :len(g), 0], w[0, I:I + len(u), 0] = g, u
    act = torch.empty(rows, I, device="cuda", dtype=torch.bfloat16)
    _, s_tok, counts, offs, _, _ = hip.moe_sort(
        torch.zeros(rows, device="cuda", dtype=torch.int32), 1, 1)
    hip.moe_wide(False, act, x.cuda(), w.cuda(), s_tok, offs, counts)
    for row in (0, rows - 1):
        check_large(act[row, :len(g)], ref)


@pytest.mark.gpu
@needs_gpu
def test_refused():
    hip = ops._load_hip()
    z = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)
    i = lambda n: torch.zeros(n, device="cuda", dtype=torch.int32)
    up = lambda x, w, E=1, n=4: hip.moe_wide(False, z(n, w.shape[1] // 2), x, w,
                                             i(n), i(E), i(E))
    up(z(4, 192), z(1, 256, 192))                     # no rows: nothing to do
    for bad in (lambda: up(z(4, 128), z(1, 256, 128)),    # two steps of k
                lambda: up(z(4, 200), z(1, 256, 200)),
                lambda: up(z(4, 192), z(257, 32, 192), 257),
                lambda: up(z(4, 256), z(1, 256, 192)),
                lambda: hip.moe_wide(True, z(4, 128), z(4, 192), z(1, 128, 192),
                                     i(4), i(1), i(1))):  # no weights
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.parametrize("E,H,I", [(128, 2048, 768), (64, 2048, 1408),
                                   (8, 4096, 14336)])
def test_rule(E, H, I):
    assert not ops.moe_wide_wins(127 * E, E, I, H, False)
    assert ops.moe_wide_wins(250 * E, E, I, H, False)
    assert ops.moe_wide_wins(250 * E, E, H, I, True)
    # two rounds for one and a third, of tiles half full
    assert not ops.moe_wide_wins(330 * 8, 8, 4096, 14336, True)
    assert not ops.moe_wide_wins(250 * 257, 257, I, H, False)
    assert not ops.moe_wide_wins(250 * E, E, I, H + 32, False)
    assert not ops.moe_wide_wins(250 * E, E, I + 4, H, False)
    # contrib past what 32 bits of offset reach
    assert not ops.moe_wide_wins(1 << 20, E, 2048, I, True)
