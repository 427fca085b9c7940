"""A decode step's rows from the projection to attention in one launch, against the row
kernel and the attention behind it, to the bit: lengths at the edges of pages, steps and
parts, whole rows and parts of a product, pools in bf16 and fp8."""
import pytest
import torch

from gpustack_amd import ops

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]
D = 128


def _step(lens, Hq, Hkv, kv="bf16", n=0, norm=False, wide=0, slots=None, seed=0):
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + Hq + n + seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    N, W = len(lens), (Hq + 2 * Hkv) * D
    pages = [(x + 15) // 16 for x in lens]
    nb = sum(pages) + 1
    pools = [rnd(nb, Hkv, 16, D) for _ in range(2)]
    pools = [t.to(torch.float8_e4m3fn) if kv == "fp8" else t.bfloat16() for t in pools]
    bt = torch.full((N, max(max(pages), wide)), nb - 1, dtype=torch.int32)
    order = torch.randperm(nb - 1, generator=torch.Generator().manual_seed(3)).int()
    at, place = 0, []
    for i, p in enumerate(pages):
        bt[i, :p] = order[at:at + p]
        at += p
        place.append(int(bt[i, p - 1]) * 16 + (lens[i] - 1) % 16)
    for i, s in (slots or {}).items():
        place[i] = s if s < 0 else (nb - 1) * 16 + s      # a page that nobody reads
    i64 = lambda v: torch.tensor(v, dtype=torch.long, device="cuda")
    pos, slot = i64([x - 1 for x in lens]), i64(place)
    bt = bt.cuda()
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    ang = torch.arange(max(lens), device="cuda")[:, None] \
        * 500.0 ** (-torch.arange(64, device="cuda") / 64.0)
    cs = torch.cat([ang.cos(), ang.sin()], 1).contiguous()
    qn, kn = ((rnd(D) + 1).bfloat16() for _ in range(2)) if norm else (None, None)
    rows = rnd(n, N, W) if n else rnd(N, W).bfloat16()
    res = []
    for fused in (False, True):
        kc, vc = (t.clone() for t in pools)
        out = torch.full((N, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
        if fused:
            ops.paged_attn_decode_rows(out, rows, Hq, Hkv, qn, kn, cs, pos, slot, kc,
                                       vc, bt, sl, 1e-5, D ** -0.5)
        else:
            qkv = torch.empty(N, W, dtype=torch.bfloat16, device="cuda") if n \
                else rows.clone()
            ops.qkv_store(qkv, Hq, Hkv, qn, kn, cs, pos, slot, kc, vc, 1e-5,
                          rows if n else None)
            ops.paged_attn_decode(out, qkv[:, :Hq * D].unflatten(1, (Hq, D)), kc, vc,
                                  bt, sl, D ** -0.5)
        res.append([out] + [t.view(torch.uint8) for t in (kc, vc)])
    assert bool(res[0][0].isfinite().all())
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens", [[1], [2, 15, 16, 17], [31, 32, 33, 63, 64, 65],
                                  [127, 128, 129, 255, 256, 257], [1000, 1, 513, 300],
                                  [4500]])
@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (8, 4), (32, 4), (14, 2), (10, 2)])
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("n,wide", [(0, 0), (4, 400)])
def test_lengths(lens, Hq, Hkv, kv, n, wide):
    _step(lens, Hq, Hkv, kv, n, wide=wide)


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("n", [0, 1, 5, 9])
@pytest.mark.parametrize("N,norm", [(48, True), (300, False)])
def test_many_rows(kv, n, N, norm):
    """More than a workgroup a CU: one page a step in bf16."""
    _step([1 + (i * 37) % 211 for i in range(N)], 32, 8, kv, n, norm)


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("wide", [0, 300])
def test_rows_that_are_not_kept(kv, wide):
    """No slot, and one outside of the sequence: attention sees what the pool holds."""
    _step([40, 17, 900, 64], 32, 8, kv, 3, wide=wide, slots={1: -1, 3: 5, 2: -1},
          seed=5)


def test_where_it_is_taken():
    def ok(N, pages, dtype=torch.bfloat16, Hq=32, Hkv=8):
        kc = torch.zeros(1, Hkv, 16, D, device="cuda").to(dtype)
        return ops.paged_attn_decode_rows_ok(
            kc, Hq, Hkv, D, kc, kc, torch.zeros(N, pages, dtype=torch.int32))

    assert ok(1, 4) and ok(128, 7) and not ok(129, 7) and ok(129, 8)
    fp8 = torch.float8_e4m3fn
    assert ok(64, 4, fp8) and not ok(65, 400, fp8) and ok(128, 4, fp8, 32, 4)
    assert not ok(1, 4, Hq=24) and not ok(1, 4, Hq=8) and not ok(1, 4, Hq=72)


@pytest.mark.parametrize("skew", [0, 1, 4])
def test_head_norms_elsewhere(skew):
    """An attention layer whose head norms lie at any address takes a step of rows of
    their own, as it takes the same without saying that they are."""
    from types import SimpleNamespace

    from gpustack_amd.models.llama import Attention, ForwardMeta

    Hq, Hkv, N, H = 8, 2, 3, 256
    g = torch.Generator(device="cuda").manual_seed(skew)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    a = Attention.__new__(Attention)
    torch.nn.Module.__init__(a)
    a.spec = SimpleNamespace(qk_norm=True, qk_norm_full=False, qk_norm_after_rope=False,
                             rope_mode="neox", rms_norm_eps=1e-5, attn_temp_scale=0)
    a.comm = SimpleNamespace(all_reduce=lambda x: x)
    a.hq, a.hkv, a.d, a.rot_dim, a.scale = Hq, Hkv, D, D, D ** -0.5
    a.use_rope, a.sinks, a.window, a.softcap = True, None, 0, None
    a.qkv_w, a.o_w = rnd((Hq + 2 * Hkv) * D, H) / 16, rnd(H, Hq * D) / 32
    a.qkv_b = a.o_b = a.qkv_pack = a.o_pack = None
    a.q_norm, a.k_norm = (rnd(D + 8)[skew:skew + D] for _ in range(2))
    x, cs = rnd(N, H), torch.randn(64, D, generator=g, device="cuda")
    pools = [rnd(4, Hkv, 16, D) for _ in range(2)]
    pos = torch.tensor([5, 15, 0], device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    res = []
    for own in (False, True):
        kc, vc = (t.clone() for t in pools)
        meta = ForwardMeta(is_prefill=False, positions=pos,
                           slot_mapping=pos + torch.arange(N, device="cuda") * 16,
                           logits_indices=None, block_tables=i32([[0], [1], [2]]),
                           seq_lens=(pos + 1).int(), own_rows=own)
        res.append((a(x, meta, cs, kc, vc), kc, vc))
    for u, v in zip(*res):
        assert torch.equal(u, v)


def test_other_heads_are_refused():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    for Hq, Hkv, d in ((4, 4, 128), (6, 2, 128), (8, 2, 64)):
        kc = z(2, Hkv, 16, d)
        rows = z(1, (Hq + 2 * Hkv) * d)
        one = torch.ones(1, dtype=torch.int32, device="cuda")
        assert not ops.paged_attn_decode_rows_ok(rows, Hq, Hkv, d, kc, kc,
                                                 one.view(1, 1))
        with pytest.raises(RuntimeError, match="paged_attn_decode_rows"):
            ops.paged_attn_decode_rows(
                z(1, Hq, d), rows, Hq, Hkv, None, None,
                torch.zeros(4, d, device="cuda"), one.long() - 1, one.long() - 1, kc,
                kc.clone(), one.view(1, 1) - 1, one, 1e-5, 0.1)
