"""Row kernels of prompts in stacks of recurrent layers: parts of a wave, value pages by
16 bytes, embeddings, convolutions inside one sequence and across several, and the
activation that they share."""
import math

import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.ops import torch_ref

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _rnd(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return lambda *s: torch.randn(*s, generator=g, device="cuda")


@pytest.mark.parametrize("gs,groups", [(264, 3), (504, 2), (512, 8), (520, 2),
                                       (1016, 3), (1024, 2)])
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("T", [1, 7])
def test_parts_of_a_wave(gs, groups, first, T):
    _parts(gs, groups, first, T)


@pytest.mark.parametrize("gs,groups", [(264, 3), (512, 8), (520, 2), (1024, 2)])
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_many_parts(gs, groups, first, more):
    """Around 6144 of them, from where on a wave has a part; the last workgroup full and
    not."""
    _parts(gs, groups, first, 6144 // groups + more)


def _parts(gs, groups, first, T):
    rnd, C = _rnd(gs + groups), gs * groups
    y, gate, w = rnd(T, C) * 3, rnd(T, C + 16).bfloat16()[:, 8:8 + C], rnd(C)
    o = torch.zeros(T, C, dtype=torch.bfloat16, device="cuda")
    ops.gated_group_norm(o, y, gate, w, groups, 1e-5, first)
    u, z = y.double(), gate.double()
    if first:
        u = u * z * torch.sigmoid(z)
    v = u.view(T, groups, gs)
    v = (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-5)).reshape(T, C) * w.double()
    if not first:
        v = v * torch.sigmoid(z)
    assert bool(((o.double() - v).abs() <= v.abs() * (2.0 ** -8 + 1e-5)).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("G,VW,skew", [(4, 128, 0), (3, 24, 0), (5, 13, 0), (9, 128, 0),
                                       (4, 128, 1), (3, 24, 2), (9, 128, 4)])
def test_value_pages(dtype, G, VW, skew):
    """By 16 bytes and (odd widths, rows at other addresses) value by value; whole
    pages, a page's part, rows without a slot."""
    D, nq, nb, T = 64, 64, 9, 40
    nk, nv, rnd = G * D, G * VW, _rnd(G + VW)
    rows = rnd(T, nq + nk + nv).to(dtype)
    flat = torch.empty(rows.numel() + 8, dtype=dtype, device="cuda")
    slots = torch.full((T,), -1, dtype=torch.long, device="cuda")
    slots[:16] = torch.arange(48, 64, device="cuda")
    slots[16:32] = torch.arange(96, 112, device="cuda")
    slots[32:37] = torch.arange(130, 135, device="cuda")
    groups = torch.tensor([[0, 16], [16, 16], [32, 5], [37, 3]], dtype=torch.int32,
                          device="cuda")
    pos = torch.arange(T, dtype=torch.int32, device="cuda")
    w = torch.ones(D, device="cuda")
    res = []
    for impl in (ops, torch_ref):
        q = torch.zeros(T, nq, dtype=dtype, device="cuda")
        kc = torch.zeros(nb, G, 16, D, dtype=dtype, device="cuda")
        vc = torch.zeros(nb, G, VW, 16, dtype=dtype, device="cuda")
        qkv = flat[skew:skew + rows.numel()].view_as(rows)
        qkv.copy_(rows)
        assert qkv.data_ptr() % 16 == skew * qkv.element_size() % 16
        args = (q, qkv, nq, nk, w, w, D, 0.0, 0, pos, None, None, kc, vc, slots, 1e-5)
        if impl is ops:
            ops.head_norm_store(*args, page_groups=groups)
        else:
            impl.head_norm_store(*args)
        res.append(vc)
    assert torch.equal(*res)


@pytest.mark.parametrize("W", [8, 264, 2048, 2056, 1030])
def test_embedding(W):
    table = _rnd(W)(11, W).bfloat16()
    ids = torch.tensor([0, 10, 3, -2, 12], device="cuda")
    x = torch.empty(5, W, device="cuda")
    ops.embed_rows_scaled(x, ids, table, 1.7)
    assert torch.equal(x, table.float()[ids.clamp(0, 10)] * torch.tensor(1.7).cuda())


@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("news,C", [
    ([8, 8], 264), ([1, 40, 2, 3, 21, 8, 16], 264), ([300], 264),
    # from 2^20 numbers on eight rows a lane: groups that begin 0 to 7 rows into a
    # sequence, lie across two or more of them, and end behind the last row
    ([300], 4096), ([16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27], 4104),
    ([1, 40, 2, 3, 21, 8, 16, 1, 1, 1, 5, 60, 64, 40], 4096), ([1] * 37, 30000)])
@pytest.mark.parametrize("silu", [True, False])
def test_convolution(taps, news, C, silu):
    rnd = _rnd(sum(news) + taps)
    T, S = sum(news), len(news)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    first = [sum(news[:i]) for i in range(S)]
    hists = [(i % 3) * 2 for i in range(S)]
    view = (i32(first), i32(news), i32(list(range(S))),
            i32([s for s, n in enumerate(news) for _ in range(n)]),
            i32([h + j for h, n in zip(hists, news) for j in range(n)]))
    src, w, b = rnd(T, C + 8).bfloat16(), rnd(C, taps), rnd(C)
    st = rnd(S, taps - 1, C).bfloat16()
    out = torch.zeros(T, C, dtype=torch.bfloat16, device="cuda")
    ops.short_conv(out, src, 8, w, b, st.clone(), view[0], view[1], view[2], view[3],
                   view[4], silu=silu)
    for s, n in enumerate(news):
        old = st[s].double().clone()
        if hists[s] < taps - 1:
            old[:taps - 1 - hists[s]] = 0
        x = torch.cat([old, src[first[s]:first[s] + n, 8:].double()])
        v = b.double() + sum(x[k:k + n] * w[:, k].double() for k in range(taps))
        if silu:
            v = v * torch.sigmoid(v)
        e = (out[first[s]:first[s] + n].double() - v).abs()
        assert bool((e <= v.abs() * 2.0 ** -8 + 1e-5).all())


def test_activation_of_all_sizes():
    """Through the convolution of one tap: to an ulp of bf16 and, where nothing rounds,
    the limits."""
    z = torch.tensor([0.0, -0.0, 1e-3, -1e-3, 1.0, -1.0, 20.0, -20.0, -80.0, -88.5, -89.0,
                      -127.0, -1e30, 88.0, 1e30, math.inf, math.nan] + [2.0] * 7)
    C = z.numel()
    src = z.bfloat16().cuda().view(1, C).repeat(24, 1).contiguous()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    out = torch.zeros(24, C, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(C, 2, device="cuda")
    w[:, 1] = 1
    ops.short_conv(out, src, 0, w, None, torch.zeros(1, 1, C, dtype=torch.bfloat16,
                                                     device="cuda"),
                   i32([0]), i32([24]), i32([0]), i32([0] * 24), i32(list(range(24))),
                   silu=True)
    x = src.double()
    want = torch.where(x < -700, torch.zeros_like(x), x / (1 + torch.exp(-x)))
    rows = out[1:].double()               # an infinity times the weight 0 is none
    ok = torch.isfinite(src[1:].float())
    e = (rows - want[1:]).abs()
    assert bool((e[ok] <= want[1:].abs()[ok] * 2.0 ** -8 + 1e-36).all())
    assert bool(rows[src[1:].isnan()].isnan().all())


def test_activation_in_fp32():
    """Every result that fp32 holds to within three halves of its last place (the power
    of two has one, the quotient one half), those near the end of the range, where the
    exponential is largest, too; normal numbers on average nearer than expf and a division
    bring these (3.95e-8)."""
    g = torch.Generator().manual_seed(4)
    z = torch.cat([torch.randn(1 << 18, generator=g),
                   torch.rand(1 << 17, generator=g) * 176 - 88,
                   torch.rand(1 << 14, generator=g) * 1.4 - 88.7,
                   torch.linspace(-17, -16, 1 << 15)]).cuda()
    C, i32 = z.numel(), lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    src = torch.cat([torch.zeros(1, C, device="cuda"), z[None]])
    w = torch.zeros(C, 2, device="cuda")
    w[:, 1] = 1
    out = torch.zeros(2, C, device="cuda")
    ops.short_conv(out, src, 0, w, None, torch.zeros(1, 1, C, device="cuda"), i32([0]),
                   i32([2]), i32([0]), i32([0, 0]), i32([0, 1]), silu=True)
    want = z.double() / (1 + torch.exp(-z.double()))
    e = (out[1].double() - want).abs()
    assert bool((e <= want.abs() * 1.5 * 2.0 ** -23).all()), \
        float((e / want.abs()).max())
    n = 1 << 18
    assert float(e[:n].norm() / want[:n].norm()) <= 3.9e-8
