"""Prompt attention at the edges of its tiles (128 query rows, 64 keys, 32
rows a wave, 16 a page), whole prompts as views of a fused projection and rows
behind a cached history in shuffled pages."""
import math

import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _check(out, q, k, v, hist, scale):
    """out / q [n, Hq, D] of one sequence, k / v [hist + n, G, D]."""
    n, Hq, _ = q.shape
    rep = Hq // k.shape[1]
    k = k.double().repeat_interleave(rep, 1).transpose(0, 1)
    v = v.double().repeat_interleave(rep, 1).transpose(0, 1)
    s = torch.matmul(q.double().transpose(0, 1),
                     k.transpose(1, 2).contiguous()) * scale
    hide = torch.arange(k.shape[1], device=q.device)[None, :] > \
        torch.arange(hist, hist + n, device=q.device)[:, None]
    p = s.masked_fill(hide, float("-inf")).softmax(-1)
    ref = torch.matmul(p, v).transpose(0, 1)
    # weights are rounded to bf16 (2^-8 of each at most), the result once more;
    # the rest is fp32
    bound = torch.matmul(p, v.abs()).transpose(0, 1) * 2.0 ** -8 \
        + ref.abs() * 2.0 ** -8 + 1e-4
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (32, 8), (16, 2), (6, 2)])
@pytest.mark.parametrize("lens", [
    [1], [31, 32, 33], [63, 64, 65, 2], [127, 128, 129], [200, 1, 257, 16],
    [1000]])
def test_whole_prompts(Hq, Hkv, lens):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(sum(lens) + Hq)
    qkv = torch.randn(sum(lens), (Hq + 2 * Hkv) * 128, generator=g,
                      device="cuda").bfloat16()
    q, k, v = (qkv[:, a * 128:b * 128].unflatten(1, (b - a, 128))
               for a, b in ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    q = q * 3          # scores whose maximum moves by more than the slack
    out = torch.full((sum(lens), Hq, 128), 9.0, device="cuda").bfloat16()
    scale = 1 / math.sqrt(128)
    ops.varlen_prefill_attn(out, q, k, v, lens, scale)
    at = 0
    for n in lens:
        _check(out[at:at + n], q[at:at + n], k[at:at + n], v[at:at + n], 0,
               scale)
        at += n


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (8, 8)])
@pytest.mark.parametrize("seqs", [
    [(0, 1)], [(1, 127), (15, 129)], [(16, 64), (17, 33), (63, 1)],
    [(64, 200)], [(1000, 130), (0, 300)]])
def test_rows_behind_history(Hq, Hkv, seqs):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(seqs[0][0] + Hq)
    need = [(h + n + 15) // 16 for h, n in seqs]
    pools = [torch.randn(sum(need) + 1, Hkv, 16, 128, generator=g,
                         device="cuda").bfloat16() for _ in range(2)]
    pages = torch.randperm(sum(need), generator=g, device="cuda")
    bt = torch.full((len(seqs), max(need)), sum(need), dtype=torch.int32,
                    device="cuda")
    at, starts, rows = 0, [], 0
    for i, (n, (_, new)) in enumerate(zip(need, seqs)):
        bt[i, :n] = pages[at:at + n].int()
        at += n
        starts.append(rows)
        rows += new
    # what lies behind a sequence's end in its last page is not its own
    for i, (h, n) in enumerate(seqs):
        if (h + n) % 16:
            pools[0][bt[i, need[i] - 1].long(), :, (h + n) % 16:] = float("nan")
            pools[1][bt[i, need[i] - 1].long(), :, (h + n) % 16:] = float("nan")
    q = (torch.randn(rows, Hq, 128, generator=g, device="cuda") * 3).bfloat16()
    out = torch.full_like(q, 9.0)
    scale = 1 / math.sqrt(128)
    ops.paged_prefill_attn(out, q, *pools, bt, starts, [h for h, _ in seqs],
                           [n for _, n in seqs], scale)
    for i, (h, n) in enumerate(seqs):
        j = torch.arange(h + n, device="cuda")
        blk = bt[i, j // 16].long()
        st = starts[i]
        _check(out[st:st + n], q[st:st + n], pools[0][blk, :, j % 16],
               pools[1][blk, :, j % 16], h, scale)


@pytest.mark.parametrize("rows", [64, 128])
def test_tile_lists_of_either_size(rows):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(rows)
    lens = [1, 64, 65, 193]
    q = torch.randn(sum(lens), 8, 128, generator=g, device="cuda").bfloat16()
    k, v = (torch.randn(sum(lens), 2, 128, generator=g,
                        device="cuda").bfloat16() for _ in range(2))
    out = torch.full_like(q, 9.0)
    ops.varlen_prefill_attn(out, q, k, v, lens, 0.1, tiles=ops.
                            build_prefill_tiles(lens, "cuda", rows))
    at = 0
    for n in lens:
        _check(out[at:at + n], q[at:at + n], k[at:at + n], v[at:at + n], 0,
               0.1)
        at += n


@pytest.mark.parametrize("pad,scale", [(0, 0.1), (8, 0.1), (4, 0.1), (1, 0.1),
                                       (0, -0.1), (0, 0.0)])
def test_rows_and_factors_of_either_kernel(pad, scale):
    """Key and value rows at 16-byte addresses or not, and factors under which
    the largest unscaled score is not the largest one."""
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(pad)
    lens, Hq, Hkv = [1, 95, 96, 97, 385], 8, 2
    qkv = torch.randn(sum(lens), (Hq + 2 * Hkv) * 128 + pad, generator=g,
                      device="cuda").bfloat16()
    q, k, v = (qkv[:, pad + a * 128:pad + b * 128].unflatten(1, (b - a, 128))
               for a, b in ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    q = (q * 3).contiguous()
    out = torch.full((sum(lens), Hq, 128), 9.0, device="cuda").bfloat16()
    ops.varlen_prefill_attn(out, q, k, v, lens, scale)
    at = 0
    for n in lens:
        _check(out[at:at + n], q[at:at + n], k[at:at + n], v[at:at + n], 0,
               scale)
        at += n


@pytest.mark.parametrize("n", [40, 200])
@pytest.mark.parametrize("at", range(0, 32, 4))
def test_one_key_far_above_the_others(n, at):
    """Four keys of 32 whose scores are 300 above all others (more than the
    exponent of a float holds): whichever lanes hold them."""
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(at)
    q, k, v = (torch.randn(n, h, 128, generator=g, device="cuda")
               for h in (8, 2, 2))
    q[..., 0] = 64.0
    k[..., 0] = 0.0
    k[at:at + 4, :, 0] = 64.0
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    out = torch.full_like(q, 9.0)
    ops.varlen_prefill_attn(out, q, k, v, [n], 0.1)
    _check(out, q, k, v, 0, 0.1)


def _check_variant(out, q, k, v, hist, scale, sinks, window, softcap):
    """out [n, Hq, DV], q [n, Hq, D] of one sequence, k / v [hist + n, G, .]"""
    n, Hq, _ = q.shape
    rep = Hq // k.shape[1]
    k, v = (t.double().repeat_interleave(rep, 1).transpose(0, 1)
            for t in (k, v))
    s = torch.matmul(q.double().transpose(0, 1),
                     k.transpose(1, 2).contiguous()) * scale
    if softcap:
        s = torch.tanh(s / softcap) * softcap
    at = torch.arange(hist, hist + n, device=q.device)[:, None]
    kv = torch.arange(hist + n, device=q.device)[None, :]
    hide = (kv > at) | (kv <= at - window if window else kv < 0)
    s = s.masked_fill(hide, float("-inf"))
    if sinks is not None:
        s = torch.cat([s, sinks.double()[:, None, None].expand(Hq, n, 1)], -1)
    p = s.softmax(-1)[:, :, :hist + n]
    ref = torch.matmul(p, v).transpose(0, 1)
    # as in _check
    bound = torch.matmul(p, v.abs()).transpose(0, 1) * 2.0 ** -8 \
        + ref.abs() * 2.0 ** -8 + 1e-4
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


_VARIANTS = pytest.mark.parametrize("sink,window,softcap", [
    (False, 0, 0.0), (True, 0, 0.0), (False, 1, 0.0), (True, 128, 0.0),
    (False, 65, 30.0), (True, 0, 30.0)])
_HEADS = pytest.mark.parametrize("D,Hq,Hkv", [(64, 16, 2), (128, 8, 4),
                                              (256, 4, 2)])


@_VARIANTS
@_HEADS
@pytest.mark.parametrize("lens", [
    [1], [31, 33, 64], [65, 77, 2], [127, 128, 129], [300]])
def test_variants_of_whole_prompts(monkeypatch, D, Hq, Hkv, lens, sink, window,
                                   softcap):
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    T = sum(lens)
    q, k, v = rnd(T, Hq, D) * 3, rnd(T, Hkv, D), rnd(T, Hkv, D)
    sinks = torch.randn(Hq, generator=g, device="cuda") * 3 if sink else None
    out = torch.full_like(q, 9.0)
    scale = 1 / math.sqrt(D)
    ops.varlen_prefill_attn(out, q, k, v, lens, scale, sinks=sinks,
                            window=window, softcap=softcap)
    at = 0
    for n in lens:
        r = slice(at, at + n)
        _check_variant(out[r], q[r], k[r], v[r], 0, scale, sinks, window,
                       softcap)
        at += n


@_VARIANTS
@_HEADS
@pytest.mark.parametrize("seqs", [
    [(0, 1)], [(1, 127), (15, 129)], [(17, 33), (63, 1), (64, 64)],
    [(500, 77), (0, 130)]])
def test_variants_behind_history(monkeypatch, D, Hq, Hkv, seqs, sink, window,
                                 softcap):
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    g = torch.Generator(device="cuda").manual_seed(seqs[0][0] + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    nb = max((h + n + 15) // 16 for h, n in seqs)
    kc, vc = (rnd(nb * len(seqs), Hkv, 16, D) for _ in range(2))
    bt = torch.randperm(nb * len(seqs), generator=g, device="cuda").int() \
        .view(len(seqs), nb)
    starts = [sum(n for _, n in seqs[:i]) for i in range(len(seqs))]
    # what lies behind a sequence's end in its last page is not its own
    for i, (h, n) in enumerate(seqs):
        j = torch.arange(h + n, (h + n + 15) // 16 * 16, device="cuda")
        for pool in (kc, vc):
            pool[bt[i, j // 16].long(), :, j % 16] = float("nan")
    q = rnd(sum(n for _, n in seqs), Hq, D) * 3
    sinks = torch.randn(Hq, generator=g, device="cuda") * 3 if sink else None
    out = torch.full_like(q, 9.0)
    scale = 1 / math.sqrt(D)
    ops.paged_prefill_attn(out, q, kc, vc, bt, starts, [h for h, _ in seqs],
                           [n for _, n in seqs], scale, sinks=sinks,
                           window=window, softcap=softcap)
    for i, (h, n) in enumerate(seqs):
        j = torch.arange(h + n, device="cuda")
        blk = bt[i, j // 16].long()
        r = slice(starts[i], starts[i] + n)
        _check_variant(out[r], q[r], kc[blk, :, j % 16], vc[blk, :, j % 16], h,
                       scale, sinks, window, softcap)


@pytest.mark.parametrize("lens", [[1], [33, 64, 65], [129, 200]])
def test_keys_wider_than_values(monkeypatch, lens):
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_MLA_KERNEL", "1")
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    T = sum(lens)
    q, k, v = rnd(T, 16, 192) * 3, rnd(T, 16, 192), rnd(T, 16, 128)
    out = torch.full_like(v, 9.0)
    scale = 1 / math.sqrt(192)
    ops.varlen_prefill_attn(out, q, k, v, lens, scale)
    at = 0
    for n in lens:
        r = slice(at, at + n)
        _check_variant(out[r], q[r], k[r], v[r], 0, scale, None, 0, 0.0)
        at += n


# launches of one tile more than the chip takes at a time, of twice as many and one more
# (256 workgroups, a tile is one a head), whose tiles start in another order
@pytest.mark.parametrize("Hq,Hkv,lens", [
    (32, 8, [1025]), (32, 8, [700, 1, 1200]), (32, 8, [2048]), (32, 8, [2049]),
    (64, 8, [513]), (64, 8, [500, 500]), (16, 2, [4100]), (28, 4, [1300])])
def test_every_tile_of_a_launch_that_fills_the_chip(Hq, Hkv, lens):
    test_whole_prompts(Hq, Hkv, lens)
