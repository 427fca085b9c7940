"""The prompt kernel of ops.paged_attention: which rows take it, and its
results at the edges of its tiles (128 query rows, 32 rows a wave, 64 keys in
two turns, 16 a page), windows, slopes and sinks."""
import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.models.llama import RaggedMeta

GPU = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(),
                                           reason="needs a GPU")]


def _meta(seqs):
    news = [n for _, n in seqs]
    starts = [sum(news[:i]) for i in range(len(news))]
    z = torch.zeros(1, 1, dtype=torch.int32)
    return RaggedMeta(z, z, z, z, starts, [h for h, _ in seqs], news,
                      max_ctx=max(h + n for h, n in seqs))


@pytest.mark.parametrize("seqs", [
    [(0, 1)], [(0, 31)], [(0, 32)], [(5, 1), (0, 300), (7, 1)],
    [(3000, 200)], [(3000, 200), (0, 700), (9, 31), (100, 1)],
    [(2000, 32)] * 8, [(2000, 16)] * 32])
@pytest.mark.parametrize("heads,kv_heads", [(16, 4), (8, 8), (6, 2)])
@pytest.mark.parametrize("window", [0, 100, 1024])
def test_every_row_and_head_has_one_tile(seqs, heads, kv_heads, window):
    m = _meta(seqs)
    prompt = m.prompt_tiles(heads, window)
    tiles = m.attn_tiles(heads, kv_heads, 1, short=prompt is not None)
    seen = torch.zeros(sum(m.seq_news), heads, dtype=torch.int64)
    for row0, n, a0, na, seq, step in tiles.tolist():
        assert m.seq_starts[seq] <= row0
        assert row0 + n <= m.seq_starts[seq] + m.seq_news[seq]
        seen[row0:row0 + n, a0:a0 + na * step:step] += 1
    if prompt is not None:
        for row0, q0, hist, new, seq in prompt.T.tolist():
            assert (row0, hist, new) == (m.seq_starts[seq], m.seq_hists[seq],
                                         m.seq_news[seq])
            seen[row0 + q0:row0 + min(q0 + 128, new)] += 1
    assert bool((seen == 1).all())


@pytest.mark.parametrize("news,ctx,heads,window,wins", [
    ([512], 1512, 16, 0, False), ([512], 4512, 16, 0, False),
    ([512], 8512, 16, 1024, False), ([1000], 9000, 16, 0, True),
    ([700], 1700, 16, 0, False), ([300, 300], 8300, 16, 0, False),
    ([768], 1768, 16, 0, True), ([200] * 8, 2200, 8, 1024, True),
    ([128] * 8, 8128, 8, 0, False), ([100], 300, 16, 0, False),
    ([300], 300, 16, 0, False), ([64], 64, 16, 0, True), ([31], 31, 64, 0, False),
    ([1] * 512, 9000, 64, 0, False)])
def test_where_the_prompt_kernel_runs(news, ctx, heads, window, wins):
    assert ops.prompt_kernel_wins(news, ctx, heads, window) == wins


@pytest.mark.parametrize("heads,kv_heads", [(16, 4), (3, 1)])
@pytest.mark.parametrize("window", [0, 1, 33, 64, 200])
@pytest.mark.parametrize("option", ["", "slopes", "sinks"])
@pytest.mark.parametrize("seqs", [
    [(0, 1)], [(0, 32), (15, 33)], [(1, 127), (64, 129), (0, 96)],
    [(1000, 65), (0, 513)], [(31, 400)]])
class TestPrompts:
    pytestmark = GPU

    def test_against_float64(self, seqs, option, window, heads, kv_heads):
        g = torch.Generator(device="cuda").manual_seed(window + heads)
        rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
        m = _meta(seqs)
        need = [(h + n + 15) // 16 for h, n in seqs]
        kc = rnd(sum(need) + 1, kv_heads, 16, 128).bfloat16()
        vc = rnd(sum(need) + 1, kv_heads, 128, 16).bfloat16()
        pages = torch.randperm(sum(need), generator=g, device="cuda").int()
        bt = torch.full((len(seqs), max(need)), sum(need), dtype=torch.int32,
                        device="cuda")
        at = 0
        for i, (n, (h, new)) in enumerate(zip(need, seqs)):
            bt[i, :n] = pages[at:at + n]
            at += n
            if (h + new) % 16:        # not the sequence's: never multiplied
                last = int(bt[i, n - 1])
                kc[last, :, (h + new) % 16:] = float("nan")
                vc[last, :, :, (h + new) % 16:] = float("nan")
        T = sum(m.seq_news)
        q = (rnd(T, heads, 128) * 3).bfloat16()
        slopes = 2.0 ** (-8.0 * (torch.arange(heads, device="cuda") + 1.0)
                         / heads) if option == "slopes" else None
        sinks = rnd(heads) * 3 if option == "sinks" else None
        scale = 128 ** -0.5
        old = ops.PROMPT_PORTION
        try:
            ops.PROMPT_PORTION = 1
            prompt = ops.build_prompt_tiles(m.seq_starts, m.seq_hists,
                                            m.seq_news, "cuda")
        finally:
            ops.PROMPT_PORTION = old
        out = torch.full_like(q, 9.0)
        none = torch.empty(0, 6, dtype=torch.int32, device="cuda")
        pos = torch.zeros(T, dtype=torch.int32, device="cuda")
        ops.paged_attention(out, q, kc, vc, bt, None, pos, scale,
                            window=window, sinks=sinks, tiles=none,
                            slopes=slopes, prompt_tiles=prompt)
        for i, (h, n) in enumerate(seqs):
            j = torch.arange(h + n, device="cuda")
            blk = bt[i, j // 16].long()
            rep = heads // kv_heads
            k = kc[blk, :, j % 16].double().repeat_interleave(rep, 1)
            v = vc[blk, :, :, j % 16].double().repeat_interleave(rep, 1)
            s = m.seq_starts[i]
            x = torch.matmul(q[s:s + n].double().transpose(0, 1),
                             k.permute(1, 2, 0).contiguous()) * scale
            p = torch.arange(h, h + n, device="cuda")
            away = (p[:, None] - j[None, :]).double()
            if slopes is not None:
                x = x - slopes.double()[:, None, None] * away
            hide = (away < 0) | ((away >= window) if window else away < 0)
            x = x.masked_fill(hide, float("-inf"))
            if sinks is not None:
                x = torch.cat([x, sinks.double()[:, None, None]
                               .expand(-1, n, 1)], -1)
            w = x.softmax(-1)[..., :h + n]
            vt = v.transpose(0, 1).contiguous()
            ref = torch.matmul(w, vt).transpose(0, 1)
            # weights are rounded to bf16 (2^-8 of each at most), the result
            # once more; the rest is fp32
            bound = torch.matmul(w, vt.abs()).transpose(0, 1) * 2.0 ** -8 \
                + ref.abs() * 2.0 ** -8 + 1e-4
            err = (out[s:s + n].double() - ref).abs()
            assert bool((err <= bound).all()), (i, float((err - bound).max()))
