"""Paged attention of heads of 128 channels, a wave to its own 32 keys: contexts at the
edges of the tiles and of the waves' shares, against the fp32 path, with every option of
the two, and the number of parts that a batch takes."""
import pytest
import torch

from gpustack_amd import ops

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(),
                                           reason="needs a GPU")]


def _run(hists, news, H, G, VW, nsplit, maps=1, fp32=False, **kw):
    D, A = 128, H * maps
    g = torch.Generator(device="cuda").manual_seed(sum(hists) + VW + nsplit)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    pages = [(h + n + 15) // 16 for h, n in zip(hists, news)]
    kc, vc = (rnd(sum(pages) + 1, G, *s).bfloat16()
              for s in ((16, maps * D), (VW, 16)))
    bt = torch.zeros(len(hists), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(1))
    at = starts = 0
    start = []
    for i, n in enumerate(pages):
        bt[i, :n] = order[at:at + n].int()
        at += n
        start.append(starts)
        starts += news[i]
    q = rnd(starts, A, D).bfloat16()
    pos = torch.tensor([h + j for h, n in zip(hists, news) for j in range(n)],
                       dtype=torch.int32, device="cuda")
    tiles = ops.build_attn_tiles(start, hists, news, H, G, maps, "cuda")
    outs = []
    k = ops._paged_backend(q)
    for exact in (False, True):
        out = torch.full((starts, A, VW), 7.0, device="cuda",
                         dtype=torch.float32 if fp32 else torch.bfloat16)
        k.paged_attention(out, q, kc, vc, bt.cuda(), tiles, pos, D ** -0.5, maps,
                          kw.get("window", 0), kw.get("keep_first", 0),
                          kw.get("sinks"), exact, nsplit, kw.get("slopes"),
                          kw.get("softcap", 0.0), kw.get("chunk", 0), kw.get("gate"))
        outs.append(out.double())
    # weights rounded to bf16 (2^-8 of each at most, of values up to 6), results too
    assert float((outs[0] - outs[1]).abs().max()) < 6 * 2.0 ** -8 \
        + 2.0 ** -8 * float(outs[1].abs().max())
    rel = float((outs[0] - outs[1]).norm() / outs[1].norm())
    assert rel < 2.0 ** -7, rel


@pytest.mark.parametrize("hists", [[0], [30, 31, 32, 33], [126, 127, 128, 129],
                                   [15, 16, 63, 64, 65], [1000, 3, 517]])
@pytest.mark.parametrize("nsplit", [1, 2, 5])
@pytest.mark.parametrize("H,G,VW", [(16, 4, 128), (4, 4, 80), (32, 2, 112)])
class TestEdges:
    pytestmark = gpu

    def test_decode_rows(self, hists, nsplit, H, G, VW):
        _run(hists, [1] * len(hists), H, G, VW, nsplit)

    def test_a_few_rows(self, hists, nsplit, H, G, VW):
        _run(hists, [3 + 20 * (i % 2) for i in range(len(hists))], H, G, VW, nsplit)


@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("kw", [
    {"window": 100}, {"window": 64, "keep_first": 5}, {"chunk": 96}, {"softcap": 20.0},
    {"maps": 2}, {"fp32": True}, {"sinks": True}, {"slopes": True}, {"gate": True}],
    ids=str)
class TestOptions:
    pytestmark = gpu

    def test_as_the_fp32_path(self, nsplit, kw):
        hists, news, H = [0, 97, 411, 1300], [1, 5, 1, 33], 16
        g = torch.Generator(device="cuda").manual_seed(4)
        per_head = lambda: torch.rand(H, generator=g, device="cuda")
        kw = dict(kw)
        if kw.get("gate"):
            kw["gate"] = torch.randn(sum(news), H, generator=g, device="cuda").bfloat16()
        for name in ("sinks", "slopes"):
            if name in kw:
                kw[name] = per_head()
        _run(hists, news, H, 4, 128, nsplit, **kw)


@pytest.mark.parametrize("S", [408, 409, 592, 593])
@pytest.mark.parametrize("VW", [128, 80])
class TestManyTiles:
    pytestmark = gpu

    def test_as_the_fp32_path(self, S, VW):
        """Two kv heads: 816, 818, 1184 and 1186 tiles, the edges between which each
        tile of channels is behind a branch."""
        _run([(i * 37) % 300 for i in range(S)], [1] * S, 8, 2, VW, 1, window=128)


@pytest.mark.parametrize("nsplit", [1, 2, 5])
@pytest.mark.parametrize("last", [32, 64, 96, 192])
class TestNotANumber:
    pytestmark = gpu

    @pytest.mark.parametrize("first", [True, False])
    def test_a_key_alone_in_a_share_shows(self, nsplit, last, first):
        """Key `last` begins a tile of 32: with no other in it, it may be the only
        one of a wave's share or of a part."""
        g = torch.Generator(device="cuda").manual_seed(last)
        rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
        H, G, n, at = 4, 2, last // 16 + 1, 0 if first else last
        kc, vc, q = rnd(2 * n, G, 16, 128), rnd(2 * n, G, 128, 16), rnd(2, H, 128)
        kc[at // 16, :, at % 16] = float("nan")
        bt = torch.arange(2 * n, dtype=torch.int32, device="cuda").view(2, n)
        pos = torch.full((2,), last, dtype=torch.int32, device="cuda")
        tiles = ops.build_attn_tiles([0, 1], [last, last], [1, 1], H, G, 1, "cuda")
        out = torch.zeros(2, H, 128, device="cuda", dtype=torch.bfloat16)
        ops._paged_backend(q).paged_attention(
            out, q, kc, vc, bt, tiles, pos, 128 ** -0.5, 1, 0, 0, None, False, nsplit,
            None, 0.0, 0, None)
        assert bool(out[0].isnan().all()) and bool(out[1].isfinite().all())


@pytest.mark.parametrize("ctx,window", [(8000, 0), (3000, 0), (20000, 4096)])
def test_parts_leave_few_cus_without_work(monkeypatch, ctx, window):
    taken = []

    class Kernel:
        def paged_attention(self, *a):
            taken.append(a[13])

    monkeypatch.setattr(ops, "_paged_backend", lambda t: Kernel())
    q = torch.zeros(1, 4, 128, dtype=torch.bfloat16)
    span = min(ctx, window or ctx)
    for nt in [1, 4, 60, 100, *range(128, 260, 4), 300, 400, 520, 800, 1500, 2047]:
        ops.paged_attention(q, q, None, None, None, None, None, 1., window=window,
                            tiles=torch.zeros(nt, 6, dtype=torch.int32), max_ctx=ctx)
        parts = taken.pop()
        assert 1 <= parts <= 16 and span // parts >= 128
        # partial sums of no more workgroups than with 64 keys to a tile
        assert parts == 1 or nt * parts <= 2048
        # whole rounds of the 256 CUs; a few tiles have a CU each
        rounds = -(-nt * parts // 256)
        assert nt * parts >= .7 * 256 * rounds or nt < 60
    ops.paged_attention(q, q, None, None, None, None, None, 1., max_ctx=500,
                        tiles=torch.zeros(132, 6, dtype=torch.int32))
    assert taken == [1]
