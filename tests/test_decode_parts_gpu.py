"""Decode attention whose keys are cut into parts: lengths at the edges of a
step (32 keys) and of a part (128), every group size, both cache types, and
batches large enough to stay whole."""
import math

import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _reference(q, kc, vc, bt, lens, scale):
    N, Hq, D = q.shape
    G = kc.shape[1]
    out = torch.empty(N, Hq, D, dtype=torch.float64, device=q.device)
    for i, n in enumerate(lens):
        j = torch.arange(n, device=q.device)
        blk = bt[i, j // 16].long()
        k = kc[blk, :, j % 16].double().repeat_interleave(Hq // G, 1)
        v = vc[blk, :, j % 16].double().repeat_interleave(Hq // G, 1)
        p = ((q[i].double() * k).sum(-1) * scale).softmax(0)
        out[i] = (p[:, :, None] * v).sum(0)
    return out


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (8, 4), (32, 8), (10, 2), (12, 2),
                                    (28, 4), (32, 4)])
@pytest.mark.parametrize("lens", [
    [1], [31, 32, 33], [127, 128, 129], [4095, 1, 300], [2049],
    [1 + 7 * i for i in range(300)], [1 + 61 * i for i in range(70)],
    [900 - 43 * i for i in range(20)]])
def test_parts_against_double(fp8, Hq, Hkv, lens):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(len(lens) + Hq + lens[0])
    maxb = (max(lens) + 15) // 16 + 3
    need = [(n + 15) // 16 for n in lens]
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    kc = rnd(sum(need) + 1, Hkv, 16, 128).bfloat16()
    vc = rnd(sum(need) + 1, Hkv, 16, 128).bfloat16()
    if fp8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    pages = torch.randperm(sum(need), generator=g, device="cuda").int()
    bt = torch.full((len(lens), maxb), sum(need), dtype=torch.int32,
                    device="cuda")
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = pages[at:at + n]
        at += n
    # what lies behind a sequence's end in its last page is not its own
    for i, n in enumerate(lens):
        if n % 16:
            for pool in (kc, vc):
                (pool.view(torch.uint8) if fp8 else pool)[
                    bt[i, need[i] - 1].long(), :, n % 16:] = \
                    0x7f if fp8 else float("nan")
    q = rnd(len(lens), Hq, 128).bfloat16()
    out = torch.empty_like(q)
    scale = 1 / math.sqrt(128)
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32,
                                       device="cuda"), scale)
    f = lambda t: t.float() if fp8 else t
    ref = _reference(q, f(kc), f(vc), bt, lens, scale)
    # the result is rounded to bf16 once (8 significant bits: half a step is at
    # most 2^-8 of the value);
    # everything before it is fp32, whose sums over n keys of size <= 5 and
    # exponentials stay within 1e-5 * 5 of the exact ones
    err = (out.double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 1e-4).all()), \
        float((err - ref.abs() * 2.0 ** -8).max())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("window", [1, 33, 128, 129, 1000])
def test_parts_of_a_window(monkeypatch, D, window):
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    lens = [4095, 1, 300, 1001, 1000, 160]
    g = torch.Generator(device="cuda").manual_seed(window + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    nb = (max(lens) + 15) // 16
    kc, vc = rnd(nb * len(lens), 2, 16, D), rnd(nb * len(lens), 2, 16, D)
    bt = torch.arange(nb * len(lens), device="cuda").int().view(len(lens), nb)
    # nothing outside the window counts: behind the end, in front of the first
    for i, n in enumerate(lens):
        j = torch.arange(nb * 16, device="cuda")
        j = j[(j >= n) | (j < n - window)]
        for pool in (kc, vc):
            pool[bt[i, j // 16].long(), :, j % 16] = float("nan")
    q = rnd(len(lens), 8, D)
    out = torch.empty_like(q)
    scale = 1 / math.sqrt(D)
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32,
                                       device="cuda"), scale, window=window)
    for i, n in enumerate(lens):
        j = torch.arange(max(0, n - window), n, device="cuda")
        k = kc[bt[i, j // 16].long(), :, j % 16].double()
        v = vc[bt[i, j // 16].long(), :, j % 16].double()
        p = ((q[i].double() * k.repeat_interleave(4, 1)).sum(-1) * scale)
        ref = (p.softmax(0)[:, :, None] * v.repeat_interleave(4, 1)).sum(0)
        err = (out[i].double() - ref).abs()
        # as above: one rounding to bf16, fp32 before it
        assert bool((err <= ref.abs() * 2.0 ** -8 + 1e-4).all()), (i, n)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,Hq,Hkv", [(64, 16, 2), (128, 8, 2), (128, 2, 2),
                                      (256, 8, 2)])
@pytest.mark.parametrize("lens", [[100, 1, 77], [2500, 1, 300, 1001, 160]])
@pytest.mark.parametrize("sink,window,softcap", [
    (True, 0, 0.0), (True, 129, 0.0), (False, 0, 20.0), (True, 129, 20.0)])
def test_sinks_and_softcap(monkeypatch, fp8, D, Hq, Hkv, lens, sink, window,
                           softcap):
    """In the one part of short sequences, and where the join adds the sink."""
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    g = torch.Generator(device="cuda").manual_seed(D + Hq + lens[0])
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    nb = (max(lens) + 15) // 16
    kc, vc = (rnd(nb * len(lens), Hkv, 16, D) for _ in range(2))
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
    bt = torch.randperm(nb * len(lens), generator=g, device="cuda").int() \
        .view(len(lens), nb)
    q = rnd(len(lens), Hq, D) * 3
    sinks = torch.randn(Hq, generator=g, device="cuda") * 3 if sink else None
    out = torch.empty_like(q)
    scale = 1 / math.sqrt(D)
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32,
                                       device="cuda"), scale, sinks=sinks,
                          window=window, softcap=softcap)
    rep = Hq // Hkv
    for i, n in enumerate(lens):
        j = torch.arange(max(0, n - window) if window else 0, n, device="cuda")
        k, v = (t.float()[bt[i, j // 16].long(), :, j % 16].double()
                .repeat_interleave(rep, 1) for t in (kc, vc))
        s = (q[i].double() * k).sum(-1) * scale              # [keys, Hq]
        if softcap:
            s = torch.tanh(s / softcap) * softcap
        if sink:
            s = torch.cat([s, sinks.double()[None]])
        p = s.softmax(0)[:len(j)]
        ref = (p[:, :, None] * v).sum(0)
        err = (out[i].double() - ref).abs()
        # as above: one rounding to bf16, fp32 before it
        assert bool((err <= ref.abs() * 2.0 ** -8 + 1e-4).all()), (i, n)
