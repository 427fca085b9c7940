"""Decode attention of grouped heads at the edges of its steps: pages of 16 keys, one
page a wave (64 keys), one step of one and of two pages a wave (64 and 128), in batches
on both sides of the line between the two; pools that its direct loads do not take."""
import pytest
import torch

from test_decode_parts_gpu import _reference

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]

EDGES = [1, 15, 16, 17, 63, 64, 65, 79, 80, 81, 127, 128, 129, 191, 193, 257]


def _pools(lens, Hkv, D, fp8, seed, offset=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    need = [(n + 15) // 16 for n in lens]
    pools = []
    for _ in range(2):
        t = torch.randn(sum(need) + 1, Hkv, 16, D, generator=g, device="cuda") \
            .to(torch.float8_e4m3fn if fp8 else torch.bfloat16)
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda")
        flat[offset:].view(torch.uint8 if fp8 else t.dtype).copy_(
            t.view(torch.uint8 if fp8 else t.dtype).flatten())
        pools.append(flat[offset:].view(t.shape))
    # more columns than the sequences have pages: of a page that is none of theirs
    bt = torch.full((len(lens), max(need) + 9), sum(need), dtype=torch.int32,
                    device="cuda")
    pages = torch.randperm(sum(need), generator=g, device="cuda").int()
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = pages[at:at + n]
        at += n
        if lens[i] % 16:      # behind the end in the last page, and that page
            for pool in pools:
                (pool.view(torch.uint8) if fp8 else pool)[
                    bt[i, n - 1].long(), :, lens[i] % 16:] = \
                    0x7f if fp8 else float("nan")
    for pool in pools:
        (pool.view(torch.uint8) if fp8 else pool)[-1] = 0x7f if fp8 else float("nan")
    q = torch.randn(len(lens), 4 * Hkv, D, generator=g, device="cuda").bfloat16()
    return *pools, bt, q


def _check(out, q, kc, vc, bt, lens, fp8, rows):
    f = lambda t: t.float() if fp8 else t
    ref = _reference(q[rows], f(kc), f(vc), bt[rows], [lens[i] for i in rows],
                     q.shape[-1] ** -0.5)
    # one rounding to bf16 (half a step is at most 2^-8 of the value) of sums that
    # are fp32 or as good: within 1e-5 * 5 over values of size <= 5
    err = (out[rows].double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 1e-4).all()), \
        float((err - ref.abs() * 2.0 ** -8).max())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("copies", [1, 20])
def test_steps(monkeypatch, fp8, D, copies):
    """16 and 320 sequences (2 kv heads): up to and above one workgroup a CU; equal
    sequences give equal results."""
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    kc, vc, bt, q = _pools(EDGES, 2, D, fp8, D + copies)
    bt, q, lens = bt.repeat(copies, 1), q.repeat(copies, 1, 1), EDGES * copies
    out = torch.full_like(q, float("nan"))
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32, device="cuda"),
                          D ** -0.5)
    _check(out, q, kc, vc, bt, lens, fp8, list(range(len(EDGES))))
    assert bool((out.view(copies, len(EDGES), -1) == out[:16].view(16, -1)).all())


@pytest.mark.parametrize("lens", [[4000, 65, 1], [700] * 40])
@pytest.mark.parametrize("fp8", [False, True])
def test_pools_at_odd_places(lens, fp8):
    """Pools that begin at no multiple of 16 bytes, whole and in parts."""
    from gpustack_amd import ops

    kc, vc, bt, q = _pools(lens, 2, 128, fp8, len(lens), offset=1)
    assert kc.data_ptr() % 16
    out = torch.full_like(q, float("nan"))
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32, device="cuda"),
                          128 ** -0.5)
    _check(out, q, kc, vc, bt, lens, fp8, list(range(len(lens)))[:4])


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("lens", [[1, 40, 200, 1000], [150] * 300])
@pytest.mark.parametrize("G", [1, 4])
def test_infinite_values(monkeypatch, lens, D, G):
    """An infinity in the values comes out, whatever its key's weight (the largest one's
    is exactly 1), and a NaN only where two of them meet; one head a kv head or four."""
    from gpustack_amd import ops

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    kc, vc, bt, q = _pools(lens, 2, D, False, D + len(lens))
    q = q[:, :2 * G].contiguous()
    rows = list(range(min(len(lens), 4)))
    for i in rows:
        def at(j):                      # the place of key j
            return bt[i, j // 16].long(), slice(None), j % 16
        s = (q[i].view(2, G, D)[:, :, None].float() * torch.stack(
            [kc[at(j)] for j in range(lens[i])], 1)[:, None].float()).sum(-1)
        top = s[0, 0].argmax().item()   # the largest weight of the first head
        vc[at(top)][:, 3] = float("inf")
        vc[at(lens[i] - 1)][:, 5] = float("-inf")
        vc[at(0)][:, 7], vc[at(lens[i] // 2)][:, 9] = float("inf"), float("inf")
        vc[at(lens[i] - 1)][:, 9] = float("-inf")
    out = torch.full_like(q, float("nan"))
    ops.paged_attn_decode(out, q, kc, vc, bt,
                          torch.tensor(lens, dtype=torch.int32, device="cuda"),
                          D ** -0.5)
    ref = _reference(q[rows], kc, vc, bt[rows], [lens[i] for i in rows], D ** -0.5)
    out = out[rows].double()
    odd = ~ref.isfinite()
    assert int(odd.sum()) >= 4 * len(rows) * 2 * G
    assert torch.equal(out[odd].nan_to_num(nan=5.0), ref[odd].nan_to_num(nan=5.0))
    assert bool((out - ref)[~odd].abs().le(ref[~odd].abs() * 2.0 ** -8 + 1e-4).all())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("pages", [4, 5, 16, 17])
@pytest.mark.parametrize("copies", [1, 64, 65])
@pytest.mark.parametrize("extra", [False, True])
def test_two_heads(monkeypatch, fp8, D, pages, copies, extra):
    """Two query heads a kv head, behind tables up to and above 64 keys (pairs of 64
    channels) and 256 (parts of 128 keys); 8, 512 and 520 groups; with a window and sinks."""
    from gpustack_amd import ops
    from gpustack_amd.ops import torch_ref

    monkeypatch.setenv("GPUSTACK_AMD_OSS_KERNELS", "1")
    lens = [1, 33, 16 * pages - 15, 16 * pages]
    kc, vc, bt, q = _pools(lens, 2, D, fp8, D + pages)
    q = q[:, :4].repeat(copies, 1, 1)
    bt = bt[:, :pages].repeat(copies, 1)
    lens = lens * copies
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    more = {"window": 40, "sinks": torch.tensor([.5, -1., 3., 0.], device="cuda")} \
        if extra else {}
    out = torch.full_like(q, float("nan"))
    ops.paged_attn_decode(out, q, kc, vc, bt, sl, D ** -0.5, **more)
    if not extra:
        _check(out, q, kc, vc, bt, lens, fp8, [0, 1, 2, 3])
    ref = torch.empty_like(q[:4])
    clean = [t.float().nan_to_num().bfloat16() for t in (kc, vc)]
    torch_ref.paged_attn_decode(ref, q[:4], *clean, bt[:4], sl[:4], D ** -0.5, **more)
    assert bool(((out[:4] - ref).abs().float()         # both rounded to bf16
                 <= ref.abs().float() * 2.0 ** -7 + 1e-4).all())
    assert bool((out.view(copies, 4, -1) == out[:4].view(4, -1)).all())
