"""Head norms and cache write of a projection that comes as fp32 parts, against the same
on the rows that a product's join leaves."""
import pytest
import torch

from gpustack_amd import ops

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("HQ,G,D,VW", [(4, 2, 64, 64), (16, 4, 128, 128),
                                       (3, 3, 256, 24), (5, 1, 128, 136)])
@pytest.mark.parametrize("T,n", [(1, 1), (21, 4), (128, 5), (37, 9)])
@pytest.mark.parametrize("mix", [False, True])
@pytest.mark.parametrize("later", [False, True])
def test_parts(HQ, G, D, VW, T, n, mix, later):
    nq, nk, nv, BS, nb = HQ * D, G * D, G * VW, 16, 30
    g = torch.Generator(device="cuda").manual_seed(T + n + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    parts = rnd(n, T, nq + nk + nv)
    x = parts[0].clone()
    for i in range(1, n):
        x += parts[i]
    rows = x.bfloat16()
    vf = rnd(T, nq + nk + nv).bfloat16()[:, nq + nk:] if mix else None
    lam = torch.tensor([0.3], device="cuda") if mix else None
    qw, kw = rnd(D) + 1, rnd(D) + 1
    pos = torch.arange(T, dtype=torch.int32, device="cuda") * 50
    slots = torch.arange(T, device="cuda") * 3 + 1
    slots[-1] = -1
    groups = torch.tensor([[t, 1] for t in range(T)], dtype=torch.int32,
                          device="cuda") if later else None
    outs = []
    for p in (None, parts):
        qkv = rows.clone() if p is None else torch.full_like(rows, 7.0)
        q = torch.zeros(T, nq, dtype=torch.bfloat16, device="cuda")
        kc = torch.zeros(nb, G, BS, D, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(nb, G, VW, BS, dtype=torch.bfloat16, device="cuda")
        ops.head_norm_store(q, qkv, nq, nk, qw, kw, D, 0.25, 1024, pos, vf, lam,
                            kc, vc, slots, 1e-5, page_groups=groups, parts=p)
        # values that were not mixed are what a later layer's mix reads
        outs.append((q, kc, vc) + (() if mix else (qkv[:, nq + nk:],)))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_heads_of_other_sizes_are_refused():
    T, D = 3, 40
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    w = torch.ones(D, device="cuda")
    i = torch.arange(T, device="cuda")
    with pytest.raises(RuntimeError, match="parts"):
        ops.head_norm_store(z(T, D), z(T, 3 * D), D, D, w, w, D, 0.0, 0, i.int(),
                            None, None, z(1, 1, 16, D), z(1, 1, D, 16), i, 1e-5,
                            parts=torch.zeros(2, T, 3 * D, device="cuda"))
    assert not ops.head_norm_parts_ok(T, D, D, z(16))


def test_pools_elsewhere():
    """Parts only where the key pool is at a 16-byte address; else rows, as before."""
    T, D, rnd = 5, 64, torch.randn(5, 192, device="cuda").bfloat16()
    pool = torch.zeros(16 * D + 8, dtype=torch.bfloat16, device="cuda")
    kc, res = pool[3:3 + 16 * D].view(1, 1, 16, D), []
    assert ops.head_norm_parts_ok(T, D, D, pool)
    assert not ops.head_norm_parts_ok(T, D, D, kc)
    w, i = torch.ones(D, device="cuda"), torch.arange(T, device="cuda")
    for k in (kc, torch.zeros(1, 1, 16, D, dtype=torch.bfloat16, device="cuda")):
        q, vc = torch.zeros(T, D, device="cuda").bfloat16(), kc.new_zeros(1, 1, D, 16)
        ops.head_norm_store(q, rnd.clone(), D, D, w, w, D, 0.0, 0, i.int(), None, None,
                            k, vc, i, 1e-5)
        res.append((q, k, vc))
    for a, b in zip(*res):            # the sum of the squares in another order
        assert bool(((a - b).abs().float() <= b.abs().float() * 2.0 ** -7).all())
