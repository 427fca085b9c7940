"""Head norm, rotation and cache write in one launch against the steps one by
one: every head size, with and without norms, both caches, rows without a
slot, and head counts that leave a workgroup part empty."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("D,Hq,Hk,T", [(128, 32, 8, 77), (128, 1, 1, 1),
                                       (64, 5, 5, 33), (256, 8, 2, 9),
                                       (128, 28, 4, 300)])
def test_against_single_steps(fp8, norm, D, Hq, Hk, T):
    from gpustack_amd import ops
    from gpustack_amd.ops import torch_ref as R

    g = torch.Generator(device="cuda").manual_seed(T * D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    qkv = rnd(T, (Hq + 2 * Hk) * D).bfloat16()
    qw, kw = ((1 + 0.1 * rnd(D)).bfloat16() for _ in range(2))
    cs = ops.build_cos_sin_cache(D, D, 4096).cuda()
    pos = torch.randint(0, 4096, (T,), generator=g, device="cuda")
    nb = T // 16 + 2
    slots = torch.randperm(nb * 16, generator=g, device="cuda")[:T]
    slots[T // 2] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = (torch.zeros(nb, Hk, 16, D, device="cuda").to(dt)
              for _ in range(2))
    x = qkv.double().view(T, -1, D).clone()
    if norm:
        for a, b, w in ((0, Hq, qw), (Hq, Hq + Hk, kw)):
            h = x[:, a:b]
            x[:, a:b] = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True)
                                        + 1e-5) * w.double()
    c, s = cs[pos][:, None, :D // 2].double(), cs[pos][:, None, D // 2:].double()
    a, b = x[:, :Hq + Hk, :D // 2].clone(), x[:, :Hq + Hk, D // 2:].clone()
    x[:, :Hq + Hk, :D // 2] = a * c - b * s
    x[:, :Hq + Hk, D // 2:] = b * c + a * s
    assert ops.qkv_store_ok(qkv, D, D, "neox")
    ops.qkv_store(qkv, Hq, Hk, qw if norm else None, kw if norm else None, cs,
                  pos, slots, kc, vc, 1e-5)
    # one rounding to bf16, at most 2^-8 of the value; fp32 before it
    assert bool(((qkv.double().view(T, -1, D) - x).abs()
                 <= x.abs() * 2.0 ** -8 + 1e-5).all())
    # the pools hold what the row now holds
    kr, vr = torch.zeros_like(kc), torch.zeros_like(vc)
    h = qkv.view(T, -1, D)
    u = (lambda t: t.view(torch.uint8)) if fp8 else (lambda t: t)
    R.reshape_and_cache(u(h[:, Hq:Hq + Hk].contiguous().to(dt)),
                        u(h[:, Hq + Hk:].contiguous().to(dt)),
                        u(kr), u(vr), slots)
    assert torch.equal(u(kc), u(kr)) and torch.equal(u(vc), u(vr))
