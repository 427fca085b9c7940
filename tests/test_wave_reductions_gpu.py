"""Row kernels whose sums cross the wave without the LDS, at widths that leave lanes,
waves and register chunks without numbers, with one to eight parts and more."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("H", [8, 72, 512, 2048, 2056, 4104, 8192, 8200])
@pytest.mark.parametrize("T,parts", [(1, 1), (3, 4), (3, 5), (2, 8), (2, 9),
                                     (600, 2)])
def test_norm_of_parts(H, T, parts):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(H + T + parts)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p, res, w = rnd(parts, T, H), rnd(T, H).bfloat16(), rnd(H).bfloat16()
    # the parts are added in their order and rounded, as a product's join does it
    x = p[0].clone()
    for i in range(1, parts):
        x += p[i]
    s = x.bfloat16().double() + res.double()
    want = s * torch.rsqrt((s * s).mean(1, keepdim=True) + 1e-5) * w.double()
    res2 = res.clone()
    out = ops.add_rms_norm(p, res2, w, 1e-5)
    assert torch.equal(res2, s.float().bfloat16())
    # rows of more than 8192 are normed from the rounded sum (2^-8 of a value)
    eps = 2.0 ** -8 if H <= 8192 else 2.0 ** -7
    assert bool(((out.double() - want).abs() <= want.abs() * eps + 1e-6).all())
    plain = x.bfloat16()
    res3 = res.clone()
    ops.fused_add_rms_norm(plain, res3, w, 1e-5)
    assert torch.equal(plain, out) and torch.equal(res3, res2)


@pytest.mark.parametrize("H", [8, 2048, 8192])
@pytest.mark.parametrize("T", [1, 600])
@pytest.mark.parametrize("parts", [0, 2, 6])
def test_order_of_squares(T, H, parts):
    """A thread's squares are one chain of multiply-adds from its first number on. Taken
    so, the squares of these three are 8 in fp32 (worked out in fractions), with the
    second one rounded in front of the first 8 + 2^-20. The probe behind them lies
    halfway between two bf16 numbers where the norm is exactly a power of two."""
    from gpustack_amd import ops

    h = float.fromhex
    x, res = torch.zeros(T, H).bfloat16(), torch.zeros(T, H).bfloat16()
    x[:, 0], res[:, 0] = h("0x1.4ep-9"), h("0x1.46p+0")
    x[:, 1], res[:, 1] = h("0x1.4ap-9"), h("0x1.8cp+0")
    x[:, 2], res[:, 2] = h("0x1.8ap-6"), h("0x1.f8p+0")
    w = torch.ones(H).bfloat16()
    res[:, 3], w[3] = 3 * 2.0 ** -30, 129 * 2.0 ** -7
    x, res, w = x.cuda(), res.cuda(), w.cuda()
    if parts:
        x = torch.cat([x.float()[None], torch.zeros(parts - 1, T, H, device="cuda")])
    out = ops.add_rms_norm(x, res, w, 0.0)
    # to even: 194 for 193.5; below it 193
    assert bool((out[:, 3].float() == 388 * 2.0 ** -37 * (H / 8) ** 0.5).all())
