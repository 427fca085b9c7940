"""Norms of rows at the edges of what a workgroup holds: a row's result does not
depend on how many rows there are."""
import pytest
import torch

from gpustack_amd import ops

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


@pytest.mark.parametrize("form", ["rows", "parts", "experts", "picked"])
@pytest.mark.parametrize("T", [1, 512, 513])
@pytest.mark.parametrize("H", [8192, 8200, 16384, 16392])
def test_the_sum_is_rounded_alike_at_any_number_of_rows(form, T, H):
    g = torch.Generator(device="cuda").manual_seed(H)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    w = rnd(H).bfloat16()
    x, res = rnd(1, H).bfloat16(), rnd(1, H).bfloat16()
    many = lambda t: t.expand(T, H).contiguous()
    added = res.double() + x.double()
    inv = (added.square().mean() + 1e-5).rsqrt()
    # up to 8192 the sum itself is scaled, wider rows read it back from bf16
    kept = added if H <= 8192 else added.float().bfloat16().double()
    want = (kept * inv * w.double()).bfloat16()
    if form == "rows":
        got = ops.add_rms_norm(many(x), many(res), w, 1e-5)
    elif form == "parts":
        got = ops.add_rms_norm(many(x).float()[None], many(res), w, 1e-5)
    elif form == "experts":
        got = ops.add_rms_norm(many(x)[:, None].contiguous(), many(res), w, 1e-5)
    else:
        got = ops.add_rms_norm_rows(many(x), many(res), w, 1e-5,
                                    torch.arange(T, device="cuda"))
    # fp32 sums of H squares move the scale by less than 1e-6, which a bf16
    # rounding (2^-9 of the value) notices in less than 1 of 1000 values; the sum
    # unrounded instead of rounded changes a third of them
    assert float((got != want).double().mean()) <= 5e-3
