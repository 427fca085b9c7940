"""Tiled product with packed int4 weights: rows at the edges of its row tiles and
above one workgroup's 64, steps of one block at the end, several chunks of staged
scales, four and eight waves, parts over k, and the activation behind it, against
float64; the forms that the launch chooses between agree with each other."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _hip():
    from gpustack_amd import ops

    return ops._load_hip()


def _case(M, N, K, size=1.0):
    """x, the packed weight, the weight in float64 and a bound for the sums: they
    run over 128 + q and are corrected by 128 times the sum of x."""
    import gpustack_amd.engine  # noqa: F401  (package import order)
    from gpustack_amd.models.quantized import pack_w4_runtime

    g = torch.Generator(device="cuda").manual_seed(M + N)
    q = torch.randint(0, 16, (N, K), generator=g, device="cuda")
    sc = (torch.rand(N, K // 128, generator=g, device="cuda") * 0.05 + 0.01) * size
    zr = torch.randint(0, 16, (N, K // 128), generator=g, device="cuda").float()
    pack = pack_w4_runtime(q, sc, zr, 128)
    x = (torch.randn(M, K, generator=g, device="cuda") + 0.5).bfloat16()
    wide = lambda t: t.double().repeat_interleave(128, 1)
    s, z = wide(pack[1]), wide(pack[2])
    return x, pack, q.double() * s - z, x.double().abs() @ (s * 144 + z.abs()).T


@pytest.mark.parametrize("M", [1, 8, 16, 17, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("N,K", [(32768, 384), (33024, 4480), (32832, 2176),
                                 (4096, 3328), (1088, 12416)])
def test_product(M, N, K):
    x, (qw, s, z), w, size = _case(M, N, K)
    ref = x.double() @ w.T
    out = torch.full((M, N), 9.0, device="cuda").bfloat16()
    _hip().w4_gemm(out, x, qw, s, z)
    # rounded to bf16 once; fp32 sums
    assert bool(((out.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + size * 2.0 ** -18).all())
    parts = _hip().w4_parts(x, qw, s, z)
    cut = N < 30000 and (M >= 8 or K >= 8192)
    assert (parts is not None) == cut
    if cut:
        assert parts.dtype == torch.float32 and parts.shape[1:] == out.shape
        assert bool(((parts.double().sum(0) - ref).abs()
                     <= size * 2.0 ** -18).all())
    # the general form, which operands at other than 16-byte addresses take
    y = torch.empty(M * K + 4, device="cuda", dtype=torch.bfloat16)[4:].view(M, K)
    y.copy_(x)
    general = torch.full_like(out, 9.0)
    _hip().w4_gemm(general, y, qw, s, z)
    assert _hip().w4_parts(y, qw, s, z) is None
    assert bool(((general.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + size * 2.0 ** -18).all())


@pytest.mark.parametrize("M", [1, 16, 17, 33, 65])
@pytest.mark.parametrize("N,K", [(22016, 384), (24576, 4352)])
def test_product_ends_in_the_activation(M, N, K):
    x, (qw, s, z), w, size = _case(M, N, K, 1 / 16)
    act = _hip().w4_silu(x, qw, s, z)
    h, n = x.double() @ w.T, N // 2
    g, u = h[:, :n], h[:, n:]
    ref = torch.nn.functional.silu(g) * u
    eg, eu = (size[:, :n] * 2.0 ** -18, size[:, n:] * 2.0 ** -18)
    # silu's slope is under 1.1 and it is no larger than its argument; the
    # exponential's own error is a few units of fp32
    bound = ref.abs() * (2.0 ** -8 + 2.0 ** -20) + 1.1 * eg * (u.abs() + eu) \
        + g.abs() * eu
    assert bool(((act.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K,wins", [
    (17, 16640, 4096, True), (192, 22016, 12288, True),   # whole tiles anyway
    (1, 32768, 4096, True), (1, 32768, 8192, False),      # cut from 8192 k on
    (64, 16384, 4096, False), (16, 22016, 8192, False),   # cut over k
    (1, 22016, 6144, False), (2, 17920, 5120, False),     # the rows' form
    (1, 22016, 4096, True), (2, 24576, 4096, True), (8, 17920, 5120, True),
    (16, 22016, 4096, True), (1, 28672, 4096, True), (1, 22016, 2048, True),
    (1, 8192, 128, False)])
def test_where_it_ends_in_the_activation(monkeypatch, M, N, K, wins):
    """The route, and both ways the same result up to the rounding of the
    product that the activation reads."""
    from gpustack_amd import ops
    from gpustack_amd.models.llama import W4Pack, _gate_up_silu, qlinear

    assert _hip().w4_silu_wins(M, N, K) == wins
    if N * K > 1 << 27:
        return                             # the two forms have tests above
    x, (qw, s, z), _, _ = _case(M, N, K, 1 / 16)
    pack = W4Pack(qw, s, z)
    got = _gate_up_silu(x, None, pack)
    assert (got is not None) == wins
    if not wins:
        return
    want = torch.empty(M, N // 2, device="cuda", dtype=torch.bfloat16)
    ops.silu_and_mul(want, qlinear(x, None, pack))
    # gate and up rounded to bf16 here and not there, the result in both; silu's
    # slope is under 1.1
    assert float((got.double() - want.double()).norm()
                 / want.double().norm()) < 3 * 2.0 ** -8


def test_none_where_there_is_no_such_form():
    x, (qw, s, z), _, _ = _case(4, 192, 256)
    assert _hip().w4_silu(x, qw, s, z) is None
    assert _hip().w4_parts(x, qw, s, z) is None


# about the four steps of 256 k from which two waves share a step, the four buffers that
# a workgroup with a CU of its own has, and the 16 steps whose scales are staged at once
@pytest.mark.parametrize("M", [1, 16, 32, 64])
@pytest.mark.parametrize("K", [768, 896, 1024, 1152, 1280, 4096, 4224, 4736, 8320])
def test_steps_of_a_workgroup(M, K):
    test_product_ends_in_the_activation(M, 8192, K)


@pytest.mark.parametrize("M", [5, 64])
def test_scales_that_lie_one_by_one(M):
    x, (qw, s, z), w, size = _case(M, 33024, 2048)
    odd = lambda t: torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)
    out = torch.full((M, 33024), 9.0, device="cuda").bfloat16()
    same = torch.full_like(out, 9.0)
    assert odd(s).data_ptr() % 4 == 2
    _hip().w4_gemm(out, x, qw, odd(s), odd(z))
    _hip().w4_gemm(same, x, qw, s, z)
    assert torch.equal(out, same)
    ref = x.double() @ w.T
    assert bool(((out.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + size * 2.0 ** -18).all())
