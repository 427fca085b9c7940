"""The product of many rows that ends in silu(gate) * up, at the edges of its tiles
(256 rows, 128 columns, steps of 64 k), and the rule that takes it."""
import pytest
import torch

from gpustack_amd import ops



def _operands(M, N, K, pad=0):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    x = torch.randn(M, K + pad, generator=g, device="cuda").bfloat16()[:, :K]
    w = torch.randn(2 * N, K, generator=g, device="cuda")
    return x, (w * K ** -0.5).bfloat16()


def _check(out, x, w):
    N, K = w.shape[0] // 2, w.shape[1]
    xd, wd = x.double(), w.double()
    g, u = (torch.matmul(xd, wd.T.contiguous()[:, at:at + N])
            for at in (0, N))
    ref = g * torch.sigmoid(g) * u
    # fp32 sums of K products, each sum off by K 2^-24 of its terms' sizes at most;
    # |silu'| < 1.1. The result is rounded once, its functions 2^-20 of it
    size = torch.matmul(xd.abs(), wd.abs().T.contiguous())
    off = size * (K * 2.0 ** -24)
    bound = 1.1 * off[:, :N] * u.abs() + g.abs() * off[:, N:] \
        + ref.abs() * (2.0 ** -8 + 2.0 ** -20) + 1e-30
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("M,N,K,pad", [
    (1, 8, 128, 0),               # one row, one store of a lane
    (255, 120, 128, 8), (256, 128, 192, 0), (257, 136, 256, 64),
    (300, 1000, 64 * 7, 0), (513, 384, 4096, 0),
    # two and three rounds of tiles: 9 x 33, 17 x 33
    (2100, 4104, 128, 0), (4100, 4200, 192, 0)])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_product_ends_in_the_activation(M, N, K, pad):
    x, w = _operands(M, N, K, pad)
    # rows beyond the result keep what they hold
    room = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.bfloat16)
    ops._load_hip().wide_silu(room[1:M + 1], x, w)
    assert bool((room[0] == 7).all()) and bool((room[M + 1] == 7).all())
    _check(room[1:M + 1], x, w)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_refused_operands():
    x, w = _operands(256, 128, 128)
    out = torch.empty(256, 128, device="cuda", dtype=torch.bfloat16)
    hip = ops._load_hip()
    for bad in (lambda: hip.wide_silu(out, x[:, :64], w[:, :64].contiguous()),
                lambda: hip.wide_silu(out, x[:255], w),
                lambda: hip.wide_silu(out, x.float(), w),
                lambda: hip.wide_silu(out[:, :124], x, w[:248])):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_linear_silu_takes_it():
    x, w = _operands(512, 8192, 1024)
    assert ops._wide_silu_wins(512, 16384, 1024)
    _check(ops.linear_silu(x, w), x, w)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("M,N,K,parts,pad", [
    (1, 8, 128, 1, 0), (257, 264, 64 * 17, 8, 8),     # parts of two and three steps
    (300, 1000, 1024, 3, 0), (513, 520, 4096, 5, 0),
    (2100, 2056, 64 * 11, 5, 64)])                    # 405 tiles: two a workgroup
def test_product_in_parts(M, N, K, parts, pad):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + pad, generator=g, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    got = ops._load_hip().wide_parts(x, w, parts)
    assert got.shape == (parts, M, N) and got.dtype == torch.float32
    n = K // 64
    for p in range(parts):
        k = slice(n * p // parts * 64, n * (p + 1) // parts * 64)
        a, b = x[:, k].double(), w[:, k].double().T.contiguous()
        # fp32 sums, each off by 2^-24 of its terms' sizes a step at most
        bound = torch.matmul(a.abs(), b.abs()) * (K * 2.0 ** -24) + 1e-30
        assert bool(((got[p].double() - torch.matmul(a, b)).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("M", [640, 1100])
def test_the_norm_behind_adds_the_parts_up(M):
    N, K = 4096, 11008
    g = torch.Generator(device="cuda").manual_seed(M)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, res = rnd(M, K).bfloat16(), rnd(M, N).bfloat16()
    w, nw = (rnd(N, K) * K ** -0.5).bfloat16(), rnd(N).bfloat16()
    parts = ops.linear_auto(x, w, True)
    assert parts.shape == (ops._wide_parts(M, N, K), M, N)
    total = torch.matmul(x.double(), w.double().T.contiguous())
    assert float((parts.double().sum(0) - total).abs().max()) < 1e-4
    got, ref = ops.add_rms_norm(parts, res.clone(), nw, 1e-5), \
        ops.add_rms_norm(parts.sum(0).bfloat16(), res.clone(), nw, 1e-5)
    for a, b in zip(got, ref):
        # the same but for the order of the parts' sum, half an ulp at a rounding
        assert float(((a.float() - b.float()).abs()
                      > b.float().abs() * 2.0 ** -7 + 2.0 ** -7).sum()) == 0


@pytest.mark.parametrize("M", [257, 400, 512, 513, 700, 1024, 2048, 4000])
@pytest.mark.parametrize("K", [4096, 7168, 8192, 11008, 14336])
def test_parts_fill_the_workgroups_once(M, K):
    for N in range(1024, 10752, 256):
        parts = ops._wide_parts(M, N, K)
        tiles = -(-M // 256) * -(-N // 256)
        if parts:
            assert K >= 7168 and 2 <= parts <= 8 and tiles * parts <= 256
            assert M * N * parts * 4 <= 67 << 20          # bytes of the parts
            assert K // 64 // parts >= 2
    assert not ops._wide_parts(256, 4096, K)
    assert not ops._wide_parts(1024, 4096, K + 32)


@pytest.mark.parametrize("K", [1024, 2048, 4096, 8192])
def test_rule_by_filled_rounds(K):
    """Full rounds are taken, rounds for the sake of a few tiles not."""
    for N in range(1024, 57345, 512):
        cols = N // 2 / 128
        for M in (129, 256, 512, 1000, 2048, 4096, 8192):
            got = ops._wide_silu_wins(M, N, K)
            tiles = -(-M // 256) * -(-int(cols * 128) // 128)
            filled = M * (N // 2) / (256 * 128 * 256 * -(-tiles // 256))
            assert got or filled < .8
            assert not got or filled >= .5
    assert not ops._wide_silu_wins(128, 28672, K)
    assert not ops._wide_silu_wins(8192, 28672, K + 32)
    assert not ops._wide_silu_wins(8192, 28672 + 8, K)
    # offsets inside the weights are 32 bits of bytes
    assert not ops._wide_silu_wins(8192, 1 << 20, 8192)
