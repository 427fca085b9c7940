"""Products of many rows, whole, ended in silu(gate) * up or in fp32 parts, at the edges
of their tiles (32 rows and 32 weight rows times a tile's numbers, steps of 64 k), and
the rules that take them."""
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


SIZES = [
    (1, 8, 128, 0),               # one row, one store of a lane
    (255, 120, 128, 8), (256, 128, 192, 0), (257, 136, 256, 64),
    (300, 1000, 64 * 7, 0), (513, 384, 4096, 0),
    # two and three rounds of 256 x 256: 9 x 33, 17 x 33
    (2100, 4104, 128, 0), (4100, 4200, 192, 0)]


@pytest.mark.parametrize("M,N,K,pad", SIZES)
@pytest.mark.parametrize("tile", ops._WIDE_SILU)
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_product_ends_in_the_activation(M, N, K, pad, tile):
    x, w = _operands(M, N, K, pad)
    # rows beyond the result keep what they hold
    room = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.bfloat16)
    ops._load_hip().wide_rows(room[1:M + 1], x, w, *tile, silu=True)
    assert bool((room[0] == 7).all()) and bool((room[M + 1] == 7).all())
    _check(room[1:M + 1], x, w)


def large_pairs():
    """Gates and ups whose product leaves fp32, or that are not finite, all by all in
    bf16, and silu(gate) * up of them; e^-g is infinite where it leaves fp32."""
    inf, nan = float("inf"), float("nan")
    g = torch.tensor([-inf, -1e38, -1e30, -1e3, -100., -60., -1., 0., 1., 60., 1e30,
                      inf, nan]).bfloat16()
    u = torch.tensor([0., 1., -3., 1e30, -1e36, 1e37, inf, -inf, nan]).bfloat16()
    g, u = (t.flatten() for t in torch.meshgrid(g, u, indexing="ij"))
    gd, ud = g.double(), u.double()
    return g, u, (gd / (1 + torch.exp(-gd).float().double()) * ud).float()


def check_large(out, ref):
    """`out` against large_pairs' `ref`: rounded to bf16 once, its functions 2^-20 of
    it; e^-g of 60 is off by 60 2^-24 of it."""
    out, ref = out.double().cpu(), ref.double()
    assert torch.equal(out.isnan(), ref.isnan())
    # no finite result becomes infinite or the other way round
    assert torch.equal(out.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert torch.equal(out[~ok & ~ref.isnan()], ref[~ok & ~ref.isnan()])
    bound = ref.abs() * (2.0 ** -8 + 2.0 ** -17) + 1e-38
    assert bool(((out - ref).abs() <= bound)[ok].all())


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("tile", ops._WIDE_SILU)
def test_gate_and_up_beyond_fp32(tile):
    g, u, ref = large_pairs()
    N, K = -(-len(g) // 16) * 16, 128
    x = torch.zeros(130, K, dtype=torch.bfloat16)
    x[:, 0] = 1
    w = torch.zeros(2 * N, K, dtype=torch.bfloat16)
    w[:len(g), 0], w[N:N + len(u), 0] = g, u
    out = torch.empty(130, N, device="cuda", dtype=torch.bfloat16)
    ops._load_hip().wide_rows(out, x.cuda(), w.cuda(), *tile, silu=True)
    for row in (0, 129):
        check_large(out[row, :len(g)], ref)


@pytest.mark.parametrize("M,N,K,pad", SIZES)
@pytest.mark.parametrize("tile", [t for t in ops._WIDE_ROWS if t != (8, 8)])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_product(M, N, K, pad, tile):
    x, w = _operands(M, N, K, pad)
    w = w[:N]
    room = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.bfloat16)
    ops._load_hip().wide_rows(room[1:M + 1], x, w, *tile)
    assert bool((room[0] == 7).all()) and bool((room[M + 1] == 7).all())
    xd, wd = x.double(), w.double().T.contiguous()
    ref = torch.matmul(xd, wd)
    # an fp32 sum of K products, off by K 2^-24 of its terms' sizes at most, rounded
    bound = torch.matmul(xd.abs(), wd.abs()) * (K * 2.0 ** -24) \
        + ref.abs() * 2.0 ** -8 + 1e-30
    assert bool(((room[1:M + 1].double() - ref).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("M,N,tile,silu", [
    (700, 2008, (8, 6), True), (2000, 1080, (8, 4), True), (520, 2136, (6, 8), True),
    (2000, 1032, (4, 4), False), (1500, 1032, (6, 6), False), (700, 5000, (8, 7), False)])
def test_equal_rows_are_equal_anywhere(M, N, tile, silu):
    # tiles of one column on two XCDs, eight row tiles a block and more; sums of which
    # nothing but their roundings is left
    x, w = _operands(1, N, 2048)
    x = torch.cat([x, x], 1).expand(M, 4096).contiguous()
    w = torch.cat([w, -w], 1)
    out = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    ops._load_hip().wide_rows(out, x, w if silu else w[:N], *tile, silu=silu)
    assert bool((out == out[:1]).all())


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_refused_operands():
    x, w = _operands(256, 128, 128)
    out = torch.empty(256, 128, device="cuda", dtype=torch.bfloat16)
    hip = ops._load_hip()
    for bad in (lambda: hip.wide_rows(out, x[:, :64], w[:, :64].contiguous(), 8, 8, True),
                lambda: hip.wide_rows(out, x[:255], w, 8, 8, True),
                lambda: hip.wide_rows(out, x.float(), w, 8, 8, True),
                lambda: hip.wide_rows(out[:, :124], x, w[:248], 8, 8, True),
                lambda: hip.wide_rows(out, x, w[:128], 8, 8),
                lambda: hip.wide_rows(out, x, w, 8, 3, True)):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_linear_silu_takes_it():
    x, w = _operands(512, 8192, 1024)
    assert ops._wide_silu_tile(512, 16384, 1024)
    _check(ops.linear_silu(x, w), x, w)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("tile", ops._WIDE_PARTS)
@pytest.mark.parametrize("M,N,K,parts,pad", [
    (1, 8, 128, 1, 0), (257, 264, 64 * 17, 8, 8),     # parts of two and three steps
    (300, 1000, 1024, 3, 0), (513, 520, 4096, 5, 0),
    (2100, 2056, 64 * 11, 5, 64)])                    # two tiles a workgroup and more
def test_product_in_parts(M, N, K, parts, pad, tile):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + pad, generator=g, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    got = ops._load_hip().wide_parts(x, w, parts, *tile)
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
@pytest.mark.parametrize("M,N,K", [(136, 4096, 4096), (512, 6144, 4096),
                                   (640, 4096, 11008), (1100, 4096, 11008)])
def test_the_norm_behind_adds_the_parts_up(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, res = rnd(M, K).bfloat16(), rnd(M, N).bfloat16()
    w, nw = (rnd(N, K) * K ** -0.5).bfloat16(), rnd(N).bfloat16()
    parts = ops.linear_auto(x, w, True)
    assert parts.shape == (ops._wide_parts_plan(M, N, K)[1], M, N)
    total = torch.matmul(x.double(), w.double().T.contiguous())
    assert float((parts.double().sum(0) - total).abs().max()) < 1e-4
    got, ref = ops.add_rms_norm(parts, res.clone(), nw, 1e-5), \
        ops.add_rms_norm(parts.sum(0).bfloat16(), res.clone(), nw, 1e-5)
    for a, b in zip(got, ref):
        # the same but for the order of the parts' sum, half an ulp at a rounding
        assert float(((a.float() - b.float()).abs()
                      > b.float().abs() * 2.0 ** -7 + 2.0 ** -7).sum()) == 0


@pytest.mark.parametrize("M", [129, 257, 400, 512, 513, 700, 1024, 2048, 4000])
@pytest.mark.parametrize("K", [2048, 2560, 4096, 7168, 8192, 11008, 14336])
def test_parts_fill_the_workgroups_once(M, K):
    taken = 0
    for N in range(1024, 10752, 256):
        plan = ops._wide_parts_plan(M, N, K)
        if plan:
            tile, parts = plan
            tiles = -(-M // (32 * tile[0])) * -(-N // (32 * tile[1]))
            assert K >= 2560 and 2 <= parts <= 8 and tiles * parts <= 256
            assert tile in ops._WIDE_PARTS and K // 64 // parts >= 2
            assert M * N * parts * 4 <= 67 << 20          # bytes of the parts
            taken += 1
    assert taken or K < 4096 or M == 4000
    assert not ops._wide_parts_plan(128, 4096, K)
    assert not ops._wide_parts_plan(512, 4096, K + 32)
    assert not ops._wide_parts_plan(512, 4100, K)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_linear_auto_takes_it():
    x, w = _operands(2039, 2048, 4096)
    assert ops._wide_rows_tile(2039, 4096, 4096)
    got = ops.linear_auto(x, w)
    ref = torch.matmul(x.double(), w.double().T.contiguous())
    assert float((got.double() - ref).abs().max()) < 2.0 ** -8 * float(ref.abs().max())
    # rows further apart than a tile's offsets reach are the library's
    far = torch.empty((1 << 22) + 8192, device="cuda", dtype=torch.bfloat16) \
        .as_strided((2, 4096), ((1 << 22) + 8, 1))
    assert not ops._wide_take(far, w) and ops._wide_take(x, w)


@pytest.mark.parametrize("rule,tiles", [(ops._wide_silu_tile, ops._WIDE_SILU),
                                        (ops._wide_rows_tile, ops._WIDE_ROWS)])
@pytest.mark.parametrize("K", [1024, 2048, 4096, 14336])
def test_the_tile_fills_its_rounds(rule, tiles, K):
    def filled(tile, M, N):
        n = -(-M // (32 * tile[0])) * -(-N // (32 * tile[1]))
        return M * N / (-(-n // 256) * 256 * 1024 * tile[0] * tile[1])

    taken = 0
    for N in range(1024, 57345, 512):
        for M in (264, 512, 1000, 2048, 4096, 8192):
            tile = rule(M, N, K)
            taken += tile is not None
            if tile:
                assert tile in tiles
                # no larger one that fills its rounds as well
                assert all(filled(tile, M, N) > .93 * filled(t, M, N) for t in tiles
                           if t[0] >= tile[0] and t[1] >= tile[1])
            if rule is ops._wide_silu_tile and filled((8, 8), M, N) > .8 \
                    and M * N > 1 << 23:
                assert tile
            if rule is ops._wide_rows_tile:
                assert tile != (8, 8)
    assert taken > 100
    assert rule(8192, 28672 + 16, K)
    assert rule(128, 28672, K) is None
    assert rule(8192, 28672, K + 32) is None
    assert rule(8192, 28672 + 4, K) is None
    # offsets inside the weights are 32 bits of bytes
    assert rule(8192, 1 << 21, K) is None
