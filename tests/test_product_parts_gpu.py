"""Products cut over k whose parts the next kernel adds up: the same bits as
the product's own join and that kernel; and the layer-norm rows of 16-byte
loads at the edges of their lanes."""
import pytest
import torch

from gpustack_amd import ops

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _gen(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return lambda *s: torch.randn(*s, generator=g, device="cuda")


def _joined(parts):
    v = parts[0].clone()
    for p in parts[1:]:
        v += p
    return v.bfloat16()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 11])
@pytest.mark.parametrize("T,H", [(1, 64), (17, 2048), (48, 4096), (3, 8200)])
def test_add_rms_norm(n, T, H):
    rnd = _gen(n + T)
    parts, res = rnd(n, T, H), rnd(T, H).bfloat16()
    w = rnd(H).bfloat16()
    x, r1, r2 = _joined(parts), res.clone(), res.clone()
    ops.fused_add_rms_norm(x, r1, w, 1e-5)
    got = ops.add_rms_norm(parts, r2, w, 1e-5)
    assert torch.equal(got, x) and torch.equal(r1, r2)


@pytest.mark.parametrize("n", [2, 4, 7])
@pytest.mark.parametrize("D,Hq,Hk", [(64, 4, 4), (128, 32, 8), (256, 3, 1)])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float8_e4m3fn])
def test_qkv_store(n, D, Hq, Hk, norm, kv):
    rnd = _gen(n + D)
    T = 21
    parts = rnd(n, T, (Hq + 2 * Hk) * D)
    qw, kw = (rnd(D).bfloat16(), rnd(D).bfloat16()) if norm else (None, None)
    cs = ops.build_cos_sin_cache(D, D, 64).cuda()
    pos = torch.arange(T, device="cuda") + 5
    slots = torch.arange(T, device="cuda") * 2 - 1
    slots[0] = -1
    got = []
    for given in (None, parts):
        pools = [torch.zeros(8, Hk, 16, D, device="cuda").to(kv)
                 for _ in range(2)]
        qkv = _joined(parts) if given is None \
            else torch.full(parts.shape[1:], 9.0, device="cuda").bfloat16()
        ops.qkv_store(qkv, Hq, Hk, qw, kw, cs, pos, slots, *pools, 1e-5, given)
        got.append([qkv] + [p.view(torch.uint8) for p in pools])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("T", [1, 65])
@pytest.mark.parametrize("W", [8, 1000, 1004, 2048, 2056, 4096, 4104, 8192,
                               8200])
@pytest.mark.parametrize("add", ["nothing", "bf16", "fp32", "parts"])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_add_layer_norm(T, W, add, out):
    rnd = _gen(W)
    x = rnd(T, W) + 3
    w, b = rnd(W), rnd(W)
    a = {"nothing": None, "bf16": rnd(T, W).bfloat16(), "fp32": rnd(T, W),
         "parts": rnd(3, T, W)}[add]
    if add == "parts" and (W % 8 or W > 8192):
        with pytest.raises(RuntimeError):
            ops.add_layer_norm(x, a, w, b, 1e-5, torch.empty_like(x))
        return
    one = _joined(a) if add == "parts" else a
    want = x.double() if one is None else x.double() + one.double()
    ref = torch.nn.functional.layer_norm(want, (W,), w.double(), b.double(),
                                         1e-5)
    h = torch.full((T, W), 9.0, device="cuda").to(out)
    ops.add_layer_norm(x, a, w, b, 1e-5, h)
    # one fp32 addition; sums of W of them, then bf16 once
    assert torch.equal(x, want.float()) if one is not None else True
    err = (h.double() - ref).abs()
    eps = 2.0 ** -8 if out == torch.bfloat16 else 0.0
    assert bool((err <= ref.abs() * eps + 2e-5).all()), float(err.max())
    y = x.clone()
    ops.add_layer_norm(y, a, None, None, 1e-5, None)
    if a is not None:
        assert torch.equal(y, (x + one.float()))


@pytest.mark.parametrize("M", [1, 17, 48, 128])
@pytest.mark.parametrize("N,K", [(4096, 14336), (4096, 4096), (2048, 8192),
                                 (1024, 1024), (16384, 2048)])
def test_products_come_in_parts(M, N, K):
    rnd = _gen(M)
    x, w = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16()
    got = ops.linear_auto(x, w, parts=True)
    # parts exactly where the plan cuts the product: of its own for consumers of
    # parts, or the product's
    plan = ops._parts_plan(M, N, K) or ops._rows_tile_plan(M, N, K)
    if plan is None or plan[1] == 1:
        assert got.shape == (M, N) and got.dtype == torch.bfloat16
    else:
        assert got.shape == (plan[1], M, N) and got.dtype == torch.float32
        got = _joined(got)
    if ops._parts_plan(M, N, K) is None:
        assert torch.equal(got, ops.linear_auto(x, w))
        return
    # another cut than without parts: fp32 sums, rounded to bf16 once
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    assert bool(((got.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + size * 2.0 ** -18).all())


@pytest.mark.parametrize("M", [1, 16, 33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("N,K,cols", [(128, 64, 64), (64, 256, 128),
                                      (1000, 192, 64), (1000, 192, 128),
                                      (36, 128, 128), (8192, 2048, 64)])
def test_product_ends_in_the_activation(M, N, K, cols):
    rnd = _gen(M + N)
    x, w = rnd(M, K).bfloat16(), (rnd(2 * N, K) * K ** -0.5).bfloat16()
    out = torch.full((M, N), 9.0, device="cuda").bfloat16()
    ops._load_hip().rows_tile(out, x, w, cols, 1, silu=True)
    h = x.double() @ w.double().T
    ref = torch.nn.functional.silu(h[:, :N]) * h[:, N:]
    # rounded to bf16 once; fp32 sums of K products of size K^-1/2
    assert bool(((out.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + 1e-4).all())


def test_no_activation_where_there_is_no_such_product():
    w = torch.zeros(64, 1024, device="cuda", dtype=torch.bfloat16)
    x = torch.zeros(4, 1024, device="cuda", dtype=torch.bfloat16)
    assert ops.linear_silu(x, w) is None
    assert ops.linear_silu(x.cpu(), w.cpu()) is None


@pytest.mark.parametrize("M", [129, 255, 257, 385, 512])
@pytest.mark.parametrize("N,K", [(1024, 6144), (1032, 7168), (4096, 11008),
                                 (5120, 6208)])
def test_tall_products_in_parts(M, N, K):
    plan = ops._rows_tile_plan(M, N, K)
    wins = N <= 4096 or M < 385
    assert (plan is not None) == wins
    if not wins:
        return
    assert plan[1] > 1
    wide = ops._wide_parts_plan(M, N, K)
    assert (wide is not None) == (N > 1280)
    rnd = _gen(M + N)
    x, w = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16()
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    parts = ops.linear_auto(x, w, parts=True)
    assert parts.shape == ((wide or plan)[1], M, N) and parts.dtype == torch.float32
    # fp32 sums of terms that add up to `size`, then rounded to bf16 once
    assert bool(((parts.double().sum(0) - ref).abs()
                 <= size * 2.0 ** -18).all())
    out = ops.linear_auto(x, w)
    assert bool(((out.double() - ref).abs()
                 <= ref.abs() * 2.0 ** -8 + size * 2.0 ** -18).all())


@pytest.mark.parametrize("M,N,K", [(1, 1024, 3072), (8, 2048, 2048),
                                   (17, 1032, 1024), (64, 2048, 1088),
                                   (65, 4096, 1024), (128, 3072, 2048),
                                   (33, 6136, 3136), (16, 5120, 2048),
                                   (16, 1160, 4160), (2, 6144, 4096),
                                   (64, 8192, 8192), (5, 5000, 10240),
                                   (3, 3072, 1088), (1, 2304, 8192),
                                   (16, 3600, 8192), (24, 6144, 2112),
                                   (96, 2560, 3072), (128, 8192, 2112)])
def test_small_products_in_parts(M, N, K):
    plan = ops._parts_plan(M, N, K)
    assert plan is not None
    rnd = _gen(M + N)
    x, w = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16()
    parts = ops.linear_auto(x, w, parts=True)
    assert parts.shape == (plan[1], M, N) and parts.dtype == torch.float32
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    # fp32 sums of terms that add up to `size`
    assert bool(((parts.double().sum(0) - ref).abs()
                 <= size * 2.0 ** -18).all())
    assert ops.linear_auto(x, w).shape == (M, N)


@pytest.mark.parametrize("T,H", [(1, 64), (17, 4096), (3, 8200)])
def test_embedding_under_the_first_norm(T, H):
    rnd = _gen(T + H)
    embed, w = rnd(50, H).bfloat16(), rnd(H).bfloat16()
    ids = torch.arange(T, device="cuda") * 7 % 50
    x, h = ops.embed_rms_norm(ids, embed, w, 1e-5)
    ref = torch.empty_like(x)
    ops.rms_norm(ref, embed[ids], w, 1e-5)
    assert torch.equal(x, embed[ids]) and torch.equal(h, ref)
    # callers refuse such ids (test_refused_ids.py); the kernel stays in bounds
    bad = ids.clone()
    bad[-1] = 50
    x, h = ops.embed_rms_norm(bad, embed, w, 1e-5)
    assert torch.equal(x[:-1], embed[ids[:-1]]) and torch.equal(h[:-1], ref[:-1])
    assert not x[-1].any() and not h[-1].any()


@pytest.mark.parametrize("n", [0, 1, 3, 8])
@pytest.mark.parametrize("T,H", [(1, 64), (17, 4096), (9, 8200)])
def test_the_last_norm_of_picked_rows(n, T, H):
    rnd = _gen(n + T)
    res, w = rnd(T, H).bfloat16(), rnd(H).bfloat16()
    a = rnd(n, T, H) if n else rnd(T, H).bfloat16()
    rows = torch.tensor([T - 1, 0, -1], device="cuda")[: 1 + 2 * (T > 1)]
    x, r = (_joined(a) if n else a.clone()), res.clone()
    ops.fused_add_rms_norm(x, r, w, 1e-5)
    got = ops.add_rms_norm_rows(a, res, w, 1e-5, rows)
    assert torch.equal(got, x[rows])


@pytest.mark.parametrize("kind,T,W", [
    (kind, T, W) for kind in ("parts", "bf16", "fp32")
    for T, W in ((1, 64), (17, 2048), (9, 8192), (5, 100))
    if kind != "parts" or W % 8 == 0])     # products give other rows whole
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_last_layer_norm_of_picked_rows(kind, T, W, dtype):
    rnd = _gen(T + W)
    x, w, b = rnd(T, W), rnd(W), rnd(W)
    a = rnd(3, T, W) if kind == "parts" else rnd(T, W)
    if kind == "bf16":
        a = a.bfloat16()
    rows = torch.tensor([T - 1, 0, 0], device="cuda")
    y, ref = x.clone(), torch.empty(T, W, device="cuda", dtype=dtype)
    ops.add_layer_norm(y, a, w, b, 1e-5, ref)
    got = ops.add_layer_norm_rows(x, a, w, b, 1e-5, rows, dtype)
    assert torch.equal(got, ref[rows])


@pytest.mark.parametrize("k", [1, 3, 4, 8, 9])
@pytest.mark.parametrize("T,H", [(1, 64), (17, 2048), (3, 8200)])
def test_the_norm_adds_up_the_experts(k, T, H):
    rnd = _gen(k + T)
    rows, res, w = rnd(T, k, H).bfloat16(), rnd(T, H).bfloat16(), rnd(H).bfloat16()
    x = torch.empty_like(res)
    ops._load_hip().moe_sum(x, rows.view(T * k, H), k)
    pick = torch.tensor([T - 1, 0], device="cuda")
    picked = ops.add_rms_norm_rows(rows, res, w, 1e-5, pick)
    r1, r2 = res.clone(), res.clone()
    ops.fused_add_rms_norm(x, r1, w, 1e-5)
    assert torch.equal(ops.add_rms_norm(rows, r2, w, 1e-5), x)
    assert torch.equal(r1, r2) and torch.equal(picked, x[pick])
