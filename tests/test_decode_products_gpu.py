"""Decode products of few rows, bf16 and packed int4: rows and columns at the
edges of their 16-wide tiles, block counts that the 8 waves do not divide, and
every column width that the launch chooses between; the argmax over a row."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _hip():
    from gpustack_amd import ops

    return ops._load_hip()


def _close(out, ref, size):
    # rounded to bf16 once (at most 2^-8 of the value); fp32 sums of terms
    # that add up to `size` in absolute value are off by less than 2^-18 of it
    err = (out.double() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + size * 2.0 ** -18
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("M", [1, 15, 16])
@pytest.mark.parametrize("N,K", [(16, 128), (100, 1152), (4096, 1024),
                                 (16400, 256)])
def test_rows_gemm(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * N)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    out = torch.full((M, N), 9.0, device="cuda").bfloat16()
    _hip().rows_gemm(out, x, w)
    _close(out, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("M", [1, 32, 33, 64, 65, 97, 128])
@pytest.mark.parametrize("N,K,cols,parts", [
    (8, 64, 32, 1), (136, 128, 64, 2), (260, 640, 128, 3), (4096, 1088, 32, 5),
    (33000, 448, 128, 1), (20000, 576, 32, 1)])
def test_rows_tile(M, N, K, cols, parts):
    g = torch.Generator(device="cuda").manual_seed(M * N)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    out = torch.full((M, N), 9.0, device="cuda").bfloat16()
    _hip().rows_tile(out, x, w, cols, parts)
    _close(out, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("M,N,K", [(1, 28672, 4096), (48, 4096, 14336),
                                   (17, 1024, 4096), (96, 10240, 3072),
                                   (64, 5128, 1024), (128, 3072, 3072)])
def test_linear_auto_takes_the_tiles(M, N, K):
    from gpustack_amd import ops

    assert ops._rows_tile_plan(M, N, K) is not None
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    _close(ops.linear_auto(x, w), x.double() @ w.double().T,
           x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("N,K", [(64, 128), (128, 1152), (14400, 256),
                                 (28736, 384)])
def test_w4_rows(M, N, K):
    import gpustack_amd.engine  # noqa: F401  (package import order)
    from gpustack_amd.models.quantized import pack_w4_runtime

    g = torch.Generator(device="cuda").manual_seed(M + N)
    q = torch.randint(0, 16, (N, K), generator=g, device="cuda")
    sc = torch.rand(N, K // 128, generator=g, device="cuda") * 0.05 + 0.01
    zr = torch.randint(0, 16, (N, K // 128), generator=g, device="cuda").float()
    qw, s, z = pack_w4_runtime(q, sc, zr, 128)
    x = (torch.randn(M, K, generator=g, device="cuda") + 0.5).bfloat16()
    out = torch.full((M, N), 9.0, device="cuda").bfloat16()
    _hip().w4_gemm(out, x, qw, s, z)
    wide = lambda t: t.double().repeat_interleave(128, 1)
    w = q.double() * wide(s) - wide(z)
    # sums run over 128 + q and are corrected by 128 times the sum of x
    size = x.double().abs() @ (wide(s) * 144 + wide(z).abs()).T
    _close(out, x.double() @ w.T, size)


@pytest.mark.parametrize("V", [7, 1000, 32776, 128256])
def test_argmax_of_a_row(V):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(V)
    x = torch.randn(9, V, generator=g, device="cuda")
    x[0] = -1.0                           # all alike: the first
    x[1, -1] = 50.0
    x[2, V // 2:] = 60.0                  # the first of many
    x[3] = float("-inf")
    x[3, V // 3] = -1e30
    for t in (x.bfloat16(), x):
        ref = torch.stack([(r == r.max()).nonzero()[0, 0] for r in t.float()])
        assert torch.equal(ops.greedy_sample(t), ref)


@pytest.mark.parametrize("M,N,K", [(4, 4096, 2048), (48, 4096, 4096),
                                   (512, 4096, 8192), (300, 256, 256)])
def test_products_without_the_main_library(monkeypatch, M, N, K):
    """A checkout that has built only the libraries of one model."""
    from pathlib import Path

    from gpustack_amd import ops

    exists = Path.exists
    monkeypatch.setattr(Path, "exists", lambda p: exists(p)
                        and p.name != "_hip_ops.so")
    monkeypatch.setattr(ops, "_HIP", None)
    monkeypatch.setattr(ops, "_HIP_ERR", None)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16()
    for _ in range(2):
        assert torch.equal(ops.linear_auto(x, w),
                           torch.nn.functional.linear(x, w))
    with pytest.raises(ImportError):
        ops._load_hip()


@pytest.mark.parametrize("N,K", [(96, 256), (8, 128), (64, 256)])
def test_packed_weights_of_any_column_count(N, K):
    from gpustack_amd.models.llama import W4Pack, qlinear
    from gpustack_amd.models.quantized import (dequant_w4_runtime,
                                               pack_w4_runtime)

    g = torch.Generator(device="cuda").manual_seed(N)
    pack = W4Pack(*pack_w4_runtime(
        torch.randint(0, 16, (N, K), generator=g, device="cuda"),
        torch.rand(N, K // 128, generator=g, device="cuda") * 0.05 + 0.01,
        torch.full((N, K // 128), 8.0, device="cuda"), 128))
    x = torch.randn(5, K, generator=g, device="cuda").bfloat16()
    w = dequant_w4_runtime(pack.qw, pack.sc, pack.zs).double()
    size = x.double().abs() @ w.abs().T
    # the expansion rounds a weight to bf16 (2^-9 of it), the result once more
    err = (qlinear(x, None, pack).double() - x.double() @ w.T).abs()
    assert bool((err <= size * 2.0 ** -7).all())


@pytest.mark.parametrize("M,N,K,own", [
    (65, 16384, 2048, True), (65, 16376, 2048, False),
    (96, 22024, 6144, True), (97, 32896, 6144, False),
    (97, 32768, 8192, True), (128, 16384, 10240, False),
    (80, 16384, 3072, False)])
def test_rule_of_tiles_for_many_columns(M, N, K, own):
    from gpustack_amd import ops

    assert (ops._rows_tile_plan(M, N, K) is not None) == own
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    _close(ops.linear_auto(x, w), x.double() @ w.double().T,
           x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("M,N,K,own", [
    (17, 49152, 8192, True), (64, 49160, 8192, False),
    (32, 81920, 8192, False), (32, 81928, 8192, True),
    (48, 57344, 6144, True), (65, 65536, 6144, True),
    (65, 65544, 6144, False), (96, 98176, 8192, False),
    (96, 98304, 8192, True), (65, 131080, 8192, False),
    (96, 73728, 4096, True), (97, 73728, 4096, False),
    (97, 32896, 4096, False), (128, 38400, 4096, True),
    (128, 73728, 2048, True)])
def test_rule_of_tiles_by_rounds(M, N, K, own):
    from gpustack_amd import ops

    assert (ops._rows_tile_plan(M, N, K) is not None) == own
