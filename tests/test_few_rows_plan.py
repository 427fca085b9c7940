"""The form of whole products of few rows: what the rules beside it decide stays where
parts, other lengths or more rows are concerned, and the forms give one product."""
import pytest
import torch

from gpustack_amd import ops


@pytest.mark.parametrize("M,N,K", [(65, 8192, 2048), (8, 8192, 4160), (8, 8192, 960),
                                   (8, 1000, 2048), (8, 8196, 2048), (8, 8192, 2080),
                                   (0, 8192, 2048)])
def test_other_products_stay(M, N, K):
    for plan, rows in (((64, 1), False), (None, True), (None, False)):
        assert ops._few_rows_plan(M, N, K, plan, rows) == (plan, rows)
    assert ops._few_rows_plan(8, 8192, 2048, (64, 4), False) == ((64, 4), False)


def test_forms():
    f = lambda M, N, K: ops._few_rows_plan(
        M, N, K, ops._rows_tile_plan(M, N, K), ops._rows_gemm_wins(M, N, K))
    assert f(16, 151936, 2048)[0] is not None           # in rows_gemm's place
    assert f(16, 8192, 2048) == ((32, 1), False)
    assert any(f(8, 10304, 2048))                       # in the library's
    assert f(32, 14336, 1024)[0] is not None
    assert f(1, 4096, 2048) == (None, True)             # as before
    assert f(64, 8192, 4096) == (None, False)           # the library
    # few workgroups beyond 16 rows, where the library cuts k
    for M, N, K in ((32, 1536, 2816), (32, 2560, 3072), (17, 2560, 2304), (48, 1536, 1536)):
        assert f(M, N, K) == (None, False)
    assert f(32, 3072, 3072)[0] is not None
    for N in range(1024, 40000, 1000):
        for K in range(1024, 4097, 64):
            plan, rows = f(8, N - N % 8, K)
            assert not (rows and K % 128)
            assert plan is None or plan[0] in (32, 64, 128)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(10304, 2048), (8192, 2048), (9224, 1088), (14336, 1536),
                                 (1032, 1024), (32008, 2560), (5120, 4096)])
def test_products(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    out = ops.linear_auto(x, w)
    want = x.double() @ w.double().T
    # bf16 of an fp32 sum of K products
    size = x.double().abs() @ w.double().abs().T
    assert bool(((out.double() - want).abs()
                 <= want.abs() * 2.0 ** -8 + size * K * 2.0 ** -24).all())
