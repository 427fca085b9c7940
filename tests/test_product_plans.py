"""The rules that choose a product's tiles and parts: neighbouring sizes are
treated alike (plain arithmetic; the products themselves are tested on the GPU)."""
import pytest

from gpustack_amd import ops


@pytest.mark.parametrize("M", [129, 256, 257, 384, 385, 512])
def test_tall_products_take_even_parts(M):
    for N in range(1024, 10241, 8):
        plan = ops._tall_tile_plan(M, N, 8192)
        if plan is not None:
            assert plan[1] <= 4 or plan[1] % 2 == 0
            assert plan[1] * -(-M // 128) * -(-N // plan[0]) <= 576


@pytest.mark.parametrize("M", [129, 256, 300, 384, 400, 512])
@pytest.mark.parametrize("K", [5120, 6144, 6208, 7168, 11008, 14336])
def test_tall_products_from_some_length_and_up_to_some_width(M, K):
    """One line in N: what is cut stays cut for fewer columns."""
    cut = [ops._tall_tile_plan(M, N, K) is not None
           for N in range(1024, 10752, 8)]
    changes = sum(a != b for a, b in zip(cut, cut[1:]))
    # at 5120 k two row tiles want 3072 columns besides
    assert changes <= (2 if K < 6144 else 1), changes


@pytest.mark.parametrize("M", [129, 192, 256, 264, 384, 400, 512])
@pytest.mark.parametrize("N", [1408, 2056, 2560, 4096, 5120, 6144, 8192])
def test_parts_of_the_wide_tiles_have_no_line_in_long_rows(M, N):
    """What the tiles of few rows cut over k, the wide ones do at any length."""
    for K in range(5120, 16385, 512):
        if ops._tall_tile_plan(M, N, K):
            assert ops._wide_parts_plan(M, N, K), K
    # narrow products stay with the others
    assert ops._wide_parts_plan(M, 1280, 6144) is None


@pytest.mark.parametrize("M", [129, 256, 400, 512, 640, 1024])
def test_no_parts_of_less_than_1024_k(M):
    for N in range(1024, 8193, 256):
        assert not ops._wide_parts_plan(M, N, 3520)
        for K in range(3584, 8193, 256):
            plan = ops._wide_parts_plan(M, N, K)
            assert plan is None or K // plan[1] >= 1024
            assert plan is None or M > 512 or N > 2048 or K >= 5120


def test_products_that_the_library_fills_are_its_own():
    """Sizes at which it is the faster one, and ones at which it is not."""
    for M, N, K in ((384, 3584, 2560), (768, 2048, 2560), (1536, 1024, 2560),
                    (384, 8192, 3072)):
        assert ops._wide_rows_tile(M, N, K) is None, (M, N, K)
    for M, N, K in ((768, 1536, 1024), (2039, 4096, 4096), (2039, 6144, 4096),
                    (7000, 3584, 2560), (300, 24576, 7168), (5000, 8192, 14336)):
        assert ops._wide_rows_tile(M, N, K), (M, N, K)


def test_products_shorter_than_a_call_of_the_library():
    """They are taken though some take the device a little longer."""
    for M, N, K in ((312, 3072, 2048), (500, 3072, 2048), (646, 2048, 2048)):
        assert ops._wide_rows_tile(M, N, K), (M, N, K)
    assert ops._wide_silu_tile(768, 1344, 1024)
    # longer ones, by the device alone
    assert ops._wide_rows_tile(384, 4096, 2560) is None
    assert ops._wide_silu_tile(144, 11264, 1536) is None


@pytest.mark.parametrize("M", [1, 8, 16, 17, 64, 65, 128])
def test_tiles_that_end_in_the_activation(M):
    """Uncut tiles of 64 or 128 columns do; of 64 not where two runs of 32 rows
    meet on the memory channels."""
    for N in range(8192, 65537, 256):
        for K in (2048, 4096, 6144, 8192):
            plan = ops._rows_tile_plan(M, N, K)
            whole = plan is not None and plan[1] == 1 and plan[0] >= 64
            meet = whole and plan[0] == 64 and K == 4096
            assert ops._silu_plan(M, N, K) == (
                plan if whole and not meet else None)


@pytest.mark.parametrize("M", [1, 8, 16])
@pytest.mark.parametrize("N", [1024, 2048, 2304, 3072, 4096, 4104, 5120, 6144,
                               8192])
def test_parts_of_long_rows_at_every_length(M, N):
    """From 4096 k to where the whole product is cut anyway."""
    for K in range(4096, 11008, 64):
        plan = ops._parts_plan(M, N, K)
        assert plan is not None, K
        assert 1 < plan[1] <= 8 and plan[1] <= K // 64
        assert plan[1] * -(-N // plan[0]) <= 256


@pytest.mark.parametrize("M", [1, 8, 16, 17, 24, 64, 65, 128])
def test_parts_of_short_rows_at_every_width(M):
    """Products that only the library is beside are cut up to 4096 columns; with
    the decode product, from one length of rows on."""
    for N in range(1024, 4097, 8):
        for K in (1088, 1984, 2624):
            assert ops._parts_plan(M, N, K) is not None, (N, K)
        for K in range(1024, 4096, 128):
            if M > 16 and (M <= 64 or K < 3072) or M <= 16 and K >= 3072:
                assert ops._parts_plan(M, N, K) is not None, (N, K)
