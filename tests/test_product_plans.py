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
