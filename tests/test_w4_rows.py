"""How many rows the packed int4 product takes before the weight is expanded."""
from types import SimpleNamespace

import pytest

import gpustack_amd.engine  # noqa: F401  (package import order)
from gpustack_amd.models.llama import _w4_takes


def _takes(M, N, K, **kw):
    x = SimpleNamespace(is_cuda=True, dim=lambda: 2, shape=(M, K), **kw)
    return _w4_takes(x, SimpleNamespace(shape=(N, K)))


@pytest.mark.parametrize("M,N,K,takes", [
    (1, 64, 128, True), (0, 64, 128, False), (192, 28672, 4096, True),
    (193, 28672, 4096, False), (64, 96, 128, False), (64, 64, 131072, True),
    (64, 64, 131200, False),
    # a last round of 4 to 40 workgroups behind 512
    (128, 22016, 4096, True), (129, 22016, 4096, True),
    (192, 21888, 2048, True), (160, 23552, 4096, True),
    (160, 21760, 4096, True), (160, 24576, 4096, True),
    (160, 22016, 5120, True)])
def test_rows_of_a_packed_product(monkeypatch, M, N, K, takes):
    monkeypatch.delenv("GPUSTACK_AMD_W4_KERNEL", raising=False)
    assert _takes(M, N, K) == takes
    monkeypatch.setenv("GPUSTACK_AMD_W4_KERNEL", "1")
    assert _takes(M, N, K) == (0 < M <= 1024 and N % 64 == 0 and K <= 131072)
