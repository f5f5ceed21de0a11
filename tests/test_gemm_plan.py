"""Which GEMM kernel the entry points run for a shape (host-side planner, no GPU code runs)."""
import pytest


@pytest.mark.parametrize("N,K,M,want", [
    (4096, 3584, 17, 10), (28672, 4096, 17, 18), (37888, 3584, 64, 5), (37888, 3584, 129, 6),
    (2048, 1024, 700, 17), (2048, 768, 700, 5), (1024, 640, 1100, 5), (512, 512, 400, 12),
    (512, 384, 17, 5)])
def test_default_variant(lib, N, K, M, want):
    """The K-splitting kernel (9 + tile shape) in one round, its two largest tiles from K = 1024 on."""
    for token in (0, 1):
        assert lib.fp8kv_gemm_plan(N, K, M, token) == want
