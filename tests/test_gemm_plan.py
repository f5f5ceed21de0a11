"""Which GEMM kernel the entry points run for a shape (host-side planner, no GPU code runs)."""
import pytest


@pytest.mark.parametrize("N,K,M,want", [
    (4096, 3584, 17, 10), (28672, 4096, 17, 18), (37888, 3584, 64, 5), (37888, 3584, 129, 6),
    (2048, 1024, 700, 17), (2048, 768, 700, 5), (1024, 640, 1100, 5), (512, 512, 400, 12),
    (512, 384, 17, 5),
    (3584, 1536, 1000, 19), (3584, 1152, 1000, 5), (3584, 512, 1000, 5), (3584, 1536, 1100, 5), (8192, 1536, 1100, 6)])
def test_default_variant(lib, N, K, M, want):
    """The K-splitting kernel (9 + tile shape) in one round, its two largest tiles from K = 1024 on; then
    variant 6 past one round of its tiles, K groups where 128 x 128 tiles get a CU each and K has the halves, 5."""
    for token in (0, 1):
        assert lib.fp8kv_gemm_plan(N, K, M, token) == want


@pytest.mark.parametrize("variant", [0, 4, 5, 6, 8, 9, 18, 19])
@pytest.mark.parametrize("N,K,M", [(4096, 3584, 300), (3584, 1536, 1000), (256, 512, 16)])
def test_a_forced_variant_is_the_one_that_runs(lib, variant, N, K, M):
    try:
        lib.fp8kv_gemm_tune(variant, 0)
        assert lib.fp8kv_gemm_plan(N, K, M, 0) == variant
        default = lib.fp8kv_gemm_plan(N, K, M, 1)
        lib.fp8kv_gemm_tune(-1, 0)
        assert default == (variant if variant in (5, 6) or variant >= 9 else lib.fp8kv_gemm_plan(N, K, M, 1))
    finally:
        lib.fp8kv_gemm_tune(-1, 0)
