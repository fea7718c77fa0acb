"""Which tile the prefill GEMMs take for a shape (host rules, through the library's test hooks; no GPU): properties that the
results rest on, and the choices that the rules' comments state with their measurements."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def L():
    import ling_gemm
    for name, n in (("lq_debug_prefill_fp8_tile", 4), ("lq_debug_prefill_nvfp4_tile", 5)):
        fn = getattr(ling_gemm.lib, name)
        fn.argtypes, fn.restype = [ctypes.c_int] * n, ctypes.c_int
    return ling_gemm.lib


@pytest.mark.parametrize("cus", [256, 228, 64])
@pytest.mark.parametrize("swiglu", [0, 1])
def test_nvfp4_waves_along_k_do_not_depend_on_m(L, swiglu, cus):
    """The order of a row's sums is that of the waves along K: a matter of the matrix alone."""
    both = set()
    for N in (128, 384, 640, 1152, 2048, 2688, 4224, 5120, 6528, 7168, 8320, 13824, 17408, 34816):
        for K in (128, 512, 1024, 1152, 2688, 5120, 7552, 17408):
            waves = {L.lq_debug_prefill_nvfp4_tile(swiglu, M, N, K, cus) % 16
                     for M in (1, 17, 63, 64, 65, 81, 128, 200, 300, 777, 1000, 2048, 4096, 10000)}
            assert len(waves) == 1, f"N={N} K={K}: {waves}"
            both |= waves
    assert both == {1, 2}


@pytest.mark.parametrize("swiglu,M,N,K,tile", [
    (0, 128, 5120, 5120, (4, 1)), (0, 300, 5120, 5120, (8, 1)), (0, 128, 5120, 17408, (4, 1)), (0, 500, 2048, 4096, (4, 1)),
    (0, 2048, 7168, 5120, (8, 1)), (0, 2048, 34816, 5120, (8, 2)), (1, 2048, 17408, 5120, (8, 2)),
    (1, 2048, 6144, 2048, (8, 2)), (1, 2048, 5120, 5120, (8, 1))])
def test_nvfp4_choices_as_measured(L, swiglu, M, N, K, tile):
    assert divmod(L.lq_debug_prefill_nvfp4_tile(swiglu, M, N, K, 256), 16) == tile


@pytest.mark.parametrize("M,N,K,tile,parts", [
    (200, 2048, 4096, 1, 1), (200, 7168, 5120, 2, 1), (300, 5120, 17408, 2, 1), (512, 5120, 5120, 3, 1),
    (1500, 5120, 17408, 4, 1), (1000, 5120, 17408, 0, 3), (500, 17408, 5120, 0, 1), (4096, 34816, 5120, 0, 1),
    (4096, 5120, 17408, 0, 4)])
def test_fp8_choices_as_measured(L, M, N, K, tile, parts):
    assert divmod(L.lq_debug_prefill_fp8_tile(M, N, K, 256), 8) == (tile, parts)


@pytest.mark.parametrize("cus", [256, 64, 8])
def test_256_tiles_only_where_their_offsets_stay_within_the_operands(L, cus):
    """The 256 x 256 tile's scalar offsets need 129 tokens and 256 weight rows."""
    taken = 0
    for M in (1, 17, 64, 81, 128, 129, 192, 256, 1000, 100000):
        for N in (128, 256, 384, 5120, 34816, 151936):
            for K in (128, 1024, 5120, 17408):
                whole = L.lq_debug_prefill_fp8_tile(M, N, K, cus) // 8 == 0
                assert not whole or (M >= 129 and N >= 256), f"{M} x {N} x {K}"
                taken += whole
    assert taken
