"""Which kernel a linear layer's launch takes, by its sizes. The choices are host code in the library and need no GPU;
every kernel gives a row the same bits (test_gpu_kernels.py), so only the time depends on them. Each line of a table was
measured on both sides, W from HBM."""
import ctypes

import pytest

from ember_amd import _lib


def _gemv_args(M, N, K, packed, lda=None):
    g = _lib.GemvArgs()
    g.M, g.N, g.K, g.lda, g.ldc, g.w_packed = M, N, K, lda or K, N, int(packed)
    return g


def _host(symbol, restype, *argtypes):
    fn = _lib.lib()[symbol]
    fn.restype, fn.argtypes = restype, list(argtypes)
    return fn


@pytest.mark.parametrize("M,N,K,packed,tiles", [
    # up to 16 rows, and one round of work-groups: the decode-sized kernel
    (16, 151936, 1024, True, False), (16, 24576, 4096, False, False), (64, 4096, 2048, True, False),
    (33, 4096, 2048, False, False),
    # staged activations: tiles for large packed W only
    (32, 12288, 2048, True, True), (17, 151936, 1024, True, True), (64, 151936, 1024, True, True),
    (64, 6144, 1024, True, False), (32, 5120, 2048, True, False), (32, 12288, 2048, False, False),
    # too many to stage, more than 8192 features: tiles for either layout (17 x 9728 x 2560, row-major: 22.5 -> 20.6 us)
    (17, 9728, 2560, False, True), (17, 9728, 2560, True, True), (33, 9728, 1376, False, True),
    # up to 8192: few rows and row-major W stay (us, GEMV against tiles: 17 x 6144 x 2560, row-major, 15.5 / 19.6; 24 x
    # 5120 x 2560 16.8 / 19.8; 17 x 8192 x 3072, packed, 14.7 / 16.5)
    (17, 6144, 2560, False, False), (24, 5120, 2560, False, False), (32, 8192, 4096, False, False),
    (17, 8192, 3072, True, False), (20, 8192, 3072, True, False),
    (32, 4112, 4096, True, True), (33, 4112, 2560, True, True), (40, 4112, 2560, False, True),
    # rows of A that are not whole 128-byte lines (us: 33 x 4112 x 2080, packed, 11.2 / 12.9)
    (33, 4112, 2080, True, False), (64, 5000, 1376, True, False), (33, 5000, 2080, False, False),
])
def test_batches_of_17_to_64_on_tiles(M, N, K, packed, tiles):
    fn = _host("_ZN5ember3hip13gemv_on_tilesERK13EmberGemvArgsb", ctypes.c_bool, ctypes.c_void_p, ctypes.c_bool)
    g = _gemv_args(M, N, K, packed)
    assert fn(ctypes.addressof(g), False) is tiles
    assert fn(ctypes.addressof(g), True) is False  # a K split stays
    if tiles and N <= 8192:
        g.lda = K + 32
        assert fn(ctypes.addressof(g), False) is False


@pytest.mark.parametrize("R,N,K,one", [
    # up to 512 work-groups: one launch (us, two launches against one: 4 x 4096 x 1024 5.7 / 4.2, 4 x 8192 x 2048 0.96)
    (1, 4096, 1024, True), (4, 6144, 1024, True), (4, 8192, 2048, True), (4, 2048, 128, True), (5, 4096, 1024, False),
    (4, 8192, 128, False), (1, 4096, 2176, False),
    # up to 1024: where W takes long enough to hide the repeated norm (4 x 12288 x 512 6.6 / 7.8)
    (4, 12288, 2048, True), (1, 12288, 512, True), (2, 16384, 512, True), (3, 16384, 1024, True),
    (3, 12288, 512, False), (4, 12288, 512, False), (4, 12288, 1024, False), (4, 12288, 1536, False), (2, 16384, 128, False),
    # beyond: two (4 x 65520 x 1024 25.3 / 35.6)
    (1, 16400, 2048, False), (4, 65520, 1024, False),
])
def test_the_norm_inside_the_projection(R, N, K, one):
    fn = _host("_ZN5ember3hip14gemv_norm_fitsERK13EmberGemvArgsRK13EmberNormArgs", ctypes.c_bool, ctypes.c_void_p,
               ctypes.c_void_p)
    g, n = _gemv_args(R, N, K, True), _lib.NormArgs()
    n.R, n.hidden = R, K
    assert fn(ctypes.addressof(g), ctypes.addressof(n)) is one
    g.w_packed = 0
    assert fn(ctypes.addressof(g), ctypes.addressof(n)) is False


@pytest.mark.parametrize("M,N,K,split,gemv", [
    # us, W from HBM, tiles against two launches: 65 x 1024 x 2048 10.5 / 7.8, 128 x 1024 x 3072 16.0 / 10.9
    (65, 1024, 2048, False, True), (128, 1024, 3072, False, True), (128, 512, 1024, False, True),
    (128, 1024, 4096, False, True), (128, 2048, 1024, False, True), (96, 2048, 2048, False, True),
    (128, 1536, 2048, False, True), (96, 3072, 512, False, True), (65, 2048, 6144, True, True), (128, 1024, 12288, True, True),
    # 97 x 2048 x 2048 0.94, 65 x 2048 x 3072 0.87, 65 x 4096 x 1024 8.1 / 8.2, 65 x 6144 x 1024 8.7 / 12.8
    (97, 2048, 2048, False, False), (65, 2048, 3072, False, False), (65, 4096, 1024, False, False),
    (65, 6144, 1024, False, False), (128, 3072, 512, False, False), (65, 2560, 6144, True, False),
    # up to 64 rows there is nothing to choose; from 129 on the tiles (129 x 1024 x 2048 10.5 / 11.9)
    (64, 1024, 2048, False, False), (129, 1024, 2048, False, False), (1800, 1024, 2048, False, False),
])
def test_products_of_65_to_128_rows(M, N, K, split, gemv):
    fn = _host("_ZN5ember3hip12gemm_by_gemvERK13EmberGemvArgs", ctypes.c_bool, ctypes.c_void_p)
    g = _gemv_args(M, N, K, True)
    need = _lib.lib().ember_hip_gemv_workspace_bytes(64, N, K)
    assert (need > 0) == split
    g.workspace, g.workspace_bytes = 256, need  # an address that nothing reads
    assert fn(ctypes.addressof(g)) is gemv
