"""The prompt GEMM's tile choice (``qwen_gemm_tile``): host arithmetic, no GPU."""

import os

import pytest

from qwen_hip import _lib, ops

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libqwen_hip.so not built")


def test_a_tile_for_every_size():
    for N in (128, 384, 640, 1280, 2560, 6144, 19456):
        for K in (64, 128, 192, 2560, 9728, 1 << 22, (1 << 22) + 64, 1 << 27):
            for M in (1, 2, 15, 16, 17, 255, 1551, 16384):
                if M * K < 2 ** 31 - 1:
                    bm, bn = ops.gemm_tile(M, N, K, 256)
                    assert N % bn == 0 and bm % 32 == 0


def test_refused_sizes():
    for M, N, K in ((0, 128, 64), (1, 64, 64), (1, 192, 64), (1, 128, 32), (1, 128, 96), (1 << 21, 128, 1 << 10)):
        assert _lib.query("qwen_gemm_tile", M, N, K, 256) == 0


def test_long_k_leaves_out_only_what_32_bit_offsets_do_not_reach():
    """A wavefront of the 256 x 256 tile addresses 16 n-tiles from one base, of the 32 x 128 tile two, of all others
    one: k alone does not change the choice before that."""
    for M, N in ((2, 128), (17, 19456), (250, 2560), (250, 1 << 16)):
        a, b = ((1 << 21) - 64, (1 << 22) + 128 * 5)
        if M * b < 2 ** 31 - 1:
            assert ops.gemm_tile(M, N, a, 256) == ops.gemm_tile(M, N, a + 128 * 7, 256)
            assert ops.gemm_tile(M, N, b, 256) == ops.gemm_tile(M, N, (1 << 22) - 128, 256)
    assert ops.gemm_tile(250, 1 << 16, 1 << 22, 256) == (256, 256)
    assert ops.gemm_tile(200, 1 << 16, 9 << 20, 256) != (256, 256)
    assert ops.gemm_tile(17, 19456, 1 << 26, 256) == (32, 128)
    assert ops.gemm_tile(15, 19456, (1 << 27) + 128, 256) != (32, 128)
