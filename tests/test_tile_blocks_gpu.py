"""GPU test of the 128 x 128 blocks of the prompt products: output widths that no bigger block divides (640 = 5 x 128 features), ragged last
row blocks, the shortest K, each epilogue that has them.  The reference is the chunked kernel."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(129, 640, 128), (257, 640, 384), (300, 640, 1024), (1, 128, 128), (128, 128, 4096), (257, 6144, 1024), (513, 1024, 3072)])
@pytest.mark.parametrize("mode,packed", [(0, 0), (2, 0), (2, 1)])
def test_small_blocks_equal_the_chunked_kernel(M, N, K, mode, packed):
    from nano_vllm_candle_amd import _lib, layers

    ctx = layers.default_context()
    d, r, u0, u1 = C.c_float(), C.c_float(), C.c_float(), C.c_float()
    _lib.check(_lib.lib().nvllm_debug_gemm_tile_check(ctx.h, M, N, K, mode, packed, 2, C.byref(d), C.byref(r), C.byref(u0), C.byref(u1)), ctx.h)
    assert r.value > 0
    # the same products summed in the same order; K splits meet in f32: K / 32 sums of 2^-24
    assert d.value <= K / 32 * 2.0 ** -24 * r.value + (2.0 ** -16 * r.value if mode else 0), (d.value, r.value)
