"""GPU test of the 128 x 128 blocks of the prompt products: output widths that no bigger block divides (640 = 5 x 128 features), ragged last
row blocks, the shortest K: f32 sums and SwiGLU by themselves, squared ReLU and GELU through a decoder.  The reference is the chunked kernel."""
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


@pytest.mark.parametrize("rows", [129, 257, 400, 513])
@pytest.mark.parametrize("ff", [4608, 1152])
@pytest.mark.parametrize("act", ["squared ReLU", "GELU"])
def test_activation_by_epilogue_and_by_launch(rows, ff, act):
    """a decoder's activation in the product's epilogue (whenever the shape fits: 128 x 128 blocks here), as the rule has it (a launch
    of its own behind a product with split K for the fewer rows), and from the chunked kernel"""
    import numpy as np

    import nano_vllm_candle_amd as pkg
    from nano_vllm_candle_amd.gopunex import LightningConfig
    from nano_vllm_candle_amd.lefalix import DeltaConfig, DenseConfig

    if act == "GELU":
        m = pkg.LefalixForCausalLM.from_random(pkg.LefalixConfig(512, 1024, [((DeltaConfig(4, 4, 64, 64, 4, 64, 64),), DenseConfig(ff))]))
    else:
        m = pkg.GopunexForCausalLM.from_random(pkg.GopunexConfig(512, 1024, [(LightningConfig(4, 64, 64, (0.9, 0.95, 0.98, 0.99)), ff)], 1e-6, 1.0, 0.5))
    m.kv_alloc(8, 3, 1024)
    toks = [np.random.default_rng(rows).integers(0, 512, rows)]
    want = [[0, rows // 2, rows - 1]]
    out = {}
    for wgs in (0, 1, 64):
        m.set_option("tile_min_wgs", wgs)
        out[wgs] = m.step_score([0], toks, True, want)
    m.close()
    # sums of up to 4608 f32 in other orders, values as two 16-bit planes (2^-17) that may round the other way, through one layer
    for wgs in (1, 64):
        assert np.abs(out[wgs] - out[0]).max() < 2.0 ** -14 * np.abs(out[0]).max(), wgs
