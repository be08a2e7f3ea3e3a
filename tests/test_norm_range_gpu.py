"""GPU test of the norm of rows whose sum of squares lies between half of a float's range and all of it, over the widths where the kernel's forms change."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3, 130])
@pytest.mark.parametrize("width", [512, 1024, 2048, 4096, 8192])
def test_a_sum_above_half_the_range(width, rows):
    from nano_vllm_candle_amd import layers

    rng = np.random.default_rng(width)
    x = rng.uniform(0.9, 1.1, (rows, width)) * rng.choice([-1, 1], (rows, width))
    x = (x * np.sqrt(2.6e38 / np.square(x).sum(1, keepdims=True))).astype(np.float32)  # the largest float is 3.4e38
    w = rng.uniform(0.5, 1.5, width).astype(np.float32)
    y, _ = layers.RMSNorm.from_weight(w, 1e-6)(x)
    want = x.astype(np.float64) / np.sqrt(np.square(x.astype(np.float64)).mean(1, keepdims=True)) * w
    # a sum by halves of up to 8192 squares, four more roundings: 2^-24 each
    assert np.abs(y / want - 1).max() < 20 * 2.0 ** -24
