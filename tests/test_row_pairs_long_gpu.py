"""GPU test of the register-direct products of more than 256 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def model(pkg, rows, bits=16, inter=3072, heads=16, kv=8):
    cfg = pkg.Qwen3Config.tiny(vocab_size=1024, hidden_size=1024, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128, num_hidden_layers=2)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.kv_alloc(rows + 16, rows + 1, 1024)
    return cfg, m


# gate/up, then q/k/v, of 24 MB and more: not this kernel's, and tile products with the residual in o and down all the same; the last two are just below
@pytest.mark.parametrize("inter,heads,kv,pairs", [(6144, 16, 8, 0), (6912, 16, 8, 0), (3072, 64, 16, 0), (5760, 16, 8, 3), (3072, 60, 15, 3)])
@pytest.mark.parametrize("rows", [300, 481, 640, 896])
def test_matrices_of_24_mb(inter, heads, kv, pairs, rows):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4, 16, inter, heads, kv)
    t = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows)
    n = m.counter("row_pair_launches")
    got = m.step_score([0], [t], True, [[rows // 2, rows - 1]])
    if rows > 480:
        assert m.counter("row_pair_launches") - n == pairs and m.counter("tile_resid_launches") > 0
    m.enable_taps()
    want = m.step_score([0], [t], True, [[rows // 2, rows - 1]])
    # products summed in another order; a cached f16 key or value may round the other way: 2^-11 of the largest logit
    assert np.isfinite(got).all() and np.abs(got - want).max() < 2.0 ** -11 * np.abs(want).max()
    m.close()
