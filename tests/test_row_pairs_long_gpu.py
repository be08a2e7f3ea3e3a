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


def prompt(m, cfg, rows):
    """logits of a prompt, products of row pairs"""
    t = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows)
    n, r = m.counter("row_pair_launches"), m.counter("tile_resid_launches")
    got = m.step_score([0], [t], True, [[rows // 2, rows - 1]])
    pairs = m.counter("row_pair_launches") - n
    assert (m.counter("tile_resid_launches") > r) == (rows > 480)
    m.enable_taps()  # slabs and norm launches
    want = m.step_score([0], [t], True, [[rows // 2, rows - 1]])
    m.enable_taps(False)
    # products summed in another order; a cached f16 key or value may round the other way: 2^-11 of the largest logit
    assert np.isfinite(got).all() and np.abs(got - want).max() < 2.0 ** -11 * np.abs(want).max()
    return pairs


# gate/up, then q/k/v, of 24 MB and more: not this kernel's, and tile products with the residual in o and down all the same; gate/up just below
@pytest.mark.parametrize("inter,heads,kv,pairs", [(6144, 16, 8, 0), (6912, 16, 8, 0), (3072, 64, 16, 0), (5760, 16, 8, 3)])
@pytest.mark.parametrize("rows", [300, 481, 640, 896])
def test_matrices_of_24_mb(inter, heads, kv, pairs, rows):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4, 16, inter, heads, kv)
    got = prompt(m, cfg, rows)
    assert rows == 300 or got == (pairs if rows == 481 else 0)
    m.close()


# the last row count whose workgroups the CUs hold at once and the next: gate/up of 9216, 11520 and 6912 features, q/k/v of 5120 and 6144, q/k/v of 9216, which are never that few, and both as narrow as
# the rows go on
@pytest.mark.parametrize("inter,heads,kv,last", [(4608, 16, 8, 512), (5760, 16, 8, 512), (3456, 16, 8, 768), (3072, 24, 8, 768), (3072, 16, 16, 512), (3072, 24, 24, 480), (3072, 16, 8, 896)])
def test_one_round_of_workgroups(inter, heads, kv, last):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4, 16, inter, heads, kv)
    # two layers, the last one's gate/up on the rows that are asked for alone
    assert last == 480 or prompt(m, cfg, last) == 3
    assert prompt(m, cfg, last + 1) == 0
    m.close()
