"""GPU test of the register-direct products of more than 256 rows, against the tile products: both ends of the ranges and of a round of row blocks,
the norms of more blocks than a workgroup has waves, rows that end within a block, prompts of one and of several sequences, a decode step, 16- and 24-bit caches, and widths whose grids leave other numbers of blocks to a workgroup."""
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


def compare(m, call, bits=16):
    got, tiles = call(), m.counter("tile_gemm_launches")
    m.set_option("no_fused", 1)
    m.set_option("tile_min_wgs", 1)  # tile products wherever they fit
    want = call()
    m.set_option("no_fused", 0)
    m.set_option("tile_min_wgs", 64)
    # products summed in another order; a cached f16 key or value may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    assert np.isfinite(got).all() and np.abs(got - want).max() < 2.0 ** (-11 if bits == 16 else -14) * np.abs(want).max()
    return tiles


@pytest.mark.parametrize("rows,bits", [(256, 16), (257, 16), (272, 24), (273, 16), (384, 16), (385, 24), (479, 16), (480, 16), (481, 16), (512, 24), (513, 16), (640, 16), (641, 16), (768, 16), (895, 24), (896, 16), (897, 16)])
def test_a_prompt(rows, bits):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4, bits)
    t = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows)
    want = [0, 15, 16, rows // 2, rows - 2]  # (the head's buffers hold five rows)
    tiles = compare(m, lambda: m.step_score([0], [t], True, [want]), bits)
    assert (tiles == 0) == (rows <= 480)
    m.close()


@pytest.mark.parametrize("inter,heads,kv,lens", [(3072, 16, 8, [100, 1, 230]), (1024, 8, 2, [300]), (2048, 8, 8, [17] * 28), (3072, 24, 4, [90, 380]), (3072, 16, 8, [400, 1, 260]), (3072, 24, 4, [520])])
def test_prompts_of_other_widths(inter, heads, kv, lens):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, len(lens), 16, inter, heads, kv)
    rng = np.random.default_rng(inter)
    seqs = [rng.integers(0, cfg.vocab_size, n) for n in lens]
    compare(m, lambda: m.step_score(list(range(len(lens))), seqs, True, [[n - 1] for n in lens]))
    m.close()


@pytest.mark.parametrize("rows", [257, 300, 480])
def test_a_decode_step(rows):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, rows)
    rng = np.random.default_rng(rows)
    seqs = [rng.integers(0, cfg.vocab_size, 2 + i % 3) for i in range(rows)]
    ids = list(range(rows))
    m.step(ids, [s[:-1] for s in seqs], True)
    assert compare(m, lambda: m.step_score(ids, seqs, False, [[len(s) - 1] for s in seqs])) >= 0
    m.close()
