"""GPU test of the register-direct products of more than 256 rows, against the tile products: both ends of the ranges and of a round of row blocks,
the norms of more blocks than a workgroup has waves, rows that end within a block, prompts of one and of several sequences, a decode step, 16- and 24-bit caches, and widths whose grids leave other numbers of
blocks to a workgroup.  Which form ran is counted: q/k/v, o, gate/up and down of two layers, past 480 rows q/k/v and the first layer's gate/up."""
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


def compare(m, call, pairs, bits=16):
    def counted():
        n, t = m.counter("row_pair_launches"), m.counter("tile_gemm_launches")
        return call(), m.counter("row_pair_launches") - n, m.counter("tile_gemm_launches") - t

    got, taken, tiles = counted()
    m.set_option("no_fused", 1)
    m.set_option("tile_min_wgs", 1)  # tile products wherever they fit
    want, none, all_tiles = counted()
    m.set_option("no_fused", 0)
    m.set_option("tile_min_wgs", 64)
    assert taken == pairs and none == 0 and all_tiles > 0 and (tiles == 0) == (pairs == 8)
    # products summed in another order; a cached f16 key or value may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    assert np.isfinite(got).all() and np.abs(got - want).max() < 2.0 ** (-11 if bits == 16 else -14) * np.abs(want).max()


@pytest.mark.parametrize("rows,bits", [(256, 16), (257, 16), (272, 24), (273, 16), (384, 16), (385, 24), (479, 16), (480, 16), (481, 16), (512, 24), (513, 16), (640, 16), (641, 16), (768, 16), (895, 24), (896, 16), (897, 16)])
def test_a_prompt(rows, bits):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4, bits)
    t = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows)
    want = [0, 15, 16, rows // 2, rows - 2]  # (the head's buffers hold five rows)
    compare(m, lambda: m.step_score([0], [t], True, [want]), 8 if rows <= 480 else 3 if rows <= 896 else 0, bits)
    m.close()


# gate/up of 2048 and 4096 features are no multiple of 96: tile products
@pytest.mark.parametrize("inter,heads,kv,lens,pairs", [(3072, 16, 8, [100, 1, 230], 8), (1024, 8, 2, [300], 0), (2048, 8, 8, [17] * 28, 0), (3072, 24, 4, [90, 380], 8), (3072, 16, 8, [400, 1, 260], 3),
                                                       (3072, 24, 4, [520], 3), (3072, 24, 24, [300], 8), (1536, 16, 8, [500], 3)])
def test_prompts_of_other_widths(inter, heads, kv, lens, pairs):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, len(lens), 16, inter, heads, kv)
    rng = np.random.default_rng(inter)
    seqs = [rng.integers(0, cfg.vocab_size, n) for n in lens]
    compare(m, lambda: m.step_score(list(range(len(lens))), seqs, True, [[n - 1] for n in lens]), pairs)
    m.close()


@pytest.mark.parametrize("rows", [257, 300, 480])
def test_a_decode_step(rows):
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, rows)
    rng = np.random.default_rng(rows)
    seqs = [rng.integers(0, cfg.vocab_size, 2 + i % 3) for i in range(rows)]
    ids = list(range(rows))
    m.step(ids, [s[:-1] for s in seqs], True)
    compare(m, lambda: m.step_score(ids, seqs, False, [[len(s) - 1] for s in seqs]), 8)
    m.close()


@pytest.mark.parametrize("rows", [257, 480])
def test_row_major_planes(rows):
    # row pairs read packed planes: without them tile products, as past 480 rows
    import nano_vllm_candle_amd as pkg

    cfg, m = model(pkg, 4)
    t = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows)
    m.set_option("no_xpack", 1)
    n, tiles = m.counter("row_pair_launches"), m.counter("tile_gemm_launches")
    got = m.step_score([0], [t], True, [[rows - 1]])
    assert m.counter("row_pair_launches") == n and m.counter("tile_gemm_launches") > tiles
    m.set_option("no_xpack", 0)
    want = m.step_score([0], [t], True, [[rows - 1]])
    # as in compare()
    assert m.counter("row_pair_launches") == n + 8 and np.abs(got - want).max() < 2.0 ** -11 * np.abs(want).max()
    m.close()
