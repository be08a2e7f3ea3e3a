"""GPU test of the q-tiles that a prompt's attention walks with one to a workgroup: those with rows, whatever fills up the groups of the other form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def model(heads, kv, blocks, seqs, rows=4096, **kw):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=256, head_dim=kw.get("hd", 128), num_attention_heads=heads, num_key_value_heads=kv, max_position_embeddings=8192)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if kw.get("bits") == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.kv_alloc(blocks, seqs, rows)
    return cfg, m


@pytest.mark.parametrize("heads,kv,tile", [(16, 8, 16), (8, 8, 32), (16, 2, 4)])
@pytest.mark.parametrize("cached,new", [(100, [5, 6, 7, 9]), (0, [65, 33, 2, 200]), (300, [17])])
def test_tiles_with_rows_alone(heads, kv, tile, cached, new):
    cfg, m = model(heads, kv, 16, len(new))
    m.set_option("prefill_deal", 1)
    m.set_option("last_rows", 0)
    rng = np.random.default_rng(tile)
    seqs = [rng.integers(0, cfg.vocab_size, cached + n) for n in new]
    ids = list(range(len(new)))
    if cached:
        m.step(ids, [s[:cached] for s in seqs], True)
    before = m.counter("prefill_dealt_tiles")
    m.step(ids, seqs, not cached)
    assert m.counter("prefill_dealt_tiles") - before == cfg.num_hidden_layers * sum(-(-n // tile) for n in new)
    m.close()


@pytest.mark.parametrize("new,every", [([70] * 8, 1), ([80] * 7 + [16] * 2, 1), ([70] * 6, 0), ([70] * 9, 0)])
def test_groups_stay_whole_where_all_fit_at_once(new, every):
    # 8 key heads: more than 32 q-tiles with rows (a CU's two workgroups), at most 64 with those that fill up the groups
    cfg, m = model(16, 8, 16, len(new))
    m.set_option("prefill_deal", 1)
    m.set_option("last_rows", 0)
    rng = np.random.default_rng(2)
    m.step(list(range(len(new))), [rng.integers(0, cfg.vocab_size, n) for n in new], True)
    tiles = [-(-n // 16) for n in new]
    assert m.counter("prefill_dealt_tiles") == cfg.num_hidden_layers * sum(-(-t // 4) * 4 if every else t for t in tiles)
    m.close()


# many contexts behind cached prefixes, on both sides of the rule: contexts but the longest in an XCD's L2 or not (key heads / 8 x tokens x 512 bytes against 5.5 MB, 20 MB with more than
# 256 workgroups of the shared form), K/V tiles of all q-tiles against 512 x 1.2 and x 2 those of the longest; heads of 64, whose line is 96 + half of the longest
@pytest.mark.parametrize("heads,kv,hd,bits,cached,new,seqs,dealt", [
    (16, 2, 128, 16, 500, 20, 64, 0), (16, 2, 128, 16, 500, 20, 16, 1), (8, 8, 128, 16, 1000, 60, 64, 0), (8, 8, 128, 16, 1000, 60, 8, 1), (32, 8, 128, 16, 2000, 100, 8, 0),
    (16, 8, 128, 16, 2000, 100, 8, 1), (32, 2, 128, 24, 500, 20, 64, 0), (16, 8, 128, 24, 1000, 16, 40, 1), (14, 2, 64, 16, 0, 264, 8, 0), (14, 2, 64, 16, 0, 264, 6, 1)])
def test_the_rule_behind_prefixes(heads, kv, hd, bits, cached, new, seqs, dealt):
    cfg, m = model(heads, kv, seqs * (-(-(cached + new) // 256)), seqs, 8192, hd=hd, bits=bits)
    m.set_option("last_rows", 0)
    rng = np.random.default_rng(1)
    toks = [rng.integers(0, cfg.vocab_size, cached + new) for _ in range(seqs)]
    ids = list(range(seqs))
    for i in range(0, seqs if cached else 0, 4):
        m.step(ids[i:i + 4], [t[:cached] for t in toks[i:i + 4]], True)
    before = m.counter("prefill_dealt_launches")
    m.step(ids, toks, False)
    assert m.counter("prefill_dealt_launches") - before == dealt * cfg.num_hidden_layers
    m.close()
