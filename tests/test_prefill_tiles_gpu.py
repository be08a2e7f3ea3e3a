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
