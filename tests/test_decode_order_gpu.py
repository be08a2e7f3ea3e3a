"""GPU test of the decode attention's launch order: kv heads fastest, rows longest context first and every other run of 256 workgroups
backwards.  Each row must be visited once whatever the rows and the kv heads of a run are: a row left out keeps what its memory held."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 256 / kv rows to a run: 32 rows of 8 heads, 85 of 3, 256 of one; the fused step takes up to 256 rows
@pytest.mark.parametrize("kv,heads", [(8, 8), (3, 6), (1, 4)])
@pytest.mark.parametrize("rows", [31, 33, 65, 86, 171, 256, 257])
def test_every_row_of_a_decode_batch_is_its_own_answer(kv, heads, rows):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=256, num_attention_heads=heads, num_key_value_heads=kv)  # (256: the head in slices of 64 rows)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(rows + 3, rows + 1, 512)
    rng = np.random.default_rng(rows + kv)
    seqs = [rng.integers(0, cfg.vocab_size, int(n)) for n in rng.permutation(np.arange(rows) % 97 + 1)]
    m.step(list(range(rows)), seqs, True, want_logits=False)
    lists = [np.append(s, 5) for s in seqs]
    _, got = m.step(list(range(rows)), lists, False, want_logits=True)
    # the same rows in the reverse order: another order of launch positions, the same arithmetic per row
    _, back = m.step(list(range(rows))[::-1], lists[::-1], False, want_logits=True)
    assert np.array_equal(got, back[::-1])
    # and the shortest, a middle and the longest one as a prompt of their own (two 16-bit planes against one step: 2^-15 a product)
    by = np.argsort([len(s) for s in seqs])
    for i in (by[0], by[rows // 2], by[-1]):
        _, one = m.step([rows], [lists[i]], True, want_logits=True)
        m.seq_free(rows)
        assert np.abs(one[0] - got[i]).max() < 5e-4 * np.abs(got[i]).max()
    m.close()


def test_more_rows_than_a_grid_axis_takes():
    """a decode step of more than 65535 sequences, against the same sequences in steps of 4097"""
    import nano_vllm_candle_amd as pkg

    rows, part = 65600, 4097
    cfg = pkg.Qwen3Config.tiny(vocab_size=256, num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=1, max_position_embeddings=256)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(rows, rows, 512)
    toks = np.random.default_rng(0).integers(0, cfg.vocab_size, (rows, 2)).astype(np.uint32)
    m.step(list(range(rows)), [t[:1] for t in toks], True)
    _, got = m.step(list(range(rows)), list(toks), False, want_logits=True)
    for a in range(0, rows, part):
        ids = list(range(a, min(rows, a + part)))
        m.step(ids, [t[:1] for t in toks[ids]], True)
        _, want = m.step(ids, list(toks[ids]), False, want_logits=True)
        # other kernels for the products, and q through memory: their rounding, two 16-bit planes a product (2^-15), one layer
        assert np.abs(got[ids] - want).max() < 5e-4 * np.abs(want).max(), a
    m.close()
