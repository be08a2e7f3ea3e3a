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
