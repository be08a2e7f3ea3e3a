"""GPU test of the streaming products of 17 to 64 decode rows (matrices of 24 MB and more): both row counts of a tile (up to 32, up to 64)
at their edges, layers whose column tiles leave a remainder for every number of waves, and the combine inside the launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,heads,kv", [(4096, 12288, 32, 8), (2560, 9856, 32, 2), (5120, 6528, 24, 4)])
@pytest.mark.parametrize("combine", [0, 1])
def test_rows_of_a_batch_equal_the_rows_alone(hidden, inter, heads, kv, combine):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128, num_hidden_layers=2)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(66, 65, 512)
    rng = np.random.default_rng(hidden)
    seqs = [rng.integers(0, cfg.vocab_size, int(n)) for n in rng.integers(1, 7, 64)]
    m.step(list(range(64)), seqs, True)
    lists = [np.append(s, 5) for s in seqs]
    # one row: the kernels of up to 16 rows, the same planes and weights summed in another order; an f16 key or value may round the other
    # way (2^-11 of itself, as often up as down), which moves a logit by less than 2^-11 of the largest
    alone = {i: m.step([i], [lists[i]], False, want_logits=True)[1][0] for i in (0, 15, 16, 30, 31, 32, 47, 48, 63)}
    m.set_option("stream_combine", combine)
    for rows in (17, 31, 32, 33, 48, 49, 64):
        _, got = m.step(list(range(rows)), lists[:rows], False, want_logits=True)
        for i, want in alone.items():
            if i < rows:
                assert np.abs(got[i] - want).max() < 2.0 ** -11 * np.abs(want).max(), (rows, i)
        assert np.isfinite(got).all()
    m.close()


@pytest.mark.parametrize("rows", [17, 33, 40, 48])
def test_planes_that_end_with_the_batch(rows):
    """a pool of as many rows as the batch has: row blocks past the planes are not read, and nothing else is"""
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=4096, intermediate_size=12288, num_attention_heads=32, num_key_value_heads=8, head_dim=128, num_hidden_layers=1)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    seqs = [np.random.default_rng(i).integers(0, cfg.vocab_size, 1 + i % 3) for i in range(rows)]
    out = []
    for most in (rows, 256):
        m.kv_alloc(rows, rows, most)
        for i, s in enumerate(seqs):  # one by one: the same cache in both pools
            m.step([i], [s], True)
        out.append(m.step(list(range(rows)), [np.append(s, 5) for s in seqs], False, want_logits=True)[1])
    m.close()
    assert np.array_equal(out[0], out[1])
