"""GPU test of few decode rows: the planes between the kernels are row-major below four rows and in fragment order from there on,
padded to sixteen rows whose memory holds whatever was there.  A row must not depend on its neighbours nor on the padding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,heads,kv", [(1024, 3072, 16, 8), (1024, 1024, 8, 8), (2048, 2048, 16, 4)])
def test_rows_alone_and_together(hidden, inter, heads, kv):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(33, 33, 512)
    rng = np.random.default_rng(hidden + inter)
    seqs = [rng.integers(0, cfg.vocab_size, int(n)) for n in rng.integers(1, 60, 33)]
    m.step(list(range(33)), seqs, True)  # many rows have left their values in the padding
    lists = [np.append(s, 5) for s in seqs]
    alone = [m.step([i], [lists[i]], False, want_logits=True)[1][0] for i in range(33)]
    for rows in (2, 3, 4, 5, 15, 16, 17, 31, 32, 33):  # one, two and three row blocks have shapes of their own
        _, got = m.step(list(range(rows)), lists[:rows], False, want_logits=True)
        for i in range(rows):
            # the same products in another order; an f16 key or value may round the other way: 2^-11 of the largest logit
            assert np.abs(got[i] - alone[i]).max() < 2.0 ** -11 * np.abs(alone[i]).max(), (rows, i)
    m.close()
