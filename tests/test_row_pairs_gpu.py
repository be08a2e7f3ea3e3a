"""GPU test of the products of 65 to 256 rows that take two row blocks at a time: row counts at the edges of a block and of a workgroup's share,
K of 1024, 2048 and 3072, against the same step on row-major planes (which the 16-wave kernels take)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,inter,hidden", [(16, 3072, 1024), (8, 2048, 1024), (8, 3072, 512)])
@pytest.mark.parametrize("rows", [64, 65, 80, 81, 117, 128, 129, 144, 145, 200, 240, 255, 256])
def test_rows(heads, inter, hidden, rows):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=4096, hidden_size=hidden, head_dim=128, num_hidden_layers=2, num_attention_heads=heads, num_key_value_heads=8, intermediate_size=inter)
    rng = np.random.default_rng(rows)
    seqs = [rng.integers(0, cfg.vocab_size, int(n)) for n in rng.integers(2, 5, rows)]
    out = []
    for row_major in (0, 1):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        m.set_option("no_xpack", row_major)
        m.kv_alloc(rows, rows, 1024)
        m.step(list(range(rows)), [s[:-1] for s in seqs], True)
        # decode: residual, norm and gate / up in the epilogues; then the prompt form, as one chunk of `rows` rows
        _, step = m.step(list(range(rows)), seqs, False, want_logits=True)
        prompt = m.step_score([0], [np.concatenate(seqs)[:rows]], True, [[0, rows // 2, rows - 1]])
        out.append(np.concatenate([step, prompt]))
        m.close()
    # f32 sums of the same products in another order, each result to two 16-bit planes (2^-16) and keys whose f16 may round the other way (2^-11)
    assert np.abs(out[0] - out[1]).max() < 2.0 ** -11 * np.abs(out[1]).max()
