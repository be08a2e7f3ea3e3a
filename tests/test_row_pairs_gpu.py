"""GPU test of the products of 65 to 256 rows that take two row blocks at a time: row counts at the edges of a block and of a workgroup's share,
K of 1024, 2048 and 3072, both sides of the rule, against the same step on row-major planes (which the 16-wave kernels take)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


LAYERS = 2


def expected(heads, inter, hidden, rows):
    """launches of two row blocks at a time: of a decode step, of a prompt"""
    if rows <= 64 or hidden != 1024:  # 512: no register-direct form for K 512, and o and down have a workgroup for every block
        return 0, 0
    blocks, features = -(-rows // 16), (heads + 16) * 128
    qkv = blocks > 256 // (features // 64)
    gate_up = 2 * inter % 96 == 0 and blocks > 256 // (2 * inter // 96)
    whole = 128 < features // 128 * blocks <= 256  # a prompt's q/k/v with norm, rotation and cache writes in its epilogue
    return LAYERS * (qkv + 2 + gate_up), LAYERS * ((qkv and not whole) + 2 + gate_up)


@pytest.mark.parametrize("heads,inter,hidden", [(16, 3072, 1024), (8, 2048, 1024), (24, 3072, 1024), (8, 3072, 512)])
@pytest.mark.parametrize("rows", [64, 65, 80, 81, 117, 128, 129, 144, 145, 200, 240, 255, 256])
def test_rows(heads, inter, hidden, rows):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=4096, hidden_size=hidden, head_dim=128, num_hidden_layers=LAYERS, num_attention_heads=heads, num_key_value_heads=8, intermediate_size=inter)
    rng = np.random.default_rng(rows)
    seqs = [rng.integers(0, cfg.vocab_size, int(n)) for n in rng.integers(2, 5, rows)]
    out = []
    for row_major in (0, 1):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        m.set_option("no_xpack", row_major)
        m.kv_alloc(rows, rows, 1024)
        m.step(list(range(rows)), [s[:-1] for s in seqs], True)
        # decode: residual, norm and gate / up in the epilogues; then the prompt form, as one chunk of `rows` rows
        n = [m.counter("row_pair_launches")]
        _, step = m.step(list(range(rows)), seqs, False, want_logits=True)
        n.append(m.counter("row_pair_launches"))
        prompt = m.step_score([0], [np.concatenate(seqs)[:rows]], True, [[0, rows // 2, rows - 1]])
        n.append(m.counter("row_pair_launches"))
        assert (n[1] - n[0], n[2] - n[1]) == ((0, 0) if row_major else expected(heads, inter, hidden, rows))
        out.append(np.concatenate([step, prompt]))
        m.close()
    # f32 sums of the same products in another order, each result to two 16-bit planes (2^-16) and keys whose f16 may round the other way (2^-11)
    assert np.abs(out[0] - out[1]).max() < 2.0 ** -11 * np.abs(out[1]).max()


# a workgroup for every block up to 6 of 3840 features and 5 of 4608; three blocks in two rounds: 5 of 9216
@pytest.mark.parametrize("ff,rows,pairs", [(1920, 65, 0), (1920, 96, 0), (1920, 97, 1), (1920, 128, 1), (2304, 80, 0), (2304, 81, 1), (4608, 65, 0), (4608, 80, 0), (4608, 81, 1)])
def test_gate_up_of_a_layered_decoder(ff, rows, pairs):
    import nano_vllm_candle_amd as pkg
    from tests import tafopel_util as T

    cfg = T.config([T.mamba(inner=1024, state=16, conv=4, rank=32, mlp=T.dense(ff))] * LAYERS, width=1024, vocab=1024)
    m = pkg.TafopelForCausalLM.from_state_dict(pkg.TafopelConfig.from_dict(cfg), T.weights(cfg, 12, gain=1.5))
    m.kv_alloc(rows, rows, 1024)
    rng = np.random.default_rng(rows)
    seqs, ids = [rng.integers(0, 1024, int(n)) for n in rng.integers(3, 6, rows)], list(range(rows))
    want = m.step_score(ids, seqs, True, [[len(s) - 1] for s in seqs])
    m.step(ids, [s[:-1] for s in seqs], True)
    n = m.counter("row_pair_launches")
    _, got = m.step(ids, seqs, False, want_logits=True)
    assert m.counter("row_pair_launches") - n == LAYERS * pairs
    assert np.abs(got - want).max() < 4e-3 * np.abs(want).max()  # the tolerance of this decoder's parity tests
    m.close()
