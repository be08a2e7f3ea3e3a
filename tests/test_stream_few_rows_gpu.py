"""GPU test of the streaming products of one to 16 rows: Qwen3 layers whose four products stream, and where two do beside others, with planes of one row and of a whole row block, against the oracle, and a layer of another design,
whose gated feed-forward streams, against the same rows in a batch of 17."""
import numpy as np
import pytest

from tests.util import LOGITS_TOL, oracle_config, row_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,heads,kv,streams", [(4096, 12288, 32, 8, 4), (5120, 6528, 40, 8, 2)])
def test_qwen_layers_against_the_oracle(oracle, hidden, inter, heads, kv, streams):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=1024, hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128, num_hidden_layers=1)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 0)
    m.kv_alloc(20, 16, 256)
    om = oracle.Model(oracle_config(oracle, cfg)).fill_synthetic(0)
    rng = np.random.default_rng(hidden)
    seqs = [rng.integers(0, cfg.vocab_size, 2 + i % 3).tolist() for i in range(16)]
    for i, s in enumerate(seqs):  # (prompts of one to three rows)
        m.step([i], [s[:-1]], True)
    _, want = om.run_greedy(seqs)
    for rows in (1, 3, 4, 15, 16):
        n = m.counter("stream_launches")
        _, got = m.step(list(range(rows)), seqs[:rows], False, want_logits=True)
        assert m.counter("stream_launches") - n == streams
        assert row_rel_err(got, want[:rows]) < LOGITS_TOL, rows
    m.close()


def test_a_gated_feed_forward(oracle):
    import nano_vllm_candle_amd as pkg
    from bench_berevik import SIZES, berevik_config

    z = dict(SIZES["4k"], layers=1)
    m = pkg.BerevikForCausalLM.from_random(berevik_config(pkg, z, 1024, 1 << 20))
    m.kv_alloc(20, 17, 256)
    rng = np.random.default_rng(1)
    seqs = [rng.integers(0, 1024, 3).astype(np.uint32) for _ in range(17)]
    m.step(list(range(17)), [s[:2] for s in seqs], True)
    want = m.step_score(list(range(17)), seqs, False, [[2]] * 17)
    for rows in (1, 3, 4, 16):
        n = m.counter("stream_launches")
        got = m.step_score(list(range(rows)), seqs[:rows], False, [[2]] * rows)
        assert m.counter("stream_launches") - n == 4
        # the same products of the same planes, summed in another order; a cached key or value may round the other way (2^-11 of itself)
        assert np.abs(got - want[:rows]).max() < 2.0 ** -11 * np.abs(want).max(), rows
    m.close()


@pytest.mark.parametrize("tp,launches", [(1, 1), (2, 0)])
def test_a_shard_keeps_its_own_rule(tp, launches):
    # gate/up of 80 MB with no row form: slabs and an activation launch on one GPU, of a shard of two (communication left out) one product with the activation in its epilogue, up to 16 rows
    import nano_vllm_candle_amd as pkg
    from bench_berevik import SIZES, berevik_config

    z = dict(SIZES["4k"], width=5120, ff=4096 * tp, layers=1)
    ctx = pkg.Context(0, tp_rank=0, tp_size=tp, null_comm=True)
    m = pkg.BerevikForCausalLM.from_random(berevik_config(pkg, z, 1024, 1 << 20), ctx=ctx)
    m.kv_alloc(20, 17, 256)
    seqs = [[1 + i, 2, 3] for i in range(17)]
    m.step(list(range(17)), [s[:2] for s in seqs], True)
    for rows in (1, 8, 16, 17):
        m.profile_kernel("silu")
        m.step(list(range(rows)), seqs[:rows], False)
        assert m.profile_read()[1] == (launches if rows <= 16 else 1), rows
        m.profile_kernel(None)
    m.close()
    ctx.close()
