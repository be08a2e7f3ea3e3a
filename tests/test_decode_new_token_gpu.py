"""GPU test of the token that a fused decode step adds: it goes into its tile from the wave that made it, and into the cache for the steps
that follow.  Every place of a tile (both halves, each lane group and halfword), the edges of tiles, waves, blocks and of a context in parts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = list(range(1, 34)) + [63, 64, 95, 96, 127, 128, 129, 159, 160, 254, 255, 256, 257, 511, 512, 513, 640, 1023, 1024]


@pytest.mark.parametrize("hd,bits", [(64, 16), (128, 16), (128, 24)])
@pytest.mark.parametrize("rows", [1, 3, 0])  # 1 and 3 rows: contexts in parts from 513 tokens on
def test_steps_equal_the_prompt(hd, bits, rows):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=256, head_dim=hd, num_attention_heads=8, num_key_value_heads=4)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    n = len(LENGTHS)
    m.kv_alloc(2 * n + 12, n + 1, 2048)
    rng = np.random.default_rng(hd + bits)
    tokens = [rng.integers(0, cfg.vocab_size, k + 3) for k in LENGTHS]
    m.step(list(range(n)), [t[:-3] for t in tokens], True)
    # the prompt's kernels sum the same products in another order and from keys whose f16 may round the other way: 2^-11 of the largest logit.
    # With 24 bits the residual products keep an eighth of what 2^-12 leaves, in the prompt's kernel as in the decode one: 2^-14
    bound = 2.0 ** (-11 if bits == 16 else -14)
    worst = 0.0
    want = {}
    for i in range(n):
        for k in (1, 2, 3):
            _, lg = m.step([n], [tokens[i][:len(tokens[i]) - 3 + k]], True, want_logits=True)
            want[i, k] = lg[0]
            m.seq_free(n)
    groups = [list(range(n))] if not rows else [list(range(i, min(n, i + rows))) for i in range(0, n, rows)]
    for g in groups:
        for k in (1, 2, 3):
            _, got = m.step(g, [tokens[i][:len(tokens[i]) - 3 + k] for i in g], False, want_logits=True)
            for r, i in enumerate(g):
                worst = max(worst, np.abs(got[r] - want[i, k]).max() / np.abs(want[i, k]).max())
                assert worst < bound, (LENGTHS[i], k)
    print(f"[parity] {hd} {bits} {rows}: worst {worst:.3e}, bound {bound:.3e}")
    m.close()
