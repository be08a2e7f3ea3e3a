"""GPU test of the decode attention's two workgroup sizes (eight waves where a launch is one workgroup per CU at most, four above) and of its
shared prologue: heads of a group that fit the rounds loaded up front and that do not, contexts on both sides of a wave's, a part's and the
unsplit form's ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1, 31, 33, 126, 127, 128, 159, 255, 256, 257, 510, 511, 512, 1021, 1022, 1023, 1024]


def check(hd, kv, heads, lens, bits, eight, ahead=0):
    import nano_vllm_candle_amd as pkg

    rows = len(lens)
    cfg = pkg.Qwen3Config.tiny(hidden_size=256, head_dim=hd, num_attention_heads=heads, num_key_value_heads=kv)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.kv_alloc(sum(n // 256 + 1 for n in lens) + 8, rows + 1, 2048)
    rng = np.random.default_rng(rows + heads)
    seqs = [rng.integers(0, cfg.vocab_size, n + 1) for n in lens]
    m.step(list(range(rows)), [s[:-1] for s in seqs], True, want_logits=False)
    _, got = m.step(list(range(rows)), seqs, False, want_logits=True)
    assert m.counter("eight_wave_launches") == eight * cfg.num_hidden_layers
    assert m.counter("tiles_ahead_launches") == ahead * cfg.num_hidden_layers
    # the prompt's kernels sum in another order, from keys whose f16 may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    bound = 2.0 ** (-11 if bits == 16 else -14)
    for i in range(min(rows, 34)):
        _, want = m.step([rows], [seqs[i]], True, want_logits=True)
        m.seq_free(rows)
        assert np.abs(got[i] - want[0]).max() < bound * np.abs(want).max(), (i, lens[i])
    m.close()


# workgroups: 256 and 264 of 8 kv heads; 128 and 124 of 4 (whole and in parts from 513 tokens on); 2 and 257 of one, whose 18 heads take
# more rounds of four waves than are loaded up front; 8 heads of 64; 3 to 14 query heads a group, whose rows lie beside each other in LDS
@pytest.mark.parametrize("hd,kv,heads,rows,bits,eight", [(128, 8, 16, 32, 16, 1), (128, 8, 16, 33, 16, 0), (128, 4, 8, 32, 16, 1), (128, 4, 8, 31, 24, 1), (128, 1, 16, 2, 16, 1),
                                                         (128, 1, 16, 257, 16, 0), (128, 1, 8, 17, 24, 1), (64, 1, 8, 17, 16, 0), (64, 1, 16, 3, 16, 0),
                                                         (128, 2, 6, 3, 16, 0), (128, 8, 40, 33, 16, 0), (128, 1, 7, 5, 24, 0), (128, 2, 28, 129, 24, 0), (64, 2, 10, 9, 16, 0)])
def test_a_step_equals_the_prompt(hd, kv, heads, rows, bits, eight):
    check(hd, kv, heads, [LENGTHS[(i * 7) % len(LENGTHS)] for i in range(rows)], bits, eight)


# both sides of each line of the rule: whole contexts by workgroups, cache and query heads, parts of a tile a wave, ragged contexts whose parts leave CUs idle
@pytest.mark.parametrize("kv,heads,lens,bits,eight", [
    (8, 16, [256], 16, 0), (8, 16, [300] * 20, 16, 0), (8, 16, [511], 16, 0), (8, 32, [300] * 10, 16, 0), (1, 14, [300], 16, 0),
    (1, 15, [127], 16, 0), (1, 15, [128], 16, 1), (1, 16, [300] * 128, 16, 1), (1, 16, [300] * 129, 16, 0),
    (8, 16, [127], 24, 0), (8, 16, [128], 24, 1), (8, 16, [255] * 32, 24, 1), (8, 16, [256] * 32, 24, 0), (8, 16, [300] * 20, 24, 1), (8, 16, [300] * 21, 24, 0),
    (8, 16, [512], 16, 0), (8, 16, [1279], 16, 0), (8, 16, [1280], 16, 1), (8, 16, [1279], 24, 0), (8, 16, [1280], 24, 1),
    (8, 16, [895] * 3, 16, 0), (8, 16, [896] * 3, 16, 1), (8, 16, [671] * 6, 16, 0), (8, 16, [672] * 6, 16, 1), (8, 16, [512] * 8, 16, 1),
    (8, 16, [256, 1024] * 12, 16, 1), (8, 16, [256, 1023] * 12, 24, 1), (8, 16, [256, 1024] * 12, 24, 0), (8, 16, [512, 1024] * 12, 24, 1), (8, 16, [1024] * 24, 24, 1),
    (8, 16, [256, 1024] * 14, 24, 1), (8, 16, [256, 1535] * 6, 24, 1), (8, 16, [256, 1536] * 6, 24, 0)])
def test_the_rule(kv, heads, lens, bits, eight):
    check(128, kv, heads, lens, bits, eight)


# a wave's second tile asked for with its first: from 512 workgroups and more than 512 tokens a row on average, four waves, 16 bits, heads of 128
@pytest.mark.parametrize("hd,kv,heads,lens,bits,ahead", [
    (128, 8, 16, [512] * 64, 16, 1), (128, 8, 16, [511] * 64, 16, 0), (128, 8, 16, [512] * 63, 16, 0), (128, 8, 16, [1, 1100] * 32, 16, 1), (128, 8, 16, [1, 1020] * 32, 16, 0),
    (128, 16, 80, [530] * 33, 16, 1), (128, 32, 64, [640, 700] * 8, 16, 1), (128, 8, 16, [520] * 64, 24, 0), (64, 8, 16, [520] * 64, 16, 0)])
def test_two_tiles_ahead(hd, kv, heads, lens, bits, ahead):
    check(hd, kv, heads, lens, bits, 0, ahead)
