"""GPU test of the q/k norm, rotation and cache writes of prompts by 16 rows and head: row counts at the edges of 16 rows and of the rule, sequences
that begin anywhere in them, both cache forms, deferred norms of one and of many groups, against the same in a product's epilogue and by a wave
per row and head."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS = 2


def model(bits, blocks, seqs, rows=4096, fuse=1):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=2048, hidden_size=1024, head_dim=128, num_hidden_layers=LAYERS, num_attention_heads=16, num_key_value_heads=8, intermediate_size=3072)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.set_option("tile_fuse_qk", fuse)
    m.kv_alloc(blocks, seqs, rows)
    return m


def tokens(lens):
    rng = np.random.default_rng(sum(lens))
    return [rng.integers(0, 2048, n + 1).astype(np.uint32) for n in lens]


def bound(bits, a):
    """f32 sums in another order, keys and values whose f16 may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals"""
    return 2.0 ** (-11 if bits == 16 else -14) * np.abs(a).max()


@pytest.mark.parametrize("bits", [16, 24])
@pytest.mark.parametrize("lens,form", [([1], 0), ([2], 0), ([15], 0), ([17], 0), ([64], 0), ([129], 0), ([144], 0), ([145], 1), ([90, 55], 1), ([255], 1), ([33, 1, 2, 300], 1), ([255, 257], 1), ([1040, 5], 1), ([2040], 1)])
def test_prompt_equals_its_portions(lens, form, bits):
    """the prompts in one chunk, and in portions of up to 100 rows, which never take 16 rows and a head (65 rows and more: the product's epilogue)"""
    seqs, ids = tokens(lens), list(range(len(lens)))
    m = model(bits, sum(n // 256 + 2 for n in lens), len(lens))
    _, prompt = m.step(ids, [s[:-1] for s in seqs], True, want_logits=True)
    assert m.counter("qk_rows16_launches") == form * LAYERS
    _, after = m.step(ids, seqs, False, want_logits=True)
    m.close()
    m = model(bits, sum(n // 256 + 2 for n in lens), len(lens))
    want = []
    for i, n in zip(ids, lens):
        for k in list(range(100, n, 100)) + [n]:
            _, lg = m.step([i], [seqs[i][:k]], k <= 100, want_logits=True)
        want.append(lg)
    assert m.counter("qk_rows16_launches") == 0
    want = np.concatenate(want)
    assert np.abs(prompt - want).max() < bound(bits, want)
    _, then = m.step(ids, seqs, False, want_logits=True)
    assert np.abs(after - then).max() < bound(bits, then)
    m.close()


@pytest.mark.parametrize("bits", [16, 24])
@pytest.mark.parametrize("lens,form", [([66], 0), ([90, 27], 0), ([128], 0), ([2500], 1), ([4000, 33], 1)])
def test_prompt_equals_the_epilogue(lens, form, bits):
    """row counts where the option chooses between the product's epilogue and the row kernels"""
    seqs, ids, out = tokens(lens), list(range(len(lens))), []
    for fuse in (0, 1):
        m = model(bits, sum(n // 256 + 2 for n in lens), len(lens), fuse=fuse)
        m.profile_kernel("qk")
        _, prompt = m.step(ids, [s[:-1] for s in seqs], True, want_logits=True)
        assert m.profile_read()[1] == (0 if fuse else LAYERS)  # launches of the row kernels
        m.profile_kernel(None)
        assert m.counter("qk_rows16_launches") == (0 if fuse else form * LAYERS)
        _, after = m.step(ids, seqs, False, want_logits=True)
        out.append(np.concatenate([prompt, after]))
        m.close()
    assert np.abs(out[0] - out[1]).max() < bound(bits, out[1])
