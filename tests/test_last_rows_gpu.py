"""GPU test of the last layer of a prompt, which goes on past its mixer with the rows whose logits are wanted alone: the same positions' logits
as when every position is wanted (then all rows go on), chunks that hold no wanted row, and the step that follows."""
import numpy as np
import pytest

from tests import berevik_util, gopunex_util, lefalix_util, tafopel_util

pytestmark = pytest.mark.gpu

# (lengths, rows of a chunk): just above and below where the rule begins (129 rows, half of them wanted), ragged ones, chunks that end inside
# sequences and one of them without a wanted row
SHAPES = [([129], 2048), ([1, 128], 2048), ([3] * 100, 2048), ([2] * 66, 2048), ([300, 17, 45, 1, 133], 2048), ([700, 33], 256), ([257, 600], 512)]


@pytest.mark.parametrize("rows", [130, 255, 300])
def test_many_wanted_rows(rows):
    """wanted rows enough for the prompt product, with a split of K of their own beside the chunk's"""
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=1024, hidden_size=512, head_dim=128, num_attention_heads=8, num_key_value_heads=8, intermediate_size=3072)
    check(pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3), [2 + i % 3 for i in range(rows)], 2048, 2.0 ** -11)


def check(m, lens, chunk, bound):
    """wanted: the last position, the last and a middle one, or none, by sequence; against all positions"""
    n = len(lens)
    m.kv_alloc(sum(k // 256 + 2 for k in lens), max(n + 1, min(sum(lens), chunk)), chunk)
    rng = np.random.default_rng(sum(lens))
    seqs = [rng.integers(0, m.vocab_size, k + 1).astype(np.uint32) for k in lens]
    ids = list(range(n))
    prompts = [s[:-1] for s in seqs]
    whole = m.step_score(ids, prompts, True, [list(range(k)) for k in lens])
    _, after = m.step(ids, seqs, False, want_logits=True)
    first = np.cumsum([0] + lens)
    for wanted in ([[k - 1] for k in lens], [sorted({k // 2, k - 1}) for k in lens], [[k - 1] if i % 2 else [] for i, k in enumerate(lens)]):
        if not any(wanted):
            continue
        got = m.step_score(ids, prompts, True, wanted)
        want = whole[[first[i] + p for i, w in enumerate(wanted) for p in w]]
        assert np.abs(got - want).max() < bound * np.abs(want).max(), (lens, wanted)
        _, then = m.step(ids, seqs, False, want_logits=True)
        assert np.abs(then - after).max() < bound * np.abs(after).max(), lens
    m.close()


@pytest.mark.parametrize("lens,chunk", SHAPES)
@pytest.mark.parametrize("width,bits", [(256, 16), (256, 24), (1024, 16)])
def test_qwen3(width, bits, lens, chunk):
    import nano_vllm_candle_amd as pkg

    cfg = (pkg.Qwen3Config.tiny(hidden_size=256, head_dim=128, num_attention_heads=4, num_key_value_heads=2) if width == 256 else
           pkg.Qwen3Config.tiny(vocab_size=8192, hidden_size=1024, head_dim=128, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=8, intermediate_size=3072))
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    # other kernels for the last layer, and chunks cut elsewhere: sums in another order, keys whose f16 may round the other way, 2^-11 of the
    # largest logit (2^-14 with the residuals)
    check(m, lens, chunk, 2.0 ** (-11 if bits == 16 else -14))


_T = tafopel_util
LAYERED = {
    "gopunex attention": ("Gopunex", gopunex_util.EVEN, gopunex_util.sharp_weights),
    "gopunex no feed-forward": ("Gopunex", gopunex_util.MIXED, gopunex_util.sharp_weights),
    "gopunex delta rule": ("Gopunex", gopunex_util.STATE, gopunex_util.sharp_weights),
    "tafopel attention": ("Tafopel", _T.config([_T.mamba(mlp=_T.dense()), _T.attn(mlp=_T.dense(200))]), _T.weights),
    "tafopel scan": ("Tafopel", _T.config([_T.attn(mlp=_T.dense()), _T.mamba(mlp=_T.dense(140))]), _T.weights),
    "tafopel experts": ("Tafopel", _T.config([_T.mamba(), _T.attn(mlp=_T.moe())]), _T.weights),
    "lefalix": ("Lefalix", lefalix_util.MIXED, lefalix_util.weights),
    "lefalix even": ("Lefalix", lefalix_util.EVEN, lefalix_util.weights),
    "berevik": ("Berevik", berevik_util.MIXED, berevik_util.sharp_weights),
}


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("name", sorted(LAYERED))
def test_layered(name, dtype):
    import nano_vllm_candle_amd as pkg

    design, cfg, weights = LAYERED[name]
    w = weights(cfg)
    shapes = ({k: np.shape(v) for k, v in w.items()},) if design in ("Gopunex", "Lefalix") else ()
    c = getattr(pkg, design + "Config").from_dict(cfg, *shapes)
    for lens, chunk in (([129], 512), ([64, 65], 512), ([300, 17, 45, 1, 133], 256)):
        m = getattr(pkg, design + "ForCausalLM").from_state_dict(c, w, dtype=dtype)
        check(m, lens, chunk, {"bfloat16": 4e-3, "float32": 3e-5}[dtype])  # the tolerances of these decoders' parity tests


def forced(make, lens, chunk, bound):
    """the prompt product on every projection that fits it, of the last layer's gathered rows too"""
    m = make()
    m.set_option("tile_min_wgs", 1)
    m.set_option("last_rows", 1)
    check(m, lens, chunk, bound)
    # launches of one prompt by the option: 0 keeps all rows, 1 the wanted ones, -1 all while the product is forced
    counts = {}
    for option in (0, 1, -1):
        m = make()
        m.set_option("tile_min_wgs", 1)
        m.set_option("last_rows", option)
        m.kv_alloc(sum(n // 256 + 1 for n in lens), len(lens), sum(lens))
        rng = np.random.default_rng(1)
        m.step(list(range(len(lens))), [rng.integers(0, m.vocab_size, n) for n in lens], True)
        counts[option] = m.counter("tile_gemm_launches")
        m.close()
    return counts


# wanted: one row, and 140 rows, which the prompt product takes as well
@pytest.mark.parametrize("lens,rest", [([700, 33], 1), ([3] * 140, 4)])
@pytest.mark.parametrize("fuse", [0, 1])
def test_forced_products(lens, rest, fuse):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=8192, hidden_size=1024, head_dim=128, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=8, intermediate_size=3072)

    def make():
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        m.set_option("tile_fuse_qk", fuse)
        return m

    assert forced(make, lens, 4096, 2.0 ** -11) == {0: 8, 1: 4 + rest, -1: 8}


_B, _G, _L = berevik_util, gopunex_util, lefalix_util
WIDE = {
    "berevik": ("Berevik", _B.config([_B.layer(heads=16, dim=64, rot=64, vdim=128, rank=256, ff=3072)] * 2, width=1024, vocab=1024), lambda c: _B.sharp_weights(c, 12, gain=1.5)),
    "gopunex": ("Gopunex", _G.config([_G.light(heads=8, dim=128, vdim=128, ff=3072), _G.attn(heads=8, kv=4, dim=128, vdim=128, ff=3072, far=120)], width=1024, vocab=1024), lambda c: _G.sharp_weights(c, 12, gain=1.5)),
    "gopunex delta rule": ("Gopunex", _G.config([_G.attn(heads=8, kv=4, dim=128, vdim=128, ff=3072, far=120), _G.delta(heads=8, kv=8, dim=128, vdim=128, ff=3072)], width=1024, vocab=1024), lambda c: _G.sharp_weights(c, 12, gain=1.5)),
    "tafopel": ("Tafopel", _T.config([_T.attn(heads=8, dim=128, rot=64, vdim=128, rank=512, q_rank=768, mlp=_T.dense(3072)), _T.mamba(inner=2048, state=16, conv=4, rank=64, mlp=_T.dense(3072))], width=1024, vocab=1024), lambda c: _T.weights(c, 12, gain=1.5)),
    "lefalix": ("Lefalix", _L.config([_L.delta(_L.dense(3072), heads=8, kv=8, dim=128, vdim=128), _L.par(_L.win(heads=8, kv=4, dim=128, vdim=128, window=100, rot=64, scale=0.2), _L.rule(heads=8, kv=4, dim=128, vdim=128), _L.dense(3072))], width=1024, vocab=1024), lambda c: _L.weights(c, 12)),
}


@pytest.mark.parametrize("lens", [[700, 33], [3] * 140])
@pytest.mark.parametrize("name", sorted(WIDE))
def test_forced_products_of_layered_decoders(name, lens):
    import nano_vllm_candle_amd as pkg

    design, cfg, weights = WIDE[name]
    w = weights(cfg)
    shapes = ({k: np.shape(v) for k, v in w.items()},) if design in ("Gopunex", "Lefalix") else ()
    c = getattr(pkg, design + "Config").from_dict(cfg, *shapes)
    counts = forced(lambda: getattr(pkg, design + "ForCausalLM").from_state_dict(c, w), lens, 4096, 4e-3)
    assert counts[0] == counts[-1] >= counts[1] > 0
    assert (counts[1] < counts[0]) == (len(lens) <= 128)  # more rows than that take the product as well
