"""GPU test of the 32-bit products at the row counts where their kernels change (16, 32, 64 rows of the decode form, blocks of 64 rows of the
prompt form) and with ragged features, against the oracle in 64 bits."""
import numpy as np
import pytest

from oracle import gopunex_oracle as G
from tests.berevik_util import row_err
from tests.gopunex_util import CONFIGS, TOL, attn, config, light, sharp_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["mixed", "sizes", "wide"])
@pytest.mark.parametrize("rows", [16, 17, 32, 33, 64, 65, 127, 128, 129, 193])
def test_prompt_of_rows(name, rows):
    import nano_vllm_candle_amd as pkg

    cfg = CONFIGS[name]
    w = sharp_weights(cfg)
    c = pkg.GopunexConfig.from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    m = pkg.GopunexForCausalLM.from_state_dict(c, w, dtype="float32")
    m.kv_alloc(4, 2, max_batched_tokens=256)
    toks = np.random.default_rng(rows).integers(0, cfg["vocab"], rows).tolist()
    ask = [0, rows // 2, rows - 1]
    got, ref = m.step_score([0], [toks], True, [ask]), np.asarray(G.forward(cfg, w, toks))[ask]
    # what the layer tests allow this decoder's 32-bit mode: a few hundred f32 sums through a handful of layers
    assert row_err(got, ref) < TOL["float32"]
    m.close()


@pytest.mark.parametrize("rows", [64, 65, 130])
def test_infinite_weights(rows):
    """a product with an infinite weight is infinite on both sides of the row count where the kernel changes, and nothing else is touched"""
    import nano_vllm_candle_amd as pkg

    cfg = CONFIGS["mixed"]
    w = sharp_weights(cfg)
    c = pkg.GopunexConfig.from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    toks = np.random.default_rng(1).integers(0, cfg["vocab"], rows).tolist()

    def logits(weights):
        m = pkg.GopunexForCausalLM.from_state_dict(c, weights, dtype="float32")
        m.kv_alloc(140, 130, max_batched_tokens=256)
        out = m.step_score([0], [toks], True, [list(range(rows))])
        m.close()
        return out

    want = logits(w)
    head = np.array(w["head"], np.float32)
    head[5, 7], head[300, 70] = np.inf, -np.inf
    got = logits({**w, "head": head})
    assert np.isinf(got[:, [5, 300]]).all()
    keep = [i for i in range(cfg["vocab"]) if i not in (5, 300)]
    assert np.array_equal(got[:, keep], want[:, keep])


# K in parts of unlike length (1056, 2080, 4608 in 2, 4, 4), a head of K 128, by the kernel for short K, and of 1024, walked by workgroups with the rows
# held (512 workgroups a few tiles each) up to 16 rows; all with ragged rows
@pytest.mark.parametrize("width,ffs,vocab", [(72, (1056, 2080), 16400), (1000, (4608, 1024), 16390)])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 64])
def test_deep_products_and_many_features(width, ffs, vocab, rows):
    import nano_vllm_candle_amd as pkg

    cfg = config([light(ff=ffs[0]), attn(ff=ffs[1])], width=width, vocab=vocab)
    w = sharp_weights(cfg)
    c = pkg.GopunexConfig.from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    m = pkg.GopunexForCausalLM.from_state_dict(c, w, dtype="float32")
    m.kv_alloc(4, 66, max_batched_tokens=256)
    toks = np.random.default_rng(rows).integers(0, vocab, rows).tolist()
    got, ref = m.step_score([0], [toks], True, [list(range(rows))]), np.asarray(G.forward(cfg, w, toks))  # every row through the head: 1 to 64
    assert row_err(got, ref) < TOL["float32"]
    ids, logits = m.step([0], [toks], True, want_logits=True)
    assert ids[0] == np.flatnonzero(logits[0] == logits[0].max())[-1]
    m.close()


# a head walked by workgroups with the rows held (up to 16 rows): 8, 12, 28 and 32 k-tiles over eight waves that hold four each, so all but the last leave
# places empty, 12 and 28 not in every wave alike; a last tile of 7 features
@pytest.mark.parametrize("width", [250, 384, 890, 1024])
@pytest.mark.parametrize("rows", [1, 15, 16, 17])
def test_head_of_many_features(width, rows):
    import nano_vllm_candle_amd as pkg

    cfg = config([light(ff=64)], width=width, vocab=16391)
    w = sharp_weights(cfg)
    c = pkg.GopunexConfig.from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    m = pkg.GopunexForCausalLM.from_state_dict(c, w, dtype="float32")
    m.kv_alloc(4, 66, max_batched_tokens=256)
    toks = np.random.default_rng(rows).integers(0, 16391, rows).tolist()
    got, ref = m.step_score([0], [toks], True, [list(range(rows))]), np.asarray(G.forward(cfg, w, toks))
    assert row_err(got, ref) < TOL["float32"]
    m.close()


# the same for prompts, whose products are cut over workgroups of 64 rows: K of 1056, 2080 and 4608 in two and four parts, one of them short
@pytest.mark.parametrize("width,ffs", [(72, (1056, 2080)), (1000, (4608, 1024))])
@pytest.mark.parametrize("rows", [65, 128, 193])
def test_deep_products_of_prompts(width, ffs, rows):
    import nano_vllm_candle_amd as pkg

    cfg = config([light(ff=ffs[0]), attn(ff=ffs[1])], width=width)
    w = sharp_weights(cfg)
    c = pkg.GopunexConfig.from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    m = pkg.GopunexForCausalLM.from_state_dict(c, w, dtype="float32")
    m.kv_alloc(4, 2, max_batched_tokens=256)
    toks = np.random.default_rng(rows).integers(0, cfg["vocab"], rows).tolist()
    ask = [0, rows // 2, rows - 1]
    got, ref = m.step_score([0], [toks], True, [ask]), np.asarray(G.forward(cfg, w, toks))[ask]
    assert row_err(got, ref) < TOL["float32"]
    m.close()


# input projections in parts: every row kernel behind them reads two slabs of a prompt's rows
@pytest.mark.parametrize("name", ["gopunex", "lefalix"])
@pytest.mark.parametrize("rows", [65, 130])
def test_split_input_projections_of_prompts(name, rows):
    import nano_vllm_candle_amd as pkg
    from oracle import lefalix_oracle as LO
    from tests import gopunex_util as GU, lefalix_util as LU

    if name == "gopunex":
        cfg = config([light(ff=0), attn(ff=0), GU.delta(ff=0)], width=1024)
        w, tol, make, conf = sharp_weights(cfg), TOL["float32"], pkg.GopunexForCausalLM, pkg.GopunexConfig
    else:
        cfg = LU.config([LU.par(mlp=LU.dense(1024)), LU.delta(LU.dense(1100))], width=1024)
        w, tol, make, conf = LU.weights(cfg), LU.TOL["float32"], pkg.LefalixForCausalLM, pkg.LefalixConfig
    m = make.from_state_dict(conf.from_dict(cfg, {k: np.shape(v) for k, v in w.items()}), {k: np.asarray(v, np.float32) for k, v in w.items()}, dtype="float32")
    m.kv_alloc(4, 2, max_batched_tokens=256)
    toks = np.random.default_rng(rows).integers(0, cfg["vocab"], rows).tolist()
    ask = [0, 1, rows // 2, rows - 2, rows - 1]
    ref = np.asarray(G.forward(cfg, w, toks) if name == "gopunex" else LO.run(cfg, w, toks)[0])
    assert row_err(m.step_score([0], [toks], True, [ask]), ref[ask]) < tol
    assert row_err(m.step([0], [toks + [3]], False, want_logits=True)[1], (G.forward(cfg, w, toks + [3]) if name == "gopunex" else LO.run(cfg, w, toks + [3])[0])[-1:]) < tol
    m.close()
