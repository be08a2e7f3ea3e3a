"""GPU test of the decode products that share a launch (output projection and down_proj of a layer, output projections of two mixers): row counts at
the edges of 16 and of the rule (64), K of 1024, 2048 and 3072 in both places, against the same positions of a prompt, whose products are separate."""
import numpy as np
import pytest

from tests import lefalix_util as L
from tests import tafopel_util as T

pytestmark = pytest.mark.gpu


def _tafopel():
    cfg = T.config([T.mamba(inner=1024, mlp=T.dense(3072)), T.attn(heads=16, dim=32, vdim=128, rank=64, mlp=T.dense(1024)), T.mamba(inner=2048, mlp=T.dense(2048)),
                    T.attn(heads=24, dim=32, vdim=128, rank=64, mlp=T.dense(2048))], width=256)
    return "Tafopel", cfg, T.weights(cfg), ()


def _lefalix():
    cfg = L.config([L.par(L.win(heads=8, kv=2, dim=64, vdim=128), L.rule(heads=16, kv=4, dim=32, vdim=128), L.dense(256)),
                    L.par(L.win(heads=24, kv=2, dim=64, vdim=128), L.rule(heads=8, kv=4, dim=32, vdim=128))], width=256)
    w = L.weights(cfg)
    return "Lefalix", cfg, w, ({k: np.shape(v) for k, v in w.items()},)


@pytest.mark.parametrize("make,pairs,products", [(_tafopel, 4, 23), (_lefalix, 2, 9)])
def test_steps_equal_the_prompt(make, pairs, products):
    import nano_vllm_candle_amd as pkg

    design, cfg, w, shapes = make()
    c = getattr(pkg, design + "Config").from_dict(cfg, *shapes)
    m = getattr(pkg, design + "ForCausalLM").from_state_dict(c, w)
    m.kv_alloc(70, 66, 8192)
    rng = np.random.default_rng(1)
    seqs = [rng.integers(0, cfg["vocab"], 66 + i % 5) for i in range(65)]
    for rows in (3, 4, 16, 17, 33, 64, 65):
        ids = list(range(rows))
        want = m.step_score(ids, seqs[:rows], True, [[len(s) - 1] for s in seqs[:rows]])
        m.step(ids, [s[:-1] for s in seqs[:rows]], True)
        before = m.counter("two_product_launches")
        m.profile_kernel("gemm")
        _, got = m.step(ids, seqs[:rows], False, want_logits=True)
        launches = m.profile_read()[1]
        m.profile_kernel(None)
        shared = m.counter("two_product_launches") - before
        assert shared == (pairs if rows <= 64 else 0), rows
        assert launches == products - shared, rows  # an event pair to every launch made, none to one that was not
        assert np.abs(got - want).max() < 4e-3 * np.abs(want).max(), rows  # the tolerance of these decoders' parity tests
    m.close()
