"""GPU test of the plain attention's form with a wave to each row: 32 heads, row counts around 256, where it takes over, and none a multiple of
four above it, every width of a value, distance biases, windows inside and across 64 tokens, 32-bit and 16-bit caches, against the oracles."""
import numpy as np
import pytest

from oracle import gopunex_oracle as G
from oracle import lefalix_oracle as L
from tests import gopunex_util as GU
from tests import lefalix_util as LU
from tests.berevik_util import row_err

pytestmark = pytest.mark.gpu


def run(design, cfg, w, oracle, tol, dtype):
    import nano_vllm_candle_amd as pkg

    c = getattr(pkg, design + "Config").from_dict(cfg, {k: np.shape(v) for k, v in w.items()})
    m = getattr(pkg, design + "ForCausalLM").from_state_dict(c, {k: np.asarray(v, np.float32) for k, v in w.items()}, dtype=dtype)
    m.kv_alloc(8, 2, max_batched_tokens=512)
    m.set_option("bias_attn_plain", 1)
    for rows in (255, 256, 257, 262, 331):
        toks = np.random.default_rng(rows).integers(0, cfg["vocab"], rows).tolist()
        ask = sorted({0, 1, 62, 63, 64, 65, 254, rows - 4, rows - 3, rows - 2, rows - 1})
        assert row_err(m.step_score([0], [toks], True, [ask]), np.asarray(oracle(cfg, w, toks))[ask]) < tol, rows
        m.seq_free(0)
    m.close()


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("dim, vdim", [(17, 16), (40, 100), (96, 250), (300, 280)])
def test_values_of_every_width(dim, vdim, dtype):
    cfg = GU.config([GU.attn(heads=32, kv=4, dim=dim, vdim=vdim, ff=0, far=70)], width=64, vocab=200)
    run("Gopunex", cfg, GU.sharp_weights(cfg), lambda c, w, t: G.forward(c, w, t), GU.TOL[dtype], dtype)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("window", [1, 63, 64, 65, 200])
def test_windows(window, dtype):
    cfg = LU.config([LU.par(LU.win(heads=32, kv=4, window=window), LU.rule(heads=1, kv=1, dim=8, vdim=8, conv=1))], vocab=64)
    run("Lefalix", cfg, LU.weights(cfg), lambda c, w, t: L.run(c, w, t)[0], LU.TOL[dtype], dtype)
