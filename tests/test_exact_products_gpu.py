"""GPU test of the 32-bit products at the row counts where their kernels change (16, 32, 64 rows of the decode form, blocks of 64 rows of the
prompt form) and with ragged features, against the oracle in 64 bits."""
import numpy as np
import pytest

from oracle import gopunex_oracle as G
from tests.berevik_util import row_err
from tests.gopunex_util import CONFIGS, TOL, sharp_weights

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
