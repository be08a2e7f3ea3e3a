"""GPU test of the selective scan's pieces: prompts of unlike length in one chunk, the longest on both sides of the one and a half pieces up to which
nothing is cut, channels that are and are not a multiple of four, every group of states a lane holds, from a fresh state and in portions."""
import numpy as np
import pytest

from oracle import tafopel_oracle as O
from tests import tafopel_util as T
from tests.berevik_util import row_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("inner, state", [(70, 4), (100, 8), (66, 16), (64, 64), (33, 256)])
@pytest.mark.parametrize("lengths", [(33, 96, 1, 64, 95), (64, 97, 33, 1, 95), (5, 130, 31, 250, 32)])
def test_prompts_of_unlike_length(lengths, inner, state, dtype):
    import nano_vllm_candle_amd as pkg

    cfg = T.config([T.mamba(inner=inner, state=state)])
    w = T.weights(cfg)
    m = pkg.TafopelForCausalLM.from_state_dict(pkg.TafopelConfig.from_dict(cfg), w, dtype=dtype)
    m.kv_alloc(16, 8, max_batched_tokens=512)
    rng = np.random.default_rng(sum(lengths))
    seqs = [rng.integers(0, cfg["vocab"], n + 40).tolist() for n in lengths]
    ids = list(range(len(lengths)))
    want = [np.asarray(O.run(cfg, w, s)[0]) for s in seqs]
    ask = [sorted({0, n // 2, max(n - 2, 0), n - 1}) for n in lengths]
    got = m.step_score(ids, [s[:n] for s, n in zip(seqs, lengths)], True, ask)
    assert row_err(got, np.concatenate([x[a] for x, a in zip(want, ask)])) < T.TOL[dtype]
    got = m.step_score(ids, seqs, False, [[n, n + 39] for n in lengths])  # from the states that the pieces left
    assert row_err(got, np.concatenate([x[[n, n + 39]] for x, n in zip(want, lengths)])) < T.TOL[dtype]
    m.close()
