"""GPU test of where a decode step's selective scan makes its step sizes, in the scan or by a launch before it: row counts on both sides of the
rule's lines, in 16 and 32 bits, against the same positions of a prompt."""
import numpy as np
import pytest

from tests import tafopel_util as T

pytestmark = pytest.mark.gpu


# 2048 channels x 256 numbers are 1 / 24 of the line at 12 Mi, 1 / 56 of that at 28 and 1 / 144 of that at 72
@pytest.mark.parametrize("dtype,rows,launches", [("bfloat16", 1, 0), ("bfloat16", 23, 0), ("bfloat16", 24, 1), ("bfloat16", 65, 1), ("float32", 1, 0), ("float32", 55, 0), ("float32", 56, 1), ("float32", 64, 1),
                                                 ("float32", 65, 0), ("float32", 143, 0), ("float32", 144, 1)])
def test_a_step_equals_the_prompt(dtype, rows, launches):
    import nano_vllm_candle_amd as pkg

    cfg = T.config([T.mamba(inner=2048, rank=256, mlp=T.dense()), T.mamba(inner=2048, rank=230)], width=96)
    m = pkg.TafopelForCausalLM.from_state_dict(pkg.TafopelConfig.from_dict(cfg), T.weights(cfg), dtype=dtype)
    m.kv_alloc(rows, rows, 4096)
    rng = np.random.default_rng(rows)
    seqs, ids = [rng.integers(0, cfg["vocab"], 7 + i % 5) for i in range(rows)], list(range(rows))
    want = m.step_score(ids, seqs, True, [[len(s) - 1] for s in seqs])
    m.step(ids, [s[:-1] for s in seqs], True)
    assert m.counter("scan_gate_launches") == 0
    _, got = m.step(ids, seqs, False, want_logits=True)
    assert m.counter("scan_gate_launches") == launches * len(cfg["layers"])
    assert np.abs(got - want).max() < {"bfloat16": 4e-3, "float32": 3e-5}[dtype] * np.abs(want).max()  # the tolerances of this decoder's parity tests
    m.close()
