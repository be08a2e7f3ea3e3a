"""GPU tests of a step's metadata: more chunks than the ring of pinned blocks, arrays that start anywhere, block tables after steps that
took blocks and failed.  The reference is the same call on a model that has run nothing else: bits are equal."""
import numpy as np
import pytest

from oracle import gopunex_oracle as G
from tests.gopunex_util import MIXED

pytestmark = pytest.mark.gpu


def _model(design, max_seqs, blocks, rows):
    import nano_vllm_candle_amd as pkg

    if design == "qwen3":
        m = pkg.Qwen3ForCausalLM.from_synthetic(pkg.Qwen3Config.tiny(), seed=3)
    else:
        w = G.random_weights(MIXED, 3)
        shapes = {k: v.shape for k, v in w.items()}
        m = pkg.GopunexForCausalLM.from_state_dict(pkg.GopunexConfig.from_dict(MIXED, shapes), w)
    m.kv_alloc(blocks, max_seqs, rows)
    return m


@pytest.mark.parametrize("design", ["qwen3", "gopunex"])
@pytest.mark.parametrize("max_seqs,rows", [(1, 16), (3, 33), (6, 64)])
def test_many_chunks_and_tables_after_failed_steps(design, max_seqs, rows):
    from nano_vllm_candle_amd._lib import NvllmError

    blocks = max_seqs + 2
    m = _model(design, max_seqs, blocks, rows)
    rng = np.random.default_rng(max_seqs)
    # every retry releases the first sequence's blocks, takes them again in another order and fails on the second one; a model of one
    # sequence fails as its metadata is sent.  Until there are more new entries than the pinned block has room for: the whole table goes
    m.set_option("stage_fail", 1 << 30 if max_seqs == 1 else 0)
    for k in range(100 * blocks):
        n = [256 * (1 + k % blocks) - 5, 256 * blocks][:max_seqs]
        with pytest.raises(NvllmError):
            m.step(list(range(len(n))), [rng.integers(0, 300, x) for x in n], True)
    m.set_option("stage_fail", 0)
    for s in (0, 1):
        m.seq_free(s)
    prompts = [rng.integers(0, 300, int(x)) for x in rng.integers(1, 250, max_seqs)]
    prompts[0] = rng.integers(0, 300, 300)  # 300 tokens: many chunks of `rows`
    ids = list(range(max_seqs))
    # as many wanted rows as the head's buffers hold, and more
    for wanted in ([[len(p) - 1] for p in prompts], [list(range(max(0, len(p) - 3), len(p))) for p in prompts]):
        fresh = _model(design, max_seqs, blocks, rows)
        got, want = (x.step_score(ids, prompts, True, wanted) for x in (m, fresh))
        assert np.array_equal(got, want)
        assert m.counter("table_copies") > 0 and fresh.counter("table_copies") == 0
        if design == "qwen3":
            lists = [np.append(p, 7) for p in prompts]
            a, b = (x.step(ids, lists, False, want_logits=True) for x in (m, fresh))
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("design", ["qwen3", "gopunex"])
def test_tables_after_a_failed_launch(design):
    """a step whose metadata launch fails has taken its blocks: the next one must still tell the device of them"""
    from nano_vllm_candle_amd._lib import NvllmError

    m, fresh = _model(design, 3, 8, 64), _model(design, 3, 8, 64)
    rng = np.random.default_rng(0)
    prompts = [rng.integers(0, 300, n) for n in (20, 300, 7)]
    ids = [0, 1, 2]
    m.set_option("stage_fail", 1)
    with pytest.raises(NvllmError):
        m.step(ids, prompts, True)
    want = fresh.step(ids, prompts, True, want_logits=True)
    got = m.step(ids, prompts, False, want_logits=True)  # nothing is cached: the same rows, in the blocks of the failed step
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    m.close(), fresh.close()
