"""GPU test of decode steps of one to eight rows in one launch (resident.hip): every number of rows, both sides of a tile's, a wave's, a block's and a part's ends, against the step
as launches and the CPU oracle; what is not taken; a launch that gives up; two models at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def config(heads=16, kv=8, inter=3072, layers=4, hidden=1024):
    import nano_vllm_candle_amd as pkg

    kw = dict(vocab_size=512, hidden_size=hidden, head_dim=128, num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv, intermediate_size=inter)
    return pkg.Qwen3Config.tiny(**kw), kw


def run(cfg, lens, resident, steps=3, bits=16, spins=None):
    """logits of every step, launches taken"""
    import nano_vllm_candle_amd as pkg

    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, seed=4)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.set_option("resident", resident)
    if spins is not None:
        m.set_option("resident_spins", spins)
    ids = list(range(len(lens)))
    m.kv_alloc(sum(-(-(n + steps + 2) // 256) for n in lens), len(lens), 4096)
    rng = np.random.default_rng(len(lens))
    seqs = [rng.integers(0, 512, n).tolist() for n in lens]
    m.step(ids, seqs, True)
    out, before = [], m.counter("resident_launches")  # (prompts of one token each are such a step too)
    for k in range(steps):
        for i, s in enumerate(seqs):
            s.append(11 + k + i)
        out.append(m.step(ids, seqs, False, want_logits=True)[1].copy())
    taken = m.counter("resident_launches") - before
    m.close()
    return out, taken, seqs


# the same sums in another order: an f16 key or value may round the other way, 2^-11 of the largest logit
def close(a, b):
    return all(np.isfinite(x).all() and np.abs(x - y).max() < 2.0 ** -11 * np.abs(y).max() for x, y in zip(a, b))


@pytest.mark.parametrize("heads,kv,inter", [(16, 8, 3072), (8, 4, 1024), (16, 4, 2048), (8, 8, 3072), (16, 8, 1024)])
@pytest.mark.parametrize("lens", [[1], [30], [137], [255], [256], [700], [2100], [31, 32], [3, 300, 64], [129, 130, 31, 500], [600, 20, 700, 513, 5], [96, 127, 128, 254, 255, 256],
                                  [8, 16, 24, 33, 40, 48, 56], [10, 20, 255, 256, 257, 100, 1030, 80], [900] * 8])
def test_equals_the_launches(heads, kv, inter, lens):
    from oracle import oracle as O

    cfg, kw = config(heads, kv, inter)
    got, taken, seqs = run(cfg, lens, 1)
    want, none, _ = run(cfg, lens, 0)
    assert taken == 3 and none == 0 and close(got, want)
    if max(lens) <= 300:
        om = O.Model(O.make_config(max_position_embeddings=cfg.max_position_embeddings, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, bos_token_id=cfg.bos_token_id,
                                   eos_token_id=cfg.eos_token_id, **kw)).fill_synthetic(4)
        truth = om.run_greedy(seqs)[1]
        assert np.abs(got[-1] - truth).max() < 2.0 ** -10 * np.abs(truth).max()  # f16 keys and values, four layers


def test_numbers_of_rows_in_turn():
    # what a launch leaves of its last layer is emptied by the next one, whatever rows either has
    import nano_vllm_candle_amd as pkg

    cfg, _ = config()
    rng = np.random.default_rng(0)
    seqs = [rng.integers(0, 512, 40 + 9 * i) for i in range(8)]
    out = {}
    for resident in (1, 0):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, seed=4)
        m.set_option("resident", resident)
        m.kv_alloc(16, 8, 1024)
        m.step(list(range(8)), seqs, True)
        out[resident] = [m.step(list(range(n)), [np.append(s, 5) for s in seqs[:n]], False, want_logits=True)[1].copy() for n in (8, 1, 4, 8, 3, 7, 2, 2, 6, 1, 5)]
        m.close()
    assert close(out[1], out[0])


@pytest.mark.parametrize("layers,hidden,inter,bits,rows", [(3, 1024, 3072, 16, 1), (4, 2048, 3072, 16, 1), (4, 1024, 4096, 16, 1), (4, 1024, 1536, 16, 1), (4, 1024, 3072, 24, 1), (4, 1024, 3072, 16, 9)])
def test_what_stays_launches(layers, hidden, inter, bits, rows):
    assert run(config(inter=inter, layers=layers, hidden=hidden)[0], [20] * rows, 1, 1, bits)[1] == 0


def greedy(m, seqs, n, enqueued=False):
    """ids of n steps behind a prompt, one row of them a sequence"""
    ids = list(range(len(seqs)))
    for i in ids:
        m.seq_free(i)
    m.step(ids, seqs, True)
    if enqueued:
        for _ in range(n):
            m.decode_enqueue()
    out = [(m.decode_collect() if enqueued else m.decode_next())[:len(seqs)].tolist() for _ in range(n)]
    return np.array(out).T


def test_steps_that_are_not_waited_for_stay_launches():
    import nano_vllm_candle_amd as pkg

    m = pkg.Qwen3ForCausalLM.from_synthetic(config()[0], seed=4)
    m.kv_alloc(8, 3, 256)
    seqs = [[1, 2, 3], [7, 5], [40] * 30]
    first = greedy(m, seqs, 4)
    assert m.counter("resident_launches") == 4
    second = greedy(m, seqs, 4, enqueued=True)
    assert m.counter("resident_launches") == 4
    m.set_option("resident", 0)
    assert np.array_equal(second, greedy(m, seqs, 4))  # the same launches
    # the ids of the one launch by the logits that launches give behind the same tokens (the prompt's own id is not among decode_next's): either may be off by the bound of close()
    ids = list(range(3))
    for i in ids:
        m.seq_free(i)
    start = m.step(ids, seqs, True)[0]
    for k in range(4):
        logits = m.step(ids, [s + [int(start[i])] + first[i, :k].tolist() for i, s in enumerate(seqs)], False, want_logits=True)[1]
        for i in ids:
            assert logits[i, first[i, k]] >= logits[i].max() - 2 * 2.0 ** -11 * np.abs(logits).max(), (i, k)
    m.close()


@pytest.mark.parametrize("seqs", [[[1, 2, 3]], [[9] * 600, [4, 4], [7] * 300]])
def test_decode_next_with_a_launch_that_gives_up(seqs):
    import nano_vllm_candle_amd as pkg

    m = pkg.Qwen3ForCausalLM.from_synthetic(config()[0], seed=4)
    m.kv_alloc(12, 3, 1024)
    m.set_option("resident_spins", 0)
    got = greedy(m, seqs, 4)
    assert m.counter("resident_launches") == 1 and m.counter("resident_give_ups") == 1
    m.set_option("resident", 0)
    assert np.array_equal(got, greedy(m, seqs, 4))
    m.close()


@pytest.mark.parametrize("lens", [[137], [600, 20, 300]])
def test_a_launch_that_gives_up(lens):
    # no turn but the first of any wait: the step is run again as launches, and so are those after it
    cfg, _ = config()
    got, taken, _ = run(cfg, lens, 1, spins=0)
    want, _, _ = run(cfg, lens, 0)
    assert taken == 1 and all(np.array_equal(a, b) for a, b in zip(got, want))


def test_giving_up_is_not_for_good():
    # counted, and after some steps as launches (the one that is run again is the first), twice as many each time, the model tries again
    import nano_vllm_candle_amd as pkg

    m = pkg.Qwen3ForCausalLM.from_synthetic(config()[0], seed=4)
    m.kv_alloc(2, 1, 256)
    m.step([0], [[1, 2, 3]], True)

    def launches_until_the_next():
        at, n = m.counter("resident_launches"), 0
        while m.counter("resident_launches") == at:
            m.step([0], [[1, 2, 3, 4]], False)
            n += 1
        return n - 1

    m.set_option("resident_spins", 0)
    assert launches_until_the_next() == 0 and m.counter("resident_give_ups") == 1
    assert launches_until_the_next() == 1023 and m.counter("resident_give_ups") == 2
    m.set_option("resident_spins", 1000000)
    assert launches_until_the_next() == 2047 and m.counter("resident_give_ups") == 2
    assert launches_until_the_next() == 0
    m.close()


def test_a_step_that_gives_up_and_then_fails():
    # the next step is a prompt of several chunks: it is not that step's to run again, nor is the first decode step a launch that may read what is left
    import nano_vllm_candle_amd as pkg

    cfg, _ = config()
    rng = np.random.default_rng(2)
    first, prompt = rng.integers(0, 512, 30), rng.integers(0, 512, 200)
    out = []
    for fails in (1, 0):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, seed=4)
        m.kv_alloc(8, 2, 64)
        m.step([0], [first], True)
        if fails:
            m.set_option("resident_spins", 0)
            m.set_option("leave_fail", 1)
            with pytest.raises(pkg._lib.NvllmError, match="leave_fail"):
                m.step([0], [np.append(first, 7)], False)
            m.set_option("resident_spins", 1000000)
            assert m.counter("resident_launches") == 1
        else:
            m.set_option("resident", 0)
        steps = [m.step([1], [prompt], True, want_logits=True)[1].copy()]
        for k in (1, 2):
            steps += [m.step([1], [np.append(prompt, [3] * k)], False, want_logits=True)[1].copy(), m.step([0], [np.append(first, [7] * k)], False, want_logits=True)[1].copy()]
        out.append(steps)
        m.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def test_two_models_at_once():
    # each on its own thread and stream: their launches take turns
    import nano_vllm_candle_amd as pkg

    cfg, _ = config(layers=8)
    lens = {0: [137], 1: [40, 60, 300]}
    want, got = {}, {}

    def work(k, into):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, seed=k)
        m.kv_alloc(8, 4, 512)
        rng = np.random.default_rng(k)
        seqs = [rng.integers(0, 512, n) for n in lens[k]]
        ids = list(range(len(seqs)))
        m.step(ids, seqs, True)
        grown = [np.append(s, 7) for s in seqs]
        out = [m.step(ids, grown, False, want_logits=True)[1].copy() for _ in range(40)]
        into[k] = out, m.counter("resident_launches")
        m.close()

    for k in lens:
        work(k, want)
    threads = [threading.Thread(target=work, args=(k, got)) for k in lens]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for k in lens:
        assert got[k][1] == 40 and all(np.array_equal(a, b) for a, b in zip(got[k][0], want[k][0]))


def test_a_turn_does_not_wait_for_other_work():
    # behind the other context's last one-launch step comes its queue of many rows: only the former is waited for
    import time

    import nano_vllm_candle_amd as pkg

    rows = 200
    one = pkg.Qwen3ForCausalLM.from_synthetic(config()[0], seed=4)
    one.kv_alloc(2, 1, 256)
    many = pkg.Qwen3ForCausalLM.from_synthetic(config(layers=28)[0], seed=4)
    many.kv_alloc(rows + 1, rows + 1, 1024)
    alone, ids = many.max_seqs - 1, list(range(rows))
    one.step([0], [[1, 2, 3]], True)
    many.step([alone], [[1, 2, 3]], True)
    for k in range(2):  # both have made such steps, each behind the other's
        one.decode_next()
        many.step([alone], [[1, 2, 3, 4]], False)
    assert one.counter("resident_launches") == 2 and many.counter("resident_launches") == 2
    many.step(ids, [[1 + i, 2, 3] for i in ids], True)
    shares = []
    for _ in range(5):
        many.step([alone], [[1, 2, 3, 4]], False)
        many.step(ids, [[1 + i, 2, 3, 4] for i in ids], False)
        t0 = time.perf_counter()
        for _ in range(4):
            many.decode_enqueue()
        one.decode_next()
        t1 = time.perf_counter()
        for _ in range(4):
            many.decode_collect()
        shares.append((t1 - t0) / (time.perf_counter() - t0))
    assert one.counter("resident_launches") == 7 and many.counter("resident_launches") == 7 and one.counter("resident_give_ups") == 0
    assert sorted(shares)[2] < 0.7, shares  # all of it, where the queue is waited for
    one.close()
    many.close()
