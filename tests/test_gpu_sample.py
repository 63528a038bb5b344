"""GPU parity of token sampling (ar_hip_sample, ar_hip_qwen3_set_sampling) against the CPU oracle.

The oracle (oracle/sample_oracle.c, pinned in tests/test_sample_oracle.py) runs on the same fp32
logits with java.util.Random generators of the same seeds.  The bar is the same index for every
draw, except where the oracle's uniform draw r lies within MARGIN of a boundary of the cumulative
intervals (the device groups its partial sums differently, ~1e-16; the nucleus cut is decided in
2^-60 fixed point): such draws are counted and must stay rare.  Generator states must match
exactly after every call (one nextDouble per sampled token, none for greedy temperatures).
"""
import dataclasses
import time

import numpy as np
import pytest

import oracle
from common_amd import config as C
from common_amd import hardware as hw
from common_amd import synthetic
from common_amd.qwen3 import Qwen3

pytestmark = pytest.mark.gpu
MARGIN = 1e-12


def _oracle_draw(mode, logits_row, temperature, top_p, g):
    if mode == hw.SAMPLE_TOKEN:
        return oracle.sample_token(logits_row.astype(np.float64), temperature, top_p, g)
    return oracle.model_sample(logits_row.astype(np.float64), temperature, g)


def _run_op(ctx, logits, mode, temperature, top_p, seeds, calls):
    rows, n = logits.shape
    lg = ctx.to_device(logits.astype(np.float32))
    st = ctx.to_device(np.array([hw.java_random_state(s) for s in seeds], dtype=np.uint64))
    out = ctx.allocate(rows * 4)
    gens = [oracle.JavaRandom(s) for s in seeds]
    near, got_all = 0, []
    for _ in range(calls):
        ctx.sample(lg, rows, n, mode, temperature, top_p, st, out)
        ctx.synchronize()
        got = out.download(np.int32, rows)
        for b in range(rows):
            k, r, margin = _oracle_draw(mode, logits[b], temperature, top_p, gens[b])
            if margin < MARGIN:
                near += 1
                continue
            assert got[b] == k, f"row {b}: device {got[b]} oracle {k} (r={r}, margin={margin})"
        got_all.append(got)
        dev_state = st.download(np.uint64, rows)
        assert [int(x) for x in dev_state] == [g.state.value for g in gens]
    for buf in (lg, st, out):
        buf.free()
    return near, np.stack(got_all)


CASES = [
    (hw.SAMPLE_TOKEN, 0.7, 1.0),
    (hw.SAMPLE_TOKEN, 1.3, 0.9),
    (hw.SAMPLE_TOKEN, 1.0, 0.5),
    (hw.SAMPLE_TOKEN, 0.8, 0.0),
    (hw.SAMPLE_MODEL, 0.7, 1.0),
    (hw.SAMPLE_MODEL, 2.0, 1.0),
]


@pytest.mark.parametrize("n", [37, 1024, 151936])
@pytest.mark.parametrize("mode,temperature,top_p", CASES)
def test_sample_op_matches_oracle(ctx, n, mode, temperature, top_p):
    print(f"[sample op] n={n} mode={mode} T={temperature} top_p={top_p}", flush=True)
    rng = np.random.default_rng(n + int(temperature * 10))
    rows = 8
    logits = rng.normal(0.0, 2.0, (rows, n)).astype(np.float32)
    logits[1, : n // 3] = 0.0  # exact zeros: the model function's ignore-zero path
    near, got = _run_op(ctx, logits, mode, temperature, top_p, seeds=[3 * b + 1 for b in range(rows)], calls=4)
    assert near <= 1
    assert got.min() >= 0 and got.max() < n


@pytest.mark.parametrize("n", [1024, 151936])
@pytest.mark.parametrize("top_p", [0.3, 0.6, 0.95])
def test_sample_op_nucleus_with_ties(ctx, n, top_p):
    # integer logits: thousands of exactly equal probabilities, the cut falls inside a tie group
    print(f"[sample ties] n={n} top_p={top_p}", flush=True)
    rng = np.random.default_rng(11)
    rows = 4
    logits = np.round(rng.normal(0.0, 1.5, (rows, n))).astype(np.float32)
    logits[2] = 1.0  # one row entirely tied
    near, _ = _run_op(ctx, logits, hw.SAMPLE_TOKEN, 1.0, top_p, seeds=[101, 202, 303, 404], calls=6)
    assert near <= 1


@pytest.mark.parametrize("n,top_p", [(63, 0.9), (4097, 0.7), (151936, 0.5), (151936, -1.0)])
def test_sample_op_nucleus_buckets(ctx, n, top_p):
    """The cut inside a bucket of the first pass that holds a whole row of distinct values (more than the
    drawing block keeps in LDS at the largest n), a row with one certain value (p = 1, the last bucket),
    one spread over more octaves than there are buckets, and a vocabulary with empty chunks."""
    print(f"[sample buckets] n={n} top_p={top_p}", flush=True)
    rng = np.random.default_rng(n)
    logits = rng.uniform(0.0, 0.02, (4, n)).astype(np.float32)
    logits[1] = 0.0
    logits[1, n // 2] = 100.0
    logits[2] = np.linspace(-120.0, 0.0, n)
    logits[3] = rng.permutation(np.linspace(-4.0, 4.0, n))
    near, _ = _run_op(ctx, logits, hw.SAMPLE_TOKEN, 0.9, top_p, seeds=[7, 8, 9, 10], calls=4)
    assert near <= 1


@pytest.mark.parametrize("n,top_p", [(4201, 0.5), (32001, 0.9), (151936, 0.3), (151936, 0.97)])
def test_sample_op_nucleus_in_a_crowded_bucket(ctx, n, top_p):
    """More values around the cut than the drawing block holds in LDS: every value equal; nearly equal ones
    (one round of ranges); half of them equal between nearly equal ones (the range of the equal ones
    alone overflows LDS); equal ones with a few a unit of the last place away.  (n * top_p is not whole:
    where it is, top_p equals a partial sum of the equal row, and the 2^-60 fixed point and the oracle's
    sequential sum, both within 1e-13 of it, may fall on different sides.)"""
    print(f"[sample crowded] n={n} top_p={top_p}", flush=True)
    rng = np.random.default_rng(n)
    logits = np.zeros((4, n), np.float32)
    logits[1] = rng.normal(0.0, 0.001, n)
    logits[2] = np.where(rng.random(n) < 0.5, 0.0, rng.normal(0.0, 0.001, n))
    logits[3] = 1.0
    logits[3, rng.integers(0, n, 500)] = np.nextafter(np.float32(1.0), np.float32(2.0))
    logits[3, rng.integers(0, n, 500)] = np.nextafter(np.float32(1.0), np.float32(0.0))
    near, _ = _run_op(ctx, logits, hw.SAMPLE_TOKEN, 1.0, top_p, seeds=[21, 22, 23, 24], calls=4)
    assert near <= 1


def test_sample_op_equal_logits_take_no_multiple_of_the_time(ctx):
    """Equal logits put the whole row into one bucket of the nucleus search; the draw must not go over them
    once per digit of the search (an ordinary row's time without; 40 times that with a pass, and its atomics
    on one address, per digit)."""
    n, best = 151936, {}
    out, st = ctx.allocate(4), ctx.to_device(np.array([hw.java_random_state(1)], dtype=np.uint64))
    rows = {"spread": np.random.default_rng(1).normal(0.0, 2.0, n), "equal": np.zeros(n)}
    for name, row in rows.items():
        lg, times = ctx.to_device(row.astype(np.float32)), []
        for _ in range(12):
            ctx.synchronize()
            t0 = time.perf_counter()
            for _ in range(4):
                ctx.sample(lg, 1, n, hw.SAMPLE_TOKEN, 1.0, 0.9, st, out)
            ctx.synchronize()
            times.append(time.perf_counter() - t0)
        best[name] = min(times)
        lg.free()
    out.free()
    st.free()
    assert best["equal"] <= 10 * best["spread"], best


@pytest.mark.parametrize("mode,temperature", [(hw.SAMPLE_MODEL, 0.0), (hw.SAMPLE_TOKEN, 0.0),
                                              (hw.SAMPLE_TOKEN, -1.0)])
def test_sample_op_greedy_temperatures_draw_nothing(ctx, mode, temperature):
    rng = np.random.default_rng(2)
    logits = rng.normal(0, 1, (3, 500)).astype(np.float32)
    logits[0, 10] = logits[0, 20] = 9.0  # first maximum wins
    lg = ctx.to_device(logits)
    st = ctx.to_device(np.array([hw.java_random_state(5)] * 3, dtype=np.uint64))
    out = ctx.allocate(12)
    ctx.sample(lg, 3, 500, mode, temperature, 0.5, st, out)
    ctx.synchronize()
    np.testing.assert_array_equal(out.download(np.int32, 3), np.argmax(logits, axis=1))
    assert out.download(np.int32, 3)[0] == 10
    assert all(int(x) == hw.java_random_state(5) for x in st.download(np.uint64, 3))


def test_sample_op_errors(ctx):
    lg = ctx.allocate(64)
    out = ctx.allocate(16)
    with pytest.raises(hw.HardwareException):
        ctx.sample(lg, 1, 16, 7, 1.0, 1.0, None, out)
    with pytest.raises(hw.HardwareException):  # a sampled temperature needs a generator
        ctx.sample(lg, 1, 16, hw.SAMPLE_TOKEN, 1.0, 1.0, None, out)


# ---- the model's token loop -------------------------------------------------------------
def _step_all(m, steps):
    am = m.model
    fed, logits = [], []
    for _ in range(steps):
        t, lg = am.next(return_logits=True)
        fed.append(t)
        logits.append(lg)
    return np.stack(fed, axis=1), np.stack(logits, axis=1)


def _check_loop(fed, logits, n_prompt, mode, temperature, top_p, seeds):
    """The token fed at each step past the prompt is the oracle's draw from the previous step's
    device logits with generators advanced only past the prompt."""
    near = 0
    for b in range(fed.shape[0]):
        g = oracle.JavaRandom(seeds[b])
        for s in range(n_prompt, fed.shape[1]):
            k, r, margin = _oracle_draw(mode, logits[b, s - 1], temperature, top_p, g)
            if margin < MARGIN:
                near += 1
                continue
            assert fed[b, s] == k, f"seq {b} step {s}: fed {fed[b, s]} oracle {k}"
    assert near <= 1


@pytest.mark.parametrize("mode,temperature,top_p", [(hw.SAMPLE_MODEL, 0.8, 1.0), (hw.SAMPLE_TOKEN, 0.9, 0.8)])
@pytest.mark.parametrize("graph", [True, False])
def test_model_samples_each_step_from_its_logits(ctx, mode, temperature, top_p, graph):
    cfg = dataclasses.replace(C.C1_TINY, max_batch=2)
    sd = synthetic.state_dict(C.C1_TINY, seed=0)
    prompt = synthetic.prompt_ids(C.C1_PROMPT, cfg.vocab_size, seed=0)
    seeds = [17, 29]
    with Qwen3(cfg, sd, ctx) as m:
        am = m.model
        am.use_graph(graph)
        am.set_sampling(mode, temperature, top_p, seeds=seeds)
        am.reset()
        for b in range(2):
            am.set_prompt(prompt, seq=b)
        fed, logits = _step_all(m, len(prompt) + 24)
        _check_loop(fed, logits, len(prompt), mode, temperature, top_p, seeds)
        assert not np.array_equal(fed[0, len(prompt):], fed[1, len(prompt):])  # independent generators
        # run() draws the same tokens from freshly seeded generators
        am.set_sampling(mode, temperature, top_p, seeds=seeds)
        am.reset()
        for b in range(2):
            am.set_prompt(prompt, seq=b)
        toks = am.run(len(prompt) + 24)
        np.testing.assert_array_equal(toks, fed)
        # back to greedy: temperature 0 (AutoregressiveModel.setTemperature)
        am.set_temperature(0.0)
        am.reset()
        am.set_prompt(prompt, seq=0)
        am.set_prompt(prompt, seq=1)
        g_fed, g_logits = _step_all(m, len(prompt) + 4)
        for s in range(len(prompt), g_fed.shape[1]):
            assert g_fed[0, s] == int(np.argmax(g_logits[0, s - 1]))


def test_prefill_draws_the_first_generated_token(ctx):
    cfg = dataclasses.replace(C.C1_TINY, weight_dtype=C.DTYPE_BF16)
    sd = synthetic.state_dict(cfg, seed=0)
    prompt = synthetic.prompt_ids(C.C1_PROMPT, cfg.vocab_size, seed=0)
    with Qwen3(cfg, sd, ctx) as m:
        am = m.model
        am.set_sampling(hw.SAMPLE_TOKEN, 0.9, 0.9, seeds=[4])
        am.reset()
        am.set_prompt(prompt)
        last = am.prefill(return_logits=True)
        fed, logits = _step_all(m, 10)
    g = oracle.JavaRandom(4)
    k, _, margin = oracle.sample_token(last[0].astype(np.float64), 0.9, 0.9, g)
    if margin >= MARGIN:
        assert fed[0, 0] == k
    for s in range(1, 10):
        k, _, margin = oracle.sample_token(logits[0, s - 1].astype(np.float64), 0.9, 0.9, g)
        if margin >= MARGIN:
            assert fed[0, s] == k


def test_model_sampling_vs_fp64_oracle_model(ctx):
    """End to end against the FP64 oracle model with its own logits.  The device's fp32 logits
    differ by ~1e-6, which moves the cumulative intervals of this sample function by ~1e-9: equal
    tokens until a draw comes within 1e-7 of a boundary."""
    cfg = C.C1_TINY
    sd = synthetic.state_dict(cfg, seed=0)
    prompt = synthetic.prompt_ids(C.C1_PROMPT, cfg.vocab_size, seed=0)
    n_dec = 24
    with Qwen3(cfg, sd, ctx) as m:
        am = m.model
        am.set_sampling(hw.SAMPLE_MODEL, 0.8, 1.0, seeds=[123])
        am.reset()
        am.set_prompt(prompt)
        fed, _ = _step_all(m, len(prompt) + n_dec)
    g = oracle.JavaRandom(123)
    margins = []

    def sampler(lg):
        k, _, mg = oracle.model_sample(lg, 0.8, g)
        margins.append(mg)
        return k

    ref = oracle.OracleQwen3(cfg, sd, precision="fp64")
    rf, _ = ref.generate(prompt, n_dec, want_logits=False, sampler=sampler)
    compared = 0
    for s in range(len(prompt), len(rf)):
        if margins[s - len(prompt)] < 1e-7:
            break
        assert fed[0, s] == rf[s], f"step {s}"
        compared += 1
    print(f"[sample e2e] {compared}/{n_dec} sampled tokens compared before a near-boundary draw")
    assert compared >= 8
