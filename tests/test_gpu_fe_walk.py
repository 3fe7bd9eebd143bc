"""faster-evgen runs walked on the device, at the sizes where the walk changes:
around the shortest runs that take it, runs of few segments, batches whose last
segments are cut, streams entered inside a round; against the oracle."""
import numpy as np
import pytest

import trois_photons as tp
from test_gpu_f32 import KIND, close_f32
from test_gpu_parity import RNG, acc_close

pytestmark = pytest.mark.gpu

SIZES = (8191, 8192, 8193, 16_383, 16_384, 16_385, 50_021, 262_145, 640_000)


@pytest.fixture(scope="module")
def engine():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        yield e


@pytest.fixture(scope="module")
def cfg(valeurs):
    return tp.Configuration.load(valeurs)


@pytest.mark.parametrize("rng", ["ranf", "xoshiro"])
def test_closures(engine, cfg, oracle, valeurs, rng):
    """Successive closures, each from where the previous one left the stream."""
    params = tp.params_from_config(cfg, faster_evgen=True)
    st, g = tp.rng_state(RNG[rng]), oracle.rng(rng)
    ocfg, opts = oracle.config(valeurs), oracle.opts(rng, faster_evgen=True)
    for n in SIZES:
        print(f"faster-evgen closure {rng} n={n}", flush=True)
        a = engine.simulate_batch(params, RNG[rng], st, n).as_array()
        acc_close(a, oracle.simulate_batch(ocfg, opts, g, n).as_array(), n)
        if rng == "xoshiro":
            assert list(st.s) == list(g.xs)
        else:
            assert st.index == g.index and list(st.numbers)[1:] == list(g.numbers)[1:]


@pytest.mark.parametrize("rng", ["ranf", "xoshiro"])
def test_f32_closures(engine, cfg, oracle32, valeurs, rng):
    params = tp.params_from_config(cfg, precision=tp.PREC_F32, faster_evgen=True)
    st, g = tp.rng_state(KIND[rng]), oracle32.rng(rng)
    ocfg, opts = oracle32.config(valeurs), oracle32.opts(rng, faster_evgen=True)
    for n in SIZES:
        print(f"faster-evgen f32 closure {rng} n={n}", flush=True)
        a = engine.simulate_batch(params, KIND[rng], st, n).as_array()
        close_f32(a, oracle32.simulate_batch(ocfg, opts, g, n).as_array(), n)
        if rng == "xoshiro":
            assert list(st.s) == list(g.xs32)
        else:
            assert st.index == g.index and list(st.numbers)[1:] == list(g.numbers)[1:]


@pytest.mark.parametrize("rng", ["ranf", "xoshiro"])
@pytest.mark.parametrize("seeding", ["skipahead", "jump"])
@pytest.mark.parametrize("n_events", [1, 10_001, 20_480, 1_048_577, 3_000_017])
def test_runs(engine, cfg, oracle, valeurs, rng, seeding, n_events):
    print(f"faster-evgen run {rng} {seeding} N={n_events}", flush=True)
    params = tp.params_from_config(cfg.with_events(n_events), faster_evgen=True)
    per, _, stats = engine.run(params, RNG[rng], tp.SEEDINGS[seeding], tp.rng_state(RNG[rng]), n_events)
    if n_events > 16_384:
        assert stats.host_walk_chunks == 0
    opts = oracle.opts(rng, faster_threading=seeding == "jump", threads=16, faster_evgen=True)
    _, oper = oracle.run(oracle.config(valeurs, n_events), opts, per_batch=True)
    assert len(per) == len(oper)
    for b, (a, o) in enumerate(zip(per, oper)):
        acc_close(tp.TpAcc.from_buffer_copy(a).as_array(), o.as_array(), min(tp.BATCH_SIZE, n_events - b * tp.BATCH_SIZE))
