"""Batches split over wavefronts: every run length of the xoshiro256+ lane
tables, parts that end inside a run, batches left with fewer events than one
part, against the oracle batch by batch."""
import numpy as np
import pytest

import trois_photons as tp
from test_gpu_parity import RNG, acc_close, cfg, engine  # noqa: F401

pytestmark = pytest.mark.gpu


# closure calls: one batch of n events, so the run length grows with n (1, 2,
# 4, 5, ... events per lane), with n around whole wavefronts and runs
@pytest.mark.parametrize("rng", ["ranf", "xoshiro"])
@pytest.mark.parametrize("precision", [tp.PREC_F64, tp.PREC_MIXED])
def test_closure_sizes(engine, cfg, oracle, valeurs, rng, precision):  # noqa: F811
    params = tp.params_from_config(cfg, precision=precision)
    st, g = tp.rng_state(RNG[rng]), oracle.rng(rng)
    ocfg = oracle.config(valeurs)
    for n in (1, 63, 64, 65, 127, 129, 4096, 10_000, 65_535, 131_073, 250_001, 400_000, 640_000):
        print(f"closure {rng} precision {precision} n={n}", flush=True)
        a = engine.simulate_batch(params, RNG[rng], st, n).as_array()
        b = np.asarray(oracle.simulate_batch(ocfg, oracle.opts(rng), g, n).as_array())
        if precision == tp.PREC_F64:
            acc_close(a, b, n)
        else:  # an event's f32 amplitudes hold about 60 roundings of 2^-24
            assert a[0] == b[0]
            scale = np.sqrt(n * np.abs(b[6:11])) + 1e-300
            assert np.all(np.abs(a[1:6] - b[1:6]) <= 64 * 2**-24 * scale)
            assert np.all(np.abs(a[6:] - b[6:]) <= 128 * 2**-24 * np.abs(b[6:]) + 1e-300)


# runs: from one batch over counts that leave the last round of resident
# wavefronts nearly empty without a split to several strides of the grid, the
# last batch partial
@pytest.mark.parametrize("rng", ["ranf", "xoshiro"])
@pytest.mark.parametrize("seeding", ["skipahead", "jump"])
@pytest.mark.parametrize("n_events", [640, 20_001, 1_000_063, 10_250_000, 15_360_001, 31_234_567])
def test_run_sizes(engine, cfg, oracle, valeurs, rng, seeding, n_events):  # noqa: F811
    print(f"run {rng} {seeding} N={n_events}", flush=True)
    params = tp.params_from_config(cfg.with_events(n_events))
    per, _, _ = engine.run(params, RNG[rng], tp.SEEDINGS[seeding], tp.rng_state(RNG[rng]), n_events)
    _, oper = oracle.run(oracle.config(valeurs, n_events), oracle.opts(rng, faster_threading=seeding == "jump", threads=16),
                         per_batch=True)
    assert len(per) == len(oper)
    for b, (a, o) in enumerate(zip(per, oper)):
        acc_close(tp.TpAcc.from_buffer_copy(a).as_array(), o.as_array(), min(tp.BATCH_SIZE, n_events - b * tp.BATCH_SIZE))
