"""faster-threading's RANF seeds, seed + 123456 b, pass the generator's modulus
1e9 in long runs, which leaves values outside [0, 1e9) in some batches' first
rounds.  Such a batch gives the same values in runs of every length, whose
batches and expansions are split in different places."""
import numpy as np
import pytest

import trois_photons as tp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("faster", [False, True])
@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_MIXED, tp.PREC_F32])
def test_batches_past_the_modulus_do_not_depend_on_the_split(valeurs, prec, faster):
    if faster and prec == tp.PREC_MIXED:
        pytest.skip("not offered")
    cfg = tp.Configuration.load(valeurs)
    state = tp.rng_state(tp.RNG_RANF, 1_000_000_000 - 5 * 123456)
    runs = []
    with tp.Engine(0) as engine:
        for batches in (60, 300, 1500, 5000):
            n = 10000 * batches
            print(f"precision {prec} faster {faster} N={n}", flush=True)
            params = tp.params_from_config(cfg.with_events(10**7), precision=prec, faster_evgen=faster)
            per, _, _ = engine.run(params, tp.RNG_RANF, tp.SEED_JUMP, state, n)
            runs.append(per[:60].copy())
    eps = 2.0**-52 if prec != tp.PREC_F32 else 0.0  # f32 sums are in event order
    for per in runs[1:]:
        assert np.array_equal(per["selected_events"], runs[0]["selected_events"])
        for name in ("spm2", "vars", "sigma", "variance"):
            a, b = per[name], runs[0][name]
            assert np.array_equal(np.isnan(a), np.isnan(b)), name
            # 10 000 terms summed in another order; the interference sum cancels
            scale = np.sqrt(10000 * np.abs(runs[0]["vars"])) if name == "spm2" else np.abs(b)
            ok = np.abs(a - b) <= 10000 * eps * scale
            assert np.all(ok | np.isnan(a)), name


def past(state):
    return any(not 0 <= x < 10**9 for x in list(state.numbers)[1:])


@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_MIXED, tp.PREC_F32])
def test_closures_past_the_modulus_equal_the_runs_batches(valeurs, prec):
    seed, batches, seen = 1_000_000_000 - 5 * 123456, 40, 0
    params = tp.params_from_config(tp.Configuration.load(valeurs).with_events(10**7), precision=prec)
    with tp.Engine(0) as engine:
        per, _, _ = engine.run(params, tp.RNG_RANF, tp.SEED_JUMP, tp.rng_state(tp.RNG_RANF, seed), 10000 * batches)
        for b in range(batches):
            st = tp.rng_state(tp.RNG_RANF, seed + 123456 * b)
            seen += past(st)
            print(f"precision {prec} batch {b}", flush=True)
            acc = engine.simulate_batch(params, tp.RNG_RANF, st, 10000)
            assert acc.selected_events == per[b]["selected_events"], b
    assert seen > 2


@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_F32])
def test_faster_evgen_refuses_a_state_past_the_modulus(valeurs, prec):
    states = (tp.rng_state(tp.RNG_RANF, 10**9 + 123456 * b) for b in range(100))
    st = next(s for s in states if past(s))
    before = bytes(st)
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=prec, faster_evgen=True)
    with tp.Engine(0) as engine:
        for n in (1, 10000):
            with pytest.raises(tp.TpError, match="below 1e9"):
                engine.simulate_batch(params, tp.RNG_RANF, st, n)
        with pytest.raises(tp.TpError, match="below 1e9"):
            engine.run(params, tp.RNG_RANF, tp.SEED_SKIPAHEAD, st, 100000)
    assert bytes(st) == before
