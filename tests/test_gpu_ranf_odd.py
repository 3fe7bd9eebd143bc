"""RANF states seeded past the modulus (values outside [0, 1e9)): every entry
point draws the same values from them, whatever the size of the call."""
import numpy as np
import pytest

import ranf_odd
import trois_photons as tp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        yield e


def odd_state(seed, taken=0):
    """The first odd state from `seed` on, `taken` values into its round."""
    while not ranf_odd.odd(tp.rng_state(tp.RNG_RANF, seed)):
        seed += 123456
    st = tp.rng_state(tp.RNG_RANF, seed)
    tp.rng_skip(tp.RNG_RANF, st, taken)
    return st


# around round 64 (event 293), in the first segment of 2048 rounds, past it (event 9386) and past the fourth
@pytest.mark.parametrize("n", [290, 300, 5000, 12_000, 40_000])
@pytest.mark.parametrize("seed, taken", [(1_000_987_648, 0), (1_500_000_000, 17), (2_100_000_000, 54)])
def test_events_draw_the_odd_streams_values(engine, valeurs, seed, taken, n):
    st = odd_state(seed, taken)
    print(f"events of an odd state, seed {st.seed} index {st.index} n={n}", flush=True)
    params = tp.params_from_config(tp.Configuration.load(valeurs))
    u = engine.events(params, tp.RNG_RANF, st, n)[0]
    assert np.array_equal(u.reshape(-1), ranf_odd.values(st, 12 * n) * 1e-9)


def sums(keep, m, contribs):
    """An accumulator's 13 numbers from events' cut decisions and helicity sums."""
    w = m @ contribs
    return np.concatenate([[keep.sum()], m.sum(0), (m * m).sum(0), [w.sum(), (w * w).sum()]])


def close(a, b, n):
    """Selected events exactly; sums of n terms each added in another order."""
    assert a[0] == b[0]
    assert np.array_equal(np.isnan(a), np.isnan(b))
    scale = np.abs(b)
    scale[1:6], scale[11] = np.sqrt(n * b[6:11]), np.sqrt(n * b[12])  # the interference cancels
    # n eps for the order of the sums, 16 for the weights
    assert np.all((np.abs(a - b) <= (n + 16) * 2.0**-52 * scale) | np.isnan(a)), (a, b)


# one batch, the second one's few events, many batches in several splits; a closure's 640 000 events cross 68 segments
@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_MIXED])
@pytest.mark.parametrize("seed, taken", [(1_000_987_648, 0), (1_500_000_000, 17)])
def test_runs_and_closures_simulate_those_events(engine, valeurs, seed, taken, prec):
    st = odd_state(seed, taken)
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=prec)
    print(f"events of an odd state, seed {st.seed} precision {prec}", flush=True)
    _, _, keep, m = engine.events(params, tp.RNG_RANF, st, 640_000)
    contribs = np.array(list(params.sigma_contribs))
    for n in (9_000, 10_000, 18_000, 20_001, 40_000, 123_457, 640_000):
        print(f"closure n={n}", flush=True)
        s = type(st).from_buffer_copy(st)
        close(engine.simulate_batch(params, tp.RNG_RANF, s, n).as_array(), sums(keep[:n], m[:n], contribs), n)
    for n in (10_001, 20_000, 600_000, 5_000_000, 50_000_000):
        print(f"skip-ahead run N={n}", flush=True)
        per, _, _ = engine.run(params, tp.RNG_RANF, tp.SEED_SKIPAHEAD, st, n)
        for b in range(min(64, len(per))):
            lo, hi = 10_000 * b, min(n, 10_000 * b + 10_000)
            close(tp.TpAcc.from_buffer_copy(per[b]).as_array(), sums(keep[lo:hi], m[lo:hi], contribs), hi - lo)


@pytest.mark.parametrize("seed, taken", [(1_000_987_648, 0), (1_500_000_000, 17)])
def test_f32_runs_do_not_depend_on_the_split(engine, valeurs, seed, taken):
    """f32 sums are in event order: the same bits in every run and closure."""
    st = odd_state(seed, taken)
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=tp.PREC_F32)
    runs = []
    for n in (20_000, 600_000, 5_000_000, 50_000_000):
        print(f"f32 skip-ahead run of an odd state, seed {st.seed} N={n}", flush=True)
        per, _, _ = engine.run(params, tp.RNG_RANF, tp.SEED_SKIPAHEAD, st, n)
        runs.append(per.view(np.uint64).reshape(-1, 13))
    for a, b in zip(runs, runs[1:]):
        assert np.array_equal(a, b[:len(a)])
    acc = engine.simulate_batch(params, tp.RNG_RANF, type(st).from_buffer_copy(st), 10_000)
    assert bytes(acc) == runs[0][0].tobytes()
