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
