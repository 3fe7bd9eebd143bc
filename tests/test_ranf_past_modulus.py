"""RANF states seeded past the modulus (1e9 and more, as faster-threading's long
runs do) hold values outside [0, 1e9): skips of such states keep the values
that one polynomial jump from the state gives."""
import hashlib

import trois_photons as tp


def test_skips_of_states_past_the_modulus_are_one_jump():
    h, past = hashlib.sha1(), 0
    for b in range(0, 3000, 7):
        for n in (1, 54, 55, 56, 1200, 60000, 120000, 1234567):
            st = tp.rng_state(tp.RNG_RANF, 990_000_000 + 123456 * b)
            past += any(not 0 <= x < 10**9 for x in list(st.numbers)[1:])
            tp.rng_skip(tp.RNG_RANF, st, n)
            h.update(bytes(st))
    assert past > 100
    # of the same states with x^(55 rounds) applied term by term
    assert h.hexdigest() == "e237540d8b8b698193feffdd80de8cf55e28cb71"
