"""faster-evgen with skip-ahead seeding from RANF states seeded past the
modulus: runs of 2^20 events or more are walked on the device, on the values
that every entry point draws from such a state (ranf_odd)."""
import numpy as np
import pytest

import ranf_odd
import trois_photons as tp

pytestmark = pytest.mark.gpu

RUNS = (1 << 20, 3_000_001, 20_000_000)


@pytest.fixture(scope="module")
def engine():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        yield e


def odd_state(seed, taken):
    while not ranf_odd.odd(tp.rng_state(tp.RNG_RANF, seed)):
        seed += 123456
    st = tp.rng_state(tp.RNG_RANF, seed)
    tp.rng_skip(tp.RNG_RANF, st, taken)
    return st


def events(state, n):
    """The photons' unit-disc points and other uniforms of n events (evgen.rs:143-173, 221-249)."""
    q0 = 55 - state.index
    u = ranf_odd.values(state, 20 * n) * 1e-9
    q = q0

    def take(k):  # random_array::<k> (ranf.rs:78-102)
        nonlocal q
        if 55 - q % 55 < k:
            q += 55 - q % 55
        q += k
        return u[q - q0 - k:q - q0][::-1]
    r9, xy = np.empty((n, 9)), np.empty((n, 3, 2))
    for e in range(n):
        r9[e] = take(9)
        r6 = 2 * take(6) - 1
        for i in range(3):
            x, y = r6[i], r6[3 + i]
            while x * x + y * y > 1:
                x, y = 2 * take(2) - 1
            xy[e, i] = x, y
    return r9, xy


def selected(cfg, r9, xy):
    """Which events pass the cuts (evgen.rs:89-118, evcut.rs:42-96)."""
    ct, en = 2 * r9[:, :3] - 1, -np.log(r9[:, 3:6] * r9[:, 6:] + 2.0**-1022)
    q = np.concatenate([xy / np.linalg.norm(xy, axis=2, keepdims=True) * np.sqrt(1 - ct**2)[..., None], ct[..., None]], 2)
    q = q * en[..., None]
    r, m = q.sum(1)[:, None], en.sum(1)[:, None]
    rn2 = m**2 - (r**2).sum(2)
    rq = (q * r).sum(2)
    alpha, b = cfg.e_total / rn2, rq / (np.sqrt(rn2) + m) - en
    E = alpha * (m * en - rq)
    p = alpha[..., None] * (np.sqrt(rn2)[..., None] * q + b[..., None] * r)
    ok = ~(E.min(1) < cfg.e_min) & ~(np.abs(p[:, :, 0]) > cfg.cut_beam * E).any(1)
    for i, j in ((0, 1), (0, 2), (1, 2)):
        ok &= ~((p[:, i] * p[:, j]).sum(1) > cfg.cut_pp * E[:, i] * E[:, j])
    return ok


@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_F32])
@pytest.mark.parametrize("seed, taken", [(1_000_987_648, 0), (1_500_000_000, 17)])
def test_runs_walk_the_odd_stream_on_the_device(engine, valeurs, seed, taken, prec):
    cfg = tp.Configuration.load(valeurs)
    st = odd_state(seed, taken)
    before = bytes(st)
    # (one normalisation of the weights for all)
    params = tp.params_from_config(cfg, precision=prec, faster_evgen=True)
    runs = []
    for n in RUNS:
        print(f"faster-evgen run of an odd state, seed {st.seed} precision {prec} N={n}", flush=True)
        per, _, stats = engine.run(params, tp.RNG_RANF, tp.SEED_SKIPAHEAD, st, n)
        assert stats.host_walk_chunks == 0
        runs.append(per)
    assert bytes(st) == before
    # jump seeding's batch 0 runs on the caller's state: the same events
    runs.append(engine.run(params, tp.RNG_RANF, tp.SEED_JUMP, st, 10_000)[0])
    for per in runs[1:]:
        k = min(len(runs[0]) - 1, len(per) - 1) or 1  # whole batches
        a, b = runs[0][:k], per[:k]
        assert np.array_equal(a["selected_events"], b["selected_events"])
        if prec == tp.PREC_F32:  # sums in event order: the same bits
            assert a.tobytes() == b.tobytes()
            continue
        for name in ("spm2", "vars", "sigma", "variance"):
            # 10 000 terms added in another order; the interference sums cancel
            scale = np.sqrt(10_000 * b["vars"]) if name == "spm2" else np.abs(b[name])
            ok = np.abs(a[name] - b[name]) <= 10_000 * 2.0**-52 * scale
            assert np.all(ok | (np.isnan(a[name]) & np.isnan(b[name]))), name
    if prec == tp.PREC_F64:
        # the stream itself: batches 1 and 2 (batch 0 starts among the values
        # outside [0, 1e9), whose logarithms are no number)
        with np.errstate(all="ignore"):
            ok = selected(cfg, *events(st, 30_000))
        assert np.array_equal(ok.reshape(3, -1).sum(1)[1:], runs[0]["selected_events"][1:3])
