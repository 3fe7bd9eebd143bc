"""RANF runs of more batches than one launch takes the streams' rounds of
(2^20): jump seeding, and one stream from a state past the modulus."""
import numpy as np
import pytest

import ranf_odd
import trois_photons as tp

pytestmark = pytest.mark.gpu

CHUNK = 1 << 20


@pytest.fixture(scope="module")
def engine():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        yield e


def close(a, b, n=10_000):
    """Selected events exactly; sums of n terms each added in another order."""
    assert a[0] == b[0]
    assert np.array_equal(np.isnan(a), np.isnan(b))
    scale = np.abs(b)
    scale[1:6], scale[11] = np.sqrt(n * b[6:11]), np.sqrt(n * b[12])  # the interference cancels
    assert np.all((np.abs(a - b) <= (n + 16) * 2.0**-52 * scale) | np.isnan(a)), (a, b)


def device_run(engine, params, seeding, st, n):
    """The run's accumulators, and the device memory it took beside them."""
    import torch
    per = torch.empty((n + 9_999) // 10_000, 13, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(0)[0]
    engine.run_device(params, tp.RNG_RANF, seeding, st, n, per.data_ptr(), None)
    engine.sync()
    taken = free - torch.cuda.mem_get_info(0)[0]
    return per, taken


def batch(per, b):
    return tp.TpAcc.from_buffer_copy(per[b].cpu().numpy())


@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_F32])
def test_jump_seeding(valeurs, prec):
    n = (2 * CHUNK + 3) * 10_000 - 77
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=prec)
    seed = 234612947
    print(f"jump-seeded run precision {prec} N={n}", flush=True)
    with tp.Engine(0) as engine:
        per, taken = device_run(engine, params, tp.SEED_JUMP, tp.rng_state(tp.RNG_RANF, seed), n)
        assert taken < 700 << 20  # 448 bytes a batch held at once
        for b in (0, 1, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK - 1, 2 * CHUNK, 2 * CHUNK + 2):
            count = min(10_000, n - 10_000 * b)
            acc = engine.simulate_batch(params, tp.RNG_RANF, tp.rng_state(tp.RNG_RANF, (seed + 123456 * b) % 2**32), count)
            if prec == tp.PREC_F32:
                assert bytes(acc) == bytes(batch(per, b)), b
            else:
                close(acc.as_array(), batch(per, b).as_array(), count)


def odd_uniforms(state, first, n):
    """Values first .. first + n of an odd stream, by ranf_odd's rule."""
    x0 = np.array(list(state.numbers)[1:], np.int64).astype(np.uint32)
    out, q = [], 55 - state.index + first
    s = q // (55 * ranf_odd.LATE)
    while len(out) == 0 or sum(map(len, out)) < q % (55 * ranf_odd.LATE) + n:
        low, x = s & -s, x0
        if s:
            x = ranf_odd.jump(x0, ranf_odd.jump_poly(ranf_odd.LATE * low))
        if s ^ low:
            x = ranf_odd.jump(x, ranf_odd.jump_poly(ranf_odd.LATE * (s ^ low)))
        x = x.reshape(55, 1)
        rounds = np.empty((ranf_odd.LATE, 55), np.uint32)
        for r in range(ranf_odd.LATE):
            rounds[r] = x[::-1, 0]
            x = ranf_odd.next_round(x)
        out.append(rounds.reshape(-1))
        s += 1
    at = q % (55 * ranf_odd.LATE)
    return np.concatenate(out)[at:at + n].view(np.int32) * 1e-9


def test_one_odd_stream(engine, valeurs):
    seed, n = 1_500_000_000, (CHUNK + 3) * 10_000 - 77
    while not ranf_odd.odd(tp.rng_state(tp.RNG_RANF, seed)):
        seed += 123456
    st = tp.rng_state(tp.RNG_RANF, seed)
    tp.rng_skip(tp.RNG_RANF, st, 17)
    params = tp.params_from_config(tp.Configuration.load(valeurs))
    contribs = np.array(list(params.sigma_contribs))
    print(f"one stream past the modulus, seed {seed} N={n}", flush=True)
    per, _ = device_run(engine, params, tp.SEED_SKIPAHEAD, st, n)
    for b in (0, CHUNK - 1, CHUNK, CHUNK + 2):
        count = min(10_000, n - 10_000 * b)
        if b == 0:
            acc = engine.simulate_batch(params, tp.RNG_RANF, type(st).from_buffer_copy(st), count)
            close(acc.as_array(), batch(per, b).as_array())
            continue
        u = odd_uniforms(st, 120_000 * b, 12 * count).reshape(-1, 12)
        m = engine.adjoint(params, count, tp.PREC_F64, u=u)[0] / params.ev_weight
        w = m @ contribs
        ref = np.concatenate([[np.count_nonzero(m[:, 0])], m.sum(0), (m * m).sum(0), [w.sum(), (w * w).sum()]])
        a = batch(per, b).as_array()
        # the adjoint's sums are another closed form: their own rounding beside the order's (events
        # near a collinear limit carry some 1e-10 of it)
        scale = np.abs(ref)
        scale[1:6], scale[11] = np.sqrt(count * ref[6:11]), np.sqrt(count * ref[12])
        assert a[0] == ref[0] and np.all(np.abs(a - ref) <= 1e-9 * scale), (b, a, ref)


# the last batch's seed is the last in [0, 1e9), the first past it, or one past 2^31; and the most batches that all lie inside
@pytest.mark.parametrize("prec", [tp.PREC_F64, tp.PREC_MIXED, tp.PREC_F32])
@pytest.mark.parametrize("first, batches", [(999_999_999 - 5 * 123456, 6), (10**9 - 5 * 123456, 6), (999_999_999 - 5 * 123456, 7),
                                            (2**31 - 3 * 123456, 6), (63_999, 8101), (64_000, 8101), (0, 8102)])
def test_seeds_at_the_modulus(engine, valeurs, first, batches, prec):
    """Batches' seeds first + 123456 b: each batch is the closure on its state."""
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=prec)
    print(f"jump-seeded run precision {prec} seed {first} batches {batches}", flush=True)
    per, _, _ = engine.run(params, tp.RNG_RANF, tp.SEED_JUMP, tp.rng_state(tp.RNG_RANF, first), 10_000 * batches)
    for b in sorted({0, *range(batches - 6, batches)}):
        acc = engine.simulate_batch(params, tp.RNG_RANF, tp.rng_state(tp.RNG_RANF, (first + 123456 * b) % 2**32), 10_000)
        got = tp.TpAcc.from_buffer_copy(per[b])
        if prec == tp.PREC_F32:
            assert bytes(acc) == bytes(got), b
        else:
            close(acc.as_array(), got.as_array())
