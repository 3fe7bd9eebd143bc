"""RANF streams whose state holds values outside [0, 1e9) (seeds past the
modulus), in numpy, by the rule the engine keeps for them: rounds in closed
form, whole segments of 2048 rounds each from one jump straight from round 0 by
the lowest binary digit of their number and ordinary jumps from there."""
import numpy as np

MOD, LATE = 10**9, 2048
M32, M64 = 2**32 - 1, 2**64 - 1


def odd(state):
    return any(not 0 <= x < MOD for x in list(state.numbers)[1:])


def _poly_mul(a, b):
    prod = [0] * 109
    for i, x in enumerate(a):
        for j, y in enumerate(b):
            prod[i + j] += x * y
    for d in range(108, 54, -1):  # x^55 = 1 - x^31
        prod[d - 55] += prod[d]
        prod[d - 24] -= prod[d]
    return [x % MOD for x in prod[:55]]


def jump_poly(rounds):
    r, base, n = [1] + [0] * 54, [0, 1] + [0] * 53, 55 * rounds
    while n:
        if n & 1:
            r = _poly_mul(r, base)
        base, n = _poly_mul(base, base), n >> 1
    return r


def next_round(x):
    """x: uint32 (55, streams), X[1..55] in the first axis."""
    def sub(a, b):
        t = a - b
        return np.minimum(t, t + np.uint32(MOD))
    zero = np.zeros_like(x[:1])
    b = np.concatenate([x[31:55], x[0:31]])
    c = np.concatenate([np.repeat(zero, 24, 0), x[31:55], x[0:7]])
    d = np.concatenate([np.repeat(zero, 48, 0), x[31:38]])
    v = sub(x, b) + sub(c, d)
    return np.minimum(v, v - np.uint32(MOD))


def jump(x, poly):
    """x: uint32 (55,)."""
    y = [int(v) for v in x] + [int(v) for v in next_round(x.reshape(55, 1))[:, 0]]
    out = []
    for i in range(55):
        acc = 0
        for k in range(55):  # groups of 16 products in 64 bits
            acc = (acc + poly[k] * y[i + k]) & M64
            if k % 16 == 15 or k == 54:
                acc %= MOD
        out.append(acc)
    return np.array(out, np.uint32)


def segment_starts(x, segments):
    """Round LATE * s of the stream for s < segments."""
    single, starts = {}, [x]
    for s in range(1, segments):
        low = s & -s
        if low not in single:
            single[low] = (jump(x, jump_poly(LATE * low)), jump_poly(LATE * low))
        rest, bit, y = s ^ low, low << 1, single[low][0]
        while rest:
            if rest & bit:
                if bit not in single:
                    single[bit] = (jump(x, jump_poly(LATE * bit)), jump_poly(LATE * bit))
                y = jump(y, single[bit][1])
                rest ^= bit
            bit <<= 1
        starts.append(y)
    return np.stack(starts, 1)


def values(state, n):
    """The next n values of the stream (int32), as the engine draws them."""
    first = 55 - state.index
    segments = -(-(first + n) // (55 * LATE))
    x = segment_starts(np.array(list(state.numbers)[1:], np.int64).astype(np.uint32), segments)
    rounds = min(LATE, -(-(first + n) // 55))
    out = np.empty((segments, rounds, 55), np.uint32)
    for r in range(rounds):
        out[:, r] = x[::-1].T  # a round is handed out backwards
        x = next_round(x)
    return out.reshape(-1)[first:first + n].view(np.int32)
