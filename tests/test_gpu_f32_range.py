"""The all-f32 event loop's division and square root without range scaling, and
runs whose energies take them out of the range where those are the plain ones."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import trois_photons as tp
from conftest import PKG

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


def test_division_and_root_are_the_plain_ones(tmp_path):
    """Bit for bit, for divisors and quotients 2^-100 .. 2^100 and roots of 2^-96 and more, and for 0, inf and NaN."""
    import torch
    out = tmp_path / "libf32ops.so"
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "f32ops_check.hip"), "-o", str(out)], check=True, capture_output=True)
    lib = ctypes.CDLL(str(out))
    r, n = np.random.default_rng(1), 1 << 22

    def values(exponents):
        bits = (exponents.astype(np.uint32) + np.uint32(127) << 23) | r.integers(0, 1 << 23, n, dtype=np.uint32)
        return (bits | r.integers(0, 2, n, dtype=np.uint32) << 31).view(np.float32)
    eb = r.integers(-100, 100, n)
    a, b = values(np.clip(eb + r.integers(-100, 100, n), -102, 126)), values(eb)
    special = np.array([0., -0., np.inf, -np.inf, np.nan, 1., 2., 4., 9., 2.0**-96, -1.], np.float32)
    k = len(special)
    a[:k * k], b[:k * k] = np.repeat(special, k), np.tile(special, k)
    ta, tb = (torch.from_numpy(x).to("cuda:0") for x in (a, b))
    res = torch.empty(4, n, dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    print(f"f32 division and root, {n} pairs", flush=True)
    assert lib.f32ops_run(*(ctypes.c_void_p(x.data_ptr()) for x in (ta, tb)), ctypes.c_int64(n), ctypes.c_void_p(res.data_ptr())) == 0
    q, q0, s, s0 = res.cpu().numpy()
    for got, want, on in ((q, q0, slice(None)), (s, s0, (np.abs(a) >= 2.0**-96) | ~(np.abs(a) > 0))):
        got, want = got[on], want[on]
        nan = np.isnan(want)
        assert np.array_equal(nan, np.isnan(got))
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


# e_total times 1e-6 and 1e-5: |D|^2 below f32's normal range; 1e-4: sums still normal; 1: plain kernels; 100 and
# 1000: |D|^2 up to 2^105 and past 2^126
@pytest.mark.parametrize("scale", [1e-6, 1e-5, 1e-4, 1.0, 100.0, 1000.0])
@pytest.mark.parametrize("rng,faster", [("ranf", False), ("xoshiro", False), ("ranf", True), ("xoshiro", True)])
def test_energies_near_the_ends_of_the_range(oracle32, valeurs, tmp_path, rng, faster, scale):
    lines = open(valeurs).read().splitlines()
    for at in (1, 4):  # e_total and the least photon energy
        number, rest = lines[at].split(None, 1)
        lines[at] = f"{float(number) * scale:.12f} {rest}"
    path = str(tmp_path / "valeurs")
    open(path, "w").write("\n".join(lines) + "\n")
    n, kind = 20_000, tp.RNG_RANF if rng == "ranf" else tp.RNG_XOSHIRO128
    params = tp.params_from_config(tp.Configuration.load(path).with_events(n), precision=tp.PREC_F32, faster_evgen=faster)
    _, oper = oracle32.run(oracle32.config(path, n), oracle32.opts(rng, threads=2, faster_evgen=faster), per_batch=True)
    print(f"f32 rng={rng} faster={faster} e_total={params.e_total}", flush=True)
    with tp.Engine(0) as engine:
        per, _, _ = engine.run(params, kind, tp.SEED_SKIPAHEAD, tp.rng_state(kind), n)
        # event-order sums: the same bits where a wavefront has a whole batch
        whole, _, _ = engine.run(params, kind, tp.SEED_SKIPAHEAD, tp.rng_state(kind), 100_000_000)
    assert per.tobytes() == whole[:2].tobytes()
    for b in range(2):
        got, want = tp.TpAcc.from_buffer_copy(per[b]).as_array(), oper[b].as_array()
        assert got[0] == want[0]
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)), (got, want)
        fin = np.isfinite(want)
        size = np.abs(want)
        if np.isfinite(want[10]) and want[10] > 0:  # (its squares underflow at the lowest energies)
            size[5] = np.sqrt(want[10] * want[0])  # the imaginary interference cancels
        # the f32 suite's bound for differences of an ulp in sinf, cosf and logf; 10 000 subnormal steps below 2^-126
        assert np.all(np.abs(got[fin] - want[fin]) <= 2e-5 * size[fin] + 10_000 * 2.0**-149), (got, want)
