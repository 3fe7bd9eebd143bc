"""The closed-form helicity sums of the f64 event loop (tp_helicity.h, built
for the host): no further from the spinor amplitudes in long double than the
oracle, which keeps the reference's order of operations; the spinor of a photon
along -Z; and energies far from the shipped configuration's."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def helicity(tmp_path_factory):
    out = tmp_path_factory.mktemp("helicity") / "libhelicity.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "helicity_check.cpp"), "-o", str(out)], check=True)
    lib = C.CDLL(str(out))

    def call(name, e, p, g):
        p = np.ascontiguousarray(p, np.float64)
        m = np.zeros((len(p), 5))
        fn = getattr(lib, name)
        fn.argtypes = [C.c_double] * 4 + [C.c_long, C.c_void_p, C.c_void_p]
        fn(e, *g, len(p), p.ctypes.data, m.ctypes.data)
        return m
    return call


@pytest.fixture(scope="module")
def events(oracle, valeurs):
    """(e_total, couplings, momenta (n, 3, 4), oracle's sums) of 200 000 accepted events."""
    import trois_photons as tp
    P = tp.params_from_config(tp.Configuration.load(valeurs))
    u = np.random.default_rng(11).random((285_000, 12))
    p, keep, _, m, _ = oracle.events(oracle.config(valeurs), oracle.opts("xoshiro"), u)
    k = keep.astype(bool)
    return P.e_total, (P.g_a, P.g_beta_p, P.g_beta_m), p[k][:, 2:, :], m[k]


def errors(m, ref):
    """Relative errors of the three squares, and of the interference on the scale of its amplitudes."""
    scale = 2 * np.sqrt(ref[:, :1] * ref[:, 1:2])
    return np.abs(m - ref) / np.concatenate([ref[:, :3], scale, scale], 1)


def test_closed_sums_are_no_further_off_than_the_oracle(helicity, events):
    e, g, p, om = events
    ref = helicity("tp_helicity_spinors", e, p, g)
    mine, theirs = errors(helicity("tp_helicity_closed", e, p, g), ref), errors(om, ref)
    for q in (50, 99, 100):
        a, b = np.percentile(mine, q, axis=0) / EPS, np.percentile(theirs, q, axis=0) / EPS
        print(f"percentile {q}: closed {a.round(2)} eps, oracle {b.round(2)} eps")
        assert np.all(a <= b)


def test_photon_along_minus_z(helicity, events):
    """E + Z = 0 takes the spinor (0, sqrt(2E)), E + Z < 0 gives NaN (spinor.rs:40-44)."""
    e, g, _, _ = events
    h = e / 2
    p = np.array([[[0.5 * h, 0.3 * h, 0.4 * h, 0.], [-0.5 * h, -0.3 * h, 0.3 * h, 0.], [0., 0., -0.7 * h, 0.7 * h]]] * 3)
    p[:, :2, 3] = np.linalg.norm(p[:, :2, :3], axis=2)
    p = p[np.arange(3)[:, None], [[0, 1, 2], [2, 0, 1], [1, 2, 0]]]
    m = helicity("tp_helicity_closed", e, p, g)
    assert np.all(errors(m, helicity("tp_helicity_spinors", e, p, g)) <= 64 * EPS)  # about 60 roundings, in no special place
    p[p[..., 2] < 0, 2] *= 1 + 2 * EPS
    assert np.isnan(helicity("tp_helicity_closed", e, p, g)).all()


@pytest.mark.parametrize("k", [-90, -7, 7, 90])
def test_energy_unit(helicity, events, k):
    """Momenta and e_total times 2^k give the sums times powers of two, exactly: with the factor (-RAC8) s(0,1) of
    every amplitude, sum |A|^2 goes as energy^-2, the interference as energy^4 and the other two as energy^10."""
    e, g, p, _ = events
    p, f = p[:500], 2.0 ** k
    far = helicity("tp_helicity_closed", e * f, p * f, g)
    assert np.array_equal(far, helicity("tp_helicity_closed", e, p, g) * np.exp2(k * np.array([-2, 10, 10, 4, 4])))
