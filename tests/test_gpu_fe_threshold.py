"""The shortest faster-evgen runs of each stream that the device walks:
the walk that a run takes, and closures on both sides, against the oracle."""
import pytest

import trois_photons as tp
from test_gpu_f32 import close_f32
from test_gpu_parity import acc_close

pytestmark = pytest.mark.gpu

STREAMS = {"ranf": (tp.RNG_RANF, tp.PREC_F64, 8192), "ranf-f32": (tp.RNG_RANF, tp.PREC_F32, 8192),
           "xoshiro": (tp.RNG_XOSHIRO, tp.PREC_F64, 20_000), "xoshiro-f32": (tp.RNG_XOSHIRO128, tp.PREC_F32, 8192)}


@pytest.mark.parametrize("stream", STREAMS)
def test_shortest_device_walks(oracle, oracle32, valeurs, stream):
    kind, prec, least = STREAMS[stream]
    orc, close = (oracle32, close_f32) if prec == tp.PREC_F32 else (oracle, acc_close)
    rng = stream.split("-")[0]
    params = tp.params_from_config(tp.Configuration.load(valeurs), precision=prec, faster_evgen=True)
    ocfg, opts = orc.config(valeurs), orc.opts(rng, faster_evgen=True)
    st, g = tp.rng_state(kind), orc.rng(rng)
    with tp.Engine(0) as engine:
        for n in (least - 1, least, least + 1, 2 * least + 1):
            print(f"faster-evgen {stream} n={n}", flush=True)
            a = engine.simulate_batch(params, kind, st, n).as_array()
            close(a, orc.simulate_batch(ocfg, opts, g, n).as_array(), n)
            _, _, stats = engine.run(params, kind, tp.SEED_SKIPAHEAD, tp.rng_state(kind), n)
            assert stats.host_walk_chunks == (1 if n < least else 0)
