"""The all-f32 sums of xoshiro128+ calls add a tile's accepted events side by
side, in whole groups of 16: calls at the edges of groups and tiles of 128,
with nearly all tiles partly filled, with few and with no accepted events."""
import pytest

import trois_photons as tp
from test_gpu_f32 import close_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emin", ["4.559e0", "26.e0", "30.35e0"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 385, 513, 1025])
def test_f32_slot_sums_at_tile_edges_match_oracle(tmp_path, oracle32, valeurs, n, emin):
    print(f"f32 slots n={n} emin={emin}", flush=True)
    path = tmp_path / "valeurs"
    with open(valeurs) as f:
        path.write_text(f.read().replace("4.559e0", emin))
    params = tp.params_from_config(tp.Configuration.load(str(path)), precision=tp.PREC_F32)
    st, g = tp.rng_state(tp.RNG_XOSHIRO128), oracle32.rng("xoshiro")
    with tp.Engine(0) as engine:
        for _ in range(3):
            acc = engine.simulate_batch(params, tp.RNG_XOSHIRO128, st, n)
            ref = oracle32.simulate_batch(oracle32.config(str(path)), oracle32.opts("xoshiro"), g, n)
            close_f32(acc.as_array(), ref.as_array(), n)
            assert list(st.s) == list(g.xs32)
