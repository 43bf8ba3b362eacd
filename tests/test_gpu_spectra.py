"""GPU check of the spectra at the edges of the histogram sum's tiles (16 bins
a work-group): bin counts below, at and above a tile, one to many."""
import numpy as np
import pytest

from tests.states import BOX_CONFIG, make_state, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1, 15, 16, 17, 100])
def test_spectra_at_tile_edges(oracle_mod, bins):
    import instaheat_amd as ih
    shape = (8, 16, 32)
    y = make_state(shape, seed=bins, gw=True)
    g = ih.Gpu(shape, bounds=BOX_CONFIG, gw=True, filt=True, bins=bins)
    df, dr = g.to_device(y), g.alloc(g.Ntot)
    print(f"output call, {bins} bins", flush=True)
    g.mk_rhs(df, dr, flags=ih.IHG_FILTER | ih.IHG_OUTPUT)
    got = g.observables()[28:]
    o = oracle_mod.Oracle(*shape, bounds=BOX_CONFIG, gw=True, filt=True, bins=bins)
    fo = y.copy()
    o.mk_rhs(fo, filter=1, output=1, field=fo)
    # a bin adds up to 8 * 16 * 17 = 2176 terms of one sign: rounding below
    # 2176 * 2^-52
    for a, b in zip(got.reshape(4, bins), o.obs()[28:].reshape(4, bins)):
        assert rel_l2(a, b) < 1e-9
        assert np.all(np.isfinite(a))
    g.close()
