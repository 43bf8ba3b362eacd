"""GPU check that the autotuner times the passes that the right-hand side of
its context runs: the numbers of arrays show in the times."""
import ctypes

import pytest

from tests.states import BOX_CONFIG

pytestmark = pytest.mark.gpu


def _times(ih, **kw):
    """fastest candidate along y and along x, ms"""
    g = ih.Gpu((128, 128, 128), bounds=BOX_CONFIG, bins=8, **kw)
    L, n, ms = ih.lib(), (ctypes.c_int * 2)(), (ctypes.c_float * 16)()
    ih._check(L.ihg_fft_candidates(g.ctx, n, None))
    ih._check(L.ihg_autotune(g.ctx, 10, None, ms, 16))
    g.close()
    return min(ms[:n[0]]), min(ms[n[0]:n[0] + n[1]])


def test_autotune_times_the_passes_of_the_rhs():
    import instaheat_amd as ih
    # the source's five components along x, one array along y; the filter's
    # four along y, one along x: bytes 5 : 1 and 4 : 1, asked for is 2 : 1
    y, x = _times(ih, gw=True, filt=False)
    print("GW, no filter", y, x, flush=True)
    assert x > 2 * y
    y4, x1 = _times(ih, gw=False, filt=True)
    print("filter, no GW", y4, x1, flush=True)
    assert y4 > 2 * x1
    # half the bytes with the FP32 source
    x32 = _times(ih, gw=True, filt=False, gw_fp32=True)[1]
    print("FP32 GW", x32, flush=True)
    assert x32 < 0.8 * x
