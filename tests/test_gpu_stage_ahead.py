"""GPU check of the stage sums that are started ahead (ihg_dp853_stage_ahead,
ihg_gsl_stage_ahead): every stage input equals the plain stage sum's, on
arrays below and above the streaming size, with and without the tensor
blocks."""
import ctypes

import numpy as np
import pytest

from tests.states import BOX_CONFIG

pytestmark = pytest.mark.gpu


def _ptrs(ks):
    return (ctypes.c_void_p * len(ks))(*[k.ptr for k in ks])


@pytest.mark.parametrize("method,stages", [(None, 12), (3, 13), (1, 6), (2, 6)])
@pytest.mark.parametrize("shape,gw", [((4, 4, 8), False), ((8, 4, 16), True),
                                      ((256, 256, 128), True)])
def test_stage_ahead_equals_stage(method, stages, shape, gw):
    import instaheat_amd as ih
    if shape[0] == 256 and method in (1, 2):
        pytest.skip("the 4(5) pairs take the plain sums: no streaming variant")
    L = ih.lib()
    g = ih.Gpu(shape, bounds=BOX_CONFIG, gw=gw)
    n = g.Ntot

    def state(seed):
        d = g.alloc(n)
        ih._check(L.ihg_init_gaussian(g.ctx, d.ptr, seed, 1e-3, 0.3 * seed, -0.7, 1.0 + seed, 1.0))
        if gw:  # the tensor blocks too: a copy of the first block
            ih._check(L.ihg_stream_copy(g.ctx, d.ptr + 8 * 4 * g.N, d.ptr, g.N))
        return d

    y, out1, out2 = state(1), g.alloc(n), g.alloc(n)
    slopes = [state(2 + j) for j in range(stages)]
    plain, ahead = [slopes[0]], [slopes[0]] + [g.alloc(n) for _ in range(stages - 1)]
    for s in range(2, stages + 1):
        print(f"stage {s} of {stages}, {shape}", flush=True)
        kp = _ptrs((plain + [slopes[0]] * stages)[:stages])
        if method is None:
            ih._check(L.ihg_dp853_stage(g.ctx, s, 0.01, y.ptr, kp, out1.ptr))
            ih._check(L.ihg_dp853_stage_ahead(g.ctx, s, 0.01, y.ptr, _ptrs(ahead), out2.ptr))
        else:
            ih._check(L.ihg_gsl_stage(g.ctx, method, s, 0.01, y.ptr, kp, out1.ptr))
            ih._check(L.ihg_gsl_stage_ahead(g.ctx, method, s, 0.01, y.ptr, _ptrs(ahead), out2.ptr))
        d = np.zeros(2)
        ih._check(L.ihg_diff_norms(g.ctx, out1.ptr, out2.ptr, out1.ptr, y.ptr, n,
                                   d.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        assert d[0] == 0.0 and d[1] > 0.0, (s, d)
        plain.append(slopes[s - 1])
        ih._check(L.ihg_stream_copy(g.ctx, ahead[s - 1].ptr, slopes[s - 1].ptr, n))
    for a in [y, out1, out2] + slopes + ahead:
        del a
    g.close()
