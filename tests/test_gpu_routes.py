"""GPU checks of the forms a right-hand side takes by size.  Small grids run
single-wavefront work-groups, helper wavefronts in the z pass, the TT components
side by side and the means inside the update; large ones 256 lanes a work-group,
the components in turn and the means in a launch of their own.  The single grids
of test_gpu_deriv.py are all small: here they are checked against the oracle
with the filter and on boxes of unequal spacing, and ensembles of them, large
enough for the other forms, must give the single grids' values bit for bit."""
import ctypes

import numpy as np
import pytest

from tests.states import BOX_CONFIG, blocks, make_state, rel_l2

pytestmark = pytest.mark.gpu

KINDS = {"scalar": (False, False), "gw": (True, False), "gw fp32": (True, True)}


def _white(shape, seed, gw, bounds=BOX_CONFIG, a=1.3):
    rng = np.random.default_rng(seed)
    b = blocks(shape)
    y = make_state(shape, bounds=bounds, seed=seed, gw=gw, a=a)
    for name in ("phi", "dphi", "psi", "dpsi"):
        y[b[name]] += 1e-2 * rng.standard_normal(y[b[name]].size)
    return y


# (shape, realizations): every length on every axis, an odd number of
# realizations with at least 512 work-groups of 256 lanes in the z and the
# derivative passes and 300000 modes in the TT pass; 16^3 x 2049 also has the
# 256 MB of fields from which the means are a launch of their own
ENSEMBLES = [((4, 4, 4), 6251), ((8, 8, 8), 939), ((16, 16, 16), 2049),
             ((32, 32, 32), 65), ((64, 64, 64), 9), ((128, 4, 128), 65),
             ((4, 128, 4), 513), ((256, 4, 4), 513), ((4, 256, 4), 513),
             ((4, 4, 256), 513), ((512, 4, 4), 513), ((4, 512, 4), 513),
             ((4, 4, 512), 257)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape,nreal", ENSEMBLES)
def test_large_ensemble_equals_single_grids(shape, nreal, kind):
    import instaheat_amd as ih
    gw, fp32 = KINDS[kind]
    L = ih.lib()
    p = ih.make_params(shape, BOX_CONFIG, 0.7, gw, True, 8, fp32)
    h = ctypes.c_void_p()
    ih._check(L.ihg_create_ensemble(ctypes.byref(p), nreal, ctypes.byref(h)))
    ens = (ctypes.c_long * 2)()
    ih._check(L.ihg_ensemble(h, ens))
    n = nreal * ens[1]
    pool = [_white(shape, 50 + s, gw) for s in range(3)]
    full = np.zeros((nreal, ens[1]))
    for s in range(3):
        full[s::3, :pool[s].size] = pool[s]
    ntot = pool[0].size
    full[:, ntot - 1] = 1.0 + 0.5 * np.arange(nreal) / nreal  # every one its own

    def dev():
        q = ctypes.c_void_p()
        ih._check(L.ihg_malloc(h, ctypes.byref(q), n))
        return q

    def host(q):
        out = np.empty((nreal, ens[1]))
        ih._check(L.ihg_download(h, out.ctypes.data_as(ctypes.c_void_p), q, n))
        return out

    f, r = dev(), dev()
    g = ih.Gpu(shape, bounds=BOX_CONFIG, mass=0.7, gw=gw, bins=8, gw_fp32=fp32)
    for flags in (0, 1):
        print(f"{shape} x {nreal}, {kind}, flags {flags}", flush=True)
        ih._check(L.ihg_upload(h, f, full.ctypes.data_as(ctypes.c_void_p), n))
        ih._check(L.ihg_mk_rhs_ensemble(h, 0.0, f, r, flags))
        got, filtered = host(r), host(f)
        for q in (0, 1, nreal // 2, nreal - 2, nreal - 1):
            d, s = g.to_device(full[q, :ntot]), g.alloc(ntot)
            g.mk_rhs(d, s, flags=flags)
            assert np.array_equal(got[q, :ntot], s.download()), (flags, q)
            assert np.array_equal(filtered[q, :ntot], d.download()), (flags, q)
    g.close()
    L.ihg_free(h, f)
    L.ihg_free(h, r)
    L.ihg_destroy(h)


def _against_oracle(ih, orc, shape, bounds, gw, fp32, flags):
    """White fluctuations up to the corner of the grid, h = 0 (its slopes are
    the source alone): tolerances as in test_gpu_deriv.py."""
    B = blocks(shape)
    y = _white(shape, sum(shape), False, bounds)
    g = ih.Gpu(shape, bounds=bounds, mass=0.7, gw=gw, bins=4, gw_fp32=fp32)
    d, r = g.to_device(y), g.alloc(g.Ntot)
    g.mk_rhs(d, r, flags=flags)
    got, filtered = r.download(), d.download()
    g.close()
    fo = y.copy()
    ref = orc.Oracle(*shape, bounds=bounds, mass=0.7, gw=gw, bins=4).mk_rhs(
        fo, filter=flags, output=0, field=fo)
    assert rel_l2(filtered, fo) < 1e-12
    for name in ("phi", "dphi", "psi", "dpsi", "a") + (("dh1", "dh2") if gw else ()):
        tol = 2e-6 if fp32 and name[:2] == "dh" else 1e-11
        assert rel_l2(got[B[name]], ref[B[name]]) < tol, name


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [
    (4, 4, 4), (8, 8, 8), (16, 4, 16), (32, 8, 32), (64, 4, 64), (128, 4, 128),
    (256, 4, 256), (512, 8, 4), (4, 8, 512), (4, 512, 8)])
def test_filtered_rhs_at_every_length(oracle_mod, shape, kind):
    import instaheat_amd as ih
    print(f"filtered mk_rhs {shape} {kind}", flush=True)
    _against_oracle(ih, oracle_mod, shape, BOX_CONFIG, *KINDS[kind], 1)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("lengths", [(1, 2, 0.5), (0.5, 1, 2), (2, 0.5, 1),
                                     (2, 1, 0.5), (1, 0.5, 2), (0.5, 2, 1)])
def test_source_on_unequal_spacings(oracle_mod, lengths, fp32):
    """Boxes whose smallest Nyquist wave number is that of x, y and z: each of
    the three products that can be subtracted from the others."""
    import instaheat_amd as ih
    bounds = tuple((0.0, 2 * np.pi / 0.1 * q) for q in lengths)
    for shape in ((16, 16, 16), (64, 64, 64)):
        print(f"mk_rhs {shape} lengths {lengths} fp32 {fp32}", flush=True)
        _against_oracle(ih, oracle_mod, shape, bounds, True, fp32, 0)
