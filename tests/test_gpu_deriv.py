"""GPU check of the axis derivatives, the z pass with the fused source
transforms and the update against the oracle, at every line length on every
axis, from the smallest grid on (partly filled work-groups and wavefronts):
white fluctuations, so that every mode up to the corner is live, and h = 0,
so that the slopes of h are the projected source alone."""
import numpy as np
import pytest

from tests.states import BOX_CONFIG, blocks, make_state, rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 4), (4, 8, 16), (8, 4, 32), (16, 16, 8), (16, 32, 64),
          (64, 16, 4), (4, 4, 128), (4, 128, 4), (128, 4, 8), (256, 8, 4),
          (4, 256, 4), (8, 4, 256), (512, 4, 4), (4, 512, 4), (4, 4, 512),
          (64, 64, 64)]


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("gw", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_rhs_of_white_fields(oracle_mod, shape, gw, fp32):
    import instaheat_amd as ih
    if fp32 and not gw:
        pytest.skip("the FP32 source needs the source")
    rng = np.random.default_rng(sum(shape))
    b = blocks(shape)
    y = make_state(shape, seed=3, gw=False, a=1.3)
    for name in ("phi", "dphi", "psi", "dpsi"):
        y[b[name]] += 1e-2 * rng.standard_normal(y[b[name]].size)
    print(f"mk_rhs {shape} gw {gw} fp32 {fp32}", flush=True)
    g = ih.Gpu(shape, bounds=BOX_CONFIG, mass=0.7, gw=gw, filt=False, bins=4,
               gw_fp32=fp32)
    df, dr = g.to_device(y), g.alloc(g.Ntot)
    g.mk_rhs(df, dr)
    got = dr.download()
    if gw:
        grad = [g.aux(i) for i in range(3)]
    g.close()
    o = oracle_mod.Oracle(*shape, bounds=BOX_CONFIG, mass=0.7, gw=gw, filt=False, bins=4)
    ref = o.mk_rhs(y.copy())
    # the transforms' rounding of phi ~ 1 reaches the second derivative with
    # k_max^2: eps log2(L) k_max^2 against fluctuations of 1e-2 k_max^2, that
    # is 2e-16 * 9 * 1e2 = 2e-13, with a margin of 50
    for name in ("phi", "dphi", "psi", "dpsi", "a"):
        assert rel_l2(got[b[name]], ref[b[name]]) < 1e-11, name
    if gw:
        # FP32: 2^-24 per product and per transform stage, with a margin
        tol = 2e-6 if fp32 else 1e-11
        for name in ("dh1", "dh2"):
            assert rel_l2(got[b[name]], ref[b[name]]) < tol, name
        for i in range(3):
            assert rel_l2(grad[i], o.aux(i)) < (1e-6 if fp32 else 1e-11), i
