"""The per-operator right-hand side with several variables a launch: every
output and every boundary derivative against the CPU oracle, on grids whose
axes run the sweep kernels, the general kernels (lines no chunk length cuts:
variable after variable), and both.

Bar: as for the same operators one variable at a time -- FP64, norm-wise
relative difference <= 1e-12 (the pointwise arithmetic is the oracle's, the
line solves differ by rounding)."""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel

TOL = 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(16, 16, 16), (17, 23, 32), (33, 18, 12), (130, 31, 24)])
@pytest.mark.parametrize("bc", [[[10, 10, 10], [10, 10, 10]], [[45, 10, 45], [45, 10, 45]]])
def test_viscous_rhs(oracle, dims, bc):
    import compact_schemes_amd as cs
    from compact_schemes_amd import workloads as wl
    lmx = dims[0] * dims[1] * dims[2]
    st = wl.flow_state(dims, seed=4, noise=1e-2, width=3.0)
    ctx = oracle.Context(dims, bc)
    num = cs.Numerics(dims, bc)
    num.deriv_setup()
    ph = cs.Physics(dims, True, st["umf"])
    q = dev(st["qa"])
    de, p = dev(np.zeros(5 * lmx)), dev(np.zeros(lmx))
    g = {k: dev(st[k]) for k in ("xim", "etm", "zem", "yaco", "ssk")}
    de_o, p_o = oracle.primitives(st["qa"], lmx)
    cs.primitives(dims, q, de, p)
    case(f"viscous dims={dims} bc={bc}")
    ph.calc_viscous_shear_stress(num, de, g["ssk"], g["xim"], g["etm"], g["zem"], g["yaco"])
    ctx.calc_viscous(de_o, st["ssk"], st["xim"], st["etm"], st["zem"], st["yaco"])
    S, H = ph.buffers()
    assert nrel(host(S), ctx.stress()) < TOL and nrel(host(H), ctx.heat()) < TOL
    assert nrel(host(de), de_o) < TOL
    case(f"fluxes dims={dims} bc={bc}")
    ph.calc_fluxes(num, q, p, de, g["xim"], g["etm"], g["zem"])
    ctx.calc_fluxes(1, st["qa"], p_o, de_o, st["xim"], st["etm"], st["zem"], st["umf"])
    for m in range(5):
        assert nrel(host(de)[m * lmx:(m + 1) * lmx], de_o[m * lmx:(m + 1) * lmx]) < TOL
    for a in range(3):
        assert nrel(host(num.buffers(a)[0]), ctx.drva(a)) < TOL
