"""The transposed sweeps on lines of any chunking -- equal and one row short,
8- and 16-point chunks, two chunks a line, x lines over 256 points -- against
the per-operator adjoint (mode 0).

Bar: 1e-12 norm-wise, as on equal chunks (the same operators, summed in
another order)."""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel

P, C = [45, 45], [10, 10]


def _solver(dims, nbc, filt):
    from compact_schemes_amd import workloads as wl
    from compact_schemes_amd.fused import FusedSolver
    st = wl.flow_state(dims, seed=33, noise=1e-2, width=3.0)
    return st, FusedSolver(dims, nbc, st, viscous=False, filt=filt)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(23, 31, 47), (37, 46, 16), (130, 39, 32), (300, 16, 23), (16, 63, 48)])
@pytest.mark.parametrize("faces", [(C, C, C), (P, P, P), (P, C, P)], ids=["closure", "periodic", "mixed"])
def test_rk4_vjp(dims, faces):
    nbc = [[f[i] for f in faces] for i in range(2)]
    st, sv = _solver(dims, nbc, True)
    rng = np.random.default_rng(9)
    q0 = dev(st["qa"])
    dt = sv.time_step(q0)
    lam = dev(rng.standard_normal(st["qa"].size))
    case(f"rk4 vjp dims={dims} nbc={nbc}")
    a1 = sv.rk4_vjp(q0, lam.clone(), dt).clone()
    g1 = sv.rhs_vjp(q0, lam).clone()
    sv.set_adjoint_mode(0)
    a0 = sv.rk4_vjp(q0, lam.clone(), dt).clone()
    g0 = sv.rhs_vjp(q0, lam).clone()
    assert nrel(host(g1), host(g0)) < 1e-12
    assert nrel(host(a1), host(a0)) < 1e-12
