"""Lines per workgroup do not change a result: the default of the y/z sweeps
(16, 32 along z, 64 for the one-variable filter) against 8, on faces that
those numbers do not divide and lines of 2 to 16 chunks of 16 points.

Bar: equal bits -- a line's operations and their order are the same."""
import pytest
import torch

from gpu_util import case, dev


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(19, 16, 32), (17, 48, 256), (33, 112, 48)])
@pytest.mark.parametrize("nbc", [[[10] * 3] * 2, [[45] * 3] * 2], ids=["closure", "periodic"])
@pytest.mark.parametrize("viscous", [True, False])
def test_lines_per_workgroup(dims, nbc, viscous):
    from compact_schemes_amd import workloads as wl
    from compact_schemes_amd.fused import FusedSolver
    st = wl.flow_state(dims, seed=12, noise=1e-2, width=3.0)
    sv = FusedSolver(dims, nbc, st, viscous=viscous)
    q = dev(st["qa"])
    case(f"lines per workgroup dims={dims} nbc={nbc[0]}")
    a, b = q.clone(), q.clone()
    dt = 0.5 * sv.time_step(q)
    sv.rk4_step(a, dt=dt)
    for axis in (1, 2):
        if dims[axis] % 16 == 0 and dims[axis] >= 32:
            sv.tune(axis, 2, 8, 1)
            sv.tune_filter(axis, 1, 8, 16)
    sv.rk4_step(b, dt=dt)
    assert torch.equal(a, b)
