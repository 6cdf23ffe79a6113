"""Launch shapes on uneven lines: a solver takes back the shape it reports,
its other admissible shapes give the default's results to rounding, and the
autotuner's record on such lines is what a solver created later runs.

Lengths: 47 and 154 (16-point chunks one row short), 248 (the same, divisible
by 8), 60 (8-point chunks only), 288 (16-point chunks, more than 256 points),
300 (x), 17 (no chunk one row short: tiles and the line solver's filter).

Bars: the same bits after get and set; 1e-13 norm-wise on the right-hand side
and 5e-12 on the filter's change between shapes, as on equal chunks."""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel
from test_gpu_fused import CL, PER, _state

DIMS = [(20, 47, 154), (61, 248, 17), (300, 60, 48), (23, 288, 31)]


@pytest.fixture
def tune():
    from compact_schemes_amd import tune as t
    t.clear()
    yield t
    t.clear()


def _filtered(sv, q):
    """the change the closing filter of a step makes (a step of dt -> 0 is the filter alone)"""
    f = q.clone()
    sv.rk4_step(f, dt=1e-300)
    return host(f) - host(q)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("nbc", [CL, PER], ids=["closure", "periodic"])
def test_solver_takes_back_the_shape_it_reports(tune, dims, nbc):
    from compact_schemes_amd.fused import FusedSolver
    st = _state(dims, seed=12)
    q = dev(st["qa"])
    sv = FusedSolver(dims, nbc, st)
    case(f"shape round trip dims={dims} nbc={nbc[0]}")
    d0, f0 = host(sv.rhs(q)).copy(), _filtered(sv, q)
    for a in range(3):
        shape, fshape = sv.get_tune(a)
        sv.tune(a, *shape)
        assert sv.get_tune(a)[0] == shape
        others = [(0, 8, 1)] + ([(2, 8, 0)] if shape[0] == 2 else [])
        for other in others:
            sv.tune(a, *other)
            assert nrel(host(sv.rhs(q)), d0) < 1e-13, (a, other)
        sv.tune(a, *shape)
        if fshape == (0, 0, 0):
            continue
        sv.tune_filter(a, *fshape)
        for other in [(1, 8, fshape[2]), (5, 16, fshape[2])] + ([(1, 16, 8)] if dims[a] <= 256 else []):
            sv.tune_filter(a, *other)
            assert sv.get_tune(a)[1] == other
            assert nrel(_filtered(sv, q), f0) < 5e-12, (a, other)
        sv.tune_filter(a, *fshape)
        assert sv.get_tune(a) == (shape, fshape)
    assert np.array_equal(host(sv.rhs(q)), d0)
    assert np.array_equal(_filtered(sv, q), f0)


@pytest.mark.gpu
def test_autotune_on_uneven_lines_records_and_reuses(tune):
    from compact_schemes_amd.fused import FusedSolver
    dims = (20, 47, 154)
    st = _state(dims, seed=13)
    q = dev(st["qa"])
    default = FusedSolver(dims, PER, st)
    sv = FusedSolver(dims, PER, st)
    case("autotune on uneven lines")
    sv.autotune(q, reps=2)
    for a in range(3):
        shape, fshape = sv.get_tune(a)
        assert tune.get_sweep(a, dims[a], 1, 0) == shape
        assert tune.get_filter_sweep(a, dims[a], 1) == (fshape if fshape != (0, 0, 0) else None)
    # entries by hand: applied where the lines take them, else the default stays
    tune.set_sweep(1, 47, 1, 0, 2, 8, 0)
    tune.set_filter_sweep(2, 154, 1, 5, 8, 16)
    tune.set_sweep(2, 154, 1, 0, 0, 8, 1)
    again = FusedSolver(dims, PER, st)
    assert again.get_tune(1)[0] == (2, 8, 0)
    assert again.get_tune(2) == ((0, 8, 1), (5, 8, 16))
    assert nrel(host(again.rhs(q)), host(default.rhs(q))) < 1e-13
