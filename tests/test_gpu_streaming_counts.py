"""Launches over several fields above the last-level cache (256 MB over all of
them): the five-field derivatives of the per-operator right-hand side, rows on
and off the 128-byte grid, and the transposed filter of five fields, against
the CPU oracle and the per-operator adjoint with the bars of the small grids."""
import numpy as np
import pytest

import test_gpu_adjoint_chunks as adjoint
import test_gpu_operator_rhs as rhs


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(160, 144, 152), (150, 160, 144)])
def test_five_field_derivatives_above_the_cache(oracle, dims):
    assert 5 * 16 * np.prod(dims) > 256 * 2 ** 20
    rhs.test_viscous_rhs(oracle, dims, [[10, 45, 10], [10, 45, 10]])


@pytest.mark.gpu
def test_transposed_filter_above_the_cache():
    dims = (192, 190, 188)
    assert 5 * 8 * np.prod(dims) > 256 * 2 ** 20
    adjoint.test_rk4_vjp(dims, (adjoint.C, adjoint.C, adjoint.C))
