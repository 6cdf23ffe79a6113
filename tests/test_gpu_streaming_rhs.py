"""The per-operator right-hand side on a grid whose pointwise kernels all pass
over more than the last-level cache holds (20 fields and more above 256 MB:
the streaming variants), against the CPU oracle with the bar of the small
grids."""
import pytest

import test_gpu_operator_rhs as rhs


@pytest.mark.gpu
def test_viscous_rhs_above_the_cache(oracle):
    rhs.test_viscous_rhs(oracle, (152, 120, 96), [[45, 10, 45], [45, 10, 45]])
