"""Operators with chunk lengths set by hand against the oracle, at the lengths
where a chunk length meets its limit: one chunk a line (16 points), the first
lengths of two chunks, a length that no chunk one row short cuts.

Bar: 1e-12 norm-wise, as for the other operator tests."""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel

CL = [[10, 10, 10], [10, 10, 10]]
PER = [[45, 45, 45], [45, 45, 45]]


@pytest.fixture
def tune():
    from compact_schemes_amd import tune as t
    t.clear()
    yield t
    t.clear()


@pytest.mark.gpu
@pytest.mark.parametrize("n, K", [(16, 16), (16, 8), (17, 16), (31, 16), (31, 8), (32, 16), (32, 32)])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("nbc", [CL, PER], ids=["closure", "periodic"])
def test_operators_on_chunk_lengths_set_by_hand(oracle, tune, n, K, axis, nbc):
    import torch
    import compact_schemes_amd as cs
    from compact_schemes_amd.batch import Batch
    seam = int(nbc is PER)
    for op in (tune.DERIV, tune.FILTER):
        tune.set_line(op, n, K, start=seam, end=seam)
    dims = [21, 18, 19]
    dims[axis] = n
    dims = tuple(dims)
    rng = np.random.default_rng(n + K)
    f = np.sin(0.3 * np.arange(np.prod(dims))) + 0.1 * rng.standard_normal(np.prod(dims))
    num, ctx = cs.Numerics(dims, nbc), oracle.Context(dims, nbc)
    case(f"chunks set by hand dims={dims} K={K} axis={axis} nbc={nbc[0]}")
    fd = dev(f)
    out = torch.full_like(fd, float("nan"))
    num.deriv(axis, fd, out)
    assert nrel(host(out), ctx.deriv_field(axis, f)) < 1e-12
    g = torch.full_like(fd, float("nan"))
    num.filter(axis, fd, g)
    assert nrel(host(g), ctx.filter(axis, f)) < 1e-12
    b = Batch([dims], nbc)                              # one subdomain: the same bits
    d = [torch.zeros_like(fd) for _ in range(3)]
    b.bind([fd], d)
    b.step()
    assert torch.equal(d[axis], out)
