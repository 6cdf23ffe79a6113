"""GPU parity of the single-field derivative and filter at the edges of the
chunk rule: lengths that 8- or 16-point chunks cut evenly, one row short, or
not at all (the general kernels), and the longest lines of each kernel, along
each axis.  Bars: 1e-12 norm-wise (derivative), 1e-12 (filter), as for the
other operator tests.
"""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel

CL = [[10, 10, 10], [10, 10, 10]]
PER = [[45, 45, 45], [45, 45, 45]]
LENGTHS = [16, 17, 31, 32, 57, 58, 63, 65, 100, 128, 129, 133, 154, 255, 256, 257, 292, 512, 513, 1000]


def _field(dims, seed):
    rng = np.random.default_rng(seed)
    return np.sin(0.3 * np.arange(dims[0] * dims[1] * dims[2])) + 0.1 * rng.standard_normal(np.prod(dims))


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("nbc", [CL, PER], ids=["closure", "periodic"])
def test_operators_on_line_lengths(oracle, n, axis, nbc):
    """Also the boundary derivatives that cs_deriv leaves for the
    characteristic BCs, the filter in place, and a field that starts off the
    16-byte grid."""
    import torch
    import compact_schemes_amd as cs
    dims = [21, 18, 19]
    dims[axis] = n
    dims = tuple(dims)
    lmx = int(np.prod(dims))
    f = _field(dims, n)
    num = cs.Numerics(dims, nbc)
    ctx = oracle.Context(dims, nbc)
    case(f"line sweeps dims={dims} axis={axis} nbc={nbc[0]}")
    buf = torch.zeros(lmx + 1, dtype=torch.float64, device="cuda")
    for fd in (dev(f), buf[1:]):
        fd.copy_(dev(f))
        out = torch.full_like(fd, float("nan"))
        num.deriv(axis, fd, out, var=2)
        assert nrel(host(out), ctx.deriv_field(axis, f)) < 1e-12
        d = host(out).reshape(dims[2], dims[1], dims[0])
        ends = [np.take(d, i, axis=2 - axis).reshape(-1) for i in (0, n - 1)]
        drva = host(num.buffers(axis)[0]).reshape(2, 5, -1)
        assert np.array_equal(drva[0, 2], ends[0]) and np.array_equal(drva[1, 2], ends[1])
        num.filter(axis, fd, out)
        want = ctx.filter(axis, f)
        assert nrel(host(out), want) < 1e-12
        num.filter(axis, fd, fd)
        assert np.array_equal(host(fd), host(out))


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(133, 58, 65), (292, 24, 257)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_batch_modes_equal_single_operators(dims, mode):
    """Sweep and general classes in one batch: the bits of the single calls."""
    import torch
    import compact_schemes_amd as cs
    from compact_schemes_amd.batch import Batch
    shapes = [dims, (40, 17, 600), (64, 48, 32)]
    fields = [dev(_field(d, i)) for i, d in enumerate(shapes)]
    f = [x.clone() for x in fields]
    d = [torch.zeros_like(f[i // 3]) for i in range(9)]
    b = Batch(shapes, PER)
    b.bind(f, d)
    b.set_persistent(mode)
    case(f"batch classes {dims} mode={mode}")
    b.step()
    torch.cuda.synchronize()
    for i, s in enumerate(shapes):
        num = cs.Numerics(s, PER)
        out = torch.zeros_like(fields[i])
        for axis in range(3):
            num.deriv(axis, fields[i], out)
            assert torch.equal(out, d[3 * i + axis]), (s, axis)
        g = fields[i].clone()
        for axis in range(3):
            num.filter(axis, g, g)
        assert torch.equal(g, f[i]), s
