"""The persistent batch grid where a workgroup runs several items, of blocks
that differ in size and faces: the bits of the single operators.

A CU holds at most 32 workgroups of one wave (x lines) or 8 of four (64-point
y and z lines), so the classes below have more items than workgroups."""
import pytest

from gpu_util import case

PER = [[45, 45, 45], [45, 45, 45]]
CL = [[10, 10, 10], [10, 10, 10]]


@pytest.mark.gpu
def test_persistent_workgroups_run_several_items():
    import torch
    import compact_schemes_amd as cs
    from compact_schemes_amd.batch import Batch
    shapes = [(64, 256, 300), (64, 200, 311), (256, 64, 300), (250, 64, 311), (256, 300, 64), (250, 311, 64)]
    nbc = [PER, CL] * 3
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert sum(s[1] * s[2] for s in shapes[:2]) // 8 > 2 * 32 * cus
    assert sum(s[0] * s[2] for s in shapes[2:4]) // 64 > 8 * cus
    torch.manual_seed(5)
    fields = [torch.randn(s[0] * s[1] * s[2], dtype=torch.float64, device="cuda") for s in shapes]
    f = [x.clone() for x in fields]
    d = [torch.zeros_like(f[i // 3]) for i in range(3 * len(shapes))]
    b = Batch(shapes, nbc)
    b.bind(f, d)
    b.set_persistent(1)
    case("persistent grid, several items a workgroup")
    b.step()
    torch.cuda.synchronize()
    for i, s in enumerate(shapes):
        num = cs.Numerics(s, nbc[i])
        out = torch.zeros_like(fields[i])
        for axis in range(3):
            num.deriv(axis, fields[i], out)
            assert torch.equal(out, d[3 * i + axis]), (s, axis)
        g = fields[i].clone()
        for axis in range(3):
            num.filter(axis, g, g)
        assert torch.equal(g, f[i]), s
