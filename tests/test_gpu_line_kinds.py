"""Chunk lengths per kind of line: what the batch autotuner times on x lines
does not choose the kernels of y and z lines, and an entry for one kind leaves
the other on its default, bit for bit.  Bar: 1e-12 norm-wise."""
import numpy as np
import pytest

from gpu_util import case, dev, host, nrel

PER = [[45, 45, 45], [45, 45, 45]]
N = 300      # x lines take 16-point chunks, y and z lines too; 8-point ones only x lines


@pytest.fixture
def tune():
    from compact_schemes_amd import tune as t
    t.clear()
    yield t
    t.clear()


def _operators(dims, axis):
    """derivative and filter along `axis` on a new context"""
    import torch
    import compact_schemes_amd as cs
    f = np.sin(0.3 * np.arange(np.prod(dims))) + 0.1 * np.random.default_rng(1).standard_normal(np.prod(dims))
    num = cs.Numerics(dims, PER)
    fd = dev(f)
    out, g = torch.zeros_like(fd), torch.zeros_like(fd)
    num.deriv(axis, fd, out)
    num.filter(axis, fd, g)
    return f, host(out), host(g)


@pytest.mark.gpu
def test_autotuner_records_the_kind_it_timed(tune, tmp_path):
    import torch
    from compact_schemes_amd.batch import Batch
    dims = (N, 24, 20)
    b = Batch([dims], PER)
    f = [dev(np.sin(0.1 * np.arange(np.prod(dims))))]
    b.bind(f, [torch.zeros_like(f[0]) for _ in range(3)])
    case("autotune x lines of 300 points")
    b.autotune(reps=2)
    tune.save(tmp_path / "t.txt")
    entries = [ln.split()[1:] for ln in (tmp_path / "t.txt").read_text().splitlines() if ln.startswith("line")]
    assert sorted((e[0], e[6]) for e in entries if e[1] == str(N)) == [("0", "0"), ("1", "0")]
    assert all(e[6:] == ["1"] for e in entries if e[1] != str(N))


@pytest.mark.gpu
@pytest.mark.parametrize("kind, K", [(0, 8), (0, 32), (1, 8), (1, 32)])
def test_entry_of_one_kind_leaves_the_other(oracle, tune, tmp_path, kind, K):
    xdims, ydims = (N, 18, 17), (18, N, 17)
    case(f"chunk length {K} for kind {kind}")
    before = [_operators(xdims, 0), _operators(ydims, 1)]
    path = tmp_path / "t.txt"
    path.write_text("".join(f"line {op} {N} 1 1 0 {K} {kind}\n" for op in (0, 1)))
    tune.load(path)
    after = [_operators(xdims, 0), _operators(ydims, 1)]
    for k in (1, 2):
        assert np.array_equal(before[1 - kind][k], after[1 - kind][k])
    ctx = oracle.Context((xdims, ydims)[kind], PER)
    f, d, g = after[kind]
    assert nrel(d, ctx.deriv_field(kind, f)) < 1e-12
    assert nrel(g, ctx.filter(kind, f)) < 1e-12


@pytest.mark.gpu
def test_both_kinds_of_one_length_in_one_context(oracle, tune, tmp_path):
    """One operator table for x and y lines of one length with chunk lengths of
    their own on the general kernels, FP64 and mixed precision."""
    import torch
    import compact_schemes_amd as cs
    dims = (96, 96, 17)
    f = np.random.default_rng(2).standard_normal(np.prod(dims))
    path = tmp_path / "t.txt"
    path.write_text("".join(f"line {op} 96 1 1 {prec} {K} {kind}\n"
                            for op in (0, 1) for prec in (0, 1) for kind, K in ((0, 32), (1, 16))))
    tune.load(path)
    ctx = oracle.Context(dims, PER)
    case("two chunk lengths in one table")
    for prec in (0, 1):
        num = cs.Numerics(dims, PER)
        num.set_precision(prec)
        fd = dev(f)
        out = torch.zeros_like(fd)
        for axis in (0, 1):
            num.deriv(axis, fd, out)
            assert nrel(host(out), ctx.deriv_field(axis, f)) < (1e-12 if prec == 0 else 1e-11)
            num.filter(axis, fd, out)
            assert nrel(host(out), ctx.filter(axis, f)) < (1e-12 if prec == 0 else 1e-11)
