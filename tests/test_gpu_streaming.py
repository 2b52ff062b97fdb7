"""Assembly and block moves of stacks too large for the caches, whose kernels go
around them: against the oracle at the first, a middle and the last energy, and
against the same call on slices small enough for the cached kernels (bit for bit)."""

import numpy as np
import pytest

from oracle import assembly as AS
from oracle.dsdb import OracleDSDB
from quatrex_amd import solve as S
from quatrex_amd.dsdb import DSDBCOO, DSDBCSR, densify_batch, sparsify_batch
from quatrex_amd.layout import Geometry
from tests.test_gpu_dsdb import SYMMETRY, _matrix

pytestmark = pytest.mark.gpu


def _random(shape, device, gen):
    import torch

    return torch.randn(shape, dtype=torch.complex128, device=device, generator=gen)


@pytest.mark.parametrize("per_energy_h,overlap", [(False, True), (True, False)])
def test_assembly_past_the_caches(device, per_energy_h, overlap):
    import torch

    bs = (64, 61, 50, 64, 33, 64, 65, 58)
    g = Geometry(bs)
    E = 67
    assert 4 * 16 * E * (g.diag_size + 2 * g.offdiag_size) > 256 * 2**20
    gen = torch.Generator(device=device)
    gen.manual_seed(5)
    sizes = (g.diag_size, g.offdiag_size, g.offdiag_size)
    stack = lambda: tuple(_random((E, n), device, gen) for n in sizes)
    sr, sl, sg = stack(), stack(), stack()
    h = stack() if per_energy_h else tuple(x[0].contiguous() for x in stack())
    s = tuple(x[0].contiguous() for x in stack()) if overlap else None
    v = torch.randn(g.n, dtype=torch.float64, device=device, generator=gen)
    z = torch.complex(torch.linspace(-1, 1, E, dtype=torch.float64, device=device),
                      torch.full((E,), 1e-3, dtype=torch.float64, device=device))

    def run(lo, hi):
        cut = lambda t: tuple(x[lo:hi].contiguous() for x in t)
        a = S.packed_empty(g, hi - lo, device)
        S.assemble_system(g, z[lo:hi].contiguous(), cut(h) if per_energy_h else h, a=a, overlap=s, potential=v,
                          sigma_retarded_herm=cut(sr), sigma_lesser=cut(sl), sigma_greater=cut(sg))
        return a

    a = run(0, E)
    for lo in range(0, E, 16):
        for x, y in zip(a, run(lo, min(lo + 16, E))):
            assert torch.equal(x[lo:lo + 16], y)
    at = [0, 34, E - 1]
    dense = lambda t: g.to_dense(*(x[at].cpu().numpy() for x in t))
    one = lambda t: g.to_dense(*(x[None].cpu().numpy() for x in t))[0]
    en = z.real.cpu().numpy()[at]
    ref = AS.assemble(bs, en, 1e-3, dense(h) if per_energy_h else one(h), one(s) if overlap else None,
                      v.cpu().numpy(), dense(sr), dense(sl), dense(sg))
    np.testing.assert_allclose(dense(a), ref, rtol=0, atol=1e-14 * np.abs(ref).max())


@pytest.mark.parametrize("layout", [DSDBCOO, DSDBCSR])
@pytest.mark.parametrize("symmetry,op", SYMMETRY)
def test_block_moves_past_the_caches(device, layout, symmetry, op):
    import torch

    bs = [96, 91, 100, 96, 88, 97, 99, 96]
    E, at = 129, [0, 64, 128]
    g = Geometry(bs)
    m = _matrix(bs, 43, symmetry, op)
    # map entries of the smallest part: a third of its elements
    assert 32 * E * 0.28 * g.offdiag_size > 64 * 2**20
    c = layout.from_sparray(m, bs, (E,), symmetry, op, device=device)
    gen = torch.Generator(device=device)
    gen.manual_seed(6)
    c.data.copy_(_random(tuple(c.data.shape), device, gen))
    o = OracleDSDB.from_sparray(m, bs, (3,), symmetry, op)
    o.data[...] = c.data[at].cpu().numpy()
    ctx = S.default_context(device)
    parts, _ = densify_batch(c, slice(None), g, "dul", device, ctx)
    for i in range(len(bs)):
        np.testing.assert_array_equal(g.diag(parts[0], i)[at].cpu().numpy(), o.get_block(i, i))
    for i in range(len(bs) - 1):
        np.testing.assert_array_equal(g.upper(parts[1], i)[at].cpu().numpy(), o.get_block(i, i + 1))
        np.testing.assert_array_equal(g.lower(parts[2], i)[at].cpu().numpy(), o.get_block(i + 1, i))
    x, y = layout.zeros_like(c), layout.zeros_like(c)
    sparsify_batch(x, slice(None), g, parts, "dul", device, ctx)
    for lo in range(0, E, 16):
        cut = tuple(p[lo:lo + 16].contiguous() for p in parts)
        sparsify_batch(y, slice(lo, min(lo + 16, E)), g, cut, "dul", device, ctx)
    assert torch.equal(x.data, y.data)
    assert bool(x.data.any())


def _calls(c, g, device, ctx, parts, bufs=None):
    """Densify of all energies in one call, and in slices that the caches hold (or sparsify into c)."""
    E, step = int(c.data.shape[0]), 32
    one = lambda lo, hi: (  # noqa: E731
        densify_batch(c, slice(lo, hi), g, parts, device, ctx, data=c.data[lo:hi])[0] if bufs is None else
        sparsify_batch(c, slice(lo, hi), g, tuple(p[lo:hi] for p in bufs), parts, device, ctx))
    return (lambda: one(0, E)), (lambda: [one(lo, min(lo + step, E)) for lo in range(0, E, step)])


@pytest.mark.parametrize("parts", ["dul", "d", "l"])
@pytest.mark.parametrize("symmetry,op", SYMMETRY)
def test_one_large_move_equals_its_slices(device, parts, symmetry, op):
    """Past the line of 1.5 times the caches, also for single parts; a symmetric stack's lower
    part is mirrored whole, its diagonal part half."""
    import torch

    bs, E = [96, 91, 100, 96, 88, 97, 99, 96], {"dul": 257, "d": 720, "l": 720}[parts]
    g = Geometry(bs)
    m = _matrix(bs, 47, symmetry, op)
    c = DSDBCOO.from_sparray(m, bs, (E,), symmetry, op, device=device)
    entries = 0.28 * {"dul": g.diag_size + 2 * g.offdiag_size, "d": g.diag_size, "l": g.offdiag_size}[parts]
    assert 32 * E * entries > 1.5 * 256 * 2**20
    gen = torch.Generator(device=device)
    gen.manual_seed(8)
    c.data.copy_(_random(tuple(c.data.shape), device, gen))
    ctx = S.default_context(device)
    whole, sliced = _calls(c, g, device, ctx, parts)
    a, b = whole(), sliced()
    for k, x in enumerate(a):
        if x is not None:
            assert torch.equal(x, torch.cat([s[k] for s in b]))
    x, y = DSDBCOO.zeros_like(c), DSDBCOO.zeros_like(c)
    if parts == "dul":
        _calls(x, g, device, ctx, parts, a)[0]()
        _calls(y, g, device, ctx, parts, a)[1]()
        assert torch.equal(x.data, y.data) and bool(x.data.any())


@pytest.mark.parametrize("symmetry", [False, True])
def test_one_large_move_is_no_slower_than_its_slices(device, symmetry):
    """A call past the caches against the same energies in cached calls, all entries stored; the slices
    pass through as much memory and have 16 times the launches.  (Mirrored entries written past
    the caches took 2.1 times as long.)"""
    import time

    import torch

    bs, E = (64,) * 16, 512
    g = Geometry(bs)
    i, j = np.indices((g.n, g.n), dtype=np.int64).reshape(2, -1)
    keep = (np.abs(i // 64 - j // 64) <= 1) & ((i <= j) | (not symmetry))
    i, j = i[keep], j[keep]
    order = np.lexsort((j, i, j // 64, i // 64))
    data = torch.ones((E, i.size), dtype=torch.complex128, device=device)
    c = DSDBCOO(data, i[order], j[order], bs, (E,), symmetry)
    ctx = S.default_context(device)

    def best(f):
        f()
        times = []
        for _ in range(7):
            torch.cuda.synchronize()
            t = time.perf_counter()
            f()
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        return min(times)

    whole, sliced = _calls(c, g, device, ctx, "dul")
    bufs = whole()
    assert best(whole) <= 1.3 * best(sliced)
    whole, sliced = _calls(DSDBCOO.zeros_like(c), g, device, ctx, "dul", bufs)
    assert best(whole) <= 1.3 * best(sliced)
