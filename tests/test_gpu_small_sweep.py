"""The persistent sweep at the sizes where its inversion and its products change form:
sub-panels of 8 columns (7, 8, 9, 15, 24, 25, 31), one 16 x 16 tile or four (16, 17), every
block above 16 or not, one to many blocks, blocks that need pivoting in every column, columns
of very different scale, and more energies than workgroups.  Against the dense oracle at 1e-10
per block, the bound of the other parity tests."""

import numpy as np
import pytest

from quatrex_amd.layout import Geometry
from tests.helpers import edge_case, skew_tridiagonal
from tests.test_gpu_products import _check, _dense, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [(7, 8, 9), (15, 16), (16, 1, 16, 8), (17, 32), (24, 25, 31), (32, 32, 32, 32),
                                (16, 17, 32), (31,), (9,), (18, 19, 20, 21, 22)])
def test_sizes_vs_dense(device, bs):
    print(f"small sweep bs={bs}", flush=True)
    g, A, SL, SG, obc = edge_case(bs, seed=7 + sum(bs), E=3)
    _check(g, _run(g, A, SL, SG, obc, device), _dense(g, A, SL, SG, obc))


def _pivoting_case(bs, E, seed):
    """Diagonal blocks dominated by a random permutation matrix (the largest entry of a
    column is almost never on the diagonal), small off-diagonal blocks."""
    rng = np.random.default_rng(seed)
    g = Geometry(tuple(bs))
    n, bo = g.n, g.block_offsets
    a = np.zeros((E, n, n), np.complex128)
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    for e in range(E):
        for i, b in enumerate(bs):
            s = slice(bo[i], bo[i + 1])
            a[e, s, s] = 4.0 * np.eye(b)[rng.permutation(b)] * np.exp(2j * np.pi * rng.random(b)) + 0.1 * c(b, b) / np.sqrt(b)
            if i:
                p = slice(bo[i - 1], bo[i])
                a[e, s, p] = 0.3 * c(b, bs[i - 1]) / np.sqrt(max(b, bs[i - 1]))
                a[e, p, s] = 0.3 * c(bs[i - 1], b) / np.sqrt(max(b, bs[i - 1]))
    sl, sg = (np.broadcast_to(skew_tridiagonal(bs, rng), (E, n, n)) for _ in range(2))
    return g, g.from_dense(a), g.from_dense(sl)[:2], g.from_dense(sg)[:2]


@pytest.mark.parametrize("bs,E", [((8,), 2), ((16, 13), 3), ((32, 32, 32), 4), ((25, 17, 31), 3), ((32, 9, 30), 2),
                                  ((32, 32), 600)])
def test_pivoting_vs_dense(device, bs, E):
    print(f"pivoting bs={bs} E={E}", flush=True)
    n = min(E, 5)
    g, A, SL, SG = _pivoting_case(bs, n, 11 + sum(bs))
    rep = lambda x: np.ascontiguousarray(np.resize(x, (E, *x.shape[1:])))  # noqa: E731
    got = _run(g, *(tuple(map(rep, m)) for m in (A, SL, SG)), None, device)
    _check(g, [tuple(p[:n] for p in x) for x in got], _dense(g, A, SL, SG, None))
    for x in got:  # the same energies further on in the queue
        for p in x:
            np.testing.assert_array_equal(p, np.resize(p[:n], p.shape))


@pytest.mark.parametrize("b", [11, 32])
def test_column_scales_leave_the_inverse_alone(device, b):
    """One block A' = A D with D powers of two: G' = D^-1 G.  The elimination of a column does not
    depend on the scale of the others and scaling by powers of two is exact, so the
    retarded block agrees bit for bit."""
    g, A, SL, SG = _pivoting_case((b,), 2, 3)
    d = np.exp2(np.random.default_rng(5).integers(-200, 201, b))
    ref = _run(g, A, SL, SG, None, device)[0][0].reshape(2, b, b)
    scaled = ((A[0].reshape(2, b, b) * d).reshape(2, b * b), *A[1:])
    got = _run(g, scaled, SL, SG, None, device)[0][0].reshape(2, b, b)
    np.testing.assert_array_equal(got * d[:, None], ref)


def test_current_of_more_energies_than_two_gib_hold(device):
    """One 1 x 1 block and 2^26 + 5 energies: the currents, two per energy, end beyond 2 GiB.
    Scalars: g = 1 / (a - b^R), g^<> = |g|^2 (s^<> + b^<>), J = b^> g^< - g^> b^< in both
    slots with opposite signs.  Every value is within some 20 roundings of its terms."""
    import torch

    from quatrex_amd import solve as S

    E, n = 2**26 + 5, 4096
    g = Geometry((1,))
    gen = torch.Generator(device=device)
    gen.manual_seed(17)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(E, dtype=torch.float64, device=device, generator=gen)  # noqa: E731
    none = torch.empty((E, 0), dtype=torch.complex128, device=device)
    a = torch.complex(u(-1.0, 1.0), u(0.5, 1.0))
    br = torch.complex(u(-0.1, 0.1), u(-0.2, -0.1))
    sl, sg, bl, bg = (1j * u(0.1, 1.0) * k for k in (1, -1, 1, -1))
    out = [S.packed_empty(g, E, device) for _ in range(2)]
    cur = torch.full((E, 2), float("nan"), dtype=torch.complex128, device=device)
    col = lambda x: x.reshape(E, 1)  # noqa: E731
    ob = [[x.reshape(E, 1, 1)] for x in (br, bl, bg)]
    print(f"current of {E} energies", flush=True)
    S.selected_solve(g, (col(a), none, none), (col(sl), none), (col(sg), none), g_lesser=out[0], g_greater=out[1],
                     obc=ob, current=cur)
    S.default_context(device).status()
    assert not bool(torch.isnan(cur.real).any())
    for part in (slice(0, n), slice(2**26 - n // 2, None)):
        w = 1.0 / (a[part] - br[part]).abs() ** 2
        gl, gg = w * (sl[part] + bl[part]), w * (sg[part] + bg[part])
        j = bg[part] * gl - gg * bl[part]
        tol = 40 * 2.0**-53 * (bg[part].abs() * gl.abs() + gg.abs() * bl[part].abs())
        assert bool(((cur[part, 0] - j).abs() <= tol).all())
        assert bool(((cur[part, 1] + j).abs() <= tol).all())
