"""GPU parity of the batched inverse at the sizes where its panels, sub-panels and waves
end, and on matrices whose pivots need care.

Bars: the residual max |A X - I| of each matrix within 100 n eps ||A||_F ||X||_F (the
rounding of n elimination steps, with room for their growth); scaling the columns of A
by powers of two scales the rows of the inverse by their inverses exactly (pivot choices compare
within a column, and every operation commutes with the scaling while it stays in range), so
those inverses are compared bit for bit: with a scale per column whose ratios stay in the range of a
double (a pivot row divided by its pivot holds them), and with one scale for all
columns whose square does not.
"""

import numpy as np
import pytest

from quatrex_amd import solve as S

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _inv(a, device):
    import torch

    out = S.inv(torch.as_tensor(a, device=device))
    S.default_context(device).status()
    return out.cpu().numpy()


def _random(n, E, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((E, n, n)) + 1j * rng.standard_normal((E, n, n))


def _check(a, x):
    n = a.shape[-1]
    for m, y in zip(a, x):
        bar = 100 * n * EPS * np.linalg.norm(m) * np.linalg.norm(y)
        assert np.abs(m @ y - np.eye(n)).max() <= bar


@pytest.mark.parametrize("n,E", [(33, 3), (39, 2), (40, 70), (41, 2), (63, 2), (64, 300), (65, 2), (72, 5),
                                 (127, 3), (128, 4), (129, 2), (193, 2), (255, 3), (256, 9), (257, 2), (320, 2),
                                 (511, 2), (512, 3), (513, 1)])
def test_inverse_at_panel_edges(device, n, E):
    print(f"inverse n={n} E={E}", flush=True)
    a = _random(n, E, n)
    _check(a, _inv(a, device))


@pytest.mark.parametrize("n", [33, 64, 100, 256, 300])
def test_inverse_of_permutations_and_ties(device, n):
    """Zero pivots everywhere but in one row per column; columns of equal magnitudes."""
    rng = np.random.default_rng(n)
    perm = np.zeros((n, n), complex)
    perm[np.arange(n), rng.permutation(n)] = np.exp(2j * np.pi * rng.random(n))
    ties = np.exp(2j * np.pi * np.outer(np.arange(n), np.arange(n)) / n)  # the Fourier matrix
    a = np.stack([perm, ties])
    x = _inv(a, device)
    np.testing.assert_allclose(x[0], perm.conj().T, rtol=0, atol=4 * EPS)
    _check(a, x)


@pytest.mark.parametrize("n", [40, 64, 200, 512])
@pytest.mark.parametrize("lo,hi", [(-400, 400), (520, 521), (-520, -519)])
def test_inverse_under_column_scaling(device, n, lo, hi):
    a = _random(n, 2, 7 * n)
    k = np.random.default_rng(n).integers(lo, hi, n)
    scale = np.ldexp(1.0, k)
    x, y = _inv(a, device), _inv(a * scale, device)
    np.testing.assert_array_equal(y, np.ldexp(x.real, -k[:, None]) + 1j * np.ldexp(x.imag, -k[:, None]))


@pytest.mark.parametrize("n,col", [(50, 0), (64, 17), (256, 255), (300, 100)])
def test_singular_column_is_reported(device, n, col):
    a = _random(n, 3, n + col)
    a[1, :, col] = 0.0
    with pytest.raises(S.LinAlgError, match=f"energy 1, block 0, column {col}"):
        _inv(a, device)
