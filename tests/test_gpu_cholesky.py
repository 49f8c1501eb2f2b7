"""Cholesky solve of the direct SR at the edges of its tiles (16-column
blocks, 64-row tiles, 256-column back substitution launches, panels with a
launch of their own from 40 trailing tile rows on): solution, factor, the
untouched triangle, and the first pivot that is not positive and finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import torch
    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    import mvmc_hip
    return mvmc_hip


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 129, 255, 256, 257, 321, 700, 2689])
def test_solve_and_factor(M, n):
    """Backward error of a Cholesky solve: |A - L L^T| <= (n + 1) eps |L||L^T|
    and |A x - b| <= 3 (n + 1) eps |A||x| up to small constants; a tenth of
    that bound's growth in n is never reached, sqrt(n) + 10 is taken."""
    import torch
    print(f"cholesky n={n}", flush=True)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, n + 5))
    A = X @ X.T / n + 0.01 * np.eye(n)
    A = (A + A.T) / 2
    A[0, n - 1] = A[n - 1, 0]
    b = rng.standard_normal(n)
    S = A.copy()
    S[np.triu_indices(n, 1)] = 7.0  # column-major lower triangle: not read, not written
    s, x = torch.tensor(S, device="cuda"), torch.tensor(b, device="cuda")
    assert M.sr_cholesky_solve(s, x, n) == 0
    F, x = s.cpu().numpy(), x.cpu().numpy()
    assert np.all(F[np.triu_indices(n, 1)] == 7.0)
    L = np.tril(F)
    eps = np.finfo(float).eps
    tol = (np.sqrt(n) + 10) * eps
    assert np.abs(L @ L.T - A).max() <= tol * np.abs(A).max()
    assert np.abs(A @ x - b).max() <= 3 * tol * np.abs(A).sum(1).max() * np.abs(x).max()


@pytest.mark.parametrize("n,at,value", [(4, 0, -1.0), (70, 65, 0.0), (200, 100, float("nan")), (130, 129, -2.0),
                                        (90, 17, float("inf"))])
def test_first_bad_pivot(M, n, at, value):
    import torch
    A = torch.eye(n, dtype=torch.float64)
    A[at, at] = value
    b = torch.ones(n, dtype=torch.float64, device="cuda")
    assert M.sr_cholesky_solve(A.cuda(), b, n) == at + 1
    assert bool((b == 1).all())  # no solution, right-hand side as given


@pytest.mark.parametrize("scale", [1e-300, 1e300])
def test_extreme_pivots(M, scale):
    import torch
    rng = np.random.default_rng(3)
    X = rng.standard_normal((80, 90))
    A = X @ X.T / 80 + np.eye(80)
    b = rng.standard_normal(80)
    s, x = torch.tensor(A * scale, device="cuda"), torch.tensor(b, device="cuda")
    assert M.sr_cholesky_solve(s, x, 80) == 0
    want = np.linalg.solve(A, b) / scale
    assert np.abs(x.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
