"""Factor and inverse of diagonal blocks: every number of 16-row tiles and both
sides of each edge, against numpy; the inverse from a factor made elsewhere
(its strict upper triangle holds anything), and FP32 blocks with FP64 pivots.
"""
import numpy as np
import pytest

from oracle import nd

pytestmark = pytest.mark.gpu

EDGES = [1, 7, 16, 17, 31, 32, 33, 48, 49, 64, 65, 79, 80, 81, 96, 97, 101, 112, 113, 127, 128,
         # (two halves of 16 ceil(n / 32) rows and the rest)
         129, 145, 160, 161, 192, 200, 223, 225, 255, 256]


def _spd(n, B, seed):
    rng = np.random.default_rng(seed)
    G = rng.standard_normal((B, 1, n, n)) / np.sqrt(n)
    return G @ np.swapaxes(G, -1, -2) + 2.0 * np.eye(n)  # kappa <= 4


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n", EDGES)
def test_factor_and_inverse(n, dtype, device):
    import torch
    from socu_amd.block_tridiag_solver import create_cholesky_factor_launch, create_cholesky_solve_launch

    print(f"diag n={n} {dtype}", flush=True)
    tdt = getattr(torch, dtype)
    tol = 64 * n * (2.0**-53 if dtype == "float64" else 2.0**-24)
    A = _spd(n, 3, n)
    Lr = np.linalg.cholesky(A)
    inv = np.linalg.inv(Lr)
    E = torch.zeros(3, 0, n, n, dtype=tdt, device=device)
    L = torch.tensor(np.tril(A) + np.triu(np.full((n, n), 7.0), 1), dtype=tdt, device=device)
    create_cholesky_factor_launch(L, E, dtype=tdt)()
    got = L.double().cpu().numpy()
    assert _rel(np.tril(got), Lr) < tol
    assert n == 1 or _rel(np.triu(got, 1), np.triu(np.swapaxes(inv, -1, -2), 1)) < tol
    # a factor from elsewhere
    L = torch.tensor(Lr + np.triu(np.full((n, n), 7.0), 1), dtype=tdt, device=device)
    keep = L.clone()
    x = torch.tensor(np.broadcast_to(np.eye(n), (3, 1, n, n)).copy(), dtype=tdt, device=device)
    create_cholesky_solve_launch(L, E, x, dtype=tdt)()
    assert torch.equal(L, keep)
    assert _rel(x.double().cpu().numpy(), np.linalg.inv(A)) < 4 * tol


@pytest.mark.parametrize("n", [5, 16, 33, 64, 65, 100, 128])
def test_fp64_pivots(n, device):
    import torch
    from socu_amd import problems
    from socu_amd.mixed import create_cholesky_mixed_factor_and_solve_launch

    print(f"mixed n={n}", flush=True)
    L0, E0, b0 = problems.readme_problem(n, 5, 2, alpha=16.0, seed=n)
    L, E, x = (torch.tensor(a, device=device) for a in (L0, E0, b0))
    run = create_cholesky_mixed_factor_and_solve_launch(L, E, x, tol=1e-12, max_iter=5)
    run()
    torch.cuda.synchronize()
    assert problems.rel_residual(L0, E0, x.cpu().numpy(), b0) <= 1e-12


# the sum of a Schur tile in halves and quarters of n rounded to 8, the last ones
# short or empty; FP32 with FP64 pivots takes these tiles for the small n too
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 15, 16, 17, 20, 31, 33, 40, 64, 65, 70, 73, 88, 97, 128, 130, 201, 255])
def test_schur_tiles(n, device):
    import torch
    from socu_amd import _lib
    from socu_amd.block_tridiag_solver import create_cholesky_factor_launch

    print(f"schur n={n}", flush=True)
    N = 12
    L0, E0, _ = nd.readme_problem(n, N, 1, alpha=16.0, seed=n)[:3]
    Lr, Er = L0.copy(), E0.copy()
    nd.factor(Lr, Er)
    if n > 64:
        L, E = (torch.tensor(a[None], device=device) for a in (L0, E0))
        create_cholesky_factor_launch(L, E)()
        for got, want in ((np.tril(L[0].cpu().numpy()), np.tril(Lr)), (E[0].cpu().numpy(), Er)):
            assert _rel(got, want) < 1e-11
    if n <= 128:
        L, E = (torch.tensor(a[None], dtype=torch.float32, device=device) for a in (L0, E0))
        lib = _lib.load()
        rc = lib.socu_cholesky_factor_f32(L.data_ptr(), E.data_ptr(), None, 1, N, n, _lib.PREC_FP32, None)
        torch.cuda.synchronize()
        assert rc == 0
        for got, want in ((np.tril(L[0].double().cpu().numpy()), np.tril(Lr)), (E[0].double().cpu().numpy(), Er)):
            assert _rel(got, want) < 1e-4
