"""Level-by-level sweeps of blocks of 32 < n <= 128 against the oracle: forward,
backward and the whole solve, on both sides of every 16-row tile, odd n (rows of
every alignment), one right-hand side to several 16-column chunks, horizons
with and without neighbours on either side, and a masked system, in both
precisions.
"""
import numpy as np
import pytest

from oracle import nd

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


CASES = [(33, 20, 2, 2), (47, 9, 1, 1), (48, 33, 16, 1), (49, 6, 17, 3), (64, 31, 5, 1), (65, 12, 33, 2), (79, 17, 3, 1),
         (80, 2, 16, 1), (81, 5, 1, 2), (96, 10, 8, 1), (97, 7, 15, 2), (100, 40, 8, 1), (111, 3, 2, 1), (112, 15, 1, 1),
         (113, 11, 4, 2), (127, 21, 18, 1), (128, 12, 31, 2), (128, 1, 2, 1)]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,N,m,B", CASES)
def test_sweeps_match_oracle(n, N, m, B, dtype, device, monkeypatch):
    import torch
    from socu_amd.block_tridiag_solver import (
        create_cholesky_backward_substitution_launch,
        create_cholesky_factor_launch,
        create_cholesky_forward_substitution_launch,
        create_cholesky_solve_launch,
    )

    print(f"steps n={n} N={N} m={m} B={B} {dtype}", flush=True)
    monkeypatch.setenv("SOCU_SWEEP", "level")
    tdt = getattr(torch, dtype)
    # kappa(Psi) <= 1e3: 1e3 * N * 2^-53, and 2^-24
    tol = 1e-11 if dtype == "float64" else 5e-4
    P = [nd.readme_problem(n, N, m, alpha=16.0, seed=31 + k)[:3] for k in range(B)]
    L, E, b = (torch.tensor(np.stack([p[i] for p in P]), dtype=tdt, device=device) for i in range(3))
    mask = torch.ones(B, dtype=torch.bool, device=device)
    mask[1:2] = False
    create_cholesky_factor_launch(L, E, dtype=tdt)()
    y, x = b.clone(), b.clone()
    create_cholesky_forward_substitution_launch(L, E, y, mask=mask, dtype=tdt)()
    z = y.clone()
    create_cholesky_backward_substitution_launch(L, E, z, mask=mask, dtype=tdt)()
    create_cholesky_solve_launch(L, E, x, mask=mask, dtype=tdt)()
    for k in range(B):
        if k == 1:
            assert torch.equal(y[k], b[k]) and torch.equal(z[k], b[k]) and torch.equal(x[k], b[k])
            continue
        Lr, Er, yr = (a.copy() for a in P[k])
        nd.factor(Lr, Er)
        nd.forward(Lr, Er, yr)
        xr = yr.copy()
        nd.backward(Lr, Er, xr)
        for got, want in ((y, yr), (z, xr), (x, xr)):
            assert _rel(got[k].double().cpu().numpy(), want) < tol
