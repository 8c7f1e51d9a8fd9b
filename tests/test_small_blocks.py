"""Small blocks: one launch per level, one, two or four wavefronts per node.

Every kernel variant (one per multiple of four of n up to 32, of eight up to
64, exact and padded; one wavefront up to n = 16, two up to 32), with the narrow levels in one launch
(at most 256 systems of n <= 16) and without, in both precisions, with the
right-hand sides inside the factor (m <= 32, n > 32: 64), in one or more column
chunks, or after it, out of place, and the sweeps on their own: against the
oracle.
"""
import numpy as np
import pytest

from oracle import nd

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


# (n, N, m, B): n on both sides of every tile edge, horizons of 1 .. 7 levels,
# m at the edges of the 16-column chunks, B on both sides of the tail's limit
CASES = [(1, 5, 1, 1), (4, 2, 3, 2), (5, 40, 1, 1), (8, 1, 2, 1), (11, 33, 16, 2), (12, 20, 1, 1), (15, 70, 17, 1),
         (16, 64, 16, 1), (16, 3, 33, 2), (17, 20, 1, 1), (20, 61, 4, 3), (23, 7, 32, 1), (24, 100, 1, 1),
         (25, 9, 2, 2), (28, 15, 16, 1), (31, 31, 33, 1), (32, 2, 17, 1), (32, 90, 1, 2), (6, 11, 1, 300),
         (18, 6, 2, 300), (33, 20, 1, 1), (36, 7, 17, 2), (40, 33, 3, 1), (41, 12, 64, 1), (48, 25, 16, 2), (49, 9, 1, 1),
         (56, 16, 65, 1), (60, 40, 4, 1), (64, 31, 16, 1), (64, 2, 33, 2), (57, 1, 2, 1)]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,N,m,B", CASES)
def test_variants_match_oracle(n, N, m, B, dtype, device):
    import torch
    from socu_amd import functional
    from socu_amd.block_tridiag_solver import (
        create_cholesky_backward_substitution_launch,
        create_cholesky_factor_and_solve_launch,
        create_cholesky_forward_substitution_launch,
    )

    print(f"small n={n} N={N} m={m} B={B} {dtype}", flush=True)
    tdt = getattr(torch, dtype)
    # kappa(Psi) <= 1e3 (alpha = 10, 16 above n = 32): 1e3 * N * 2^-53, and 2^-24
    tol = 1e-11 if dtype == "float64" else 5e-4
    kinds = min(B, 3)  # distinct systems, repeated over the batch
    P = [nd.readme_problem(n, N, m, alpha=10.0 if n <= 32 else 16.0, seed=17 + k)[:3] for k in range(kinds)]
    L0, E0, b0 = (np.stack([P[k % kinds][i] for k in range(B)]) for i in range(3))
    L, E, x = (torch.tensor(a, dtype=tdt, device=device) for a in (L0, E0, b0))
    E[:, N - 1:] = 3.0  # the fill-in region's contents on entry are ignored
    run = create_cholesky_factor_and_solve_launch(L, E, x, dtype=tdt, use_cuda_graph=True)
    run()
    # functional: out of place
    Lf, Ef, xf = functional.cholesky_factor_and_solve(*(torch.tensor(a, dtype=tdt, device=device)
                                                        for a in (L0, E0[:, :N - 1], b0)), pad_problem=False)
    y = torch.tensor(b0, dtype=tdt, device=device)
    create_cholesky_forward_substitution_launch(L, E, y, dtype=tdt)()
    z = y.clone()
    create_cholesky_backward_substitution_launch(L, E, z, dtype=tdt)()
    got = [t.double().cpu().numpy() for t in (L, E, x, Lf, Ef, xf, y, z)]
    for k in range(kinds):
        Lr, Er, yr = P[k][0].copy(), P[k][1].copy(), P[k][2].copy()
        nd.factor(Lr, Er)
        nd.forward(Lr, Er, yr)
        xr = yr.copy()
        nd.backward(Lr, Er, xr)
        inv = np.linalg.inv(np.tril(Lr))
        want_L = np.tril(Lr) + np.triu(np.swapaxes(inv, -1, -2), 1)
        for b in {k, k + kinds * ((B - 1 - k) // kinds)}:
            for i, want in enumerate((want_L, Er, xr, want_L, Er, xr, yr, xr)):
                assert _rel(got[i][b], want) < tol, (b, i)
