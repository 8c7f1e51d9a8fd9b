"""Which plans with one right-hand side sweep by the persistent launch."""
import pytest

pytestmark = pytest.mark.gpu


def _arrays(n, B, device, dtype):
    import torch

    return (torch.zeros(B, 3, n, n, dtype=dtype, device=device), torch.zeros(B, 2, n, n, dtype=dtype, device=device),
            torch.zeros(B, 3, n, 1, dtype=dtype, device=device))


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,B,want", [(1, 32, True), (1, 33, False), (12, 9, True), (24, 16, True), (32, 32, True),
                                      (32, 33, False), (33, 33, True), (128, 65, True), (129, 1, False)])
def test_solves_by_batch_and_block_size(n, B, want, dtype, device, monkeypatch):
    import torch
    from socu_amd.block_tridiag_solver import (
        create_cholesky_backward_substitution_launch,
        create_cholesky_forward_substitution_launch,
        create_cholesky_solve_launch,
    )

    monkeypatch.delenv("SOCU_SWEEP", raising=False)
    tdt = getattr(torch, dtype)
    L, E, x = _arrays(n, B, device, tdt)
    for create in (create_cholesky_solve_launch, create_cholesky_forward_substitution_launch,
                   create_cholesky_backward_substitution_launch):
        assert create(L, E, x, dtype=tdt).sweep_status() == (want, False)


@pytest.mark.parametrize("n,B,dtype,want", [(1, 1, "float64", False), (24, 1, "float64", False),
                                            (25, 6, "float64", True), (32, 6, "float64", True),
                                            (32, 7, "float64", False), (25, 1, "float32", False),
                                            (32, 1, "float32", False), (33, 65, "float32", True),
                                            (128, 9, "float64", True), (129, 1, "float64", False)])
def test_captured_solves_by_batch_and_block_size(n, B, dtype, want, device, monkeypatch):
    import numpy as np
    import torch
    from oracle import nd
    from socu_amd.block_tridiag_solver import create_cholesky_factor_launch, create_cholesky_solve_launch

    monkeypatch.delenv("SOCU_SWEEP", raising=False)
    tdt = getattr(torch, dtype)
    P = [nd.readme_problem(n, 5, 1, alpha=16.0, seed=70 + k)[:3] for k in range(2)]
    pick = torch.arange(B) % 2
    L, E, b = (torch.tensor(np.stack([p[i] for p in P]), dtype=tdt)[pick].to(device) for i in range(3))
    create_cholesky_factor_launch(L, E, dtype=tdt)()
    x = b.clone()
    run = create_cholesky_solve_launch(L, E, x, dtype=tdt, use_cuda_graph=True)
    # kappa(Psi) <= 1e3: 1e3 * N * 2^-53, and 2^-24
    tol = 1e-11 if dtype == "float64" else 5e-4
    for _ in range(2):
        x.copy_(b)
        run()
        assert run.sweep_status() == (want, False)
        for k in range(min(B, 2)):
            Lr, Er, xr = (a.copy() for a in P[k])
            nd.factor(Lr, Er)
            nd.solve(Lr, Er, xr)
            assert np.abs(x[pick == k].double().cpu().numpy() - xr).max() <= tol * np.abs(xr).max()


@pytest.mark.parametrize("n,B,want", [(4, 9, True), (16, 64, True), (16, 65, False), (32, 64, True), (33, 65, True)])
def test_mixed_solver_by_batch_and_block_size(n, B, want, device, monkeypatch):
    import torch
    from socu_amd.mixed import create_cholesky_mixed_factor_and_solve_launch

    monkeypatch.delenv("SOCU_SWEEP", raising=False)
    L, E, x = _arrays(n, B, device, torch.float64)
    run = create_cholesky_mixed_factor_and_solve_launch(L, E, x)
    assert run.sweep_status() == (want, False)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,N,B", [(1, 1, 1), (4, 20, 1), (12, 20, 2), (16, 70, 3), (16, 2, 1)])
def test_asked_for_by_small_factor_and_solve(n, N, B, dtype, graph, device, monkeypatch):
    """factor_and_solve of n <= 16 sweeps back inside the factor's kernels; the
    variable overrides that too."""
    import numpy as np
    import torch
    from oracle import nd
    from socu_amd.block_tridiag_solver import create_cholesky_factor_and_solve_launch

    tdt = getattr(torch, dtype)
    P = [nd.readme_problem(n, N, 1, alpha=10.0, seed=50 + k)[:3] for k in range(B)]
    for mode, want in (("persistent", True), ("level", False)):
        monkeypatch.setenv("SOCU_SWEEP", mode)
        L, E, x = (torch.tensor(np.stack([p[i] for p in P]), dtype=tdt, device=device) for i in range(3))
        run = create_cholesky_factor_and_solve_launch(L, E, x, dtype=tdt, use_cuda_graph=graph)
        run()
        assert run.sweep_status() == (want, False)
        for k in range(B):
            Lr, Er, xr = (a.copy() for a in P[k])
            nd.factor(Lr, Er)
            nd.solve(Lr, Er, xr)
            # kappa(Psi) <= 1e3: 1e3 * N * 2^-53, and 2^-24
            tol = 1e-11 if dtype == "float64" else 5e-4
            assert np.linalg.norm(x[k].double().cpu().numpy() - xr) < tol * np.linalg.norm(xr)
            assert np.linalg.norm(np.tril(L[k].double().cpu().numpy()) - np.tril(Lr)) < tol * np.linalg.norm(Lr)


@pytest.mark.parametrize("n,dtype,W", [(65, "float64", 1024), (96, "float64", 1024), (97, "float64", 320),
                                       (128, "float64", 320), (65, "float32", 320), (128, "float32", 320),
                                       (33, "float64", 64), (64, "float32", 64)])
@pytest.mark.parametrize("over", [0, 1])
def test_solve_on_both_sides_of_the_split(n, dtype, W, over, device, monkeypatch):
    """W nodes at level 0 sweep persistently, W + 1 by the level kernels and the upper
    level persistently: against the oracle (three systems, repeated over the batch)."""
    import numpy as np
    import torch
    from oracle import nd
    from socu_amd.block_tridiag_solver import create_cholesky_factor_launch, create_cholesky_solve_launch

    monkeypatch.delenv("SOCU_SWEEP", raising=False)
    tdt, B = getattr(torch, dtype), W + over  # N = 2: one node a system at level 0
    P = [nd.readme_problem(n, 2, 1, alpha=16.0, seed=60 + k)[:3] for k in range(3)]
    pick = torch.arange(B) % 3
    L, E, x = (torch.tensor(np.stack([p[i] for p in P]), dtype=tdt)[pick].to(device) for i in range(3))
    create_cholesky_factor_launch(L, E, dtype=tdt)()
    run = create_cholesky_solve_launch(L, E, x, dtype=tdt)
    run()
    assert run.sweep_status() == (True, False)
    # kappa(Psi) <= 1e3: 1e3 * N * 2^-53, and 2^-24
    tol = 1e-11 if dtype == "float64" else 5e-4
    for k in range(3):
        Lr, Er, xr = (a.copy() for a in P[k])
        nd.factor(Lr, Er)
        nd.solve(Lr, Er, xr)
        got = x[pick == k].double().cpu().numpy()
        assert np.abs(got - xr).max() <= tol * np.abs(xr).max()
