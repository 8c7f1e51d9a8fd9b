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


@pytest.mark.parametrize("n,B,want", [(4, 9, True), (16, 64, True), (16, 65, False), (32, 64, True), (33, 65, True)])
def test_mixed_solver_by_batch_and_block_size(n, B, want, device, monkeypatch):
    import torch
    from socu_amd.mixed import create_cholesky_mixed_factor_and_solve_launch

    monkeypatch.delenv("SOCU_SWEEP", raising=False)
    L, E, x = _arrays(n, B, device, torch.float64)
    run = create_cholesky_mixed_factor_and_solve_launch(L, E, x)
    assert run.sweep_status() == (want, False)
