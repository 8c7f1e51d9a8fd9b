"""Sweeps whose block rows of right-hand sides are larger than 4 GiB: every kernel
of the level sweeps (one per range of n) addresses them with 64 bits.

The columns repeat with a period of 16, so each chunk of 16 has to come out as
the same sweep of the 16 columns alone, bit for bit.
"""
import pytest

from oracle import nd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 15, 20, 23, 40, 128, 200])
def test_block_rows_above_4_gib(n, device):
    import torch
    from socu_amd.block_tridiag_solver import (
        create_cholesky_backward_substitution_launch,
        create_cholesky_factor_launch,
        create_cholesky_forward_substitution_launch,
    )

    N, dt = 2, torch.float32
    m = 16 * (2**30 // (16 * (n - 1)) + 2)  # the last row begins beyond 2^32 bytes
    print(f"many rhs n={n} m={m}", flush=True)
    L0, E0, b0 = nd.readme_problem(n, N, 16, alpha=16.0, seed=n)[:3]
    L, E, y = (torch.tensor(a, dtype=dt, device=device) for a in (L0, E0, b0))
    create_cholesky_factor_launch(L, E, dtype=dt)()
    x = torch.empty(N, n, m, dtype=dt, device=device)
    chunks = x.view(N, n, m // 16, 16)
    chunks.copy_(y[:, :, None])
    for create in (create_cholesky_forward_substitution_launch, create_cholesky_backward_substitution_launch):
        create(L, E, y, dtype=dt)()
        create(L, E, x, dtype=dt)()
        for row in range(0, n, 32):
            assert bool((chunks[:, row:row + 32] == y[:, row:row + 32, None]).all()), (create.__name__, row)
    del x, chunks
    torch.cuda.empty_cache()
