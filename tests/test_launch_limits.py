"""Systems and batches with more tasks per level than one launch takes."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,N", [(17, 4_900_000), (8, 17_000_000)])
def test_fp64_pivots_of_a_long_system(n, N, device):
    """n = 17 with 4.9 million blocks: 17 million 16x16 tiles of a level's Schur updates
    would be 2^32 threads and more (it takes 32x32 ones); n = 8 with 17 million blocks:
    so many 16x16 tiles.  Checked by the residual of a solve."""
    import torch
    from socu_amd import _lib

    print(f"long system n={n} N={N}", flush=True)
    gen = torch.Generator(device=device).manual_seed(1)
    # diagonally dominant: couplings of norm <= 2, diagonal blocks 8 I + (norm <= 1)
    C = torch.randn(N - 1, n, n, generator=gen, device=device) * 0.1
    D = torch.randn(N, n, n, generator=gen, device=device) * 0.05
    D = D + D.transpose(1, 2)
    D.diagonal(dim1=1, dim2=2).add_(8.0)
    nE = sum((N >> l) - 1 for l in range(N.bit_length()))
    L, E = D.clone(), torch.empty(nE, n, n, device=device)
    E[: N - 1] = C
    b = torch.randn(N, n, generator=gen, device=device)
    x = b.clone()
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    assert lib.socu_cholesky_factor_f32(L.data_ptr(), E.data_ptr(), None, 1, N, n, _lib.PREC_FP32, st) == 0
    assert lib.socu_cholesky_solve_with_inverses(L.data_ptr(), E.data_ptr(), x.data_ptr(), None, 1, N, n, 1,
                                                 _lib.DTYPE_F32, st) == 0
    del L, E
    step = 1 << 18
    for i in range(0, N, step):
        j = min(i + step, N)
        r = (D[i:j] * x[i:j, None]).sum(2) - b[i:j]
        lo, hi = max(i, 1), min(j, N - 1)
        r[lo - i:] += (C[lo - 1:j - 1] * x[lo - 1:j - 1, None]).sum(2)
        r[:hi - i] += (C[i:hi] * x[i + 1:hi + 1, :, None]).sum(1)
        # kappa <= 3: a few units of 2^-24 of the terms' size
        assert float(r.abs().max()) < 1e-5 * float(b.abs().max()), i


def test_bf16_schur_of_a_long_system(device):
    """n = 1 with 2^24 blocks and more: as many tasks of 256 threads.  Checked by the
    residual of a solve."""
    import torch
    from socu_amd import _lib

    N = 2**24 + 5
    print(f"long system bf16 n=1 N={N}", flush=True)
    gen = torch.Generator(device=device).manual_seed(3)
    D = 8 + torch.rand(N, generator=gen, device=device)
    C = 2 * torch.rand(N - 1, generator=gen, device=device) - 1
    b = torch.randn(N, generator=gen, device=device)
    nE = sum((N >> l) - 1 for l in range(N.bit_length()))
    L, E, x = D.clone(), torch.empty(nE, device=device), b.clone()
    E[: N - 1] = C
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    assert lib.socu_cholesky_factor_f32(L.data_ptr(), E.data_ptr(), None, 1, N, 1, _lib.PREC_BF16, st) == 0
    assert lib.socu_cholesky_solve_with_inverses(L.data_ptr(), E.data_ptr(), x.data_ptr(), None, 1, N, 1, 1,
                                                 _lib.DTYPE_F32, st) == 0
    r = D * x - b
    r[1:] += C * x[:-1]
    r[:-1] += C * x[1:]
    # products of two numbers rounded to 2^-9: of |C|^2 / D <= 1/6, two into a diagonal
    # block and one into a fill-in, 2e-3 and 7e-4 over the levels; |x| <= max |b| / 6
    assert float(r.abs().max()) < 1e-3 * float(b.abs().max())


def test_batch_of_many_block_rows(device):
    """69 million block rows in one batch: level 0 has 35 million tasks of two
    wavefronts (m > 16), 2^32 threads and more.  Equal systems, against the same
    system in a launch of its own."""
    import torch
    from socu_amd.batched import create_batched_cholesky_launch
    from socu_amd.block_tridiag_solver import calculate_off_diag_storage_len, create_cholesky_factor_and_solve_launch

    N, m, count, dt = 2**21, 17, 33, torch.float32
    print(f"batch of {count} systems n=1 N={N} m={m}", flush=True)
    gen = torch.Generator(device=device).manual_seed(2)
    nE = calculate_off_diag_storage_len(N)
    L0 = torch.rand(N, 1, 1, generator=gen, device=device) + 3.0
    E0 = torch.zeros(nE, 1, 1, device=device)
    E0[: N - 1] = torch.rand(N - 1, 1, 1, generator=gen, device=device)
    b0 = torch.randn(N, 1, m, generator=gen, device=device)
    L, E, x = (t.expand(count, *t.shape).contiguous() for t in (L0, E0, b0))
    create_batched_cholesky_launch(list(L), list(E), list(x), dtype=dt)()
    create_cholesky_factor_and_solve_launch(L0, E0, b0, dtype=dt)()
    for k in range(count):
        for got, want in ((L[k], L0), (E[k], E0), (x[k], b0)):
            assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max()), k
    del L, E, x
    torch.cuda.empty_cache()
