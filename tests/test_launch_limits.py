"""Systems and batches with more tasks per level than one launch takes."""
import pytest

pytestmark = pytest.mark.gpu


def test_fp64_pivots_of_a_long_system(device):
    """n = 17 with 4.9 million blocks: level 0 has 17 million 16x16 Schur tiles,
    2^32 threads and more.  Checked by the residual of a solve."""
    import torch
    from socu_amd import _lib

    n, N = 17, 4_900_000
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
