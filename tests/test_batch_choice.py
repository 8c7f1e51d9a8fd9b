"""Batches by one workgroup per system (short systems) or by level launches (long
ones): which is taken, and that both give the oracle's results.
"""
import numpy as np
import pytest

from oracle import nd

pytestmark = pytest.mark.gpu

OPS = ["factor_and_solve", "factor", "solve", "forward_substitution", "backward_substitution"]


def _batch(shapes, device, dtype, seed=7):
    import torch

    P = [nd.readme_problem(n, N, m, alpha=10.0, seed=seed + k)[:3] for k, (N, n, m) in enumerate(shapes)]
    return P, [[torch.tensor(p[i], dtype=dtype, device=device) for p in P] for i in range(3)]


# sizes of a batch, its horizon, systems, right-hand sides, and whether a system
# is one workgroup's work
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("ns,N,count,m,op,one", [
    (range(1, 9), 6, 12, 1, "solve", True), (range(1, 9), 15, 30, 1, "factor", True),
    (range(1, 9), 40, 80, 1, "backward_substitution", True), (range(9, 17), 7, 16, 1, "factor_and_solve", True),
    (range(17, 33), 7, 30, 1, "solve", True), (range(1, 33), 15, 16, 1, "forward_substitution", True),
    (range(1, 9), 200, 16, 1, "factor_and_solve", False), (range(9, 17), 100, 30, 1, "factor", False),
    (range(17, 33), 150, 16, 1, "solve", False), (range(1, 33), 200, 64, 1, "factor_and_solve", False),
    (range(9, 17), 10, 16, 16, "backward_substitution", False)])
def test_choice(ns, N, count, m, op, one, graph, device, monkeypatch):
    import torch
    from socu_amd.batched import create_batched_cholesky_launch
    from socu_amd.block_tridiag_solver import calculate_off_diag_storage_len

    monkeypatch.delenv("SOCU_BATCHED_WAVES", raising=False)
    nE = calculate_off_diag_storage_len(N)
    sizes = [ns[k % len(ns)] for k in range(count)]
    L, E, x = ([torch.zeros(rows, n, c or n, dtype=torch.float64, device=device) for n in sizes]
               for rows, c in ((N, 0), (nE, 0), (N, m)))
    cfg = create_batched_cholesky_launch(L, E, None if op == "factor" else x, op=op, use_cuda_graph=graph).config()
    # (level launches report one or two wavefronts per node)
    got = {bound: v["waves"] for bound, v in cfg.items() if v["systems"]}
    assert all((w == 4) == one for w in got.values()), got


SHAPES = [(1, 1, 1), (2, 8, 3), (3, 5, 1), (6, 16, 2), (5, 13, 1), (4, 32, 1), (7, 17, 2), (9, 27, 1), (12, 3, 4),
          (15, 4, 1), (8, 12, 1)]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("waves", [None, 0])
@pytest.mark.parametrize("op", OPS)
def test_short_systems_match_oracle(op, waves, dtype, device, monkeypatch):
    """The default (one workgroup per system) and, by the override, level launches."""
    import torch
    from socu_amd.batched import create_batched_cholesky_launch

    if waves is None:
        monkeypatch.delenv("SOCU_BATCHED_WAVES", raising=False)
    else:
        monkeypatch.setenv("SOCU_BATCHED_WAVES", str(waves))
    tdt = getattr(torch, dtype)
    # kappa(Psi) <= 1e3: 1e3 * N * 2^-53, and 2^-24
    tol = 1e-11 if dtype == "float64" else 5e-4
    P, (L, E, x) = _batch(SHAPES, device, tdt)
    mask = torch.tensor([k != 4 for k in range(len(SHAPES))], device=device)
    if op not in ("factor", "factor_and_solve"):
        create_batched_cholesky_launch(L, E, op="factor", dtype=tdt, tune=False)()
    before = [[t.clone() for t in a] for a in (L, E, x)]
    create_batched_cholesky_launch(L, E, None if op == "factor" else x, op=op, mask=mask, dtype=tdt, tune=False)()
    for k, (L0, E0, b0) in enumerate(P):
        if k == 4:
            assert all(torch.equal(t[k], s[k]) for t, s in zip((L, E, x), before))
            continue
        Lr, Er, y = L0.copy(), E0.copy(), b0.copy()
        nd.factor(Lr, Er)
        if op in ("factor_and_solve", "solve", "forward_substitution"):
            nd.forward(Lr, Er, y)
        if op in ("factor_and_solve", "solve", "backward_substitution"):
            nd.backward(Lr, Er, y)
        for got, want in ((np.tril(L[k].double().cpu().numpy()), np.tril(Lr)), (E[k].double().cpu().numpy(), Er),
                          (x[k].double().cpu().numpy(), y)):
            assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (k, SHAPES[k])
