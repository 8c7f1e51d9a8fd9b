"""Performance cases of the nested-dissection block-tridiagonal Cholesky.

Each case is one pass of a program that uses the public entry points: a model
writes the next problem's blocks into the arrays that a launch is bound to and
calls the launch (model-predictive control, trajectory optimisation, Kalman
smoothing), or calls the functional / differentiable interface on new tensors.

The matrices are those of the README generator (diagonal shift alpha on random
lower triangles, random couplings), drawn on the GPU.  Above n = 50 the shift
grows with sqrt(n), to 16 at n = 128: a constant shift of 10 is numerically
singular there.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from socu_amd import functional
from socu_amd.autograd import block_tridiag_solve
from socu_amd.batched import create_batched_cholesky_launch
from socu_amd.block_tridiag_solver import (
    calculate_off_diag_storage_len,
    create_cholesky_factor_and_solve_launch,
    create_cholesky_factor_launch,
    create_cholesky_solve_launch,
)
from socu_amd.mixed import create_cholesky_mixed_factor_and_solve_launch
from socu_amd.problems import MPC_BLOCK_SIZES, nd_flops

DTYPES = {"float64": torch.float64, "float32": torch.float32}


def listed():
    return [
        # one small MPC problem per control step: the smallest call, launch latency alone
        _regular("small_mpc", "factor_and_solve", 12, 20, 1),
        # the n=32, N=100 problem of the test configurations
        _regular("n32_N100", "factor_and_solve", 32, 100, 1),
        # the notebook's benchmark shape, factor and solve as two launches; n is no multiple of a tile
        _regular("notebook_n34_N128", "factor_then_solve", 34, 128, 1),
        # a long horizon with a panel of right-hand sides (sensitivities)
        _regular("n64_N1024_m16", "factor_and_solve", 64, 1024, 16),
        # the headline problem in plain FP64
        _regular("n128_N512", "factor_and_solve", 128, 512, 1),
        # the headline problem: FP32 factor, refined in FP64
        {**_regular("n128_N512_mixed", "mixed", 128, 512, 1), "precision": "float32", "max_iter": 3, "tol": 1e-10},
        # scenario MPC in single precision: equal small systems, the converged ones masked out, ragged n and N
        {**_regular("masked_f32_batch", "factor_and_solve", 20, 61, 1, B=256, dtype="float32"), "active": 0.75},
        # many solves with one factor (smoothing several signals): odd n, m > 1
        _regular("resolve_n100_N200_m8", "solve", 100, 200, 8),
        # thousands of uneven MPC systems in one launch: the largest call
        {"name": "uneven_mpc_4096", "kind": "batched", "count": 4096, "m": 1, "dtype": "float64", "graph": True},
        # a differentiable layer in training: forward and backward
        {"name": "gradient_B256_n32_N128_m4", "kind": "gradient", "B": 256, "n": 32, "N": 128, "m": 4,
         "dtype": "float64"},
        # the functional interface, eager, block size padded inside, single precision
        {"name": "functional_f32_n36_N100", "kind": "functional", "B": 8, "n": 36, "N": 100, "m": 3,
         "dtype": "float32"},
        # blocks above 128
        _regular("large_n200_N64_m2", "factor_and_solve", 200, 64, 2),
    ]


def _regular(name, kind, n, N, m, B=1, dtype="float64", graph=True):
    return {"name": name, "kind": kind, "B": B, "n": n, "N": N, "m": m, "dtype": dtype, "graph": graph}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["factor_and_solve", "factor_and_solve", "factor_then_solve", "solve", "mixed", "batched",
                       "gradient", "functional"])
    dtype = rng.choice(["float64", "float64", "float32"])
    m = rng.choice([1, 1, 1, 2, 3, 4, 8, 16])
    if kind == "batched":
        return {"kind": kind, "count": _log_int(rng, 16, 4096), "m": rng.choice([1, 1, 2, 3]), "dtype": dtype,
                "graph": rng.random() < 0.75}
    case = {"kind": kind, "B": 1, "n": _log_int(rng, 4, 128), "N": _log_int(rng, 8, 1024), "m": m, "dtype": dtype}
    if kind in ("gradient", "functional") or rng.random() < 0.4:
        case["B"] = _log_int(rng, 2, 512)
    if kind in ("factor_and_solve", "factor_then_solve", "solve"):
        case["graph"] = rng.random() < 0.75
        if rng.random() < 0.1:
            case["n"] = _log_int(rng, 129, 256)
        if case["B"] > 1 and rng.random() < 0.5:
            case["active"] = round(rng.uniform(0.4, 1.0), 2)
    if kind == "mixed":
        case.update(dtype="float64", graph=True, tol=1e-12)
        case["precision"] = rng.choice(["float32", "float32", "float32_f32_pivots", "bfloat16"])
        case["max_iter"] = 16 if case["precision"] == "bfloat16" else 5
    while case["B"] * sum(nd_flops(case["N"], case["n"], case["m"])) > 1.2e10 or \
            case["B"] * case["N"] * case["n"] ** 2 > 4e7:
        if case["B"] > 1:
            case["B"] = max(1, case["B"] // 2)
        else:
            case["N"] = max(8, case["N"] * 3 // 4)
            if case["N"] == 8:
                break
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _alpha(n):
    return max(10.0, 16.0 * math.sqrt(n / 128.0))


def _blocks(gen, lengths, n):
    """Diagonal blocks (M, n, n) of systems of the given lengths, one after
    the other, and the coupling block behind each diagonal block (zero behind
    a system's last), float64."""
    M = int(sum(lengths))
    D = torch.randn(M, n, n, generator=gen, dtype=torch.float64, device="cuda").tril_()
    D.diagonal(dim1=1, dim2=2).add_(_alpha(n))
    Ec = torch.randn(M, n, n, generator=gen, dtype=torch.float64, device="cuda")
    Ec[torch.as_tensor(np.cumsum(lengths) - 1, device="cuda")] = 0
    L = torch.bmm(D, D.transpose(1, 2).contiguous())
    L[1:] += torch.bmm(Ec[:-1], Ec[:-1].transpose(1, 2).contiguous())
    return L, torch.bmm(Ec, D.transpose(1, 2).contiguous())


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _problem(case, seed):
    """(L, E at full storage length, b) of B equal systems."""
    gen = _generator(seed)
    B, N, n, m = case["B"], case["N"], case["n"], case["m"]
    L, Ec = _blocks(gen, [N] * B, n)
    E = torch.zeros(B, calculate_off_diag_storage_len(N), n, n, dtype=torch.float64, device="cuda")
    E[:, : N - 1] = Ec.view(B, N, n, n)[:, : N - 1]
    b = torch.randn(B, N, n, m, generator=gen, dtype=torch.float64, device="cuda")
    return [t.to(DTYPES[case["dtype"]]) for t in (L.view(B, N, n, n), E, b)]


def _uneven_sizes(case):
    """The lengths and block sizes of the systems, in the order of the sizes."""
    rs = np.random.RandomState(case["count"])
    return rs.randint(10, 201, size=case["count"]), np.sort(rs.choice(MPC_BLOCK_SIZES, size=case["count"]))


def _uneven(case, seed):
    """(lengths, sizes, flat L, flat E, flat b) of `count` uneven systems, one
    after the other in the order of their sizes."""
    lengths, sizes = _uneven_sizes(case)
    gen, dt = _generator(seed), DTYPES[case["dtype"]]
    Ls, Es, bs = [], [], []
    for n in sorted(set(int(v) for v in sizes)):
        len_n = lengths[sizes == n]
        L, Ec = _blocks(gen, len_n, n)
        stored = np.array([calculate_off_diag_storage_len(int(N)) for N in len_n])
        E = torch.zeros(int(stored.sum()), n, n, dtype=torch.float64, device="cuda")
        within = np.concatenate([np.arange(N) for N in len_n])
        at = np.repeat(np.cumsum(stored) - stored, len_n) + within
        has = within < np.repeat(len_n, len_n) - 1
        E[torch.as_tensor(at[has], device="cuda")] = Ec[torch.as_tensor(has, device="cuda")]
        Ls.append(L.reshape(-1).to(dt))
        Es.append(E.reshape(-1).to(dt))
        bs.append(torch.randn(int(len_n.sum()) * n * case["m"], generator=gen, dtype=torch.float64,
                              device="cuda").to(dt))
    return lengths, sizes, torch.cat(Ls), torch.cat(Es), torch.cat(bs)


def _arena(tensors):
    """One buffer that holds the given tensors' values, each at a multiple of
    512 bytes, the views of it, and where the last one begins: a program that
    writes each new problem with one copy."""
    dt = tensors[0].dtype
    step = 512 // tensors[0].element_size()
    starts, end = [], 0
    for t in tensors:
        starts.append(end)
        end += -(-t.numel() // step) * step
    buf = torch.zeros(end, dtype=dt, device="cuda")
    views = [buf[s:s + t.numel()].view(t.shape) for s, t in zip(starts, tensors)]
    for v, t in zip(views, tensors):
        v.copy_(t)
    return buf, views, starts[-1]


def _mask(case, seed):
    if "active" not in case:
        return None
    rs = np.random.RandomState((seed + 7) % (1 << 32))
    return torch.as_tensor(rs.rand(case["B"]) < case["active"], device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "batched":
        lengths, sizes, L, E, b = _uneven(case, seed)
        data, (Ld, bd, Ed), _ = _arena([L, b, E])
        new = data.clone()
        Ls, Es, xs = [], [], []
        oL = oE = ob = 0
        for N, n in zip(lengths.tolist(), sizes.tolist()):
            nE = calculate_off_diag_storage_len(N)
            Ls.append(Ld[oL:oL + N * n * n].view(N, n, n))
            Es.append(Ed[oE:oE + nE * n * n].view(nE, n, n))
            xs.append(bd[ob:ob + N * n * case["m"]].view(N, n, case["m"]))
            oL, oE, ob = oL + N * n * n, oE + nE * n * n, ob + N * n * case["m"]
        launch = create_batched_cholesky_launch(Ls, Es, xs, dtype=DTYPES[case["dtype"]], use_cuda_graph=case["graph"])
        return {**state, "bound": data, "new": new, "launches": [launch], "out": [Ld, Ed, bd]}
    L, E, b = _problem(case, seed)
    if kind == "gradient":
        xbar = torch.randn(b.shape, generator=_generator(seed + 1), dtype=torch.float64, device="cuda").to(b.dtype)
        return {**state, "args": [t.requires_grad_() for t in (L, E, b)], "xbar": xbar}
    if kind == "functional":
        return {**state, "args": [L, E[:, : case["N"] - 1].contiguous(), b]}
    if kind == "mixed":
        x = b.clone()
        launch = create_cholesky_mixed_factor_and_solve_launch(
            L, E, x, precision=case["precision"], tol=case["tol"], max_iter=case["max_iter"],
            use_cuda_graph=case["graph"])
        return {**state, "bound": x, "new": b, "launches": [launch], "out": [x]}
    opt = {"mask": _mask(case, seed), "dtype": DTYPES[case["dtype"]], "use_cuda_graph": case["graph"]}
    if kind == "solve":
        create_cholesky_factor_launch(L, E, **{**opt, "use_cuda_graph": False})()
        x = b.clone()
        return {**state, "bound": x, "new": b, "launches": [create_cholesky_solve_launch(L, E, x, **opt)], "out": [x]}
    data, (Ld, xd, Ed), at_E = _arena([L, b, E])
    if case["B"] == 1:  # the coupling blocks lead E: the fill-in region behind them is not written
        data = data[: at_E + (case["N"] - 1) * case["n"] ** 2]
    if kind == "factor_then_solve":
        launches = [create_cholesky_factor_launch(Ld, Ed, **opt), create_cholesky_solve_launch(Ld, Ed, xd, **opt)]
    else:
        launches = [create_cholesky_factor_and_solve_launch(Ld, Ed, xd, **opt)]
    return {**state, "bound": data, "new": data.clone(), "launches": launches, "out": [Ld, Ed, xd]}


def run(state):
    if state["kind"] == "gradient":
        x = block_tridiag_solve(*state["args"])
        return [x, *torch.autograd.grad(x, state["args"], state["xbar"])]
    if state["kind"] == "functional":
        return list(functional.cholesky_factor_and_solve(*state["args"]))
    state["bound"].copy_(state["new"])  # the next problem's values into the bound arrays
    for launch in state["launches"]:
        launch()
    return state["out"]


# ---------------------------------------------------------------------------
# work and values
# ---------------------------------------------------------------------------

def _shapes(case):
    """(N, n) of every system a pass works on."""
    if case["kind"] == "batched":
        return list(zip(*(a.tolist() for a in _uneven_sizes(case))))
    return [(case["N"], case["n"])] * max(1, int(round(case["B"] * case.get("active", 1.0))))


def work(case):
    kind, m = case["kind"], case["m"]
    w = 4 if case["dtype"] == "float32" else 8
    flops = nbytes = 0.0
    for N, n in _shapes(case):
        factor, solve = nd_flops(N, n, m)
        tri, nn, nE = N * n * (n + 1) // 2, n * n, calculate_off_diag_storage_len(N)
        read_psi, vec = tri + (N - 1) * nn, N * n * m
        if kind == "solve":  # tril(L) and E of the factor, b; x
            flops += solve
            nbytes += w * (tri + nE * nn + 2 * vec)
        elif kind == "mixed":  # Psi and b; x
            flops += factor + solve
            nbytes += w * (read_psi + 2 * vec)
        elif kind == "gradient":  # Psi, b, xbar; x, the gradients (zeros in the fill-in region among them)
            flops += factor + 2 * solve + 2 * m * nn * (2 * N - 1)
            nbytes += w * (read_psi + 4 * vec + (N + nE) * nn)
        else:  # Psi and b; the factor with its inverses, the fill-in, x
            flops += factor + solve
            nbytes += w * (read_psi + 2 * vec + (N + nE) * nn)
    return {"bytes": float(nbytes), "flops": float(flops)}


def _nd_factor(L, E, lengths):
    """In-place ND block Cholesky in plain torch of systems stored one after
    the other: L (sum N, n, n), E (sum of storage lengths, n, n).  Returns the
    diagonal blocks' inverses and the levels' index arrays."""
    n = L.shape[-1]
    inv = torch.zeros_like(L)
    lengths = np.asarray(lengths)
    stored = np.array([calculate_off_diag_storage_len(int(N)) for N in lengths])
    oL, oE = np.cumsum(lengths) - lengths, np.cumsum(stored) - stored
    off, levels, s = np.zeros_like(lengths), [], 1
    eye = torch.eye(n, dtype=L.dtype, device=L.device)

    def on_gpu(a):
        return torch.as_tensor(np.ascontiguousarray(a), device=L.device)

    while s <= int(lengths.max()):
        count = np.maximum(0, (lengths - s) // (2 * s) + 1) * (lengths >= s)
        sysno = np.repeat(np.arange(len(lengths)), count)
        t = np.arange(len(sysno)) - np.repeat(np.cumsum(count) - count, count)
        i = (2 * t + 1) * s - 1
        r, c = i + s < lengths[sysno], t > 0
        node, seg = oL[sysno] + i, oE[sysno] + off[sysno]
        off = off + np.where(lengths >= s, lengths // s - 1, 0)
        lev = {"node": on_gpu(node), "R": on_gpu((seg + 2 * t)[r]), "r": on_gpu(np.flatnonzero(r)),
               "up": on_gpu((node + s)[r]), "C": on_gpu((seg + 2 * t - 1)[c]), "c": on_gpu(np.flatnonzero(c)),
               "down": on_gpu((node - s)[c]), "both": on_gpu(np.flatnonzero(r & c)),
               "F": on_gpu((oE[sysno] + off[sysno] + t - 1)[r & c]),
               "Rb": on_gpu((seg + 2 * t)[r & c]), "Cb": on_gpu((seg + 2 * t - 1)[r & c])}
        Lk = torch.linalg.cholesky(L[lev["node"]])
        Ik = torch.linalg.solve_triangular(Lk, eye.expand_as(Lk), upper=False)
        L[lev["node"]], inv[lev["node"]] = Lk, Ik
        R = torch.bmm(E[lev["R"]], Ik[lev["r"]].transpose(1, 2).contiguous())
        C = torch.bmm(Ik[lev["c"]], E[lev["C"]])
        E[lev["R"]], E[lev["C"]] = R, C
        L[lev["up"]] -= torch.bmm(R, R.transpose(1, 2).contiguous())
        L[lev["down"]] -= torch.bmm(C.transpose(1, 2).contiguous(), C)
        E[lev["F"]] = -torch.bmm(E[lev["Rb"]], E[lev["Cb"]])
        levels.append(lev)
        s *= 2
    return inv, levels


def _nd_solve(E, inv, levels, b):
    x = b.clone()
    for lev in levels:
        y = torch.bmm(inv[lev["node"]], x[lev["node"]])
        x[lev["node"]] = y
        x[lev["up"]] -= torch.bmm(E[lev["R"]], y[lev["r"]])
        x[lev["down"]] -= torch.bmm(E[lev["C"]].transpose(1, 2).contiguous(), y[lev["c"]])
    for lev in reversed(levels):
        y = x[lev["node"]]
        y[lev["r"]] -= torch.bmm(E[lev["R"]].transpose(1, 2).contiguous(), x[lev["up"]])
        y[lev["c"]] -= torch.bmm(E[lev["C"]], x[lev["down"]])
        x[lev["node"]] = torch.bmm(inv[lev["node"]].transpose(1, 2).contiguous(), y)
    return x


def _factor_and_solve(L, E, b, lengths):
    """(stored L: the factor with its transposed inverse above the diagonal,
    E, x) and what a further solve needs."""
    L, E = L.double().clone(), E.double().clone()
    inv, levels = _nd_factor(L, E, lengths)
    x = _nd_solve(E, inv, levels, b.double())
    return L.tril() + inv.tril(-1).transpose(1, 2), E, x, inv, levels


def exact(case, seed):
    kind, m = case["kind"], case["m"]
    if kind == "batched":
        lengths, sizes, L, E, b = _uneven(case, seed)
        outs, oL, oE, ob = ([], [], []), 0, 0, 0
        for n in sorted(set(int(v) for v in sizes)):
            len_n = lengths[sizes == n]
            kL, kE = int(len_n.sum()), sum(calculate_off_diag_storage_len(int(N)) for N in len_n)
            got = _factor_and_solve(L[oL:oL + kL * n * n].view(kL, n, n), E[oE:oE + kE * n * n].view(kE, n, n),
                                    b[ob:ob + kL * n * m].view(kL, n, m), len_n)
            oL, oE, ob = oL + kL * n * n, oE + kE * n * n, ob + kL * n * m
            for o, v in zip(outs, got):
                o.append(v.reshape(-1))
        return [torch.cat(o) for o in outs]
    B, N, n = case["B"], case["N"], case["n"]
    L, E, b = _problem(case, seed)
    Lf, Ef, x, inv, levels = _factor_and_solve(L.view(-1, n, n), E.view(-1, n, n), b.view(-1, n, m), [N] * B)
    Lf, Ef, x = Lf.view(L.shape), Ef.view(E.shape), x.view(b.shape)
    if kind == "gradient":
        xbar = torch.randn(b.shape, generator=_generator(seed + 1), dtype=torch.float64, device="cuda").to(b.dtype)
        bbar = _nd_solve(Ef.view(-1, n, n), inv, levels, xbar.double().view(-1, n, m)).view(b.shape)

        def outer(u, v):
            return torch.bmm(u.reshape(-1, n, m), v.reshape(-1, n, m).transpose(1, 2).contiguous()).view(B, -1, n, n)

        dL = -(outer(bbar, x) + outer(x, bbar)).tril()
        dL.diagonal(dim1=2, dim2=3).mul_(0.5)
        dE = torch.zeros_like(Ef)
        dE[:, : N - 1] = -(outer(bbar[:, 1:], x[:, :-1]) + outer(x[:, 1:], bbar[:, :-1]))
        return [x, dL, dE, bbar]
    active = _mask(case, seed)
    if active is not None:  # a masked system's arrays stay as given
        keep = active.view(-1, 1, 1, 1)
        Lf, Ef, x = (torch.where(keep, f, g.double()) for f, g in ((Lf, L), (Ef, E), (x, b)))
    return [x] if kind in ("solve", "mixed") else [Lf, Ef, x]
