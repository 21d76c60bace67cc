"""The calls of this framework that its speed is judged by.

The framework has one path: closed-shell CCSD(T). A user transforms the AO
integrals, iterates CCSD, evaluates E(T), and for properties its adjoint, on one
molecule after another. The cases below are those calls, through the Python
entry points of scess_amd, from a water-sized molecule, where every call is a
few launches long, to the o=30, v=300 and o=20, v=200 configurations of
bench.py and the GPU tests. The two largest are run as a shard of the occupied
triples (Context.set_shard), which is what one GPU of several evaluates.

Inputs follow the distribution of scess_amd/synthetic.py (uniform orbital
energies, integrals from a random symmetric factor, T2 of MP2 form), drawn on
the GPU; the factor is scaled by 0.25 so that the amplitudes have chemical size
and CCSD converges.
"""

from __future__ import annotations

import itertools
import math

import numpy as np
import torch

from scess_amd import gpu, triples
from scess_amd.synthetic import TriplesInputs

FACTOR_SCALE = 0.25


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # E(T) of a water-sized molecule (cc-pVDZ: o=5, v=19) in one call from host blocks: what a scan
        # over geometries does at every point; upload, repack and launches count
        {"name": "call_o5_v19", "kind": "call", "o": 5, "v": 19, "prec": "fp64"},
        # the same call for a medium molecule: upload, repack and contraction all count
        {"name": "call_o12_v120", "kind": "call", "o": 12, "v": 120, "prec": "fp64"},
        # E(T) and F_ijk from resident inputs at the o=20, v=200 configuration, the reference precision
        {"name": "forward_fp64_o20_v200", "kind": "forward", "o": 20, "v": 200, "prec": "fp64", "shard": 0, "nshards": 1},
        # one GPU's share of the benchmark configuration o=30, v=300, FP64
        {"name": "forward_fp64_o30_v300", "kind": "forward", "o": 30, "v": 300, "prec": "fp64", "shard": 5, "nshards": 16},
        # the same configuration with split-BF16x3 products, the fastest mode
        {"name": "forward_bf16x3_o30_v300", "kind": "forward", "o": 30, "v": 300, "prec": "bf16x3", "shard": 3, "nshards": 8},
        # and with exact int8 digits (five, the benchmark's choice)
        {"name": "forward_int8_o30_v300", "kind": "forward", "o": 30, "v": 300, "prec": "ozaki", "digits": 5, "shard": 7,
         "nshards": 16},
        # gradients of E(T) of a medium molecule with an odd number of virtuals
        {"name": "backward_o10_v75", "kind": "backward", "o": 10, "v": 75, "prec": "fp64", "shard": 0, "nshards": 1},
        # one GPU's share of the gradients at the adjoint configuration o=20, v=200
        {"name": "backward_o20_v200", "kind": "backward", "o": 20, "v": 200, "prec": "fp64", "shard": 2, "nshards": 8},
        # one CCSD residual update, Cholesky ladder, FP64 products
        {"name": "ccsd_update_fp64_o20_v200", "kind": "ccsd_update", "o": 20, "v": 200, "prec": "fp64", "vvvv": False},
        # one CCSD residual update with BF16x3 products, odd number of virtuals
        {"name": "ccsd_update_bf16x3_o16_v157", "kind": "ccsd_update", "o": 16, "v": 157, "prec": "bf16x3", "vvvv": False},
        # CCSD of a water-sized molecule to convergence (about ten DIIS iterations of small contractions)
        {"name": "ccsd_solve_o5_v19", "kind": "ccsd_solve", "o": 5, "v": 19, "prec": "fp64", "vvvv": True},
        # AO -> MO transform to <pq|rs>, as the CCSD(T) driver calls it (water cc-pVTZ size: 58 functions)
        {"name": "transform_n58", "kind": "transform", "nao": 58, "nmo": 58, "phys": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: any kind, sizes spread over their logarithm, work bounded by
    sharding as one of several GPUs would run it."""
    kind = rng.choice(["call", "forward", "forward", "forward", "backward", "backward", "ccsd_update", "ccsd_update",
                       "ccsd_solve", "transform"])
    if kind == "transform":
        nao = rng.randint(13, 64)
        return {"kind": kind, "nao": nao, "nmo": nao - rng.randint(0, 3), "phys": rng.random() < 0.5}
    if kind == "ccsd_solve":
        return {"kind": kind, "o": rng.randint(2, 6), "v": rng.randint(9, 30), "prec": "fp64", "vvvv": rng.random() < 0.5}
    if kind == "ccsd_update":
        return {"kind": kind, "o": rng.randint(5, 18), "v": _log(rng, 24, 190), "prec": rng.choice(["fp64", "fp64", "bf16x3", "fp32"]),
                "vvvv": False}
    if kind == "call":
        return {"kind": kind, "o": rng.randint(3, 12), "v": _log(rng, 10, 120), "prec": "fp64"}
    hi = 290 if kind == "forward" else 200
    o, v = rng.randint(4, 24), _log(rng, 19, hi)
    case = {"kind": kind, "o": o, "v": v, "prec": rng.choice(["fp64", "fp64", "bf16x3", "ozaki", "fp32"] if kind == "forward" else
                                                             ["fp64", "fp64", "ozaki"])}
    if case["prec"] == "ozaki":
        case["digits"] = rng.choice([5, 6, 7])
    # shards of at most a quarter second or so of FP64 work
    cost = 2.0 * (o * v) ** 3 * (o + v) * (1.0 if kind == "forward" else 3.0)
    case["nshards"] = max(1, math.ceil(cost / 1.0e13))
    case["shard"] = rng.randrange(case["nshards"])
    return case


# -------------------------------------------------------------- synthetic inputs
def _system(o, v, seed):
    """Orbital energies, the factor L[P, p, q] and t1, on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n, naux = o + v, 3 * v
    f = dict(generator=g, device="cuda", dtype=torch.float64)
    e = torch.cat([torch.sort(torch.rand(o, **f) * 1.2 - 1.5)[0], torch.sort(torch.rand(v, **f) * 2.9 + 0.1)[0]])
    L = torch.randn(naux, n, n, **f) * (FACTOR_SCALE / math.sqrt(naux))
    L = torch.triu(L) + torch.triu(L, 1).transpose(1, 2)
    t1 = torch.randn(o, v, **f) * 1e-3
    return e, L, t1


def _pair(L, s1, s2, s3, s4):
    """(pq|rs), p in s1, q in s2, r in s3, s in s4."""
    A, B = L[:, s1, s2], L[:, s3, s4]
    return (A.reshape(A.shape[0], -1).t() @ B.reshape(B.shape[0], -1)).reshape(*A.shape[1:], *B.shape[1:])


def _host(t):
    """ColMajor (Fortran-ordered) host array of a GPU tensor: the layout of the entry points."""
    return t.permute(*reversed(range(t.dim()))).contiguous().cpu().numpy().transpose()


def _denominators(e, o):
    eo, ev = e[:o], e[o:]
    return eo[:, None] - ev, eo[:, None, None, None] + eo[None, :, None, None] - ev[None, None, :, None] - ev


def _triples_tensors(case, seed):
    o, v = case["o"], case["v"]
    e, L, t1 = _system(o, v, seed)
    O, V = slice(0, o), slice(o, o + v)
    ovov = _pair(L, O, V, O, V)
    t2 = ovov.permute(0, 2, 1, 3) / _denominators(e, o)[1]
    return {"e": e, "t1": t1, "t2": t2.contiguous(), "ovvv": _pair(L, O, V, V, V), "ovoo": _pair(L, O, V, O, O), "ovov": ovov}


def _triples_inputs(case, seed):
    return TriplesInputs(o=case["o"], v=case["v"], **{k: _host(t) for k, t in _triples_tensors(case, seed).items()})


def _ccsd_tensors(case, seed):
    o, v = case["o"], case["v"]
    e, L, t1 = _system(o, v, seed)
    O, V = slice(0, o), slice(o, o + v)
    b = {"ovov": _pair(L, O, V, O, V), "oovv": _pair(L, O, O, V, V), "ovvo": _pair(L, O, V, V, O),
         "ovvv": _pair(L, O, V, V, V), "ovoo": _pair(L, O, V, O, O), "oooo": _pair(L, O, O, O, O)}
    if case["vvvv"]:
        b["vvvv"] = _pair(L, V, V, V, V)
    t2 = b["ovov"].permute(0, 2, 1, 3) / _denominators(e, o)[1]
    return e, b, L[:, O.stop:, O.stop:].permute(1, 2, 0), t1, t2.contiguous()


def _transform_tensors(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n, m = case["nao"], case["nmo"]
    L = torch.randn(2 * n, n, n, generator=g, device="cuda", dtype=torch.float64) / math.sqrt(2 * n)
    L = (L + L.transpose(1, 2)).reshape(2 * n, n * n)
    C = torch.linalg.qr(torch.randn(n, n, generator=g, device="cuda", dtype=torch.float64))[0][:, :m]
    return (L.t() @ L).reshape(n, n, n, n), C


# ------------------------------------------------------------------ prepare, run
def prepare(case, seed):
    kind = case["kind"]
    ctx = gpu.Context(0)
    state = {"kind": kind, "ctx": ctx}
    if kind == "transform":
        tei, C = _transform_tensors(case, seed)
        state.update(tei=_host(tei), C=_host(C), phys=case["phys"])
    elif kind.startswith("ccsd"):
        e, blocks, chol, t1, t2 = _ccsd_tensors(case, seed)
        ctx.set_ccsd_inputs(case["o"], case["v"], _host(e), {k: _host(b) for k, b in blocks.items()},
                            chol_vv=None if case["vvvv"] else _host(chol))
        ctx.set_ccsd_precision(case["prec"])
        if kind == "ccsd_update":
            state.update(t1=_host(t1), t2=_host(t2))
    else:
        inp = _triples_inputs(case, seed)
        state["prec"] = case["prec"]
        if kind == "call":
            state["inp"] = inp
        else:
            if case["prec"] == "ozaki":
                ctx.set_int8_digits(case["digits"])
            ctx.set_triples_inputs(inp, tuple({"fp64", case["prec"]}) if kind == "backward" else (case["prec"],))
            ctx.set_shard(case["shard"], case["nshards"])
    return state


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "call":
        return {"E": np.array([triples.triples_correction(state["inp"], precision=state["prec"], ctx=ctx)])}
    if kind == "forward":
        E, F, _ = ctx.triples_forward(state["prec"], with_F=True)
        return {"E": np.array([E]), "F": F}
    if kind == "backward":
        return ctx.triples_backward(state["prec"])
    if kind == "ccsd_update":
        t1, t2 = ctx.ccsd_update(state["t1"], state["t2"])
        return {"t1": t1, "t2": t2}
    if kind == "ccsd_solve":
        r = ctx.ccsd_solve()
        return {"E": np.array([r["E_CCSD"]]), "t1": r["t1"], "t2": r["t2"], "iterations": r["iterations"]}
    return {"tei": ctx.transform_tei(state["tei"], state["C"], chem_to_phys=state["phys"])}


def _shard(case):
    """The unique occupied triples (i >= j >= k, not all equal) of the case's shard, as (index, i, j, k)."""
    o, ns = case["o"], case.get("nshards", 1)
    every = [(i, j, k) for i in range(o) for j in range(i + 1) for k in range(j + 1)]
    todo = [(n, *t) for n, t in enumerate(every) if t[0] != t[2]]
    s = case.get("shard", 0)
    return len(every), todo[len(todo) * s // ns:len(todo) * (s + 1) // ns]


def work(case):
    """Bytes: host or resident inputs once and outputs once. Flops: the contractions of the path at 2 per
    multiply-add, half for triples with two equal indices; three times that for gradients."""
    kind = case["kind"]
    if kind == "transform":
        n, m = case["nao"], case["nmo"]
        return {"bytes": 8.0 * (n ** 4 + m ** 4 + n * m), "flops": 2.0 * (n ** 4 * m + n ** 3 * m ** 2 + n ** 2 * m ** 3 + n * m ** 4)}
    o, v = case["o"], case["v"]
    blocks = o * v ** 3 + o ** 3 * v + 2 * o * o * v * v + o * v
    if kind.startswith("ccsd"):
        # the o^2 v^4 ladder, its integrals from the factor (half by symmetry), the o^3 v^3 terms
        flops = 2.0 * o * o * v ** 4 / 2 + 2.0 * o ** 3 * v ** 3 * 8 + 2.0 * o ** 4 * v ** 2 * 2 + 2.0 * o * o * v ** 3 * 4
        flops += 0.0 if case["vvvv"] else 2.0 * v ** 4 * 3 * v / 2
        steps = 10 if kind == "ccsd_solve" else 1
        read = blocks + o * o * v * v * 2 + o ** 4 + (v ** 4 if case["vvvv"] else 3 * v ** 3)
        return {"bytes": 8.0 * steps * (read + 2 * o * o * v * v), "flops": steps * flops}
    todo = _shard(case)[1]
    units = sum(0.5 if i == j or j == k else 1.0 for _, i, j, k in todo)
    flops = units * 12.0 * v ** 3 * (o + v)
    if kind == "backward":
        return {"bytes": 8.0 * 2 * blocks, "flops": 3.0 * flops}
    size = {"fp64": 8, "fp32": 4, "bf16x3": 4, "ozaki": case.get("digits", 5)}[case["prec"]]
    return {"bytes": float(size * blocks), "flops": flops}


# --------------------------------------------------------------------- 64 bits
def _f_ijk(x, ovvv, i, j, k):
    """F_ijk = sum_abc W r3(W + V) / D of one occupied triple; ovvv: the slices (px|yf) by p."""
    e, t1, t2, o = x["e"], x["t1"], x["t2"], x["t1"].shape[0]
    v = t1.shape[1]
    W = 0.0
    for s in itertools.permutations(range(3)):
        p, q, r = ((i, j, k)[n] for n in s)
        w = (ovvv[p].reshape(v * v, v) @ t2[r, q].t()).reshape(v, v, v)
        w = w - (x["ovoo"][p, :, :, q] @ t2[:, r].reshape(o, v * v)).reshape(v, v, v)
        W = W + w.permute(*(s.index(n) for n in range(3)))
    S = lambda p, q: 0.5 * (x["ovov"][p, :, q] + x["ovov"][q, :, p].t())  # noqa: E731
    Y = W + S(i, j)[:, :, None] * t1[k] + S(i, k)[:, None, :] * t1[j][:, None] + S(j, k) * t1[i][:, None, None]
    ev = e[o:]
    D = e[i] + e[j] + e[k] - ev[:, None, None] - ev[:, None] - ev
    r3 = 4 * Y + Y.permute(2, 0, 1) + Y.permute(1, 2, 0) - 2 * (Y.permute(2, 1, 0) + Y.permute(0, 2, 1) + Y.permute(1, 0, 2))
    return (W * r3 / D).sum()


def _exact_triples(case, seed):
    x = _triples_tensors(case, seed)
    count, todo = _shard(case)
    if case["kind"] == "backward":
        ovvv = [s.clone().requires_grad_() for s in x.pop("ovvv")]
        for k in ("t1", "t2", "ovoo", "ovov"):
            x[k].requires_grad_()
        for _, i, j, k in todo:
            ((1.0 if i == j or j == k else 2.0) * _f_ijk(x, ovvv, i, j, k)).backward()
        g = {k: x[k].grad if x[k].grad is not None else torch.zeros_like(x[k]) for k in ("t1", "t2", "ovoo", "ovov")}
        g["ovvv"] = torch.stack([s.grad if s.grad is not None else torch.zeros_like(s) for s in ovvv])
        return g
    F = torch.zeros(count, dtype=torch.float64, device="cuda")
    w = torch.zeros_like(F)
    for n, i, j, k in todo:
        F[n] = _f_ijk(x, x["ovvv"], i, j, k)
        w[n] = 1.0 if i == j or j == k else 2.0
    E = (w * F).sum().reshape(1)
    return {"E": E} if case["kind"] == "call" else {"E": E, "F": F}


def _tau(t1, t2):
    return t2 + torch.einsum("ia,jb->ijab", t1, t1)


def _ccsd_update(e, b, chol, t1, t2):
    """One Jacobi update of the closed-shell CCSD amplitudes."""
    o, v = t1.shape
    ein = torch.einsum
    P = lambda X: X + X.permute(1, 0, 3, 2)  # noqa: E731
    tau = _tau(t1, t2)
    ovov, oovv, ovvo, ovvv, ovoo = (b[k] for k in ("ovov", "oovv", "ovvo", "ovvv", "ovoo"))
    Lov = 2 * ovov - ovov.permute(0, 3, 2, 1)
    Foo = ein("kcld,ilcd->ki", Lov, tau)
    Fvv = -ein("kcld,klad->ac", Lov, tau)
    Fov = ein("kcld,ld->kc", Lov, t1)
    n1 = t1 @ Fvv.t() - Foo.t() @ t1 + ein("kc,kica->ia", Fov, 2 * t2 - t2.permute(1, 0, 2, 3)) + (t1 @ Fov.t()) @ t1
    n1 = n1 + 2 * ein("kcai,kc->ia", ovvo, t1) - ein("kiac,kc->ia", oovv, t1)
    n1 = n1 + 2 * ein("kdac,ikcd->ia", ovvv, tau) - ein("kcad,ikcd->ia", ovvv, tau)
    n1 = n1 - 2 * ein("lcki,klac->ia", ovoo, tau) + ein("kcli,klac->ia", ovoo, tau)

    n2 = ovov.permute(0, 2, 1, 3).clone()
    n2 += P(ein("iacb,jc->ijab", ovvv, t1) - ein("kibj,ka->ijab", ein("kibc,jc->kibj", oovv, t1), t1))
    n2 -= P(ein("akij,kb->ijab", ein("kcai,jc->akij", ovvo, t1) + ein("iajk->akij", ovoo), t1))
    Loo = Foo + 2 * ein("lcki,lc->ki", ovoo, t1) - ein("kcli,lc->ki", ovoo, t1)
    Lvv = Fvv + 2 * ein("kdac,kd->ac", ovvv, t1) - ein("kcad,kd->ac", ovvv, t1)
    Wo = b["oooo"].permute(0, 2, 1, 3) + ein("lcki,jc->klij", ovoo, t1) + ein("kclj,ic->klij", ovoo, t1)
    Wo = Wo + ein("kcld,ijcd->klij", ovov, tau)
    n2 += ein("klij,klab->ijab", Wo, tau)
    for a in range(v):  # (ac|bd) tau_ij^cd, a slab of the v^4 integrals at a time
        slab = b["vvvv"][a] if "vvvv" in b else ein("cP,bdP->cbd", chol[a], chol)
        n2[:, :, a] += ein("cbd,ijcd->ijb", slab, tau)
    Z = ein("kdac,ijcd->kaij", ovvv, tau)
    n2 -= ein("kaij,kb->ijab", Z, t1) + ein("kbji,ka->ijab", Z, t1)
    n2 += P(ein("ac,ijcb->ijab", Lvv, t2) - ein("ki,kjab->ijab", Loo, t2))
    Wx = ein("kcai->akic", ovvo) + ein("kcad,id->akic", ovvv, t1) - ein("kcli,la->akic", ovoo, t1)
    Wx = Wx - 0.5 * ein("ldkc,ilda->akic", ovov, t2) - 0.5 * ein("lckd,ilad->akic", ovov, t2) + ein("ldkc,ilad->akic", ovov, t2)
    Wx = Wx - ein("lkci,la->akic", ein("ldkc,id->lkci", ovov, t1), t1)
    Wy = ein("kiac->akci", oovv) + ein("kdac,id->akci", ovvv, t1) - ein("lcki,la->akci", ovoo, t1)
    Wy = Wy - 0.5 * ein("lckd,ilda->akci", ovov, t2) - ein("lcki,la->akci", ein("lckd,id->lcki", ovov, t1), t1)
    n2 += P(2 * ein("akic,kjcb->ijab", Wx, t2) - ein("akci,kjcb->ijab", Wy, t2))
    n2 -= P(ein("akic,kjbc->ijab", Wx, t2) + ein("bkci,kjac->ijab", Wy, t2))
    d1, d2 = _denominators(e, o)
    return n1 / d1, n2 / d2


def exact(case, seed):
    kind = case["kind"]
    if kind == "transform":
        tei, C = _transform_tensors(case, seed)
        g = torch.einsum("abcd,ap,bq,cr,ds->pqrs", tei, C, C, C, C)
        return {"tei": g.permute(0, 2, 1, 3) if case["phys"] else g}
    if not kind.startswith("ccsd"):
        return _exact_triples(case, seed)
    e, b, chol, t1, t2 = _ccsd_tensors(case, seed)
    if kind == "ccsd_update":
        n1, n2 = _ccsd_update(e, b, chol, t1, t2)
        return {"t1": n1, "t2": n2}
    t1, t2 = torch.zeros_like(t1), b["ovov"].permute(0, 2, 1, 3) / _denominators(e, case["o"])[1]
    for _ in range(120):
        n1, n2 = _ccsd_update(e, b, chol, t1, t2)
        done = max((n1 - t1).abs().max(), (n2 - t2).abs().max()) < 1e-14
        t1, t2 = n1, n2
        if done:
            break
    g = b["ovov"].permute(0, 2, 1, 3)
    return {"E": ((2 * g - g.transpose(2, 3)) * _tau(t1, t2)).sum().reshape(1), "t1": t1, "t2": t2, "iterations": None}
