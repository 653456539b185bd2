"""Performance cases of the effective-Hamiltonian path: what a DMRG or TDVP
program has this framework do, at the sizes it does it.

Kinds of case:

* ``matvec``   one application of a planned H_eff (two-site or one-site, real
               or complex, any arithmetic mode) to a vector the caller holds;
* ``batch``    the same for several independent chains in one plan;
* ``lanczos``  one ground-state Krylov solve on a planned H_eff;
* ``expmv``    one exp(-i tau H_eff) psi on a planned H_eff (TDVP);
* ``svd``      the truncated block SVD of a two-site tensor and the product of
               its factors (the next update's starting state);
* ``env``      one environment update, planning included;
* ``sweep``    one two-site DMRG sweep of a short chain, everything included.

The operators of ``matvec`` and ``batch`` are random environments of a given
bond profile; those of ``lanczos`` and ``expmv`` are contracted from random
isometric site tensors, so that H_eff is Hermitian and on its physical scale.
"""
from __future__ import annotations

import functools
import itertools
import math

import numpy as np
import torch

from ultradmrg_amd import mpo as M
from ultradmrg_amd.solver import BatchedEffectiveHamiltonian, EffectiveHamiltonian, LanczosParams
from ultradmrg_amd.sweep import SweepParams, SweepStats, TwoSiteVMPS, block_svd, random_bonds, trivial_env
from ultradmrg_amd.tensor import IN, OUT, Axis, BlockTensor, contract, env_update
from ultradmrg_amd.workloads import gaussian_bond


def listed():
    return [
        # a bond near the end of a chain, or any bond early in a ramp of the
        # bond dimension: launches and waits count
        dict(name="matvec_heis_d32", kind="matvec", model="heis", sites=2, cplx=False, D=32, half=4, width=1.6,
             prec="fp64", call="matmul"),
        # the middle of the L=100 Heisenberg chain at the end of its ramp
        dict(name="matvec_heis_d1024", kind="matvec", model="heis", sites=2, cplx=False, D=1024, half=6, width=2.0,
             prec="fp64", call="into"),
        # the headline matvec of bench.py: many sectors, most of them narrow
        dict(name="matvec_hub_d2000", kind="matvec", model="hub", sites=2, cplx=False, D=2000, half=5, width=2.0,
             prec="fp64", call="into"),
        # a converged D=2000 state (25 sectors up to 332 states) in the split
        # mode that the D=2000 sweep comparison reports
        dict(name="matvec_hub_d2000_wide_x6", kind="matvec", model="hub", sites=2, cplx=False, D=2000, half=3,
             width=1.4, prec="bf16x6", call="into"),
        # TDVP at D=1500, complex: the forward evolution's matvec in FP64 ...
        dict(name="matvec_hub_c128_d1500", kind="matvec", model="hub", sites=2, cplx=True, D=1500, half=4, width=1.7,
             prec="fp64", call="into"),
        # ... and the one-site backward evolution's in its split mode
        dict(name="matvec_hub_c128_one_site_x6", kind="matvec", model="hub", sites=1, cplx=True, D=1500, half=4,
             width=1.7, prec="bf16x6", call="into"),
        # independent chains of mixed sizes in one launch per stage
        dict(name="batch_heis_16", kind="batch", chains=16, Dmin=128, Dmax=768, pick=7),
        # the ground-state solve of one two-site update, at its usual number
        # of iterations
        dict(name="lanczos_hub_d1600", kind="lanczos", D=1600, iters=16, prec="fp64"),
        # the exponential of one TDVP step
        dict(name="expmv_hub_c128_d600", kind="expmv", D=600, iters=10, prec="fp64"),
        # the SVD of a D=2000 update
        dict(name="svd_hub_d2000", kind="svd", model="hub", cplx=False, D=2000, half=5, width=2.0, decades=6.0),
        # the environment update of a D=2000 update
        dict(name="env_hub_d2000", kind="env", model="hub", cplx=False, D=2000, half=5, width=2.0, side="l"),
        # a whole sweep of a short chain, as in a first run on a new model
        dict(name="sweep_heis_l20_d48", kind="sweep", sites=20, D=48),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm; odd more often than not."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, v | 1) if rng.random() < 0.6 else v


def _profile(rng, model):
    if model == "heis":
        half = rng.randint(3, 12)
        return dict(half=half, width=round(rng.uniform(0.3, 0.45) * half, 3))
    half = rng.randint(3, 5)
    return dict(half=half, width=round(rng.uniform(0.38, 0.48) * half, 3))


def draw(rng):
    kind = rng.choices(["matvec", "batch", "lanczos", "expmv", "svd", "env", "sweep"], [9, 2, 2, 2, 2, 2, 1])[0]
    model = rng.choice(["heis", "hub"])
    cplx = rng.random() < 0.35
    top = 1024 if model == "heis" else 1500 if cplx else 2000
    if kind == "matvec":
        modes = ["fp64", "bf16x6", "bf16x3"] if cplx else ["fp64", "fp64", "bf16x6", "bf16x3", "fp32"]
        return dict(kind=kind, model=model, sites=rng.choice([2, 2, 1]), cplx=cplx, D=_log(rng, 24, top),
                    prec=rng.choice(modes), call=rng.choice(["into", "into", "matmul"]), **_profile(rng, model))
    if kind == "batch":
        return dict(kind=kind, chains=rng.randint(2, 16), Dmin=64, Dmax=_log(rng, 128, 768), pick=rng.randint(0, 999))
    if kind == "lanczos":
        return dict(kind=kind, D=_log(rng, 60, 1600), iters=rng.randint(8, 16),
                    prec=rng.choice(["fp64", "fp64", "bf16x6"]))
    if kind == "expmv":
        return dict(kind=kind, D=_log(rng, 60, 600), iters=rng.randint(6, 10), prec=rng.choice(["fp64", "bf16x6"]))
    if kind == "svd":
        return dict(kind=kind, model=model, cplx=cplx, D=_log(rng, 48, 600 if cplx or model == "heis" else 2000),
                    decades=round(rng.uniform(4.0, 10.0), 2), **_profile(rng, model))
    if kind == "env":
        return dict(kind=kind, model=model, cplx=cplx, D=_log(rng, 48, top), side=rng.choice("lr"),
                    **_profile(rng, model))
    return dict(kind=kind, sites=rng.randint(10, 20), D=_log(rng, 16, 48))


# ---------------------------------------------------------------------------
# block tensors
# ---------------------------------------------------------------------------
def _signed(ax, s):
    return ax.qns[s] if ax.dir == OUT else tuple(-v for v in ax.qns[s])


def _add(p, q):
    return tuple(a + b for a, b in zip(p, q))


def _allowed(axes, div):
    """Every sector combination of divergence ``div``, in lexicographic order."""
    last = {}
    for s in range(axes[-1].nsect):
        last.setdefault(_signed(axes[-1], s), []).append(s)
    out = []
    for c in itertools.product(*[range(ax.nsect) for ax in axes[:-1]]):
        q = tuple(div)
        for ax, s in zip(axes, c):
            q = tuple(a - b for a, b in zip(q, _signed(ax, s)))
        out += [c + (s,) for s in last.get(q, ())]
    return out


def _uniform(axes, div, gen, cplx):
    """All allowed blocks, filled with U[-1, 1) (real and imaginary parts)."""
    coords = _allowed(axes, div)
    n = sum(math.prod(ax.degs[s] for ax, s in zip(axes, c)) for c in coords)
    x = torch.rand(n * (2 if cplx else 1), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    return BlockTensor(axes, coords, torch.view_as_complex(x.view(-1, 2)) if cplx else x)


@functools.lru_cache(maxsize=None)
def _model(name):
    """The Hamiltonian a program works with: a chain whose middle has the full MPO bond."""
    return M.heisenberg_chain(8) if name == "heis" else M.hubbard_cylinder(4, 4)


@functools.lru_cache(maxsize=None)
def _mpo(name, cplx):
    return M.build_mpo(_model(name), dtype=torch.complex128 if cplx else torch.float64)


def _bond(case):
    return gaussian_bond(case["D"], case["half"], case["width"], 1 if case["model"] == "heis" else 2)


def _across(secs):
    """The bond on the other side of one site: a spin-1/2 chain's charges change parity from bond to bond."""
    return [((q[0] + 1,), d) for q, d in secs] if len(secs[0][0]) == 1 else secs


def _operators(model, cplx, sites, secs, gen):
    """Random L, W..., R and a state at a bond of sectors ``secs`` in the middle of the model."""
    mpo = _mpo(model, cplx)
    mid = _model(model).n // 2
    W = mpo[mid - 1:mid + 1] if sites == 2 else mpo[mid:mid + 1]
    zero = (0,) * len(secs[0][0])
    a, b = Axis.make(secs, OUT), Axis.make(secs if sites == 2 else _across(secs), OUT)
    phys = M.physical_axis(_model(model).qns, OUT)
    L = _uniform([a.inverse(), W[0].axes[0].inverse(), a], zero, gen, cplx)
    R = _uniform([b, W[-1].axes[3].inverse(), b.inverse()], zero, gen, cplx)
    psi = _uniform([a.inverse()] + [phys] * sites + [b], zero, gen, cplx)
    return [L, *W, R], psi


def _isometry(lvb, phys, rvb, div, left, rng, cplx):
    """A random site tensor, left- or right-isometric, every allowed block present."""
    axes = [lvb, phys, rvb]
    groups = {}
    for c in _allowed(axes, div):
        groups.setdefault(c[2] if left else c[0], []).append(c)
    blocks = {}
    for k, cs in groups.items():
        keep = rvb.degs[k] if left else lvb.degs[k]
        rows = [(lvb.degs[c[0]] if left else rvb.degs[c[2]]) * phys.degs[c[1]] for c in cs]
        G = rng.standard_normal((sum(rows), keep))
        if cplx:
            G = G + 1j * rng.standard_normal(G.shape)
        Q = np.linalg.qr(G)[0] if sum(rows) >= keep else G / math.sqrt(keep)
        for c, q in zip(cs, np.split(Q, np.cumsum(rows)[:-1])):
            blocks[c] = q if left else q.T
            blocks[c] = blocks[c].reshape(lvb.degs[c[0]], phys.degs[c[1]], rvb.degs[c[2]])
    return BlockTensor.from_blocks(axes, blocks, dtype=torch.complex128 if cplx else torch.float64)


def _mps(model, total, D, rng, cplx, centre):
    """Random site tensors: left-isometric before ``centre``, right-isometric from it on."""
    n, phys = model.n, M.physical_axis(model.qns, OUT)
    zero = tuple(0 for _ in total)
    bonds = [Axis.make([(zero, 1)], OUT)] + random_bonds(model, total, D) + [Axis.make([(zero, 1)], OUT)]
    out = []
    for i in range(n):
        lvb, rvb = bonds[i].inverse(), bonds[i + 1]
        out.append(_isometry(lvb, phys, rvb, total if i == 0 else zero, i < centre, rng, cplx))
    return out


def _hermitian(case, seed, cplx):
    """H_eff of the middle two sites of a half-filled 4x4 Hubbard cylinder, and a random state."""
    model, mpo = _model("hub"), _mpo("hub", cplx)
    mid, n = model.n // 2, model.n
    mps = _mps(model, (n, 0), case["D"], np.random.default_rng(seed), cplx, mid)
    dt = mps[0].data.dtype
    le = trivial_env(mps[0].axes[0], mpo[0].axes[0], "cuda", dt)
    for i in range(mid - 1):
        le = env_update(le, mps[i], mpo[i], "l")
    re = trivial_env(mps[-1].axes[2], mpo[-1].axes[3], "cuda", dt)
    for i in range(n - 1, mid, -1):
        re = env_update(re, mps[i], mpo[i], "r")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    psi = _uniform([mps[mid - 1].axes[0], mps[mid - 1].axes[1], mps[mid].axes[1], mps[mid].axes[2]], (0, 0), gen, cplx)
    psi.data /= torch.linalg.vector_norm(psi.data)
    return [le, mpo[mid - 1], mpo[mid], re], psi


def _two_site_state(case, gen):
    """A two-site tensor whose sector matrices have singular values that fall
    off like those of a correlated two-dimensional state: 10^(-decades x^(1/2))
    over x = j / rank, times the sector's weight."""
    secs, cplx = _bond(case), case["cplx"]
    a, b = Axis.make(secs, IN), Axis.make(secs, OUT)
    phys = M.physical_axis(_model(case["model"]).qns, OUT)
    psi = _uniform([a, phys, phys, b], (0,) * len(secs[0][0]), gen, cplx)
    dt = psi.data.dtype
    sizes = [psi.block_size(c) for c in psi.coords]
    weight = dict(secs)
    top = max(weight.values())
    for q, blks in _sectors(psi).items():
        rows, cols = _offsets(psi, blks)
        m, n = rows["n"], cols["n"]
        k = min(m, n)
        sv = 10.0 ** (-case["decades"] * torch.sqrt(torch.arange(k, device="cuda", dtype=torch.float64) / k))
        g = [torch.randn(s, generator=gen, device="cuda", dtype=dt) for s in ((m, k), (k, n))]
        X = (g[0] * sv) @ g[1]
        X *= weight.get(q, 1) / top / torch.linalg.vector_norm(X)
        for i in blks:
            c = psi.coords[i]
            r0, c0 = rows[c[:2]], cols[c[2:]]
            shp = psi.block_shape(c)
            blk = X[r0:r0 + shp[0] * shp[1], c0:c0 + shp[2] * shp[3]]
            psi.data[psi.offsets[i]:psi.offsets[i] + sizes[i]] = blk.reshape(-1)
    psi.data /= torch.linalg.vector_norm(psi.data)
    return psi


def _sectors(psi):
    """Blocks of a two-site tensor by the charge q that the new bond carries between (a, s1) and (s2, b)."""
    out = {}
    for i, c in enumerate(psi.coords):
        q = tuple(-v for v in _add(_signed(psi.axes[0], c[0]), _signed(psi.axes[1], c[1])))
        out.setdefault(q, []).append(i)
    return out


def _offsets(psi, blks):
    rows, cols = {"n": 0}, {"n": 0}
    for part, lo in ((rows, 0), (cols, 2)):
        for key in sorted({psi.coords[i][lo:lo + 2] for i in blks}):
            part[key] = part["n"]
            part["n"] += psi.axes[lo].degs[key[0]] * psi.axes[lo + 1].degs[key[1]]
    return rows, cols


def _members(case):
    """(D, half, width) of a batch's chains, from the case alone."""
    rng = np.random.default_rng(case["pick"])
    out = []
    for _ in range(case["chains"]):
        half = int(rng.integers(4, 9))
        D = int(round(math.exp(rng.uniform(math.log(case["Dmin"]), math.log(case["Dmax"])))))
        out.append((D, half, 0.35 * half))
    return out


# ---------------------------------------------------------------------------
# inputs and passes
# ---------------------------------------------------------------------------
def _inputs(case, seed):
    """The tensors of a case (no plans)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "matvec":
        return _operators(case["model"], case["cplx"], case["sites"], _bond(case), gen)
    if kind == "batch":
        return [_operators("heis", False, 2, gaussian_bond(D, half, width, 1), gen) for D, half, width in
                _members(case)]
    if kind in ("lanczos", "expmv"):
        return _hermitian(case, seed, kind == "expmv")
    if kind == "svd":
        return _two_site_state(case, gen)
    if kind == "env":
        secs, name, cplx = _bond(case), case["model"], case["cplx"]
        mid = _model(name).n // 2
        W = _mpo(name, cplx)[mid]
        phys = M.physical_axis(_model(name).qns, OUT)
        a, b = Axis.make(secs, OUT), Axis.make(_across(secs), OUT)
        zero = (0,) * len(secs[0][0])
        mps = _uniform([a.inverse(), phys, b], zero, gen, cplx)
        if case["side"] == "l":
            env = _uniform([a.inverse(), W.axes[0].inverse(), a], zero, gen, cplx)
        else:
            env = _uniform([b, W.axes[3].inverse(), b.inverse()], zero, gen, cplx)
        return env, mps, W
    raise ValueError(kind)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "sweep":
        # a chain in a random field, one sweep away from a random state
        rng = np.random.default_rng(seed)
        m = M.heisenberg_chain(case["sites"], fields=list(rng.uniform(-2, 2, size=case["sites"])))
        mps = _mps(m, (case["sites"] % 2,), case["D"], rng, False, 0)
        drv = TwoSiteVMPS(mps, M.build_mpo(m), SweepParams(1, case["D"], case["D"], 1e-12, LanczosParams(1e-11, 100),
                                                           verbose=False))
        drv.sweep()
        st["drv"] = drv
        st["start"] = (list(drv.mps), list(drv.lenvs), list(drv.renvs))
    elif kind == "svd":
        st["psi"] = _inputs(case, seed)
    elif kind == "env":
        st["env"], st["mps"], st["mpo"] = _inputs(case, seed)
    elif kind == "batch":
        ins = _inputs(case, seed)
        members = [EffectiveHamiltonian(eff, psi) for eff, psi in ins]
        st["H"] = BatchedEffectiveHamiltonian(members)
        st["x"] = st["H"].pack([psi for _, psi in ins])
        st["y"] = torch.zeros_like(st["x"])
    else:
        eff, psi = _inputs(case, seed)
        st["H"] = EffectiveHamiltonian(eff, psi, precision=case["prec"])
        st["psi"] = psi
        if kind == "matvec":
            st["x"], st["y"] = st["H"].adopt(psi).data, st["H"].new_vector().data
    torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matvec" and case["call"] == "matmul":
        return (state["H"] @ state["psi"]).data
    if kind in ("matvec", "batch"):
        # as in a program's own Krylov loop: the caller keeps the vectors
        state["H"].matvec_into(state["x"], state["y"], sync=False)
        return state["y"]
    if kind == "lanczos":
        res = state["H"].lanczos(state["psi"], LanczosParams(1e-30, case["iters"]))
        # an eigenvector's sign is free: take the one that points along the start
        x = res.gs_vec.data
        return {"energy": res.gs_eng, "psi": x * torch.sign(torch.dot(x, state["psi"].data))}
    if kind == "expmv":
        return state["H"].expmv(state["psi"], 0.05, LanczosParams(1e-30, case["iters"])).expmv.data
    if kind == "svd":
        psi, D = state["psi"], case["D"]
        r = block_svd(psi, 2, (0,) * psi.qn_len, 0.0, D, D)
        # the values without the zeros around them: their number does not depend on how they fall to the sectors
        return {"s": r.s.data[r.s.data != 0], "psi": contract(r.u, contract(r.s, r.vt)).data}
    if kind == "env":
        return env_update(state["env"], state["mps"], state["mpo"], case["side"]).data
    drv = state["drv"]
    drv.mps, drv.lenvs, drv.renvs = (list(v) for v in state["start"])
    drv.stats = SweepStats()
    drv.sweep()
    log = drv.stats.log
    return {"energy": np.array([u["e0"] for u in log]), "entropy": np.array([u["entropy"] for u in log])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _matvec_work(eff, psi):
    """Operands once, and the sector products of the first and the last
    contraction (the two with the MPO in between are a few percent more)."""
    L, R = eff[0], eff[-1]
    cplx = psi.is_complex
    per = 8 if cplx else 2
    wide = {}   # columns of the state per left sector
    for c in psi.coords:
        wide[c[0]] = wide.get(c[0], 0) + psi.block_size(c) // psi.axes[0].degs[c[0]]
    tall = {}   # rows of the result per right sector
    for c in psi.coords:
        tall[c[-1]] = tall.get(c[-1], 0) + psi.block_size(c) // psi.axes[-1].degs[c[-1]]
    flops = sum(per * L.block_size(c) * wide.get(c[2], 0) for c in L.coords)
    flops += sum(per * R.block_size(c) * tall.get(c[0], 0) for c in R.coords)
    item = 16 if cplx else 8
    return {"bytes": item * (sum(t.data.numel() for t in eff) + 2 * psi.data.numel()), "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "sweep":   # two products of the full state per update, about ten Krylov vectors each
        D, n = case["D"], case["sites"]
        return {"bytes": 2 * n * 8 * 12 * D * D, "flops": 2 * n * 10 * 2 * 2 * 5 * 4 * D ** 3 / 6}
    ins = _inputs(case, 1)
    if kind == "matvec":
        return _matvec_work(*ins)
    if kind == "batch":
        each = [_matvec_work(*m) for m in ins]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    if kind in ("lanczos", "expmv"):
        w = _matvec_work(*ins)
        return {"bytes": w["bytes"], "flops": w["flops"] * case["iters"]}
    if kind == "svd":
        # values and both sets of vectors of every sector, and the product of the kept ones
        item, per = (16, 4) if case["cplx"] else (8, 1)
        flops = 0
        for blks in _sectors(ins).values():
            rows, cols = _offsets(ins, blks)
            m, n = sorted((rows["n"], cols["n"]))
            flops += per * (4 * m * m * n + 8 * m ** 3)
        return {"bytes": item * 2 * ins.data.numel(), "flops": flops}
    env, mps, W = ins
    item, per = (16, 8) if case["cplx"] else (8, 2)
    far = 2 if case["side"] == "l" else 0
    near = 2 - far
    w_far = W.axes[3 if case["side"] == "l" else 0]
    cols = {}
    for c in mps.coords:
        cols[c[near]] = cols.get(c[near], 0) + mps.block_size(c) // mps.axes[near].degs[c[near]]
    flops = sum(per * env.block_size(c) * cols.get(c[2], 0) for c in env.coords)
    out_ax = [mps.axes[far], w_far, mps.axes[far].inverse()]
    if case["side"] == "l":
        out_ax = [mps.axes[2].inverse(), w_far, mps.axes[2]]
    rows = {}
    for c in mps.coords:
        rows[c[far]] = rows.get(c[far], 0) + mps.block_size(c) // mps.axes[far].degs[c[far]]
    out = [math.prod(ax.degs[s] for ax, s in zip(out_ax, c)) for c in _allowed(out_ax, (0,) * mps.qn_len)]
    flops += sum(per * math.prod(ax.degs[s] for ax, s in zip(out_ax, c)) * rows.get(c[0], 0)
                 for c in _allowed(out_ax, (0,) * mps.qn_len))
    return {"bytes": item * (env.data.numel() + mps.data.numel() + sum(out)), "flops": flops}


# About four times what each path was seen to differ by from `exact`.
_MODES = {"fp64": 1e-14, "fp32": 3e-6, "bf16x6": 3e-6, "bf16x3": 3e-5}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matvec", "batch"):
        return {"rel": _MODES[case.get("prec", "fp64")]}
    if kind == "lanczos":
        return {"rel": 1e-11 if case["prec"] == "fp64" else 1e-5}
    if kind == "expmv":
        return {"rel": 1e-12 if case["prec"] == "fp64" else 1e-5}
    if kind == "svd":   # the cut falls between values that differ by little
        return {"rel": 1e-10}
    if kind == "env":
        return {"rel": 1e-14}
    return {"rel": 1e-6}


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch
# ---------------------------------------------------------------------------
def _dense(t):
    """A block tensor as one dense array, sectors side by side."""
    start = [np.concatenate([[0], np.cumsum(ax.degs)]) for ax in t.axes]
    out = torch.zeros([ax.dim for ax in t.axes], dtype=t.data.dtype, device="cuda")
    for c, o in zip(t.coords, t.offsets):
        ix = tuple(slice(int(p[s]), int(p[s + 1])) for p, s in zip(start, c))
        out[ix] = t.data[o:o + t.block_size(c)].view(t.block_shape(c))
    return out


def _packed(d, axes, coords):
    """The listed blocks of a dense array, one after another."""
    start = [np.concatenate([[0], np.cumsum(ax.degs)]) for ax in axes]
    return torch.cat([d[tuple(slice(int(p[s]), int(p[s + 1])) for p, s in zip(start, c))].reshape(-1)
                      for c in coords])


def _apply(eff, x):
    """H_eff x on dense arrays."""
    L, R = eff[0], eff[-1]
    if len(eff) == 3:
        t = torch.tensordot(L, x, ([2], [0]))                     # a' w s b
        t = torch.tensordot(t, eff[1], ([1, 2], [0, 1]))          # a' b t z
        return torch.tensordot(t, R, ([3, 1], [1, 2]))            # a' t b'
    t = torch.tensordot(L, x, ([2], [0]))                         # a' w s1 s2 b
    t = torch.tensordot(t, eff[1], ([1, 2], [0, 1]))              # a' s2 b t1 y
    t = torch.tensordot(t, eff[2], ([4, 1], [0, 1]))              # a' b t1 t2 z
    return torch.tensordot(t, R, ([4, 1], [1, 2]))                # a' t1 t2 b'


def _krylov(eff, x, k):
    """k steps of the three-term Lanczos recurrence: basis, diagonal, off-diagonal."""
    nrm = torch.linalg.vector_norm(x)
    V, a, b = [x / nrm], [], []
    for m in range(k):
        w = _apply(eff, V[m])
        a.append(torch.vdot(V[m].reshape(-1), w.reshape(-1)).real.item())
        w = w - a[m] * V[m]
        if m:
            w = w - b[m - 1] * V[m - 1]
        if m + 1 < k:
            b.append(torch.linalg.vector_norm(w).item())
            V.append(w / b[m])
    T = np.diag(a) + np.diag(b, 1) + np.diag(b, -1)
    return V, T, nrm


def exact(case, seed):
    kind = case["kind"]
    if kind == "sweep":
        return None   # thousands of products
    ins = _inputs(case, seed)
    if kind == "matvec":
        eff, psi = ins
        return _packed(_apply([_dense(t) for t in eff], _dense(psi)), psi.axes, psi.coords)
    if kind == "batch":
        return torch.cat([_packed(_apply([_dense(t) for t in eff], _dense(psi)), psi.axes, psi.coords)
                          for eff, psi in ins])
    if kind in ("lanczos", "expmv"):
        eff, psi = ins
        V, T, nrm = _krylov([_dense(t) for t in eff], _dense(psi), case["iters"])
        w, U = np.linalg.eigh(T)
        c = U[:, 0] * np.sign(U[0, 0]) if kind == "lanczos" else (U * np.exp(-0.05j * w)) @ U[0] * nrm.item()
        x = sum(v * complex(z) if kind == "expmv" else v * float(z) for v, z in zip(V, c))
        x = _packed(x, psi.axes, psi.coords)
        if kind == "expmv":
            return x
        return {"energy": float(w[0]), "psi": x}
    if kind == "svd":
        psi, D = ins, case["D"]
        facs = {}
        for q, blks in _sectors(psi).items():
            rows, cols = _offsets(psi, blks)
            X = torch.zeros(rows["n"], cols["n"], dtype=psi.data.dtype)
            host = psi.data.cpu()
            for i in blks:
                c, shp = psi.coords[i], psi.block_shape(psi.coords[i])
                r0, c0 = rows[c[:2]], cols[c[2:]]
                X[r0:r0 + shp[0] * shp[1], c0:c0 + shp[2] * shp[3]] = \
                    host[psi.offsets[i]:psi.offsets[i] + psi.block_size(c)].view(shp[0] * shp[1], -1)
            facs[q] = (*torch.linalg.svd(X, full_matrices=False), rows, cols, blks)
        pool = torch.cat([f[1] for f in facs.values()])
        cut = torch.sort(pool, descending=True).values[min(D, pool.numel()) - 1]
        out = torch.zeros_like(psi.data, device="cpu")
        s_blocks = []
        for q in sorted(facs):
            U, S, Vh, rows, cols, blks = facs[q]
            k = int((S >= cut).sum())
            if k == 0:
                continue
            s_blocks.append(S[:k])
            X = (U[:, :k] * S[:k]) @ Vh[:k]
            for i in blks:
                c, shp = psi.coords[i], psi.block_shape(psi.coords[i])
                r0, c0 = rows[c[:2]], cols[c[2:]]
                out[psi.offsets[i]:psi.offsets[i] + psi.block_size(c)] = \
                    X[r0:r0 + shp[0] * shp[1], c0:c0 + shp[2] * shp[3]].reshape(-1)
        return {"s": torch.cat(s_blocks), "psi": out}
    env, mps, W = ins
    E, A, Wd = _dense(env), _dense(mps), _dense(W)
    if case["side"] == "l":
        t = torch.tensordot(E, A, ([2], [0]))                     # a' w s b
        t = torch.tensordot(t, Wd, ([1, 2], [0, 1]))              # a' b t z
        t = torch.tensordot(A.conj(), t, ([0, 1], [0, 2])).permute(0, 2, 1)   # b' z b
        axes = [mps.axes[2].inverse(), W.axes[3], mps.axes[2]]
    else:
        t = torch.tensordot(A, E, ([2], [2]))                     # a s b' z
        t = torch.tensordot(t, Wd, ([1, 3], [1, 3]))              # a b' w t
        t = torch.tensordot(A.conj(), t, ([1, 2], [3, 1])).permute(0, 2, 1)   # a' w a
        axes = [mps.axes[0].inverse(), W.axes[0], mps.axes[0]]
    return _packed(t, axes, _allowed(axes, (0,) * mps.qn_len))
