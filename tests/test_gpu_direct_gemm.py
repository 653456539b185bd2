"""The FP64 matvec where its GEMM can go wrong: sectors of one state and of odd
sizes, at and around the 4-deep k-steps, 16-deep slices, 16-wide blocks and
32-wide block pairs, on every tile shape, real and complex; plans that switch
between the FP64 and the reduced layouts; in-place products; batches in a split
mode.  Against the oracle; bars: FP64 1e-12 relative (sums of at most a few
thousand products of numbers in [-1, 1)), split modes their Frobenius bars."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle.bsten import OUT, BSTensor, Index
from oracle.lanczos import eff_ham_mul_two_site_state
from oracle.models import build_mpo, heisenberg_chain, phys_index
from tests.convert import to_device, to_oracle

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from ultradmrg_amd import _lib as L
    from ultradmrg_amd.solver import BatchedEffectiveHamiltonian, EffectiveHamiltonian

EDGES = [1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 49, 65]
LONG = [1, 131, 2, 257, 1]


def _problem(degs, seed, cplx=False):
    rng = np.random.default_rng(seed)
    m = heisenberg_chain(8)
    mpo = build_mpo(m)
    Wl, Wr = mpo[3], mpo[4]
    secs = [((2 * k - len(degs) // 2 * 2,), d) for k, d in enumerate(degs)]
    a, b, p = Index.make(secs, OUT), Index.make(secs, OUT), phys_index(m.qns, OUT)
    out = []
    for ixs in ([a.inverse(), Wl.indexes[0].inverse(), a], [b, Wr.indexes[3].inverse(), b.inverse()],
                [a.inverse(), p, p, b]):
        t = BSTensor(ixs, np.complex128 if cplx else np.float64, div=(0,))
        for c in t.allowed_blocks((0,)):
            t.blocks[c] = rng.uniform(-1, 1, size=t.blk_shape(c))
            if cplx:
                t.blocks[c] = t.blocks[c] + 1j * rng.uniform(-1, 1, size=t.blk_shape(c))
        out.append(t)
    if cplx:
        Ws = []
        for w in (Wl, Wr):
            c = BSTensor(w.indexes, np.complex128, w.div())
            c.blocks = {k: v + 0j for k, v in w.blocks.items()}
            Ws.append(c)
        Wl, Wr = Ws
    return [out[0], Wl, Wr, out[1]], out[2]


def _err(got, ref):
    got = to_oracle(got, ref)
    assert sorted(got.blocks) == sorted(ref.blocks)
    num = max(float(np.abs(got.blocks[k] - ref.blocks[k]).max()) for k in ref.blocks)
    return num / max(float(np.abs(v).max()) for v in ref.blocks.values())


@pytest.mark.parametrize("cplx,shape", [(False, s) for s in ("32x32", "64x32", "32x64", "64x64", "128x64", "64x128",
                                                             "128x128", "64x16", "128x16")] +
                         [(True, s) for s in ("32x32", "64x32", "32x64", "64x64")])
@pytest.mark.parametrize("degs", [EDGES, LONG], ids=["edges", "long"])
def test_edge_sectors(monkeypatch, degs, cplx, shape):
    print(f"[case] {degs} {'complex' if cplx else 'real'} {shape}", flush=True)
    monkeypatch.setenv("QLG_TILES", f"{shape},16x128,{shape}")
    eff, psi = _problem(degs, 5, cplx)
    ref = eff_ham_mul_two_site_state(eff, psi)
    H = EffectiveHamiltonian([to_device(t) for t in eff], to_device(psi))
    assert _err(H @ to_device(psi), ref) < 1e-12


@pytest.mark.parametrize("cplx,shape", [(False, s) for s in ("32x32", "64x32", "32x64", "64x64", "128x64", "64x128",
                                                             "128x128", "64x16", "128x16")] +
                         [(True, s) for s in ("32x32", "64x32", "32x64", "64x64")])
@pytest.mark.parametrize("degs", [EDGES, LONG], ids=["edges", "long"])
def test_edge_sectors_lds_kernel(monkeypatch, degs, cplx, shape):
    """The same on the LDS-staged kernel, which serves the plans whose spans the
    direct one cannot address (QLG_DIRECT=0 puts any plan there)."""
    print(f"[case] LDS kernel {degs} {'complex' if cplx else 'real'} {shape}", flush=True)
    monkeypatch.setenv("QLG_DIRECT", "0")
    test_edge_sectors(monkeypatch, degs, cplx, shape)


@pytest.mark.parametrize("shape", ["128x64", "64x128", "128x128"])
@pytest.mark.parametrize("degs", [EDGES, LONG], ids=["edges", "long"])
def test_wide_complex_tiles(monkeypatch, degs, shape):
    """Complex tiles that only the LDS-staged kernel has, pinned: it runs on the same
    k-major operands and row tables."""
    print(f"[case] {degs} complex {shape}", flush=True)
    monkeypatch.setenv("QLG_TILES", f"{shape},16x128,{shape}")
    eff, psi = _problem(degs, 5, True)
    ref = eff_ham_mul_two_site_state(eff, psi)
    H = EffectiveHamiltonian([to_device(t) for t in eff], to_device(psi))
    assert _err(H @ to_device(psi), ref) < 1e-12


@pytest.mark.parametrize("first", ["fp64", "bf16x6"])
def test_plan_switches_layouts(first):
    """One plan through FP64, both kinds of reduced layouts and back: the FP64
    results are the same bits, the reduced ones those of a plan of that mode."""
    print(f"[case] switching plan, first {first}", flush=True)
    eff, psi = _problem([7, 30, 41, 30, 7], 9)
    ref = eff_ham_mul_two_site_state(eff, psi)
    d_eff, x = [to_device(t) for t in eff], to_device(psi)
    H = EffectiveHamiltonian(d_eff, x, precision=first)
    got = {}
    for prec in (first, "fp64", "fp32", "bf16x3", "bf16x6", "fp64"):
        H.set_precision(prec)
        y = (H @ x).data
        if prec in got:
            assert torch.equal(got[prec], y), prec
        got[prec] = y
        if prec != "fp64":
            fresh = EffectiveHamiltonian(d_eff, x, precision=prec)
            assert torch.equal((fresh @ x).data, y), prec
    out = H @ x
    assert _err(out, ref) < 1e-12
    assert float(torch.linalg.vector_norm(got["bf16x6"] - out.data) / torch.linalg.vector_norm(out.data)) < 2e-6


@pytest.mark.parametrize("prec,cplx,bar", [("bf16x6", False, 2e-6), ("fp32", False, 2e-6), ("bf16x6", True, 2e-6)])
def test_reduced_padding_in_reused_memory(prec, cplx, bar):
    """The reduced operands' padding is written with them: a plan whose buffers held
    another plan's NaN gives the same bits as one on fresh buffers."""
    print(f"[case] reused buffers {prec} {'complex' if cplx else 'real'}", flush=True)
    eff, psi = _problem([3, 17, 29, 18, 2], 13, cplx)
    d_eff, x = [to_device(t) for t in eff], to_device(psi)
    bad = [to_device(t) for t in eff]
    for t in (bad[0], bad[3]):
        t.data.fill_(float("nan"))
    H = EffectiveHamiltonian(d_eff, x, precision=prec)
    want = (H @ x).data
    num = to_oracle(H @ x, psi)
    ref = eff_ham_mul_two_site_state(eff, psi)
    scale = np.sqrt(sum(float((np.abs(v) ** 2).sum()) for v in ref.blocks.values()))
    assert np.sqrt(sum(float((np.abs(num.blocks[k] - v) ** 2).sum()) for k, v in ref.blocks.items())) < bar * scale
    del H
    B = EffectiveHamiltonian(bad, x, precision=prec)
    assert torch.isnan(torch.view_as_real((B @ x).data) if cplx else (B @ x).data).any()
    B.close()
    assert torch.equal((EffectiveHamiltonian(d_eff, x, precision=prec) @ x).data, want)


def test_in_place_product():
    """qlg_matvec with one buffer as input and output."""
    print("[case] in place", flush=True)
    eff, psi = _problem([5, 21, 33, 20, 4], 11)
    H = EffectiveHamiltonian([to_device(t) for t in eff], to_device(psi))
    x = H.adopt(to_device(psi)).data.clone()
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    H.matvec_into(x, y)
    H.matvec_into(x, x)
    assert torch.equal(x, y)


def test_batch_in_split_mode():
    """A batch plan switched to a split mode (its reduced lists joined from the members')."""
    print("[case] batch bf16x6", flush=True)
    probs = [_problem(d, s) for s, d in enumerate(([3, 17, 29, 16, 2], [1, 40, 33, 1], [64, 65, 9]))]
    members = [EffectiveHamiltonian([to_device(t) for t in eff], to_device(psi)) for eff, psi in probs]
    B = BatchedEffectiveHamiltonian(members)
    x = B.pack([to_device(psi) for _, psi in probs])
    y = torch.empty_like(x)
    for prec, bar in ((L.QLG_PREC_F64, 1e-12), (L.QLG_PREC_BF16X6, 2e-6), (L.QLG_PREC_F64, 1e-12)):
        B.ctx.check(B.lib.qlg_plan_set_precision(B.h, prec))
        torch.cuda.synchronize()
        B.matvec_into(x, y)
        for (eff, psi), got in zip(probs, B.unpack(y)):
            assert _err(got, eff_ham_mul_two_site_state(eff, psi)) < bar


def test_batch_keeps_pinned_tiles(monkeypatch):
    """QLG_TILES holds for the batch of pinned plans too: the same tiles, so the same
    bits as the members' own products."""
    print("[case] pinned batch", flush=True)
    monkeypatch.setenv("QLG_TILES", "32x32,64x64,128x128")
    probs = [_problem(d, s) for s, d in enumerate(([30, 170, 290, 160, 20], [10, 140, 133, 9]))]
    members = [EffectiveHamiltonian([to_device(t) for t in eff], to_device(psi)) for eff, psi in probs]
    B = BatchedEffectiveHamiltonian(members)
    x = B.pack([to_device(psi) for _, psi in probs])
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    B.matvec_into(x, y)
    for m, (_, psi), got in zip(members, probs, B.unpack(y)):
        assert torch.equal((m @ to_device(psi)).data, got.data)
