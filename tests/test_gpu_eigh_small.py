"""Small real symmetric matrices through ``qlg_eigh_batched``: orders around the
in-LDS solver's thread counts and its upper limit (32; 33 and up run on the
library's solver), odd orders, batches, and spectra that a Jacobi method can stumble
over (graded Gram matrices, repeated and zero eigenvalues, diagonal and
indefinite matrices).

Bars: an orthogonal method's backward error is a modest multiple of n eps |A|;
values and residuals are held to 4 n eps |A|_2, orthonormality to 8 n eps, with
numpy's ``eigvalsh`` (itself n eps |A|) as the reference."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from ultradmrg_amd.sweep import eigh_batched

EPS = np.finfo(float).eps
KINDS = ["random", "graded", "rank", "diagonal", "zero", "repeated"]


def _matrix(kind, n, rng):
    if kind == "random":
        a = rng.standard_normal((n, n))
        return a + a.T
    if kind == "graded":   # a unit-norm Gram matrix, singular values over 8 decades
        x = (rng.standard_normal((n, n)) * 10.0 ** (-8.0 * np.arange(n) / n)) @ rng.standard_normal((n, 2 * n))
        x /= np.linalg.norm(x)
        return x @ x.T
    if kind == "rank":
        x = rng.standard_normal((n, max(1, n // 3)))
        return x @ x.T
    if kind == "diagonal":
        return np.diag(rng.standard_normal(n))
    if kind == "zero":
        return np.zeros((n, n))
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    return (q * np.where(np.arange(n) % 2, 2.0, -1.0)) @ q.T


@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 24, 25, 31, 32, 33, 64, 97])
def test_small_orders(n):
    print(f"[case] order {n}", flush=True)
    rng = np.random.default_rng(n)
    mats = []
    for k in KINDS:
        a = _matrix(k, n, rng)
        mats.append((a + a.T) / 2)
    dev = torch.from_numpy(np.stack(mats)).cuda()
    (w, v), = eigh_batched([dev.contiguous()])
    w, v = w.cpu().numpy(), v.cpu().numpy()
    for k, a, wi, vi in zip(KINDS, mats, w, v):
        nrm = max(np.linalg.norm(a, 2), np.finfo(float).tiny)
        assert np.all(np.diff(wi) >= 0), k
        assert np.abs(wi - np.linalg.eigvalsh(a)).max() <= 4 * n * EPS * nrm, k
        assert np.linalg.norm(a @ vi - vi * wi, 2) <= 4 * n * EPS * nrm, k
        assert np.linalg.norm(vi.T @ vi - np.eye(n), 2) <= 8 * n * EPS, k


def test_mixed_groups():
    """Small and large orders in one call, and a non-finite input beside finite ones."""
    print("[case] mixed groups", flush=True)
    rng = np.random.default_rng(0)
    groups = []
    for n, b in ((16, 5), (32, 2), (130, 3), (40, 1)):
        a = rng.standard_normal((b, n, n))
        groups.append((a + a.transpose(0, 2, 1)) / 2)
    groups[0][2, 3, 1] = groups[0][2, 1, 3] = np.nan
    out = eigh_batched([torch.from_numpy(g.copy()).cuda() for g in groups])
    for g, (w, v) in zip(groups, out):
        w, v = w.cpu().numpy(), v.cpu().numpy()
        for a, wi, vi in zip(g, w, v):
            if not np.isfinite(a).all():
                assert not np.isfinite(wi).any()
                continue
            n = a.shape[0]
            assert np.linalg.norm(a @ vi - vi * wi, 2) <= 4 * n * EPS * np.linalg.norm(a, 2)


@pytest.mark.parametrize("power", [-1030, -665, 665, 1010])
@pytest.mark.parametrize("n", [2, 17, 32])
def test_any_scale(n, power):
    """Matrices scaled by 2^power, down to denormal elements and up to where their
    squares overflow.  The bars are those of the unscaled matrix (the input's own
    rounding to denormal numbers is part of the matrix) plus the rounding of a
    value to a denormal number, 2^-1075."""
    print(f"[case] order {n} scaled by 2^{power}", flush=True)
    rng = np.random.default_rng(n)
    mats = np.stack([(lambda a: np.ldexp((a + a.T) / 2, power))(_matrix(k, n, rng)) for k in KINDS])
    (w, v), = eigh_batched([torch.from_numpy(mats.copy()).cuda()])
    w, v = np.ldexp(w.cpu().numpy(), -power), v.cpu().numpy()
    for k, a, wi, vi in zip(KINDS, np.ldexp(mats, -power), w, v):
        bar = 4 * n * EPS * max(np.linalg.norm(a, 2), np.finfo(float).tiny) + 2.0 ** max(-1075 - power, -1000)
        assert np.all(np.diff(wi) >= 0), k
        assert np.abs(wi - np.linalg.eigvalsh(a)).max() <= bar, k
        assert np.linalg.norm(a @ vi - vi * wi, 2) <= bar, k
        assert np.linalg.norm(vi.T @ vi - np.eye(n), 2) <= 8 * n * EPS, k


def test_upper_triangle_is_the_input():
    """Both solvers read the row-major upper triangle and the diagonal: with anything
    below it the results are those of the symmetric matrix, bit for bit."""
    print("[case] garbage below the diagonal", flush=True)
    rng = np.random.default_rng(1)
    groups = []
    for n, b in ((1, 2), (2, 3), (17, 4), (32, 2), (40, 2)):
        a = rng.standard_normal((b, n, n))
        groups.append((a + a.transpose(0, 2, 1)) / 2)
    whole = eigh_batched([torch.from_numpy(g.copy()).cuda() for g in groups])
    half = eigh_batched([torch.from_numpy(np.triu(g) + np.tril(np.full(g.shape, 7.5), -1)).cuda() for g in groups])
    for (w, v), (wh, vh) in zip(whole, half):
        assert torch.equal(w, wh) and torch.equal(v, vh)


@pytest.mark.parametrize("n", [16, 24, 32])
def test_no_less_accurate_than_the_library(n):
    """Residual and orthonormality of the in-LDS solver, means over 24 random and 24
    graded matrices in extended precision, against the library's solver on the same
    matrices as complex ones.  Both are orthogonal methods whose mean errors are
    those of many roundings; a quarter is allowed for the means' scatter."""
    print(f"[case] accuracy at order {n}", flush=True)
    rng = np.random.default_rng(100 + n)
    mats = [_matrix(k, n, rng) for k in ("random", "graded") for _ in range(24)]
    mats = np.stack([(a + a.T) / 2 for a in mats])
    err = {}
    for name, dt in (("small", np.float64), ("library", np.complex128)):
        (w, v), = eigh_batched([torch.from_numpy(mats.astype(dt)).cuda()])
        w, v = w.cpu().numpy().astype(np.longdouble), v.cpu().numpy().astype(np.clongdouble)
        res = [np.linalg.norm((a @ vi - vi * wi).astype(complex)) / np.linalg.norm(a, 2)
               for a, wi, vi in zip(mats, w, v)]
        orth = [np.linalg.norm((vi.conj().T @ vi - np.eye(n)).astype(complex)) for vi in v]
        err[name] = np.mean(res), np.mean(orth)
    print(f"  residual {err['small'][0]:.2e} library {err['library'][0]:.2e}, orthonormality "
          f"{err['small'][1]:.2e} library {err['library'][1]:.2e}", flush=True)
    assert err["small"][0] <= 1.25 * err["library"][0]
    assert err["small"][1] <= 1.25 * err["library"][1]
