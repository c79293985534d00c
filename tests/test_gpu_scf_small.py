"""
The single-launch SCF algebra of small matrices against numpy in FP64: Fock matrices
with energies and commutators, the Pulay step over a filling and a wrapping ring,
densities with frozen replicas, S^(-1/2); at sizes on both sides of the 16-wide tiles.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    import torch
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


def _sym(rng, *shape):
    a = rng.standard_normal(shape)
    return 0.5 * (a + a.swapaxes(-1, -2))


@pytest.mark.parametrize("ld", [1, 16, 17, 38, 49, 64])
@pytest.mark.parametrize("nspin", [1, 2])
def test_fock_commutator_and_density(ld, nspin):
    import torch
    from aimd_amd import _lib
    L = _lib.lib()
    R, g = 3, 2.0 / nspin
    rng = np.random.default_rng(ld + nspin)
    H, S, X = _sym(rng, R, ld, ld), _sym(rng, R, ld, ld), rng.standard_normal((R, ld, ld))
    D, J, K, P = (_sym(rng, R, nspin, ld, ld) for _ in range(4))
    F = H[:, None] + g * J.sum(axis=1, keepdims=True) - K
    XT = X.swapaxes(1, 2)[:, None]
    FDS = F @ D @ S[:, None]
    E = XT @ (FDS - FDS.swapaxes(2, 3)) @ X[:, None]
    Fo = XT @ F @ X[:, None]
    en = 0.5 * g * (D * (H[:, None] + F)).sum(axis=(1, 2, 3))
    M, slot = 3, 2
    t = {k: _dev(v) for k, v in dict(H=H, S=S, X=X, D=D, J=J, K=K, P=P).items()}
    Fg, ring_f = torch.zeros_like(t["D"]), torch.zeros((R, M, nspin, ld, ld), dtype=torch.float64, device="cuda")
    ring_e, energy, err = torch.zeros_like(ring_f), torch.zeros(R, device="cuda", dtype=torch.float64), None
    err = torch.zeros_like(energy)
    sl = torch.tensor([slot], device="cuda")
    vec = nspin * ld * ld
    _lib.check(L.aimdhf_small_fock(R, nspin, ld, _ptr(t["H"]), _ptr(t["S"]), _ptr(t["X"]), _ptr(t["D"]), _ptr(t["J"]),
                                   _ptr(t["K"]), _ptr(Fg), _ptr(ring_f), _ptr(ring_e), M * vec, vec, _ptr(sl),
                                   _ptr(energy), _ptr(err), _stream()))
    # each of k chained products loses at most about ld eps of the product of the Frobenius norms
    nf = lambda a: np.sqrt((a * a).sum(axis=(-1, -2))).max()
    tol = 8 * ld * EPS * nf(X) ** 2 * nf(F)
    assert np.abs(Fg.cpu().numpy() - F).max() < 8 * EPS * np.abs(F).max() + 8 * EPS * np.abs(J).max()
    assert np.abs(ring_f.cpu().numpy()[:, slot] - Fo).max() < tol
    assert np.abs(ring_e.cpu().numpy()[:, slot] - E).max() < 4 * tol * nf(D) * nf(S)
    assert float(ring_f[:, :slot].abs().max()) == 0.0 and float(ring_e[:, :slot].abs().max()) == 0.0
    assert np.abs(energy.cpu().numpy() - en).max() < 8 * ld * ld * EPS * nspin * nf(D) * (nf(H) + nf(F))
    np.testing.assert_array_equal(err.cpu().numpy(), ring_e[:, slot].abs().amax(dim=(1, 2, 3)).cpu().numpy())
    # replica 0 was frozen before, replica 1 freezes now, replica 2 takes its new density
    frozen = torch.tensor([True, False, False], device="cuda")
    prev = energy.clone()
    prev[2] += 1.0
    count = torch.tensor([3], device="cuda")
    Dg = t["D"].clone()
    _lib.check(L.aimdhf_small_density(R, nspin, ld, _ptr(t["X"]), _ptr(t["P"]), _ptr(Dg), _ptr(frozen), _ptr(energy),
                                      _ptr(err), _ptr(prev), 1e-6, 1e300, _ptr(sl), _ptr(count), M, _stream()))
    assert frozen.tolist() == [True, True, False] and torch.equal(prev, energy)
    assert sl.tolist() == [0] and count.tolist() == [3]
    Dn = X[:, None] @ P @ XT
    assert torch.equal(Dg[:2], t["D"][:2])
    assert np.abs(Dg.cpu().numpy()[2] - Dn[2]).max() < 8 * ld * EPS * nf(X) ** 2 * nf(P)


@pytest.mark.parametrize("ld", [5, 17, 64])
@pytest.mark.parametrize("m", [2, 8, 12])
def test_pulay_step_over_the_ring(ld, m):
    import torch
    from aimd_amd import _lib
    L = _lib.lib()
    R, nspin, pad = 2, 1, 7.0
    rng = np.random.default_rng(10 * ld + m)
    E, F = (torch.zeros((R, m, nspin, ld, ld), dtype=torch.float64, device="cuda") for _ in range(2))
    G = torch.full((R, m, m), float("nan"), dtype=torch.float64, device="cuda")
    Fx = torch.zeros((R, nspin, ld, ld), dtype=torch.float64, device="cuda")
    nao = torch.tensor([ld, ld - 2], dtype=torch.int32, device="cuda")
    slot, count = torch.zeros(1, dtype=torch.long, device="cuda"), torch.zeros(1, dtype=torch.long, device="cuda")
    held = []
    for it in range(m + 3):
        e, f = rng.standard_normal((R, nspin, ld, ld)), rng.standard_normal((R, nspin, ld, ld))
        s = it % m
        E[:, s], F[:, s] = _dev(e), _dev(f)
        slot.fill_(s)
        count.fill_(min(it, m))
        held = (held + [(e, f)])[-m:]
        _lib.check(L.aimdhf_small_diis(R, nspin, ld, m, _ptr(slot), _ptr(count), _ptr(E), _ptr(F), _ptr(G), _ptr(nao),
                                       pad, _ptr(Fx), _stream()))
        for r in range(R):
            d = np.array([(e2[r] - held[-1][0][r]).ravel() for e2, _ in held[:-1]]).reshape(len(held) - 1, nspin * ld * ld)
            A, b = d @ d.T, -d @ held[-1][0][r].ravel()
            c = np.linalg.solve(A, b) if len(d) else np.zeros(0)
            c = np.append(c, 1.0 - c.sum())
            ref = sum(ci * f2[r] for ci, (_, f2) in zip(c, held))
            ref = ref + pad * np.diag((np.arange(ld) >= int(nao[r])).astype(float))
            cond = np.linalg.cond(A) if len(d) else 1.0
            tol = 100 * ld * ld * EPS * cond * max(1.0, np.abs(c).max()) * 5.0
            assert np.abs(Fx[r].cpu().numpy() - ref).max() < tol, (it, r, cond)


@pytest.mark.parametrize("ld", [1, 16, 17, 50, 64])
def test_inverse_square_root(ld):
    import torch
    from aimd_amd import _lib
    rng = np.random.default_rng(ld)
    R = 3
    S, lam = np.empty((R, ld, ld)), np.empty((R, ld))
    for r in range(R):
        Q, _ = np.linalg.qr(rng.standard_normal((ld, ld)))
        lam[r] = np.sort(np.exp(rng.uniform(np.log(1e-3), np.log(2.0), ld)))
        S[r] = (Q * lam[r]) @ Q.T
    S = 0.5 * (S + S.swapaxes(1, 2))
    St = _dev(S)
    X, out = torch.empty_like(St), torch.empty((R, 2), dtype=torch.float64, device="cuda")
    _lib.check(_lib.lib().aimdhf_small_inv_sqrt(R, ld, _ptr(St), _ptr(X), 60, 1e-12, _ptr(out), _stream()))
    w, U = np.linalg.eigh(S)
    ref = (U / np.sqrt(w)[:, None, :]) @ U.swapaxes(1, 2)
    # ld eps cond |X| = 64 x 2.2e-16 x 2e3 x 32
    assert np.abs(X.cpu().numpy() - ref).max() < 1e-9
    res, low = out.cpu().numpy().T
    assert res.max() < 1e-10 and (low <= lam[:, 0] * (1 + 1e-9)).all() and (low * ld > lam[:, 0] * 0.99).all()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 65, 304])
def test_purification_step_in_one_launch(n):
    import torch
    from aimd_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    X = (Q * rng.uniform(0.0, 1.0, n)) @ Q.T
    X = 0.5 * (X + X.T)
    T = (n + 15) // 16
    Xt = _dev(X)
    out = torch.full_like(Xt, float("nan"))
    sums, sums_out = torch.empty((2, 2, T * (T + 1) // 2), dtype=torch.float64, device="cuda")
    _lib.check(L.aimdhf_tc2_sums(n, _ptr(Xt), _ptr(sums), _stream()))
    tr, err = np.trace(X), abs(np.trace(X) - (X * X).sum())
    # |X| <= 1: every sum of n products of one row and one column is below 1
    tol = 8 * n * EPS
    for nocc, freeze, ref in ((tr - 0.5, 0.0, X @ X), (tr + 0.5, 0.0, 2 * X - X @ X), (tr, 2 * err + 1.0, X)):
        _lib.check(L.aimdhf_tc2_fused(n, _ptr(Xt), _ptr(out), _ptr(sums), _ptr(sums_out), nocc, freeze, _stream()))
        o = out.cpu().numpy()
        assert np.abs(o - ref).max() <= tol
        np.testing.assert_array_equal(o, o.T)
        s = sums_out.sum(dim=1).cpu().numpy()
        assert abs(s[0] - np.trace(o)) < tol * n and abs(s[1] - (o * o).sum()) < tol * n
