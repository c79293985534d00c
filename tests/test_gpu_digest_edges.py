"""
The single-read J/K digestion at the edges of its routes: bases of one angular
momentum, integral lists past the size of one launch, direct mode's pieces,
matrices of more than 16384 orbitals, builds that a graph records, what difference
builds leave out, densities with one dominant element, coefficients of any magnitude.
"""

import numpy as np
import pytest

from tests.conftest import cluster, water_dimer

pytestmark = pytest.mark.gpu


def _table(l):
    return {"H": [[l, [1.7, 0.4], [0.6, 0.7]]]}


def _points(n, spacing=2.2, seed=0):
    """n points of a cubic lattice, shaken."""
    k = int(np.ceil(n ** (1.0 / 3.0)))
    grid = np.array([[i, j, m] for i in range(k) for j in range(k) for m in range(k)][:n], float)
    return spacing * grid + 0.2 * np.random.default_rng(seed).standard_normal((n, 3))


def _dens(n, nset, seed=0):
    import torch
    D = np.random.default_rng(seed).standard_normal((nset, n, n))
    return torch.tensor(D + D.transpose(0, 2, 1), device="cuda")


@pytest.mark.parametrize("nset", [1, 2])
@pytest.mark.parametrize("l,natm", [(0, 1), (0, 30), (1, 1), (1, 12), (2, 1), (2, 6), (2, 19), (2, 20)])
def test_bases_of_one_angular_momentum(oracle_lib, l, natm, nset):
    """One shell per atom, so one pair class and one to six quartet classes (19 and 20 d shells
    lie on both sides of the rule that launches heavy and light classes apart), against the
    oracle at 1e-11 as every other J/K test."""
    from aimd_amd.qc.basis import basis_from_table
    from aimd_amd.qc.engine import Engine
    s, x = ["H"] * natm, _points(natm)
    e = Engine(basis_from_table(s, x, _table(l)))
    e.set_jk_mode("store")
    e.set_geometry(x)
    D = _dens(e.nao, nset, l)
    J, K = e.jk(D)
    Jo, Ko = oracle_lib.Pairs(oracle_lib.make_basis(s, x, _table(l))).jk_direct(D.cpu().numpy())
    assert np.abs(Jo).max() > 1e-3 and np.abs(Ko).max() > 1e-3
    np.testing.assert_allclose(J.cpu().numpy(), Jo, rtol=0, atol=1e-11)
    np.testing.assert_allclose(K.cpu().numpy(), Ko, rtol=0, atol=1e-11)
    e.close()


@pytest.mark.parametrize("l", [0, 1, 2])
def test_batches_of_one_angular_momentum(oracle_lib, monkeypatch, l):
    import torch
    import aimd_amd.batch as batch_module
    from aimd_amd.qc.basis import basis_from_table
    monkeypatch.setattr(batch_module, "build_basis", lambda s, x, name: basis_from_table(s, x, _table(l)))
    sizes = [2, 3, 4]
    xs = [_points(n, seed=n) for n in sizes]
    batch = batch_module.ReplicaBatch([(["H"] * n, n % 2, 1) for n in sizes], jk_lanes=16)
    batch._set_geometry(np.concatenate(xs))
    n = batch.ld
    D = torch.zeros((len(sizes), 2, n, n), dtype=torch.float64, device="cuda")
    for r, nr in enumerate(batch.rep_nao):
        D[r, :, :nr, :nr] = _dens(int(nr), 2, r)
    batch._jk(D)
    for r, (nr, x) in enumerate(zip(batch.rep_nao, xs)):
        ob = oracle_lib.make_basis(["H"] * sizes[r], x, _table(l))
        Jo, Ko = oracle_lib.Pairs(ob).jk_direct(D[r, :, :nr, :nr].cpu().numpy())
        np.testing.assert_allclose(batch.J[r, :, :nr, :nr].cpu().numpy(), Jo, rtol=0, atol=1e-11)
        np.testing.assert_allclose(batch.K[r, :, :nr, :nr].cpu().numpy(), Ko, rtol=0, atol=1e-11)
    batch.close()


def test_more_contracted_quartets_than_one_launch_takes(oracle_lib):
    """220 hydrogen atoms, STO-3G, no screening: 295 million contracted (ss|ss) quartets in the
    store, more tiles than a grid of 1024-thread workgroups may have. Ten bohr apart, so
    that most pairs keep no primitive and the oracle walks them quickly."""
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    n = 220
    s, x = ["H"] * n, _points(n, 10.0)
    e = Engine(build_basis(s, x, "sto-3g"))
    e.set_jk_mode("store")
    e.set_geometry(x, 0.0)
    npair = n * (n + 1) // 2
    assert e.quartet_count() == npair * (npair + 1) // 2 > (1 << 32) // 1024 * 64
    D = _dens(n, 1, 3)
    J, K = e.jk(D)
    Jo, Ko = oracle_lib.Pairs(oracle_lib.make_basis(s, x, "sto-3g")).jk_direct(D.cpu().numpy(), 0.0)
    np.testing.assert_allclose(J.cpu().numpy(), Jo, rtol=0, atol=1e-11)
    np.testing.assert_allclose(K.cpu().numpy(), Ko, rtol=0, atol=1e-11)
    e.close()


@pytest.mark.parametrize("nset", [1, 2])
def test_direct_mode_does_not_depend_on_its_buffer(nset):
    """J and K of direct mode bit for bit the same whatever buffer the pieces are cut for: the
    smallest (64 MiB, runs of some classes longer than what is left of it), others, and one
    that holds the whole list; and again at the same geometry."""
    import torch
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    s, x = cluster("water8.xyz")
    e = Engine(build_basis(s, x, "6-31g*"))
    D = _dens(e.nao, nset, 7)
    ref = None
    for limit in (0, 1, 1, 70_000_000, 100_000_000, 0):
        e.set_jk_mode("direct", limit)
        e.set_geometry(x)
        out = e.jk(D)
        ref = ref or out
        for a, b in zip(ref, out):
            assert torch.equal(a, b), limit
    e.close()


def test_direct_mode_with_a_run_longer_than_its_buffer():
    """One far d shell with coefficients that lift only its quartets over the threshold: its
    (d d| run holds 240 thousand (s s| kets, 67 MB of integrals, more than the 64 MiB
    buffer. Direct mode takes the run whole, so it adds what store mode adds, bit for bit."""
    import torch
    from aimd_amd.qc.basis import BasisSet
    from aimd_amd.qc.engine import Engine
    n = 701
    x = np.concatenate([_points(n - 1, 1.0), [[400.0, 0.0, 0.0]]])
    b = BasisSet("custom", ["H"] * n, x, np.arange(n), [0] * (n - 1) + [2], np.arange(n + 1), [0.05] * (n - 1) + [1.0],
                 [0.07] * (n - 1) + [1e3])
    e = Engine(b)
    D = _dens(e.nao, 1, 9)
    out = []
    for mode in ("store", "direct"):
        e.set_jk_mode(mode, 1)
        e.set_geometry(x, 10.0)
        out.append(e.jk(D))
    assert e.class_counts()[0][15] * 36 * 8 > 64 << 20          # (d d|s s)
    for a, c in zip(*out):
        assert float(a.abs().max()) > 0.0 and torch.equal(a, c)
    e.close()


@pytest.mark.parametrize("mode", ["auto", "direct"])
def test_more_than_16384_orbitals(mode):
    """2732 d shells (16392 AOs, 3.7 million pairs), of which the last three sit close together
    and are the only ones tight enough for the threshold: J and K in their block equal those
    of the three atoms alone. The screening value of a lone shell grows as the fourth root
    of its exponent (products of two: 1, 2 and 4 for exponents 1 and 16)."""
    import torch
    from aimd_amd.qc.basis import BasisSet
    from aimd_amd.qc.engine import Engine
    n, tail = 2732, 3
    near = np.array([[0.0, 0.0, 0.0], [0.3, 0.1, 0.0], [0.0, 0.2, 0.25]])
    x = np.concatenate([_points(n - tail, 40.0), near - 100.0])
    ex = np.where(np.arange(n) < n - tail, 1.0, 16.0)

    def engine(pos, exps):
        m = len(exps)
        b = BasisSet("d", ["H"] * m, pos, np.arange(m), np.full(m, 2), np.arange(m + 1), exps, 0.7 * exps ** 1.75)
        e = Engine(b)
        e.set_jk_mode(mode)
        return e

    small = engine(x[-tail:], ex[-tail:])
    small.set_geometry(x[-tail:], 0.0)
    q = small.schwarz_bounds()
    thr = 0.75 * q[0] ** 2
    small.set_geometry(x[-tail:], thr)
    e = engine(x, ex)
    e.set_geometry(x, thr)
    assert e.nao == 16392 and e.quartet_count() == small.quartet_count() >= 6
    D = torch.zeros((1, e.nao, e.nao), dtype=torch.float64, device="cuda")
    m = 6 * tail
    D[0, -m:, -m:] = _dens(m, 1, 5)[0]
    J, K = e.jk(D)
    for got, ref in zip((J, K), small.jk(D[:, -m:, -m:].contiguous())):
        assert float((got[:, -m:, -m:] - ref).abs().max()) < 1e-12 * float(ref.abs().max())
        assert float(got[:, :-m].abs().max()) == 0.0
    e.close()
    small.close()


@pytest.mark.parametrize("nset", [1, 2])
@pytest.mark.parametrize("mode", ["direct", "store"])
def test_builds_recorded_in_a_graph(mode, nset):
    """A captured build replayed with other densities, with eager builds and waits between the
    replays, equals the eager one bit for bit (two densities of 152 orbitals take the
    launches per class, one the launch of all classes)."""
    import torch
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    s, x = cluster("water8.xyz")
    e = Engine(build_basis(s, x, "6-31g*"))
    e.set_jk_mode(mode, 1 if mode == "direct" else 0)
    e.set_geometry(x)
    D = _dens(e.nao, nset)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        e.jk(D)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = e.jk(D)
    for seed in range(1, 5):
        D.copy_(_dens(e.nao, nset, seed))
        ref = e.jk(D)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, ref):
            assert torch.equal(a, b), seed
    del graph
    e.close()


@pytest.mark.parametrize("name,nset", [("dimer", 1), ("water8", 2)])
def test_difference_build_skips_only_what_is_below_the_threshold(name, nset):
    """What a screened build leaves out, element by element, is at most the sum of |integral
    bounds| |dD| over the products below the threshold (Schwarz bounds and densities as given,
    not a count times the threshold); something is left out, and everything is when the threshold
    is above every product. The bounds tell a threshold that is off by a thousand. One launch
    for all classes (dimer) and launches per class."""
    import torch
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    s, x = water_dimer() if name == "dimer" else cluster("water8.xyz")
    b = build_basis(s, x, "6-31g*")
    assert b.nblock == b.nshell
    e = Engine(b)
    e.set_jk_mode("store")
    e.set_geometry(x)
    D = 1e-3 * _dens(e.nao, nset, 11)
    i = torch.arange(b.nshell)
    pair = torch.where(i[:, None] >= i[None], i[:, None] * (i[:, None] + 1) // 2 + i[None],
                       i[None] * (i[None] + 1) // 2 + i[:, None])
    ao = torch.as_tensor(b.ao_shell.copy())
    Q = torch.as_tensor(e.schwarz_bounds())[pair][ao][:, ao].cuda()
    full = e.jk_delta(D, 0.0)
    thr = 1e-8
    part = e.jk_delta(D, thr)
    off = e.jk_delta(D, 1e3 * thr)
    for s_ in range(nset):
        a = D[s_].abs()
        bound_j, bound_k = torch.empty_like(a), torch.empty_like(a)
        for m in range(e.nao):
            T = Q[m][:, None, None] * Q[None]               # (second index of the bra, k, l)
            T = torch.where(T * a.max() < thr, T, torch.zeros_like(T))
            bound_j[m] = (T * a[None]).sum(dim=(1, 2))
            # (m k|n l) D_kl: T indexed (k, n, l)
            bound_k[m] = (T * a[:, None, :]).sum(dim=(0, 2))
        for f, p, o, bound in ((full[0][s_], part[0][s_], off[0][s_], bound_j),
                               (full[1][s_], part[1][s_], off[1][s_], bound_k)):
            left = (f - p).abs()
            print(name, nset, s_, "left out", float(left.max()), "bound", float(bound.max()), flush=True)
            assert float(left.max()) > 0.0
            slack = 1e-14 * float(f.abs().max())
            assert bool((left <= bound + slack).all())
            assert bool(((f - o).abs() > bound + slack).any())
    for z in e.jk_delta(D, 1.001 * float(Q.max()) ** 2 * float(D.abs().max())):
        assert float(z.abs().max()) == 0.0
    e.close()


def test_one_dominant_density_element(oracle_lib):
    """The fixed-point words of a build have one resolution for every element, 2^-61 of a bound of
    the largest: with one density element of 1e10 the others keep an absolute error of that size
    (and of the FP64 lane sums, 2^-53 of the same bound), not a relative one."""
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    s, x = water_dimer()
    b = build_basis(s, x, "6-31g*")
    e = Engine(b)
    e.set_jk_mode("store")
    e.set_geometry(x)
    D = _dens(e.nao, 1, 13)
    D[0, 2, 2] = 1e10
    J, K = e.jk(D)
    Dh = D.cpu().numpy()
    Jo, Ko = oracle_lib.Pairs(oracle_lib.make_basis(s, x, "6-31g*")).jk_direct(Dh)
    q = e.schwarz_bounds()
    i = np.arange(b.nshell)
    hi, lo = np.maximum(i[:, None], i), np.minimum(i[:, None], i)
    Q = q[hi * (hi + 1) // 2 + lo][np.ix_(b.ao_shell, b.ao_shell)]
    a = np.abs(Dh[0])
    bound_j, bound_k = Q.max() * (Q * a).sum(), (Q ** 2).sum(axis=1).max() * a.sum(axis=1).max()
    assert np.abs(J.cpu().numpy() - Jo).max() < b.nao * 2.0 ** -53 * bound_j
    assert np.abs(K.cpu().numpy() - Ko).max() < b.nao * 2.0 ** -53 * bound_k
    e.close()


@pytest.mark.parametrize("power", [6, 10, 12, 40, -30])
def test_coefficients_of_any_magnitude(power):
    """Contraction coefficients scaled by c = 2^power scale every integral, J and K by c^4, whatever the
    magnitude of the Schwarz bounds that set the words' exponents (q grows as c^2: the sum of its
    squares passes 1e12 at 2^10)."""
    from aimd_amd.qc.basis import BasisSet, build_basis
    from aimd_amd.qc.engine import Engine
    s, x = water_dimer()
    b = build_basis(s, x, "6-31g*")
    D = _dens(b.nao, 2, 17)
    out = []
    for c in (1.0, 2.0 ** power):
        e = Engine(BasisSet("scaled", s, x, b.shell_atom, b.shell_l, b.shell_prim, b.prim_exp, c * b.prim_coef))
        e.set_jk_mode("store")
        e.set_geometry(x, 1e-12 * c ** 4)
        out.append(e.jk(D))
        e.close()
    for ref, got in zip(*out):
        assert float((got / 2.0 ** (4 * power) - ref).abs().max()) < 1e-13 * float(ref.abs().max())
