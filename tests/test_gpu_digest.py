"""
The single-read J/K digestion (jk_digest*.hip) where it can go wrong: matrices too
large for a bra's rows in LDS, densities of extreme magnitude (the fixed-point
exponents follow them), zero and NaN densities, difference builds, and replicas of
a batch that must not affect each other. J/K over ordinary sizes, both precisions
and both reference routes: test_gpu_engine.py, test_gpu_clusters.py.
"""

import numpy as np
import pytest

from tests.conftest import ANG, WATER, bohr, water_dimer

pytestmark = pytest.mark.gpu


def _engine(s, x, basis, mode="store"):
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    e = Engine(build_basis(s, x, basis))
    e.set_jk_mode(mode)
    e.set_geometry(x)
    return e


def _dens(n, nset, seed=0, scale=1.0):
    import torch
    D = np.random.default_rng(seed).standard_normal((nset, n, n))
    return torch.tensor(scale * (D + D.transpose(0, 2, 1)), device="cuda")


@pytest.mark.parametrize("nset", [1, 2])
def test_rows_that_do_not_fit_lds(oracle_lib, nset):
    """44 waters 12 angstrom apart (836 AOs): the 12 rows of a (d d) bra take more than a
    CU's LDS, the other classes' rows do not; every class against the oracle. Entries are
    sums of about 1e5 products of magnitude one: 1e-11, as the smaller systems' tests."""
    s, w = bohr(WATER)
    grid = np.array([[i, j, k] for i in range(4) for j in range(4) for k in range(3)][:44], float) * 12.0 * ANG
    x = np.concatenate([w + g for g in grid])
    e = _engine(s * 44, x, "6-31g*")
    D = _dens(e.nao, nset)
    J, K = e.jk(D)
    Jo, Ko = oracle_lib.Pairs(oracle_lib.make_basis(s * 44, x, "6-31g*")).jk_direct(D.cpu().numpy())
    np.testing.assert_allclose(J.cpu().numpy(), Jo, rtol=0, atol=1e-11)
    np.testing.assert_allclose(K.cpu().numpy(), Ko, rtol=0, atol=1e-11)
    e.close()


@pytest.mark.parametrize("scale", [1e12, 1e-12, 1e-30])
def test_density_magnitude(scale):
    """J and K are linear: scaled densities give scaled results to the resolution of the
    fixed-point words, 2^-62 of a bound within 1e5 of the largest element (1e-13)."""
    s, x = water_dimer()
    e = _engine(s, x, "6-31g**")
    D = _dens(e.nao, 2, 1)
    ref = e.jk(D)
    out = e.jk(D * scale)
    for a, b in zip(ref, out):
        assert float((a - b / scale).abs().max()) < 1e-13 * float(a.abs().max()), scale
    e.close()


def test_zero_and_nan_densities():
    import torch
    s, x = water_dimer()
    e = _engine(s, x, "6-31g*")
    D = _dens(e.nao, 2, 2)
    ref = e.jk(D)
    for z in e.jk(torch.zeros_like(D)):
        assert float(z.abs().max()) == 0.0
    bad = D.clone()
    bad[1, 3, 5] = float("nan")
    J, K = e.jk(bad)
    assert torch.isnan(J[1]).all() and torch.isnan(K[1]).all()      # flagged, and confined to its density
    assert torch.equal(J[0], ref[0][0]) and torch.equal(K[0], ref[1][0])
    bad[1, 3, 5] = float("inf")
    assert torch.isnan(e.jk(bad)[0][1]).any()
    for a, b in zip(ref, e.jk(D)):
        assert torch.equal(a, b)
    e.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_difference_build(precision):
    """Threshold 0 skips nothing; with a threshold every skipped product is below it (a row
    of n^2 products per element)."""
    import torch
    from aimd_amd.qc.basis import build_basis
    from aimd_amd.qc.engine import Engine
    s, x = water_dimer()
    e = Engine(build_basis(s, x, "6-31g*"))
    e.set_precision(precision, 1e-5, 1e-5, 1e-2)
    e.set_geometry(x)
    D = _dens(e.nao, 1, 3, 1e-3)
    full = e.jk(D)
    for a, b in zip(full, e.jk_delta(D, 0.0)):
        assert torch.equal(a, b)
    thr = 1e-7
    for a, b in zip(full, e.jk_delta(D, thr)):
        assert float((a - b).abs().max()) < 8 * thr * e.nao ** 2
    e.close()


def test_replicas_stay_apart():
    """A NaN density in one replica of a batch leaves every other replica's J and K as they
    were, bit for bit."""
    import torch
    from aimd_amd.batch import ReplicaBatch
    s, w = bohr(WATER, 0.05, 4)
    batch = ReplicaBatch([(s, 0, 1)] * 3 + [(["H", "H"], 0, 1)], basis="6-31g**", jk_lanes=16)
    h2 = np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]])
    batch._set_geometry(np.concatenate([w, w + 0.01, w - 0.02, h2]))
    n = batch.ld
    D = torch.zeros((4, 2, n, n), dtype=torch.float64, device="cuda")
    for r, nr in enumerate(batch.rep_nao):
        D[r, :, :nr, :nr] = _dens(int(nr), 2, r)
    batch._jk(D)
    J, K = batch.J.clone(), batch.K.clone()
    assert float(J[3, :, 10:, :].abs().max()) == 0.0 and float(K[3, :, :, 10:].abs().max()) == 0.0
    D[1, 0, 2, 2] = float("nan")
    batch._jk(D)
    for r in (0, 2, 3):
        assert torch.equal(batch.J[r], J[r]) and torch.equal(batch.K[r], K[r])
    assert torch.isnan(batch.J[1, 0, :25, :25]).all()
    batch.close()


@pytest.mark.parametrize("nset", [1, 2])
def test_direct_in_pieces(oracle_lib, nset):
    """Direct mode with its buffer held to 64 MiB (eight waters take several hundred MB, so
    runs and classes are cut between pieces) against the oracle (1e-11, as the other J/K
    tests); a difference build and mixed precision change nothing in direct mode."""
    import torch
    from tests.conftest import cluster
    s, x = cluster("water8.xyz")
    e = _engine(s, x, "6-31g*", "store")
    assert e.jk_info()["gather_bytes"] > 3 * (64 << 20)
    D = _dens(e.nao, nset, 5)
    e.set_jk_mode("direct", 1)
    e.set_geometry(x)
    assert not e.jk_info()["stored"]
    ref = e.jk(D)
    Jo, Ko = oracle_lib.Pairs(oracle_lib.make_basis(s, x, "6-31g*")).jk_direct(D.cpu().numpy())
    np.testing.assert_allclose(ref[0].cpu().numpy(), Jo, rtol=0, atol=1e-11)
    np.testing.assert_allclose(ref[1].cpu().numpy(), Ko, rtol=0, atol=1e-11)
    for a, b in zip(ref, e.jk_delta(D, 1e-3)):
        assert torch.equal(a, b)
    e.set_precision("mixed", 1e-5, 1e-5, 1e-2)
    e.set_geometry(x)
    for a, b in zip(ref, e.jk(D)):
        assert torch.equal(a, b)
    e.close()
