"""Half-spectrum shell sums and the marching diagnostics sums at the sizes where
their indexing can go wrong: odd extents (no Nyquist plane, an unpaired last row),
lines of 2048 points with thousands of shells, columns and planes that no tile
divides, extents below a tile."""
import numpy as np
import pytest

from droplet_amd.abi import kappa_g_from_sigma, make_config
from tests.test_gpu_spectral_diag import _grad, _lattice_with, _random_state, _shells, _spectrum_ref

pytestmark = pytest.mark.gpu


# 64-bit transforms and sums: a few hundred roundings of 1.1e-16 of the largest shell
TOL = 1e-12


@pytest.mark.parametrize("shape,nshells", [((3, 3, 3), 4), ((5, 9, 15), 8), ((6, 5, 4), 3), ((27, 16, 25), 30),
                                           ((2048, 3, 4), 1030), ((4, 6, 2048), 8192), ((4, 1500, 3), 760),
                                           ((40, 36, 50), 26)])
def test_shell_sums(shape, nshells):
    """Energy spectrum and per-scale interaction; each [z][y][x]."""
    f = _random_state(shape, 21)
    kg = 0.004
    lat = _lattice_with(f, make_config(shape[2], shape[1], shape[0], kappa_g=kg))
    E = lat.energy_spectrum(nshells)
    ref = _spectrum_ref(*f[2:], nshells)
    assert np.abs(E - ref).max() <= TOL * ref.max()
    g = _grad(f[0])
    n = f[0].size
    cross = np.zeros(shape)
    for b in range(3):
        w = sum(_grad(g[b] * g[a])[a] for a in range(3))
        cross += np.real(np.fft.fftn(f[2 + b]) * np.conj(np.fft.fftn(w))) / n ** 2
    sh = _shells(shape)
    keep = sh < nshells
    ref = kg * np.bincount(sh[keep], cross[keep], minlength=nshells)
    C = lat.scale_interaction(nshells)
    assert np.abs(C - ref).max() <= TOL * kg * np.abs(cross).sum()


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 9, 15), (27, 16, 25), (40, 36, 50)])
def test_phi_contribution(shape):
    """Half-space cross spectrum of u . grad phi and mu (drop_analysis.f90:476-578)."""
    f = _random_state(shape, 22)
    cfg = make_config(shape[2], shape[1], shape[0], kappa_g=0.004)
    lat = _lattice_with(f, cfg)
    got, _ = lat.phi_contribution()
    a, m = np.fft.fftn(lat.derived(2)), np.fft.fftn(lat.derived(0))
    nz = shape[0]
    w = np.full(shape, 2.0)
    w[0] = 1.0
    w[nz // 2 + 1:] = 0.0
    sh, nb = _shells(shape), shape[2] // 2 + 1
    keep = sh < nb
    c = np.real(a * np.conj(m)) * w
    num = np.bincount(sh[keep], c[keep], minlength=nb)
    den = np.bincount(sh[keep], w[keep], minlength=nb)
    ref = np.where(den > 0, num / np.where(den > 0, den, 1.0), 0.0)
    assert np.abs(got - ref).max() <= TOL * np.abs(c).max()


@pytest.mark.parametrize("dims", [(3, 3, 3), (3, 200, 3), (65, 9, 5), (130, 17, 33), (64, 8, 70), (16, 16, 300)])
def test_reduce(dims):
    """drp_reduce against the restatement's sums."""
    from droplet_amd.lattice import Lattice
    from oracle.pyoracle import OracleLattice
    nx, ny, nz = dims
    cfg = make_config(nx, ny, nz, kappa_g=kappa_g_from_sigma(0.01))
    rng = np.random.default_rng(23)
    shape = (nz, ny, nx)
    phi = cfg.phi1 + (cfg.phi2 - cfg.phi1) * rng.random(shape)
    u = [0.02 * rng.standard_normal(shape) + 0.01 for _ in range(3)]
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(phi, 1 / 3, *u)
    a, b = lat.reduce(), ora.reduce()
    for k in ("phi_mass", "kinetic", "dissipation", "interface_area", "free_energy", "p_mean"):
        assert abs(a[k] - b[k]) <= 1e-12 * abs(b[k]), (k, a[k], b[k])
    # the interaction sums terms of both signs
    assert abs(a["interaction"] - b["interaction"]) <= 1e-12 * a["interface_area"]
    np.testing.assert_allclose(a["momentum"], b["momentum"], rtol=1e-12)
