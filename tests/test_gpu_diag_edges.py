"""The marching diagnostics sums at the sizes where their indexing can go wrong:
columns and planes that no tile divides, extents below a tile."""
import numpy as np
import pytest

from droplet_amd.abi import kappa_g_from_sigma, make_config

pytestmark = pytest.mark.gpu


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
