"""Rows on either side of the length (16 nodes) up to which a lattice takes the
16-wide tile: ten steps bit-identical to the restatement, periodic and with walls,
forced and not."""
import numpy as np
import pytest

from droplet_amd.abi import DRP_FORCE_TAYLOR_GREEN, DRP_WALL_NONE, DRP_WALL_Y, make_config
from oracle.pyoracle import OracleLattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(wall_axis=DRP_WALL_Y, wall_u=0.01),
                                dict(wall_axis=DRP_WALL_NONE, force_kind=DRP_FORCE_TAYLOR_GREEN),
                                dict(wall_axis=DRP_WALL_NONE, les_cs=0.1, les_delta=1.0)])
@pytest.mark.parametrize("dims", [(3, 5, 9), (15, 9, 7), (16, 18, 5), (17, 6, 10)])
def test_short_rows(dims, kw):
    from droplet_amd.lattice import Lattice
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.1, **kw)
    rng = np.random.default_rng(11)
    nx, ny, nz = dims
    y = np.arange(ny)[None, :, None]
    phi = cfg.phi1 + (cfg.phi2 - cfg.phi1) * 0.5 * (1 + np.tanh(y - ny / 2)) * np.ones((nz, ny, nx))
    f = [phi, np.full(phi.shape, 1 / 3)] + [0.01 * rng.standard_normal(phi.shape) for _ in range(3)]
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=2)
    for o in (lat, ora):
        o.init_fields(*f)
        o.step(10)
    a, b = lat.fields(), ora.fields()
    for k in ("phi", "p", "u1", "u2", "u3"):
        np.testing.assert_array_equal(a[k], b[k])
