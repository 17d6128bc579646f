"""Smagorinsky tau where its workgroups march over 2, 4, 8 and 16 planes, the last
march shorter than the others, with ragged rows."""
import numpy as np
import pytest

from droplet_amd.abi import DRP_FP32_SHIFTED, DRP_WALL_Z, make_config
from oracle.pyoracle import OracleLattice

pytestmark = pytest.mark.gpu
GRIDS = [(20, 9, 5), (130, 250, 43), (256, 256, 71), (256, 256, 129)]


def _cfg(dims, **kw):
    return make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.08, wall_axis=DRP_WALL_Z, wall_u=0.01, les_cs=0.17,
                       les_delta=1.0, **kw)


def _state(cfg):
    rng = np.random.default_rng(3)
    shape = (cfg.nz, cfg.ny, cfg.nx)
    y = np.arange(cfg.ny)[None, :, None]
    phi = cfg.phi1 + (cfg.phi2 - cfg.phi1) * 0.5 * (1 + np.tanh((y - cfg.ny / 2) / 2.0)) * np.ones(shape)
    return [phi, np.full(shape, 1 / 3)] + [0.01 * rng.standard_normal(shape) for _ in range(3)]


@pytest.mark.parametrize("dims", GRIDS)
def test_les_fp64(dims):
    from droplet_amd.lattice import Lattice
    cfg = _cfg(dims)
    f = _state(cfg)
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=8)
    for o in (lat, ora):
        o.init_fields(*f)
        o.step(2)
    a, b = lat.fields(), ora.fields()
    for k in ("phi", "p", "u1", "u2", "u3"):
        np.testing.assert_array_equal(a[k], b[k])


@pytest.mark.parametrize("dims", GRIDS)
def test_les_fp32(dims):
    """Against FP64 after two steps: a few units in the last place of the shifted
    populations (of order 1e-8) apart; tau off in one plane shows as 1e-4."""
    from droplet_amd.lattice import Lattice
    out = []
    for kw in ({}, dict(precision=DRP_FP32_SHIFTED)):
        cfg = _cfg(dims, **kw)
        lat = Lattice(cfg)
        lat.init_fields(*_state(cfg))
        lat.step(2)
        out.append(lat.fields())
    for k in ("u1", "u2", "u3"):
        assert np.abs(out[0][k] - out[1][k]).max() < 2e-6
