"""The global phi range on either side of the sizes where a step folds it into one
part of its slot or into eight: phi beyond its two values at one node of the last
tile, so that the viscosity of every node hangs on that part."""
import numpy as np
import pytest

from droplet_amd.abi import DRP_FP32_SHIFTED, DRP_WALL_Z, make_config
from oracle.pyoracle import OracleLattice

pytestmark = pytest.mark.gpu
# 7936 and 8192 nodes; 524288 and 532480
GRIDS = [(16, 31, 16), (16, 32, 16), (128, 64, 64), (130, 64, 64)]


def _state(dims, phi1, phi2):
    rng = np.random.default_rng(7)
    nx, ny, nz = dims
    z = np.arange(nz)[:, None, None]
    phi = np.broadcast_to(0.5 * (phi1 + phi2) + 0.5 * (phi2 - phi1) * np.tanh((z - nz / 2) / 2.0), (nz, ny, nx)).copy()
    phi[nz - 1, ny - 1, nx - 1] = phi2 + 0.2 * (phi2 - phi1)
    phi[0, 0, 0] = phi1 - 0.2 * (phi2 - phi1)
    return [phi, np.full(phi.shape, 1 / 3)] + [0.01 * rng.standard_normal(phi.shape) for _ in range(3)]


@pytest.mark.parametrize("dims", GRIDS)
def test_range_fp64(dims):
    """Five steps bit-identical to the restatement, and the range that a reduction sees."""
    from droplet_amd.lattice import Lattice
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.2, wall_axis=DRP_WALL_Z, wall_u=0.01)
    f = _state(dims, cfg.phi1, cfg.phi2)
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(*f)
    for n in (1, 4):
        for o in (lat, ora):
            o.step(n)
        a, b = lat.fields(), ora.fields()
        for k in ("phi", "p", "u1", "u2", "u3"):
            np.testing.assert_array_equal(a[k], b[k])


@pytest.mark.parametrize("dims", GRIDS)
def test_range_fp32(dims):
    """FP32 storage against FP64 after five steps.  Velocities of 0.04 differ by a few
    units in the last place of the shifted populations (of order 1e-8) a step; a range
    that misses the two nodes puts the viscosities off by a seventh of 0.15, which
    damps this velocity noise by percents more or less (of order 1e-4)."""
    from droplet_amd.lattice import Lattice
    out = []
    for kw in ({}, dict(precision=DRP_FP32_SHIFTED)):
        cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.2, wall_axis=DRP_WALL_Z, wall_u=0.01, **kw)
        lat = Lattice(cfg)
        lat.init_fields(*_state(dims, cfg.phi1, cfg.phi2))
        lat.step(5)
        out.append(lat.fields())
    for k in ("u1", "u2", "u3"):
        assert np.abs(out[0][k] - out[1][k]).max() < 2e-6


@pytest.mark.parametrize("dims", GRIDS)
def test_range_of_a_reduction(dims):
    """What a reduction folds from all parts of a slot, whichever of them the step used:
    the restatement's range at the start and after 1, 2, 3 and 7 steps, so in each of the
    three slots, and the extremes of the field.  (The fields pass the two values at both
    ends.)"""
    from droplet_amd.lattice import Lattice
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.2, wall_axis=DRP_WALL_Z, wall_u=0.01)
    f = _state(dims, cfg.phi1, cfg.phi2)
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(*f)
    for n in (0, 1, 1, 1, 4):
        for o in (lat, ora):
            o.step(n)
        a, b = lat.reduce(), ora.reduce()
        assert (a["phi_min"], a["phi_max"]) == (b["phi_min"], b["phi_max"])
        if n > 0:
            phi = lat.fields()["phi"]
            assert a["phi_min"] == min(phi.min(), cfg.phi2) and a["phi_max"] == max(phi.max(), cfg.phi1)


# Tiles of the default shape: 225, 56, 64 and 2560 in both.
# From 64 to 2048 of them a step folds into eight parts.
@pytest.mark.parametrize("dims", [(3, 3, 900), (32, 32, 14), (32, 32, 16), (130, 62, 64)])
def test_range_tile_counts_fp64(dims):
    test_range_fp64(dims)
    test_range_of_a_reduction(dims)


@pytest.mark.parametrize("dims", [(3, 3, 900), (32, 32, 28), (32, 32, 32), (130, 128, 64)])
def test_range_tile_counts_fp32(dims):
    test_range_fp32(dims)


def test_range_keeps_its_parts_when_the_tile_shape_changes():
    """Tiles of another shape from step to step: bit-identical to the restatement, whose
    viscosity hangs on the range at every node."""
    from droplet_amd.lattice import Lattice
    dims = (32, 32, 16)
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.2, wall_axis=DRP_WALL_Z, wall_u=0.01)
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(*_state(dims, cfg.phi1, cfg.phi2))
    for shape in (0, 6, 1, 2, 4, 3):
        lat.tile_shape = shape
        for o in (lat, ora):
            o.step(1)
        a, b = lat.fields(), ora.fields()
        for k in ("phi", "p", "u1", "u2", "u3"):
            np.testing.assert_array_equal(a[k], b[k])
