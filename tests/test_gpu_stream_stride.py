"""Grids whose arrays are just long enough to be laid out apart (1 MiB), with extents
that are no multiple of a line, a row or a tile, and just short enough not to be:
host copies in and out, and every variant that reads several arrays."""
import numpy as np
import pytest

from droplet_amd.abi import (DRP_FORCE_FIELD, DRP_FP32_SHIFTED, DRP_WALL_Z, POP_MOM, POP_PHI, make_config)
from oracle.pyoracle import OracleLattice

pytestmark = pytest.mark.gpu
FIELDS = ("phi", "p", "u1", "u2", "u3")
GRIDS = [(51, 51, 51), (50, 61, 43), (47, 53, 52)]   # 132651, 131150, 129532 nodes; 1 MiB is 131072 doubles


def _state(cfg, seed):
    rng = np.random.default_rng(seed)
    shape = (cfg.nz, cfg.ny, cfg.nx)
    z, y, x = np.meshgrid(*[np.arange(n) for n in shape], indexing="ij")
    r = np.sqrt((x - cfg.nx / 2) ** 2 + (y - cfg.ny / 2) ** 2 + (z - cfg.nz / 2) ** 2)
    phi = cfg.phi1 + (cfg.phi2 - cfg.phi1) * 0.5 * (1 + np.tanh((0.3 * min(shape) - r) / 2.0))
    return [phi, np.full(shape, 1 / 3)] + [0.01 * rng.standard_normal(shape) for _ in range(3)]


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("les", [False, True])
def test_steps_and_host_copies(dims, les):
    """FP64: force field in and out, LES, ten steps bit-identical to the restatement,
    both population sets out, in again, and ten more steps."""
    from droplet_amd.lattice import Lattice
    kw = dict(les_cs=0.1, les_delta=1.0) if les else {}
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=0.08, wall_axis=DRP_WALL_Z, wall_u=0.01,
                      force_kind=DRP_FORCE_FIELD, **kw)
    f = _state(cfg, 31)
    force = [1e-5 * v for v in f[2:]]
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(*f)
        o.set_force(*force)
        o.step(10)
    for got, want in zip(lat.force(), force):
        np.testing.assert_array_equal(got, want)
    a, b = lat.fields(), ora.fields()
    for k in FIELDS:
        np.testing.assert_array_equal(a[k], b[k])
    for which in (POP_PHI, POP_MOM):
        g = lat.populations(which)
        np.testing.assert_array_equal(g, ora.populations(which))
        for o in (lat, ora):
            o.set_populations(which, g)
    for o in (lat, ora):
        o.step(10)
    a, b = lat.fields(), ora.fields()
    for k in FIELDS:
        np.testing.assert_array_equal(a[k], b[k])


@pytest.mark.parametrize("dims", [(64, 64, 64), (65, 67, 61)])   # 1 MiB is 262144 floats
def test_fp32_host_copies(dims):
    """FP32: populations survive a round trip, and the fields are their moments."""
    from droplet_amd.lattice import Lattice
    cfg = make_config(*dims, kappa_g=0.004, nu2=0.15, precision=DRP_FP32_SHIFTED)
    lat = Lattice(cfg)
    lat.init_fields(*_state(cfg, 32))
    lat.step(5)
    f, g = lat.populations(POP_PHI), lat.populations(POP_MOM)
    fields = lat.fields()
    assert np.abs(f.sum(0) - fields["phi"]).max() <= 15 * 4.9 * 2.0 ** -24
    assert np.abs(g.sum(0) / 3 - fields["p"]).max() <= 15 * 0.25 * 2.0 ** -24
    lat.set_populations(POP_PHI, f)
    lat.set_populations(POP_MOM, g)
    np.testing.assert_array_equal(lat.populations(POP_PHI), f)
    np.testing.assert_array_equal(lat.populations(POP_MOM), g)
