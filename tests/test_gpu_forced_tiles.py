"""Steps with a force field at the sizes where its default tiles change, and on either
side of them, with and without a viscosity of phi."""
import numpy as np
import pytest

from droplet_amd.abi import DRP_FORCE_FIELD, DRP_FP32_SHIFTED, DRP_WALL_Z, make_config
from oracle.pyoracle import OracleLattice

pytestmark = pytest.mark.gpu
FIELDS = ("phi", "p", "u1", "u2", "u3")


def _run(make, dims, nu2, **kw):
    cfg = make_config(*dims, kappa_g=0.004, nu1=0.05, nu2=nu2, wall_axis=DRP_WALL_Z, wall_u=0.01,
                      force_kind=DRP_FORCE_FIELD, **kw)
    rng = np.random.default_rng(11)
    nx, ny, nz = dims
    z = np.arange(nz)[:, None, None]
    phi = np.broadcast_to(0.5 * (cfg.phi1 + cfg.phi2) + 0.5 * (cfg.phi2 - cfg.phi1) * np.tanh((z - nz / 2) / 2.0),
                          (nz, ny, nx)).copy()
    u = [0.01 * rng.standard_normal(phi.shape) for _ in range(3)]
    lat = make(cfg)
    lat.init_fields(phi, np.full(phi.shape, 1 / 3), *u)
    lat.set_force(*[1e-3 * v for v in u])
    lat.step(5)
    return lat.fields()


@pytest.mark.parametrize("nu2", [0.05, 0.2])
@pytest.mark.parametrize("dims", [(32, 32, 32), (33, 33, 33), (64, 32, 32), (100, 20, 28), (60, 20, 64)])
def test_forced_fp64(dims, nu2):
    """Bit-identical to the restatement."""
    from droplet_amd.lattice import Lattice
    a, b = _run(Lattice, dims, nu2), _run(lambda c: OracleLattice(c, threads=4), dims, nu2)
    for k in FIELDS:
        np.testing.assert_array_equal(a[k], b[k])


@pytest.mark.parametrize("nu2", [0.05, 0.2])
@pytest.mark.parametrize("dims", [(32, 32, 32), (32, 32, 33)])
def test_forced_fp32(dims, nu2):
    """FP32 storage against FP64 after five steps: velocities of 0.04 differ by a few units
    in the last place of the shifted populations (of order 1e-8) a step; a force of 1e-5
    from the wrong node would move them by 3e-5 a step."""
    from droplet_amd.lattice import Lattice
    a, b = _run(Lattice, dims, nu2), _run(Lattice, dims, nu2, precision=DRP_FP32_SHIFTED)
    for k in ("u1", "u2", "u3"):
        assert np.abs(a[k] - b[k]).max() < 2e-6
