"""The adjoint at extents that are no multiple of a tile or of a padded row, with and
without walls, against the FP64 autograd reference.  Sums in another order differ by
a few units in the last place a step; the bound is the one of the cubic grids, 1e-9."""
import numpy as np
import pytest
import torch

from droplet_amd.abi import DRP_WALL_NONE, DRP_WALL_Y, DRP_WALL_Z, make_config
from oracle import torch_step as ts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [DRP_WALL_NONE, DRP_WALL_Y, DRP_WALL_Z])
@pytest.mark.parametrize("dims", [(33, 13, 17), (31, 16, 12), (51, 12, 15)])
def test_adjoint_ragged_grids(axis, dims):
    from droplet_amd import lattice as dl
    cfg = make_config(*dims, nu1=0.1, nu2=0.1, kappa_g=0.01, wall_axis=axis, wall_u=0.02, wall_start=2)
    nx, ny, nz = dims
    drops = [(0.5 * (nx - 1), 0.5 * (ny - 1) + 0.3, 0.5 * (nz - 1) - 0.2, 0.45 * min(ny, nz))]
    nsteps, w = 8, (1.0, 1.0)
    theta = torch.tensor([cfg.tau_f, cfg.kappa_g, cfg.wall_u], dtype=torch.float64, requires_grad=True)
    f, g, mac = ts.initial_state(cfg, drops, theta[1])
    for n in range(1, nsteps + 1):
        f, g, mac = ts.step(f, g, mac, cfg, theta[0], theta[1], theta[2], n)
    J_ref = w[0] * ts.deformation_inertia(mac[0], cfg) + w[1] * ts.interface_area(mac[0])
    J_ref.backward()
    want = np.array([0.0 if t is None else t for t in theta.grad.tolist()])
    lat = dl.Lattice(cfg)
    lat.init_droplets(drops)
    tape = dl.Tape(lat, 3)
    tape.step(nsteps)
    J, got = tape.backward(w)
    tape.close()
    lat.close()
    assert abs(J - J_ref.item()) <= 1e-11 * max(abs(J_ref.item()), 1.0)
    print(dims, axis, got, want)
    assert (np.abs(np.array(got) - want) <= 1e-9 * np.abs(want)).all()
