"""Grids whose rows are padded in device memory (extents that are no multiple of a
64-byte sector) and whose arrays are just long enough, or just not, to be laid out
apart (1 MiB): host copies in and out, and every kernel that reads node arrays,
against the restatement."""
import numpy as np
import pytest

from droplet_amd.abi import (DRP_FILE_FG, DRP_FORCE_FIELD, DRP_FORCE_SPECTRAL, DRP_FORCE_TAYLOR_GREEN,
                             DRP_FP32_SHIFTED, DRP_LES_NONEQ, DRP_MODEL_ALLEN_CAHN, DRP_WALL_Y, DRP_WALL_Z, POP_MOM,
                             POP_PHI, make_config)
from oracle import pyoracle, torch_step
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


# 45 -> 48 doubles per row; 61 -> 64 floats
VARIANTS = {
    "periodic": dict(nu2=0.2),
    "walls": dict(wall_axis=DRP_WALL_Y, wall_u=0.02),
    "taylor-green": dict(force_kind=DRP_FORCE_TAYLOR_GREEN, force_amp=1e-5, force_k=0.14, nu2=0.15),
    "rank blocks": dict(les_cs=0.15, les_delta=2.0, nu2=0.2, les_ranks_x=3, les_ranks_y=2, les_ranks_z=2),
    "noneq": dict(les_cs=0.17, les_delta=2.0, nu2=0.2, les_model=DRP_LES_NONEQ),
    "allen-cahn": dict(model=DRP_MODEL_ALLEN_CAHN, ac_a=0.4, ac_width=4.0, phi1=-0.5, phi2=0.5, nu2=0.2,
                       wall_axis=DRP_WALL_Z, wall_u=0.02),
    "scale": dict(advect_k_high=3, advect_k_low=0, advect_start=1),
    "spectral": dict(force_kind=DRP_FORCE_SPECTRAL, force_amp=1e-6, force_k=3.0, les_cs=0.1, les_delta=1.0),
}


@pytest.mark.parametrize("name", list(VARIANTS))
def test_padded_rows(name):
    """Fields after twelve steps: bit-identical to the restatement, or within the
    rounding of its direct DFT sums where a truncated DFT takes part (about 1e-14
    of u a step)."""
    from droplet_amd.lattice import Lattice
    cfg = make_config(45, 22, 26, kappa_g=0.004, **VARIANTS[name])
    f = _state(cfg, 33)
    lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
    for o in (lat, ora):
        o.init_fields(*f)
        o.step(12)
    a, b = lat.fields(), ora.fields()
    for k in FIELDS:
        if name in ("scale", "spectral"):
            assert np.abs(a[k] - b[k]).max() <= 1e-12 * max(1e-2, np.abs(b[k]).max()), k
        else:
            np.testing.assert_array_equal(a[k], b[k])


def test_padded_rows_hooks(tmp_path):
    """Census, deformation of both planes, derived fields, energy budget, filters and a
    restart through the reference's files."""
    from droplet_amd.lattice import Lattice
    for wall in (DRP_WALL_Y, DRP_WALL_Z):
        cfg = make_config(45, 24, 30, kappa_g=0.004, wall_axis=wall, wall_u=0.02)
        f = _state(cfg, 34)
        lat, ora = Lattice(cfg), OracleLattice(cfg, threads=4)
        for o in (lat, ora):
            o.init_fields(*f)
            o.step(10)
        for mode in (0, 1, 2):
            np.testing.assert_allclose(lat.deformation(mode), ora.deformation(mode), rtol=1e-12, atol=1e-12)
    thr = 0.5 * (cfg.phi1 + cfg.phi2)
    first, vol, labels = lat.droplet_census(labels=True)
    count, rfirst, rvol, rlab = _census(ora.macro(0), thr)
    assert len(first) == count
    np.testing.assert_array_equal(first, rfirst)
    np.testing.assert_array_equal(vol, rvol)
    np.testing.assert_array_equal(labels, rlab)
    fields = [lat.macro(k) for k in range(5)]
    for kind in range(3):
        ref = pyoracle.derived(cfg, fields, kind)
        assert np.abs(lat.derived(kind) - ref).max() <= 1e-13 * np.abs(ref).max()
    low = lat.filter_velocity(0, 4)
    k = [np.where(np.arange(m) >= m // 2 + 1, np.arange(m) - m, np.arange(m)) for m in (30, 24, 45)]
    shell = np.sqrt(k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2).astype(int)
    for got, u in zip(low, fields[2:]):
        ref = np.real(np.fft.ifftn(np.fft.fftn(u) * (shell < 4)))
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(u).max()
    terms = lat.step_energy_budget()
    ora.step(1)
    ref = pyoracle.budget_terms(cfg, fields, [ora.macro(k) for k in range(5)])
    assert np.abs(terms - ref).max() <= 1e-11 * np.abs(ref).max()
    lat.write_reference_files(str(tmp_path), 11, DRP_FILE_FG, 3, 2)
    again = Lattice(cfg)
    again.init_fields(*f)
    again.read_reference_files(str(tmp_path), 11, DRP_FILE_FG, 3, 2)
    for o in (lat, again):
        o.step(3)
    for k in range(5):
        np.testing.assert_array_equal(lat.macro(k), again.macro(k))


def _census(phi, thr):
    first, vol, labels = pyoracle.census(phi, thr)
    return len(first), first, vol, labels


def test_padded_rows_gradient():
    """Checkpointed adjoint against autograd through the torch restatement."""
    import torch
    from droplet_amd.lattice import Lattice, Tape
    cfg = make_config(45, 12, 14, kappa_g=0.01, wall_axis=DRP_WALL_Y, wall_u=0.02)
    drops = [(22.0, 5.8, 6.7, 8.0)]
    theta = torch.tensor([cfg.tau_f, cfg.kappa_g, cfg.wall_u], dtype=torch.float64, requires_grad=True)
    J, _, _, _ = torch_step.run_loss(cfg, drops, 10, theta[0], theta[1], theta[2])
    J.backward()
    lat = Lattice(cfg)
    lat.init_droplets(drops)
    tape = Tape(lat, 4)
    tape.step(10)
    loss, grad = tape.backward()
    assert abs(loss - J.item()) <= 1e-10 * abs(J.item())
    ref = theta.grad.numpy()
    assert np.abs(np.array(grad) - ref).max() <= 1e-9 * np.abs(ref).max()


@pytest.mark.parametrize("kw", [dict(nu2=0.2, wall_axis=DRP_WALL_Z, wall_u=0.01),
                                dict(les_cs=0.1, les_delta=1.0, force_kind=DRP_FORCE_SPECTRAL, force_amp=1e-6,
                                     force_k=3.0)])
def test_padded_rows_fp32(kw):
    """FP32 rows of 61 -> 64 floats: the first steps follow FP64 to FP32 rounding."""
    from droplet_amd.lattice import Batch, Lattice
    cfg = make_config(61, 22, 26, kappa_g=0.004, precision=DRP_FP32_SHIFTED, **kw)
    c64 = make_config(61, 22, 26, kappa_g=0.004, **kw)
    f = _state(cfg, 35)
    lats = [Lattice(cfg), Lattice(c64)]
    for lat in lats:
        lat.init_fields(*f)
        lat.step(10)
    a, b = lats[0].fields(), lats[1].fields()
    for k in FIELDS:
        assert np.abs(a[k] - b[k]).max() <= 2e-5 * np.abs(b[k]).max(), k
    st = [lat.reduce() for lat in lats]
    assert abs(st[0]["phi_mass"] - st[1]["phi_mass"]) <= 1e-6 * st[1]["phi_mass"]
    if "les_cs" not in kw:
        batch = Batch([cfg, make_config(19, 70, 12, kappa_g=0.004, precision=DRP_FP32_SHIFTED, **kw)])
        batch[0].init_fields(*f)
        batch[1].init_fields(*_state(batch[1].cfg, 36))
        batch.step(10)
        c = batch[0].fields()
        for k in FIELDS:
            np.testing.assert_array_equal(a[k], c[k])
