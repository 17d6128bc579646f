"""Host copies of padded lattices long enough for several threads and chunks that cross
array boundaries, alone and from several threads at once (more chunks asked for than the
process has)."""
import threading

import numpy as np
import pytest

from droplet_amd.abi import DRP_FP32_SHIFTED, POP_MOM, POP_PHI, make_config

pytestmark = pytest.mark.gpu
DIMS = (131, 70, 97)   # 131 -> 136 doubles, 144 floats a row; 13.3 million values in 15 arrays
PRECISIONS = {"fp64": {}, "fp32": dict(precision=DRP_FP32_SHIFTED)}


def _lattice(precision, seed):
    from droplet_amd.lattice import Lattice
    nx, ny, nz = DIMS
    rng = np.random.default_rng(seed)
    lat = Lattice(make_config(nx, ny, nz, kappa_g=0.004, **PRECISIONS[precision]))
    fields = [rng.uniform(2.0, 5.0, (nz, ny, nx)), np.full((nz, ny, nx), 1 / 3)]
    lat.init_fields(*fields, *[rng.uniform(-0.01, 0.01, (nz, ny, nx)) for _ in range(3)])
    return lat, rng


@pytest.mark.parametrize("precision", list(PRECISIONS))
def test_population_round_trip(precision):
    """FP64: every value comes back.  FP32 holds deviations from values below 6 in
    magnitude, so one of a number within (0, 1) is rounded by at most 2^-22; any two
    values are 0.5 apart on average."""
    lat, rng = _lattice(precision, 1)
    nx, ny, nz = DIMS
    for which in (POP_PHI, POP_MOM):
        want = rng.uniform(0.0, 1.0, (15, nz, ny, nx))
        lat.set_populations(which, want)
        got = lat.populations(which)
        if precision == "fp64":
            np.testing.assert_array_equal(got, want)
        else:
            assert np.abs(got - want).max() <= 2.0 ** -22


def test_copies_from_several_threads():
    """Five lattices, read at once by a thread each, three times: what a thread alone reads."""
    lats = [_lattice("fp32" if k % 2 else "fp64", 10 + k)[0] for k in range(5)]
    alone = [(lat.populations(POP_PHI), lat.populations(POP_MOM), lat.fields()) for lat in lats]
    start, wrong = threading.Barrier(len(lats)), []

    def read(k):
        try:
            for _ in range(3):
                start.wait(60)
                f, g, fields = lats[k].populations(POP_PHI), lats[k].populations(POP_MOM), lats[k].fields()
                ok = np.array_equal(f, alone[k][0]) and np.array_equal(g, alone[k][1])
                if not (ok and all(np.array_equal(fields[n], alone[k][2][n]) for n in fields)):
                    wrong.append(k)
        except Exception as e:   # a thread's exception would go unseen
            wrong.append((k, e))

    threads = [threading.Thread(target=read, args=(k,)) for k in range(len(lats))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
