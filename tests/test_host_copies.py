"""Copies between node arrays and host memory without a GPU: the library's host code and
its copy kernels built against a host-only double of the HIP runtime (tests/native), with
two devices, memory that runs out and streams that do not end."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "droplet_amd", "csrc")
SOURCES = ["host_io.hip", "lattice.cpp", "fp32_shifted.cpp", "deformation.cpp", "aux_kernels.hip", "aux_fp32.hip"]
CHECKS = {
    "devices": "a lattice's copies run on its own device whatever the caller's current one is",
    "visibility": "what a kernel wrote to pinned memory is visible to the thread that reads it",
    "no pinned memory": "output calls do without pinned memory",
    "no device memory": "host arrays go in and out without device memory beyond the lattice's own",
    "earlier error": "an error that an earlier call left behind does not fail a copy",
    "independence": "a copy does not wait for those of other lattices",
    "plane memory": "a deformation plane takes a plane's worth of device memory",
    "tight lattice": "a lattice that fits the device without padding is made without it",
    "range parts": "the parts of a phi-range slot follow the default shape's tiles and stay with the lattice",
    "forced tiles": "default tiles of lattices with a force field",
    "together": "the host arrays of a call go in together",
}


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("host_copies")
    flags = ["-std=c++17", "-O1", "-ffp-contract=off", "-w", "-pthread", "-fno-pie",
             "-I" + os.path.join(HERE, "native", "hip_double")]
    paths = [os.path.join(CSRC, s) for s in SOURCES] + [os.path.join(HERE, "native", "host_copies.cpp")]
    procs, objs = [], []
    for p in paths:
        objs.append(str(out / (os.path.basename(p) + ".o")))
        procs.append(subprocess.Popen([cxx, *flags, "-x", "c++", "-c", p, "-o", objs[-1]], stdout=subprocess.PIPE,
                                      stderr=subprocess.STDOUT, text=True))
    for p in procs:
        log, _ = p.communicate()
        assert p.returncode == 0, log
    exe = str(out / "host_copies")
    # (the step and the spectra are not part of the program, and nothing calls them)
    r = subprocess.run([cxx, "-no-pie", "-pthread", *objs, "-Wl,--unresolved-symbols=ignore-all", "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return exe


@pytest.mark.parametrize("name", list(CHECKS))
def test_host_copies(program, name):
    r = subprocess.run([program, name], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, errors="replace",
                       timeout=120)
    assert r.returncode == 0, f"{CHECKS[name]}: {r.returncode}\n{r.stdout[-3000:]}"
