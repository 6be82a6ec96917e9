"""Records of the brick list (mdk_brick.h), on the host: the pair passes stage as
many atoms as a brick's record counts, by indices that the list kernel wrote, and
it writes none for a brick that does not fit or has no atoms of its own.  So such
a record must count none, also where the cells around the brick hold atoms: in
voids, and in the gap beside a slab."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import brick_case
from conftest import ROOT
from moldy_amd import lattice

SRC = os.path.join(ROOT, "tests", "probe", "brick_extent_probe.cpp")


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("probe") / "brick_extent_probe")
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-x", "hip", SRC, "-o", out],
                   check=True, capture_output=True)

    def run(own, staged, threads, cap):
        txt = "".join(f"{7 * k} {o} {s} {threads} {cap}\n" for k, (o, s) in enumerate(zip(own, staged)))
        res = subprocess.run([out], input=txt, capture_output=True, text=True, check=True)
        return np.array([[int(w) for w in ln.split()] for ln in res.stdout.splitlines()])
    return run


def void_system():
    sd = lattice.make_system(nc=(54, 54, 54), sigma=0.08, temp=300.0, seed=7)
    keep = np.linalg.norm(sd.s - 0.5, axis=1) > 0.18
    return lattice.System(b0=sd.b0, s=sd.s[keep], x1=sd.x1[keep], mass=sd.mass[keep], z=sd.z[keep],
                          deltat_fs=sd.deltat_fs)


@pytest.mark.parametrize("system", [brick_case.slab_with_gap, void_system])
def test_bricks_without_own_atoms_stage_none(probe, system):
    own, staged = brick_case.extents(system())
    lone = (own == 0) & (staged > 0)
    assert lone.sum() >= 4  # the system has such bricks
    rec = probe(own, staged, 512, brick_case.CAP_MAX)
    np.testing.assert_array_equal(rec[:, 0], 7 * np.arange(len(own)))
    np.testing.assert_array_equal(rec[:, 1], own)
    np.testing.assert_array_equal(rec[:, 2], np.where(own > 0, staged, 0))


def test_bricks_that_do_not_fit_stage_none(probe):
    # own atoms at and above the threads, staged ones below, at and above the
    # capacity (the null slot takes the last one)
    own = [320, 321, 320, 320, 0, 1]
    staged = [999, 999, 1000, 1001, 1000, 1]
    rec = probe(own, staged, 320, 1000)
    np.testing.assert_array_equal(rec[:, 1:], [[320, 999], [0, 0], [0, 0], [0, 0], [0, 0], [1, 1]])
