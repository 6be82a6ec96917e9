"""Ways out of and back into the brick list (FP32 Fe, large periodic systems),
against the FP64 form with the bounds of the FP32 form (forces 1e-5 eV/A, 3e-6 of an
atom's own where it is large; energy 1e-6 eV per atom; doubled after some steps):
a slab whose bricks hold more atoms than a workgroup has threads (their mean over the
box, with its gap, fits) takes the list of indices, and tries bricks again every 32
lists; one whose bricks need larger sizes than the mean's; a list capacity to grow; an upload of light masses
between two calls, after which the general passes read the expanded list."""
import numpy as np
import pytest

import brick_case
from moldy_amd import engine, lattice

pytestmark = pytest.mark.gpu


# cells of 5.7 A along x: 8 across, rounded down from 11
THICK = (16, 95, 92)


def forms(sd, calls, between=None, **kw):
    out = []
    for prec in (engine.PREC_FP32, engine.PREC_FP64):
        eng = engine.Engine(sd, precision=prec, **kw)
        eng.linkup()
        eng.md_init()
        f, pe = [eng.forces_cart()], [eng.scalar("pe")]
        for k, steps in enumerate(calls):
            if k and between:
                between(eng)
            pe += list(eng.md_steps(steps)[:, 0])
            f.append(eng.forces_cart())
        out.append((f, np.array(pe), eng.stats()[1]))
        eng.close()
    (f32, pe32, p32), (f64, pe64, p64) = out
    assert abs(p32 - p64) <= 1e-5 * p64
    for k, (a, b) in enumerate(zip(f32, f64)):
        big = np.max(np.abs(b), axis=1, keepdims=True)
        assert np.all(np.abs(a - b) <= (2e-5 if k else 1e-5) + 3e-6 * big), k
    assert np.max(np.abs(pe32 - pe64)) <= 1e-6 * sd.n


@pytest.mark.parametrize("ivol", [0, 1])
def test_bricks_that_do_not_fit(ivol):
    print("[gpu-test] bricks that do not fit, ivol", ivol, flush=True)
    sd = brick_case.slab_with_gap(nc=THICK)
    assert sd.n >= 262144
    own, _ = brick_case.extents(sd)
    assert brick_case.threads_for(1.02 * own.mean()) and not brick_case.threads_for(own.max())
    forms(sd, [4], ivol=ivol, rebuild=1)


def test_bricks_tried_again():
    # a list every step: the try after 32 of them
    print("[gpu-test] bricks tried again", flush=True)
    forms(brick_case.slab_with_gap(nc=THICK), [36], ivol=1, ntcm=1)


def test_bricks_larger_than_the_mean():
    print("[gpu-test] bricks larger than the mean", flush=True)
    sd = brick_case.slab_with_gap()
    own, _ = brick_case.extents(sd)
    g = brick_case.grid(sd)
    assert brick_case.threads_for(1.02 * 64 * sd.n / np.prod(g)) < brick_case.threads_for(own.max())
    forms(sd, [36], ivol=1, ntcm=1)


def test_capacity_grows():
    print("[gpu-test] brick list capacity", flush=True)
    forms(lattice.make_system(nc=(52, 52, 50), sigma=0.08, temp=300.0, seed=3), [4], ivol=0, rebuild=1, max_full=8)


@pytest.mark.parametrize("ivol", [0, 1])
def test_light_masses_between_calls(ivol):
    print("[gpu-test] light masses between calls, ivol", ivol, flush=True)
    sd = lattice.make_system(nc=(52, 52, 50), sigma=0.08, temp=300.0, seed=4)

    def freeze(eng):  # too light for an acceleration, and at rest
        mass, del2 = eng.array("mass"), eng.array("del2")
        mass[[0, 1000]], del2[[0, 1000]] = 0.005, 0.0
        for k in ("x1", "y1", "z1", "x2", "y2", "z2"):
            v = eng.array(k)
            v[[0, 1000]] = 0.0
            eng.upload(k, v)
        eng.upload("mass", mass)
        eng.upload("del2", del2)

    forms(sd, [3, 3], between=freeze, ivol=ivol, rebuild=1)
