"""A call of several steps in a fixed box that stops with MDK_ERR_SKIN: the forces
and densities are those of its last step, as for calls of one step each.

An atom alone in a gap flies 0.1 A a step (0.06), so the list's bound (0.15 A) is
passed without any pair missing by the second step (the third), and the call stops
three steps later; the positions are then those of the next.  A step back (x0 - x1 - x2) a fresh evaluation gives the
forces: rounding of the positions by 1e-16 of a box edge of up to 300 A, times
stiffnesses of 10 eV/A^2 and 14 partners, stays below 1e-10 of the largest force in
FP64; FP32 1e-5 eV/A, the bound of that form, from both."""
import numpy as np
import pytest

from moldy_amd import engine, lattice

pytestmark = pytest.mark.gpu

F32 = engine.PREC_FP32


def flyer(nc, fec, light, speed):
    """A crystal in the lower 0.6 of the box, and its last atom in the gap above."""
    sd = lattice.make_system(nc=nc, a=2.87 if fec else lattice.A_FE, sigma=0.05, temp=300.0, seed=nc[0])
    scale = np.array([1.0, 1.0, 1.0 / 0.6])
    b0, s, x1, mass = sd.b0 * scale, sd.s / scale, sd.x1 / scale, sd.mass.copy()
    s[:, 2] += 0.02
    s[-1] = [0.3, 0.4, 0.82]
    x1[-1] = [speed / b0[0, 0], 0.0, 0.0]
    if light:  # immobile atoms (too light for an acceleration): the per-pair mass test
        mass[[1, 7]], x1[[1, 7]] = 0.005, 0.0
    return lattice.System(b0=b0, s=s, x1=x1, mass=mass, z=sd.z, deltat_fs=sd.deltat_fs)


# at the lower speed the list is rebuilt, and the atoms sorted again, before the last step
@pytest.mark.parametrize("speed,steps", [(0.1, 4), (0.06, 5)])
@pytest.mark.parametrize("nc,kw", [
    ((10, 10, 10), dict(ivol=1)),
    ((10, 10, 10), dict(ivol=2)),
    ((10, 10, 10), dict(ivol=1, precision=F32)),
    ((10, 10, 10), dict(ivol=1, precision=F32, light=True)),
    ((10, 10, 10), dict(ivol=1, material="iron_carbon", lookup=5000)),
    ((28, 28, 28), dict(ivol=1, precision=F32)),
    ((40, 40, 40), dict(ivol=1)),
    ((54, 54, 54), dict(ivol=1, precision=F32)),
])
def test_forces_after_a_stopped_call(nc, kw, speed, steps):
    print("[gpu-test] stopped call", nc, kw, speed, flush=True)
    kw = dict(kw)
    sd = flyer(nc, kw.get("material") == "iron_carbon", kw.pop("light", False), speed)
    eng = engine.Engine(sd, ntcm=10, **kw)
    eng.linkup()
    eng.md_init()
    with pytest.raises(engine.MdkError) as err:
        eng.md_steps(20)
    assert err.value.code == engine.MDK_ERR_SKIN and f"step {steps - 3}:" in str(err.value)
    f, rho = eng.forces_cart(), eng.array("rho")
    s, x1 = (np.stack([eng.array(a + k) for a in "xyz"], axis=1) for k in "01")
    x2 = np.stack([eng.array(a + "2") for a in "xyz"], axis=1)
    eng.close()
    assert abs((s[-1] - sd.s[-1])[0] * sd.b0[0, 0] - (steps + 1) * speed) < 0.01  # and the next drift
    back = lattice.System(b0=sd.b0, s=s - (x1 + x2), x1=x1, mass=sd.mass, z=sd.z, deltat_fs=sd.deltat_fs)
    ref = engine.Engine(back, ntcm=10, **kw)
    ref.linkup()
    ref.force()
    g, rho1 = ref.forces_cart(), ref.array("rho")
    ref.close()
    tol = 2e-5 if kw.get("precision") == F32 else 1e-10 * np.max(np.abs(g))
    assert np.max(np.abs(f - g)) <= tol
    np.testing.assert_allclose(rho, rho1, rtol=0, atol=(1e-5 if kw.get("precision") == F32 else 1e-10) * rho1.max())
