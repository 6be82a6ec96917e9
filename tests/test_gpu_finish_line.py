"""NPT steps on both sides of the line between finishing in the kick's workgroups
and in a kernel of its own (kick workgroups times those of the pair passes: 64,000),
at eight, four, two and one lanes per atom: md_steps against the step-by-step calls,
which always take the second form, bit for bit."""
import numpy as np
import pytest

from moldy_amd import engine, lattice

pytestmark = pytest.mark.gpu


# below, just below (89 x 712 and 126 x 504 workgroups), just above, and where the
# pair passes have few workgroups but the kick many
@pytest.mark.parametrize("nc,keep,kw", [
    ((16, 16, 17), 8193, dict()),
    ((25, 26, 26), 32256, dict()),
    ((25, 26, 26), 32257, dict()),
    ((25, 26, 26), 32256, dict(precision=engine.PREC_FP32)),
    ((25, 26, 26), 32257, dict(precision=engine.PREC_FP32)),
    ((28, 28, 27), 40961, dict()),
    ((32, 32, 32), 65536, dict(precision=engine.PREC_FP32)),
    ((35, 34, 35), 81921, dict()),
    ((40, 40, 40), 128000, dict()),
    ((44, 43, 44), 163841, dict(precision=engine.PREC_FP32)),
    ((23, 23, 22), 22784, dict(material="iron_carbon", lookup=5000)),
    ((23, 23, 22), 22785, dict(material="iron_carbon", lookup=5000)),
])
def test_both_finishing_forms(nc, keep, kw):
    print("[gpu-test] finishing line", nc, keep, kw, flush=True)
    a = 2.87 if kw.get("material") == "iron_carbon" else lattice.A_FE
    sd = lattice.make_system(nc=nc, a=a, sigma=0.05, temp=300.0, seed=keep)
    sd = lattice.System(b0=sd.b0, s=sd.s[:keep].copy(), x1=sd.x1[:keep].copy(), mass=sd.mass[:keep], z=sd.z[:keep],
                        deltat_fs=sd.deltat_fs)
    one, steps = (engine.Engine(sd, ivol=0, ntcm=10, **kw) for _ in range(2))
    for e in (one, steps):
        e.linkup()
        e.md_init()
    steps.md_steps(8)
    for _ in range(8):
        one.velocityverlet()
        one.update_therm_avs()
        if one.ntc == 0:
            one.relink()
    for name in ("x0", "y1", "z2", "fx", "rho"):
        np.testing.assert_array_equal(steps.array(name), one.array(name))
    for name in ("b0", "b1", "tp", "tk", "fb"):
        np.testing.assert_array_equal(steps.tensor(name), one.tensor(name))
    one.close()
    steps.close()
