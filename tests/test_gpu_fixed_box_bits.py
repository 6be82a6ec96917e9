"""MD calls in a box that does not move against calls of one step each: the fused
force pass follows the same trajectory bit for bit (positions, velocities,
accelerations, forces, densities, F'), in every form of the pass.  Only the reported
sums over atoms (energies, TK) add the same terms in another order: 1e-12 of their
largest value, as n terms of one sign round like sqrt(n) eps."""
import numpy as np
import pytest

from moldy_amd import engine, lattice

pytestmark = pytest.mark.gpu

F32 = engine.PREC_FP32
FEC = dict(material="iron_carbon")


def run(sd, kw, calls):
    eng = engine.Engine(sd, ntcm=5, **kw)
    eng.linkup()
    eng.md_init()
    trace = np.vstack([eng.md_steps(k) for k in calls])
    state = {k: eng.array(k) for k in ("x0", "y1", "z2", "fx", "fz", "rho", "dafrho")}
    state.update((t, eng.tensor(t)) for t in ("b0", "tp", "tgid"))
    sums = [trace, eng.tensor("tk")]
    eng.close()
    return state, sums


# eight, four, two and one lanes per atom, knots and tables, both packings, a
# brick list, and both forms of the finishing
@pytest.mark.parametrize("nc,kw", [
    ((6, 6, 6), dict(ivol=1)),
    ((10, 10, 10), dict(ivol=2)),
    ((10, 10, 10), dict(ivol=3, precision=F32)),
    ((10, 10, 10), dict(ivol=5, lookup=5000, precision=F32)),
    ((10, 10, 10), dict(ivol=1, **FEC)),
    ((20, 20, 20), dict(ivol=1)),
    ((20, 20, 20), dict(ivol=1, precision=F32)),
    ((32, 32, 32), dict(ivol=1)),
    ((32, 32, 32), dict(ivol=2, precision=F32)),
    ((44, 44, 44), dict(ivol=1)),
    ((44, 44, 44), dict(ivol=1, precision=F32)),
    ((42, 42, 42), dict(ivol=1, lookup=5000, **FEC)),
    ((52, 52, 52), dict(ivol=1, precision=F32)),
])
def test_same_trajectory(nc, kw):
    print("[gpu-test] fixed box bits", nc, kw, flush=True)
    sd = lattice.make_system(nc=nc, a=2.87 if "material" in kw else lattice.A_FE, sigma=0.05, temp=300.0, seed=1)
    (a, sa), (b, sb) = run(sd, kw, [12]), run(sd, kw, [1] * 12)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    for x, y in zip(sa, sb):
        np.testing.assert_allclose(x, y, rtol=0, atol=1e-12 * np.abs(y).max())
