"""mdk_batch_loss_grad_noalloc shares its handle's workspace with every other call:
after evaluations, products and losses with other knots and targets on the same
handle it still equals mdk_batch_loss_grad on a fresh one, bit for bit, and so do
the calls that follow it.  The fresh handle is given the same potentials in turn: the
sub-cells that they leave planned (which decide the order of sums) are the same."""
import numpy as np
import pytest
import torch

from moldy_amd import engine, lattice, potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [engine.PREC_FP32, engine.PREC_FP64])
def test_calls_in_turn_on_one_handle(prec):
    print("[gpu-test] no-alloc workspace, precision", prec, flush=True)
    cells = lattice.make_batch(ncell=12, seed=15, nmin=3, nmax=6, sigma=0.1)
    rng = np.random.default_rng(3)
    theta = potential.theta_vector()
    # knots near the Fe ones, and a range 6 % longer, which lays the cells out again
    sets = [potential.coeffs_from_theta(theta * (1 + rng.uniform(-0.01, 0.01, 16))) for _ in range(2)]
    sets.insert(1, dict(potential.FE_POTENTIAL, rv=potential.FE_POTENTIAL["rv"] * 1.06,
                        rp=potential.FE_POTENTIAL["rp"] * 1.06))
    one = engine.BatchEngine(cells, precision=prec)
    loss = torch.zeros(1, dtype=torch.float64, device="cuda:0")
    grad = torch.zeros(16, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    for k, c in enumerate(sets):
        et, ft = rng.standard_normal(one.ncell), rng.standard_normal((one.natom, 3))
        dE, dF = rng.standard_normal(one.ncell), rng.standard_normal((one.natom, 3))
        fresh = engine.BatchEngine(cells, precision=prec)
        for p in sets[: k + 1]:
            fresh.set_potential(p)
        fresh.set_targets(et, ft)
        l0, g0 = fresh.loss_grad()
        v0 = fresh.vjp(dE, dF)
        fresh.close()
        one.set_potential(c)
        one.set_targets(et, ft)
        if k:  # something else in the workspace first
            one.evaluate()
            one.vjp(dF.sum(axis=1)[: one.ncell], -dF)
        one.loss_grad_noalloc(loss.data_ptr(), grad.data_ptr())
        one.synchronize()
        assert float(loss.cpu()[0]) == l0
        np.testing.assert_array_equal(grad.cpu().numpy(), g0)
        np.testing.assert_array_equal(one.vjp(dE, dF), v0)
        for _ in range(3):  # direct launch, capture, replay
            l1, g1 = one.loss_grad()
            assert l1 == l0
            np.testing.assert_array_equal(g1, g0)
    one.close()
