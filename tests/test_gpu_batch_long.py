"""Batched cells with a long edge, where FP32 positions in the whole cell are off
by as much as the lists' margin (1e-4 A at an edge of some 1000 A): dimers just
inside and just outside the interaction range, against the oracle's brute-force
evaluation of the cell.

FP64 form: the pair count is exact, since every dimer is further from the range than
the 1e-12 A of the separations.  A dimer d inside the range has terms in d^2 and
d^0.5 (pair and embedding), so their relative error is 2 x 1e-12 / d; with d >= 2e-5
A and at most one partner each, 1e-6 of the largest force and density bounds them.

FP32 form: no partner in range is missing, and none is listed further past the range
than the margin for the rounding (1e-6 of the edges' sum and 1e-5 A, at least 1e-4 A)
and the rounding itself.  Its terms are not compared: so close to the range F' grows
without bound."""
import numpy as np
import pytest

from moldy_amd import engine, lattice, potential

pytestmark = pytest.mark.gpu

RC = potential.FE_INTERACTION_RANGE


# sub-cells in rows (three across) and one sub-cell across
@pytest.mark.parametrize("width", [12.6, 9.0])
@pytest.mark.parametrize("length", [90.0, 3000.0, 20000.0])
def test_dimers_at_the_range(oracle, length, width):
    print("[gpu-test] batch long cell", length, width, flush=True)
    rng = np.random.default_rng(int(length) + int(width))
    m = int(length / 14.0)  # further apart than two ranges
    b0 = np.diag([width, width, length])
    d = np.exp(rng.uniform(np.log(2e-5), np.log(9e-5), m)) * rng.choice([-1.0, 1.0], m)  # inside the range: > 0
    d[: m // 4] = rng.uniform(1.1e-4, 1.5e-4, m // 4) * -1.0
    u = rng.standard_normal((m, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    x = np.column_stack([rng.uniform(0, width, (m, 2)), 14.0 * np.arange(m) + rng.uniform(0.0, 0.5, m)])
    s = np.stack([x, x + u * (RC - d)[:, None]], axis=1).reshape(-1, 3) @ np.linalg.inv(b0)
    n = len(s)
    cell = lattice.System(b0=b0, s=s, x1=np.zeros_like(s), mass=np.full(n, lattice.FE_MASS),
                          z=np.full(n, lattice.FE_Z, dtype=np.int32), deltat_fs=1.0)
    pe, f, rho, _ = oracle.eval_cell(oracle.Potential(), cell, RC)
    assert np.sum(d > 0) >= 2 and np.max(np.abs(f)) > 0
    count, res = {}, {}
    for prec in (engine.PREC_FP64, engine.PREC_FP32):
        be = engine.BatchEngine([cell], precision=prec)
        be.evaluate()
        res[prec] = be.results()
        count[prec] = be.info()["pairs"]
        be.close()
    e64, _, f64, r64 = res[engine.PREC_FP64]
    assert count[engine.PREC_FP64] == 2 * np.sum(d > 0)
    assert np.max(np.abs(f64 - f)) <= 1e-6 * np.max(np.abs(f))
    assert np.max(np.abs(r64 - rho)) <= 1e-6 * np.max(rho)
    assert abs(e64[0] - pe) <= 1e-6 * abs(pe)
    rounding = 1e-6 * length + 1e-5
    most = 2 * np.sum(d > -max(1e-4, rounding) - rounding)
    assert 2 * np.sum(d > 0) <= count[engine.PREC_FP32] <= most
    assert np.all(res[engine.PREC_FP32][3].reshape(-1, 2)[d > 0] > 0.0)  # each has its partner's density
