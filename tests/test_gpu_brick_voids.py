"""Brick lists (FP32 Fe, large periodic systems) where some bricks hold no atoms
but have neighbours that do: a slab beside a gap.  Against the FP64 form, with the
bounds of the FP32 form (forces 1e-5 eV/A, and 3e-6 of an atom's own where it is
large; energy 1e-6 eV per atom)."""
import numpy as np
import pytest

import brick_case
from moldy_amd import engine

pytestmark = pytest.mark.gpu


def run(sd, prec, ivol, steps):
    eng = engine.Engine(sd, ivol=ivol, precision=prec, rebuild=1)
    eng.linkup()
    eng.md_init()
    out = dict(f0=eng.forces_cart(), pe0=eng.scalar("pe"), pairs=eng.stats()[1])
    out["pe"] = eng.md_steps(steps)[:, 0]
    out["f1"] = eng.forces_cart()
    out["x0"], out["z0"] = eng.array("x0"), eng.array("z0")
    eng.close()
    return out


def check(a, b, n, width):
    assert abs(a["pairs"] - b["pairs"]) <= 1e-5 * b["pairs"]  # the skin's edge, 1e-6 A of FP32 positions
    for k, tol in (("f0", 1e-5), ("f1", 2e-5)):
        big = np.max(np.abs(b[k]), axis=1, keepdims=True)
        assert np.all(np.abs(a[k] - b[k]) <= tol + 3e-6 * big), k
    assert abs(a["pe0"] - b["pe0"]) <= 1e-6 * n
    assert np.max(np.abs(a["pe"] - b["pe"])) <= 1e-6 * n
    for k in ("x0", "z0"):
        assert np.max(np.abs(a[k] - b[k])) * width <= 1e-5, k


@pytest.mark.parametrize("ivol", [0, 1])
def test_slab_with_gap(ivol):
    print("[gpu-test] brick list, slab with a gap, ivol", ivol, flush=True)
    sd = brick_case.slab_with_gap()
    own, staged = brick_case.extents(sd)
    assert np.sum((own == 0) & (staged > 0)) >= 50
    a, b = (run(sd, p, ivol, 6) for p in (engine.PREC_FP32, engine.PREC_FP64))
    check(a, b, sd.n, np.max(sd.b0))
