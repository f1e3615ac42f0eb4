"""Every form of the fast f32 kernels against the FP64 oracle, states after five
steps and od_rhs: boxes one element thin (tiles whose faces meet themselves),
channels of odd height, small (tiles) and large enough for core and shell, and the
Euler mode.

States have the other fast boxes' tolerance.  A right-hand side is a small difference
of large fluxes, whose f32 rounding depends on the box's element size and flow; the
oracle in f32 measures it.  The fast build's reciprocals and square roots are good
to one unit in the last place, the oracle's divisions to half of one, so its error
may be twice the f32 oracle's."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import rel_err_per_var, smooth_state
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-5  # max |gpu - oracle_f64| / max |oracle_f64| per variable

THIN = [(1, 4, 3), (3, 1, 2), (4, 3, 1), (1, 1, 5)]
ODD_HEIGHT = [(4, 3, 2), (3, 5, 3), (2, 3, 2)]
CORE_SHELL = [(6, 19, 10), (9, 16, 9)]  # 570 and 720 tiles: viscous boxes on core and shell


def compare(n, flux, wall, viscous, lengths):
    print(f"CASE test=fast_forms n={n} flux={flux} wall={wall} viscous={viscous}", flush=True)
    kw = dict(flux=flux, y_wall=wall, viscous=viscous, viscosity_model=1, mu_ref=2e-3)
    u = smooth_state(*n, *lengths, seed=5, amp=0.05, dtype=np.float32)
    po = O.params(*n, *lengths, u_real=8, **kw)
    with od.Solver(od.params(*n, *lengths, u_real=od.OD_F32, fast_math=1, **kw)) as s:
        s.set_state(u)
        rhs = s.rhs()
        s.step(1e-3, 5)
        state = s.get_state()
    err = rel_err_per_var(state, O.step(po, u.astype(np.float64), 1e-3, 5))
    rhs64 = O.rhs_total(po, u.astype(np.float64))
    rhs_err = rel_err_per_var(rhs, rhs64)
    rhs_err32 = rel_err_per_var(O.rhs_total(O.params(*n, *lengths, u_real=4, **kw), u), rhs64)
    print("rel err per var, state", err, "rhs", rhs_err, "of f32", rhs_err / rhs_err32, flush=True)
    assert np.all(err < TOL), err
    assert np.all(rhs_err <= 2.0 * rhs_err32), (rhs_err, rhs_err32)


@pytest.mark.parametrize("n", THIN + ODD_HEIGHT, ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("flux", ["slau2", "ausm+", "rusanov"])
@pytest.mark.parametrize("viscous", [True, False])
def test_small_boxes_against_fp64_oracle(n, flux, viscous):
    for wall in (True, False):
        compare(n, flux, wall, viscous, (2 * np.pi, 2.0, np.pi))


@pytest.mark.parametrize("n", CORE_SHELL, ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("flux", ["slau2", "ausm+", "rusanov"])
def test_core_and_shell_against_fp64_oracle(n, flux):
    for wall in (True, False):
        compare(n, flux, wall, True, tuple(float(d) for d in n))


def test_euler_core_and_shell_against_fp64_oracle():
    compare((8, 27, 15), "slau2", True, False, (8.0, 27.0, 15.0))  # 1620 tiles
