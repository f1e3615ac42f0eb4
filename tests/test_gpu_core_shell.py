"""Boxes with an odd dimension in the fast f32 build: core on 2x2x2-element
blocks and the last layers on two-element tiles in one launch.  The same flow
repeated along each odd direction fills a box with even dimensions, which runs
on blocks alone, with the same element sizes: every copy must equal the odd box
bit for bit."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state

pytestmark = pytest.mark.gpu


def repeated(u, n, times):
    """The state of the box n repeated times[d] times along direction d."""
    nx, ny, nz = n
    a = u.reshape(5, nz, ny, nx, 64)
    return np.ascontiguousarray(np.tile(a, (1, times[2], times[1], times[0], 1))).ravel()


# every combination of odd directions; shells of fewer than four tiles (a
# work-group's part), of a multiple of four and of one more; a core of one block
@pytest.mark.parametrize("n", [(3, 2, 2), (2, 3, 2), (2, 2, 3), (3, 3, 2), (3, 2, 3), (2, 3, 3), (3, 3, 3), (5, 4, 4),
                               (9, 2, 2), (7, 5, 9), (4, 11, 6)], ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("viscous", [True, False])
def test_odd_box_equals_its_repetition_on_blocks(n, viscous):
    for flux in ("slau2", "ausm+", "rusanov"):
        for wall in ((False, True) if n[1] % 2 == 0 else (False,)):
            print(f"CASE test=core_shell n={n} viscous={viscous} flux={flux} wall={wall}", flush=True)
            kw = dict(u_real=od.OD_F32, flux=flux, y_wall=wall, viscous=viscous, viscosity_model=1,
                      mu_ref=0.002 if viscous else 0.0, fast_math=1)
            times = [1 + d % 2 for d in n]
            length = [0.5 * d for d in n]  # powers of two times n: the same Jacobians in both boxes
            u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=np.float32)
            out = []
            for t in ([1, 1, 1], times):
                p = od.params(*[d * q for d, q in zip(n, t)], *[x * q for x, q in zip(length, t)], **kw)
                with od.Solver(p) as s:
                    s.set_state(repeated(u, n, t))
                    s.step(0.003, 9)
                    out.append((s.get_state(), s.rhs()))
            for small, large in zip(*out):
                assert np.isfinite(small).all()
                assert repeated(small, n, times).tobytes() == large.tobytes()


def test_eddy_viscosity_in_core_and_shell():
    """Each element's own eddy viscosity reaches it in both kernel forms."""
    n, times = (5, 4, 3), [2, 1, 2]
    print("CASE test=core_shell_mu_t", flush=True)
    kw = dict(u_real=od.OD_F32, y_wall=True, mu_ref=1e-3, fast_math=1)
    u = smooth_state(*n, 2.5, 2.0, 1.5, seed=1, amp=0.05, dtype=np.float32)
    mu = np.random.default_rng(2).uniform(0.0, 3e-3, (n[2], n[1], n[0]))
    out = []
    for t in ([1, 1, 1], times):
        p = od.params(*[d * q for d, q in zip(n, t)], 2.5 * t[0], 2.0, 1.5 * t[2], **kw)
        with od.Solver(p) as s:
            s.set_state(repeated(u, n, t))
            s.set_eddy_viscosity(np.tile(mu, (t[2], t[1], t[0])).ravel())
            s.step(0.003, 3)
            out.append(s.get_state())
    assert repeated(out[0], n, times).tobytes() == out[1].tobytes()
