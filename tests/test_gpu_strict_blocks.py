"""Strict viscous boxes large enough for the 2x2x2-element block kernels.  A
small box runs on the kernels by fours and by tiles; the same flow repeated
along each direction fills a box that runs on blocks, with the same element
sizes: every copy must equal the small box bit for bit."""
import numpy as np
import pytest

import opendynamo_amd as od
from helpers import smooth_state

pytestmark = pytest.mark.gpu

TYPES = {"f32": dict(u_real=4), "f64": dict(u_real=8),
         "f64_state": dict(u_real=8, compute_real=4, q_real=4, rhs_real=4, rk_accum=1),
         "f32_state": dict(u_real=4, compute_real=8, q_real=4, rhs_real=4)}


def repeated(u, n, times):
    """The state of the box n repeated times[d] times along direction d."""
    nx, ny, nz = n
    a = u.reshape(5, nz, ny, nx, 64)
    return np.ascontiguousarray(np.tile(a, (1, times[2], times[1], times[0], 1))).ravel()


# odd periods against the blocks' even one; boxes two elements wide, whose
# external neighbour is the block's own other element; walls at both ends of y
@pytest.mark.parametrize("n, times, wall", [((3, 3, 5), (6, 6, 4), False), ((1, 3, 3), (2, 18, 16), False),
                                            ((3, 2, 3), (16, 1, 18), False), ((5, 5, 1), (12, 12, 2), False),
                                            ((3, 2, 5), (18, 1, 10), True), ((3, 18, 3), (6, 1, 6), True)],
                         ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else None)
@pytest.mark.parametrize("types", list(TYPES))
def test_repeated_box_on_blocks_equals_the_small_one(n, times, wall, types):
    for flux, eddy in (("slau2", False), ("ausm+", True), ("rusanov", False)):
        print(f"CASE test=strict_blocks n={n} times={times} wall={wall} types={types} flux={flux}", flush=True)
        kw = dict(TYPES[types], flux=flux, y_wall=wall, viscous=True, viscosity_model=1, mu_ref=2e-3)
        length = [0.5 * d for d in n]  # powers of two times n: the same Jacobians in both boxes
        u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=np.float32 if kw["u_real"] == 4 else np.float64)
        mu = np.random.default_rng(2).uniform(0.0, 3e-3, (n[2], n[1], n[0]))
        out = []
        for t in ((1, 1, 1), times):
            p = od.params(*[d * q for d, q in zip(n, t)], *[x * q for x, q in zip(length, t)], **kw)
            with od.Solver(p) as s:
                s.set_state(repeated(u, n, t))
                if eddy:
                    s.set_eddy_viscosity(np.tile(mu, (t[2], t[1], t[0])).ravel())
                s.step(0.003, 4)
                out.append((s.get_state(), s.rhs()))
                names = set(s.time_kernels(0.003, 1))
            assert names == ({"od_visc_line_kernel", "od_update_kernel"} if len(out) == 1 else
                             {"od_visc_lines_block_kernel", "od_update_face_block_kernel"})
        for small, large in zip(*out):
            assert np.isfinite(small).all()
            assert repeated(small, n, times).tobytes() == large.tobytes()
