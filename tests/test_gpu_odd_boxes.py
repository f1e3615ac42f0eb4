"""Which kernels a fast f32 box with an odd dimension runs on, and that the forms
agree: small ones run on two-element tiles, larger ones on 2x2x2-element blocks with
the last layers on tiles in one launch.

The same flow repeated an odd number of times along x and z fills a larger box, odd
like the small one, with the same element sizes, and every copy must equal the small
box bit for bit: tiles against blocks, also in a channel of odd height, one wall of
which lies on blocks and the other on the tiles of the last layer."""
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


def update_kernel(p):
    u = np.repeat(np.array([1.0, 0.1, 0.0, 0.0, 2.0], np.float32), 64 * p.nx * p.ny * p.nz)
    with od.Solver(p) as s:
        s.set_state(u)
        return [k for k in s.time_kernels(1e-4, 1) if "update" in k][0]


# the largest box on tiles and one above it (tiles of two elements along x: 512, 513
# and 540; Euler 1500, 1512), and its smallest
@pytest.mark.parametrize("n,viscous,on_tiles", [((3, 3, 3), True, True), ((3, 16, 16), True, True),
                                                ((5, 19, 9), True, False), ((9, 9, 12), True, False),
                                                ((3, 30, 25), False, True), ((3, 27, 28), False, False)],
                         ids=str)
def test_form_of_an_odd_box(n, viscous, on_tiles):
    p = od.params(*n, 3.0, 2.0, 2.5, u_real=od.OD_F32, viscous=viscous, mu_ref=1e-3 if viscous else 0.0, fast_math=1)
    assert update_kernel(p) == ("od_update_kernel" if on_tiles else "od_update_core_shell_kernel")


# every combination of odd directions, as many times as gives core and shell; shells
# with every remainder of a work-group's three and four tiles
@pytest.mark.parametrize("n,times", [((3, 3, 3), (11, 1, 11)), ((3, 5, 3), (11, 1, 9)), ((2, 3, 2), (17, 1, 31)),
                                     ((4, 5, 2), (15, 1, 11)), ((1, 3, 1), (33, 1, 35)), ((1, 2, 5), (33, 1, 11)),
                                     ((3, 2, 2), (21, 1, 13)), ((2, 2, 3), (31, 1, 11)), ((3, 3, 2), (21, 1, 13)),
                                     ((2, 3, 3), (21, 1, 11))],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("viscous", [True, False])
def test_tiles_equal_core_and_shell(n, times, viscous):
    large = [d * q for d, q in zip(n, times)]
    length = [0.5 * d for d in n]  # elements of side 1/2 in both boxes: the same Jacobians
    for flux in ("slau2", "ausm+", "rusanov"):
        for wall in (True, False):
            print(f"CASE test=odd_boxes n={n} times={times} viscous={viscous} flux={flux} wall={wall}", flush=True)
            kw = dict(u_real=od.OD_F32, flux=flux, y_wall=wall, viscous=viscous, viscosity_model=1,
                      mu_ref=0.002 if viscous else 0.0, fast_math=1)
            u = smooth_state(*n, *length, seed=sum(n), amp=0.05, dtype=np.float32)
            out = []
            for t in ((1, 1, 1), times):
                p = od.params(*[d * q for d, q in zip(n, t)], *[x * q for x, q in zip(length, t)], **kw)
                form = update_kernel(p)
                assert form == ("od_update_kernel" if t == (1, 1, 1) else "od_update_core_shell_kernel"), (large, form)
                with od.Solver(p) as s:
                    s.set_state(repeated(u, n, t))
                    s.step(0.003, 5)
                    out.append((s.get_state(), s.rhs()))
            for a, b in zip(*out):
                assert np.isfinite(a).all()
                wrong = np.count_nonzero(repeated(a, n, times).view(np.uint32) != b.view(np.uint32))
                assert wrong == 0, wrong


def test_boxes_of_a_batch_switch_between_their_forms():
    """Box by box a small odd box runs on tiles, in batched steps its core on blocks,
    which leave out the core's internal traces; larger odd boxes and even ones keep
    their form.  Every box follows the box run alone, however the steps are made."""
    print("CASE test=odd_boxes_batch", flush=True)
    kw = dict(u_real=od.OD_F32, y_wall=True, viscosity_model=1, mu_ref=2e-3, fast_math=1)
    boxes = [(3, 3, 3, 1.5, 1.5, 1.5), (5, 19, 9, 2.5, 9.5, 4.5), (4, 4, 2, 2.0, 2.0, 1.0), (1, 5, 3, 0.5, 2.5, 1.5),
             (2, 5, 4, 1.0, 2.5, 2.0)]
    inits = [smooth_state(*x, seed=q, amp=0.04, dtype=np.float32) for q, x in enumerate(boxes)]
    plan = [(0, 2), (2, 1), (1, 1), (2, 2), (0, 1), (0, 1), (2, 1)]
    with od.Batch(od.params(1, 1, 1, 1.0, 1.0, 1.0, **kw), boxes) as b:
        for q, u in enumerate(inits):
            b.set_state(q, u)
        for order, n in plan:
            b.set_schedule(order=order)
            b.step(0.003, n)
        b.set_schedule(order=0)
        b.time_steps(0.003, 2)
        b.time_steps(0.003, 1, per_box=True)
        b.step(0.003, 1)
        got = [b.get_state(q) for q in range(len(boxes))]
    for q, x in enumerate(boxes):
        with od.Solver(od.params(*x, **kw)) as s:
            s.set_state(inits[q])
            s.step(0.003, sum(n for _, n in plan) + 4)
            want = s.get_state()
        assert np.isfinite(want).all()
        assert np.array_equal(got[q].view(np.uint32), want.view(np.uint32)), x
