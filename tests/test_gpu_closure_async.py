"""Steps with an attached network are enqueued without waiting: whole refresh
intervals run as one graph, other pieces launch by launch, and the network's
weights and scaling may change right after a step call returns."""
import numpy as np
import pytest

import opendynamo_amd as od
from opendynamo_amd import ic

pytestmark = pytest.mark.gpu

TWO_PI = 2 * np.pi
N, DT = 4, 0.01


def network(seed=0):
    rng = np.random.default_rng(seed)
    m = od.MLP(params=rng.uniform(-0.2, 0.2, od.MLP_PARAMS).astype(np.float32))
    m.set_output_scale(0.05)
    return m


def solver(real=od.OD_F32, fast=1):
    s = od.Solver(od.params(N, N, N, TWO_PI, TWO_PI, TWO_PI, u_real=real, mu_ref=1e-3, body_force_x=0.0,
                            fast_math=fast))
    s.set_state(ic.fourier_state(N, N, N, TWO_PI, TWO_PI, TWO_PI, u0=(0.05, 0.0, 0.0), amplitude=0.05, n_modes=8,
                                 seed=3, kmax=3, dtype=s.dtype))
    return s


# shorter than a graph's 8 steps, exactly 8, longer
@pytest.mark.parametrize("interval", [1, 3, 8, 9])
@pytest.mark.parametrize("kappa", [1.0, 1e-6])  # 1e-6: the budget check switches the model off now and then
@pytest.mark.parametrize("real,fast", [(od.OD_F32, 1), (od.OD_F64, 0)])
def test_split_step_calls_equal_one_call(interval, kappa, real, fast):
    print(f"CASE test=closure_split interval={interval} kappa={kappa} real={real}", flush=True)
    got = []
    for plan in ([26], [1] * 26, [5, 2, 11, 8]):
        with network() as m, solver(real, fast) as s:
            s.attach_closure(m, update_interval=interval, budget_kappa=kappa)
            for n in plan:
                s.step(DT, n)
            stats = s.closure_stats()
            assert stats["updates"] == -(-26 // interval)
            got.append((s.get_state().tobytes(), stats))
            s.attach_closure(None)
    assert got[0] == got[1] == got[2]
    assert (got[0][1]["budget_fallbacks"] > 0) == (kappa < 1.0)


@pytest.mark.parametrize("change", ["params", "scale", "step"])
def test_changes_right_after_a_step_call_do_not_reach_back(change):
    """New weights, a new output scale or a new step size, set while the steps
    are still running, leave those steps as they are."""
    print(f"CASE test=closure_change change={change}", flush=True)
    got = []
    for wait in (False, True):
        with network() as m, solver() as s:
            s.attach_closure(m, update_interval=2, budget_kappa=0.0)
            s.step(DT, 400)
            if wait:
                s.synchronize()
            dt = DT
            if change == "params":
                m.set_params(np.zeros(od.MLP_PARAMS, np.float32))
            elif change == "scale":
                m.set_output_scale(0.01)
            else:
                dt = 0.5 * DT
            s.step(dt, 6)
            got.append(s.get_state())
            s.attach_closure(None)
    assert np.isfinite(got[0]).all()
    assert got[0].tobytes() == got[1].tobytes()


def test_stats_before_and_after_an_attachment():
    with network() as m, solver() as s:
        assert all(v == 0 for v in s.closure_stats().values())
        s.features()  # allocates the closure's buffers
        assert all(v == 0 for v in s.closure_stats().values())
        s.attach_closure(m, update_interval=2)
        s.step(DT, 4)
        assert s.closure_stats()["updates"] == 2
        s.attach_closure(None)
        assert s.closure_stats()["updates"] == 2
        s.attach_closure(m, update_interval=2)
        assert all(v == 0 for v in s.closure_stats().values())
        s.attach_closure(None)
