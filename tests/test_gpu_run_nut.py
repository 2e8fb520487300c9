"""nu_t after a call of several steps, whose earlier steps leave pass B to the RHS:
the same bits as steps one call at a time, for the ways a step is launched."""
import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, FP64, NU_T, U, V, W, Channel, Ensemble
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


# nu_t = max(A v, B) of the same values by the same operations wherever it is taken
@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("mass, limit, graph", [(0, 0.0, True), (1, 0.0, True), (2, 0.25, True), (1, 0.0, False)])
def test_nu_t_after_several_steps(gpu, monkeypatch, mass, limit, graph, precision):
    monkeypatch.setenv("CHANLES_NO_GRAPH", "0" if graph else "1")
    case, field = cases.small_case(34, 17, 26, seed=9)
    kw = dict(case.kwargs(), x_mass_cte=mass)
    got = []
    for calls in ([5], [1] * 5, [3, 2]):
        g = Channel(case.x, case.y, case.z, precision=precision, **kw)
        g.set_state(*field)
        g.apply_boundary_conditions()
        g.compute_projection_step()
        g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
        g.set_wall_model(1, h_wm=case.h_wm)
        if limit:
            g.set_wall_viscosity_limit(limit)
        for n in calls:
            g.run_steps(n)
        got.append([g.get_field(w) for w in (NU_T, U, V, W)])
        g.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.isfinite(a).all() and np.array_equal(a, b)


# the same of an ensemble: two grouped members and a lone one
@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
def test_nu_t_after_several_ensemble_steps(gpu, precision):
    got = []
    for calls in ([5], [1] * 5, [3, 2]):
        chans = []
        for n, seed in (((34, 17, 26), 3), ((34, 17, 26), 4), ((18, 9, 10), 5)):
            case, field = cases.small_case(*n, seed=seed)
            g = Channel(case.x, case.y, case.z, precision=precision, **dict(case.kwargs(), x_mass_cte=2))
            g.set_state(*field)
            g.apply_boundary_conditions()
            g.compute_projection_step()
            g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx)
            g.initialize_mass_flow()
            g.set_wall_model(1, h_wm=case.h_wm)
            chans.append(g)
        e = Ensemble(chans)
        assert e.group_count() == 2
        for n in calls:
            e.run_steps(n)
        got.append([g.get_field(w) for g in chans for w in (NU_T, U, V, W)])
        e.close()
        [g.close() for g in chans]
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.isfinite(a).all() and np.array_equal(a, b)
