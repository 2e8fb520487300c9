"""The learned wall model with 16, 32 and 64 cells a wave: one, four and eight
channels of one wall in a launch, the last set partial."""
import numpy as np
import pytest

from channel_rl_amd import ALPHA_X, FP32_BULK, FP64, NU_T, U, WALL_MLP, Channel, Ensemble, WallNetwork
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


# a cell's values do not depend on the wave it shares: the same bits
@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
def test_cells_per_wave(gpu, precision):
    net = WallNetwork(seed=3)
    got = []
    for count in (1, 4, 8):
        chans = []
        for _ in range(count):
            case, field = cases.small_case(66, 9, 66, seed=9)
            g = Channel(case.x, case.y, case.z, precision=precision, **case.kwargs())
            g.set_state(*field)
            g.apply_boundary_conditions()
            g.compute_projection_step()
            g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx)
            g.initialize_mass_flow()
            g.set_wall_network(net, max_rel_err=1e30)
            g.set_wall_model(WALL_MLP, h_wm=case.h_wm)
            chans.append(g)
        e = Ensemble(chans)
        e.run_steps(1)
        got.append([chans[-1].get_field(w) for w in (ALPHA_X, NU_T, U)] + [np.array(chans[-1].wall_model_stats())])
        e.close()
        [g.close() for g in chans]
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b, equal_nan=True)
    assert np.isfinite(got[0][0]).all() and np.any(got[0][0])
