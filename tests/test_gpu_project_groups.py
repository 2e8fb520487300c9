"""The projection with four z cells a lane, which a group of FP32 channels takes
from 4096 blocks on, where the number of planes leaves two cells over: against the
same channels stepped alone, with one cell a lane."""
import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, NU_T, P, U, V, W, Channel, Ensemble
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


def _channel(n, seed, mass):
    case, field = cases.small_case(*n, seed=seed)
    g = Channel(case.x, case.y, case.z, precision=FP32_BULK, **dict(case.kwargs(), x_mass_cte=mass))
    g.set_state(*field)
    g.apply_boundary_conditions()
    g.compute_projection_step()
    g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
    if mass == 2:
        g.initialize_mass_flow()
    g.set_wall_model(1, h_wm=case.h_wm)
    return g


# the same operations a cell either way: the same bits, images and walls included.
# Blocks of 64 x 4 cells where rows fill them, 32 x 8 where those leave fewer lanes
# idle; mass 1 adds the last projection's shift
@pytest.mark.parametrize("mass", [1, 2])
@pytest.mark.parametrize("n, members, block", [((66, 33, 52), 11, (64, 4)), ((98, 30, 32), 12, (32, 8))])
def test_planes_left_over(gpu, n, members, block, mass):
    nx, ny, nz = n
    planes = nz - 2
    blocks = -(-(nx - 2) // block[0]) * -(-(ny - 1) // block[1]) * planes
    assert planes % 4 == 2 and blocks < 4096 <= blocks * members
    alone = []
    for q in range(members):
        g = _channel(n, q, mass)
        g.run_steps(2)
        alone.append([g.get_field(w) for w in (U, V, W, P, NU_T)])
        g.close()
    chans = [_channel(n, q, mass) for q in range(members)]
    e = Ensemble(chans)
    assert e.group_count() == 1
    e.run_steps(2)
    for g, want in zip(chans, alone):
        for a, b in zip([g.get_field(w) for w in (U, V, W, P, NU_T)], want):
            assert np.isfinite(a).all() and np.array_equal(a, b)
    e.close()
    [g.close() for g in chans]
