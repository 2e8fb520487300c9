"""The RHS kernel's tile and z chunk as picked by the grid (shape 0) at the edges
of that rule: one-plane chunks, both tiles with remainders in x, y and z, more
blocks than one round and a group's tiles; against a fixed tile and chunk."""
import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, FP64, KERNEL_RHS, NU_T, P, Channel
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


# every cell is computed once by the same operations, so any tile and chunk
# gives the same bits
@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("n", [(6, 4, 6), (66, 7, 38), (98, 31, 62), (130, 41, 66), (38, 100, 130)])
def test_picked_tile_agrees_bitwise(gpu, n, precision):
    case, field = cases.small_case(*n, seed=7)
    out = []
    for shape in (0, 3):
        g = Channel(case.x, case.y, case.z, precision=precision, **case.kwargs())
        g.set_state(*field)
        g.apply_boundary_conditions()
        g.compute_projection_step()
        g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
        g.set_tile_shape(shape, KERNEL_RHS)
        g.run_steps(2)
        out.append(list(g.state()) + [g.get_field(NU_T), g.get_field(P)])
        g.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
