"""The plane ratios of the dynamic Smagorinsky model from many partial sums a row:
more and fewer than a lane's loads in flight cover in one round, and the launch's
time where there are thousands."""
import pytest

from channel_rl_amd import FP64, KERNEL_DSM, NU_T, Channel
from helpers import rel
from test_gpu_parity import cases, make_pair

pytestmark = pytest.mark.gpu


# partials a row, tile by tile: ceil((nx-1)/28) * 2 * ceil((nz-1)/4), and
# ceil((nx-1)/12) * ceil((nz-1)/4) of the 12-wide tile; a round of the wave takes
# 1024.  FP64 round-off as for the other whole-field comparisons.
@pytest.mark.parametrize("shape", [1, 3])
@pytest.mark.parametrize("n", [(66, 6, 152), (290, 6, 182), (290, 6, 386)])
def test_ratio_of_many_partials_matches_oracle(gpu, n, shape):
    case, o, g, (U, V, W) = make_pair(*n)
    ref = o.compute_eddy_viscosity(U, V, W)
    g = Channel(case.x, case.y, case.z, precision=FP64, **case.kwargs())
    g.set_state(U, V, W)
    g.set_tile_shape(shape, KERNEL_DSM)
    g.compute_eddy_viscosity()
    assert rel(g.get_field(NU_T), ref) <= 1e-12


# 2716 partials in each of 192 rows (8.3 MB, 1.5 us at the memory's rate) beside a
# pass A of about 800 us: with its launch and the events around it the sum stays
# below a fortieth of the pass; a load at a time it takes more.  The least of
# several steps, so that one late launch does not decide.
def test_ratio_launch_is_short_on_a_large_grid(gpu):
    case, field = cases.small_case(386, 193, 386, seed=3)
    g = Channel(case.x, case.y, case.z, precision=FP64, **case.kwargs())
    g.set_state(*field)
    g.apply_boundary_conditions()
    g.compute_projection_step()
    g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
    g.run_steps(1)
    best = {}
    for _ in range(6):
        for name, (ms, launches) in g.profile_steps(1).items():
            best[name] = min(best.get(name, 1e9), 1e3 * ms / launches)
    g.close()
    print({q: best[q] for q in ("k_dsm_fused", "k_dsm_ratio")})
    assert best["k_dsm_ratio"] <= best["k_dsm_fused"] / 40
