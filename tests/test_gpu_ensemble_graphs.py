"""How many steps an ensemble captures: one per rotation of the states, and a
second form of each, the last of a call, only where that one differs (dynamic
Smagorinsky members, whose other steps leave nu_t to the RHS)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

SCRIPT = """
import ctypes, sys
count = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library that it counts for
from channel_rl_amd import Channel, Ensemble, cases
for models in sys.argv[2:]:
    chans = []
    for q, les in enumerate(models.split(",")):
        case, field = cases.small_case(18, 9, 10, seed=q)
        g = Channel(case.x, case.y, case.z, **dict(case.kwargs(), LES_model=int(les)))
        g.set_state(*field)
        g.apply_boundary_conditions()
        g.compute_projection_step()
        g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
        chans.append(g)
    e = Ensemble(chans)
    before = count.graphs_instantiated()
    for _ in range(3):
        e.run_steps(7)  # the last step meets each rotation once
    e.synchronize()
    print(count.graphs_instantiated() - before, flush=True)
    e.close()
    [g.close() for g in chans]
"""


# per ensemble, its members' SGS models (2: dynamic Smagorinsky, 3: AMD)
@pytest.mark.parametrize("deferred, want", [(True, [3, 6, 6]), (False, [3, 3, 3])])
def test_captured_steps(gpu, tmp_path, deferred, want):
    lib = str(tmp_path / "count_graphs.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", os.path.join(HERE, "host", "count_graphs.c"), "-o", lib,
                    "-L/opt/rocm/lib", "-Wl,--no-as-needed", "-lamdhip64", "-ldl"], check=True)
    env = dict(os.environ, CHANLES_NO_DEFERRED_NUT="0" if deferred else "1")
    r = subprocess.run([sys.executable, "-c", SCRIPT, lib, "3,3", "2,2", "3,2"], cwd=ROOT, env=env,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert [int(v) for v in r.stdout.split()] == want
