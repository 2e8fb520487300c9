"""compute_dt on its own at the edges of its tiles: rows narrower and wider than
either tile, planes left over, more tiles than blocks; the deciding component and
the place of its extreme varied, zeros and infinities among the values."""
import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, FP64
from test_gpu_parity import Channel, make_pair

pytestmark = pytest.mark.gpu


# a maximum of correctly rounded quotients, in any order: the same bits
@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("n", [(6, 4, 6), (34, 5, 10), (66, 9, 38), (92, 11, 14), (130, 41, 66)])
def test_dt_of_any_cell(gpu, n, precision):
    case, o, g, field = make_pair(*n, CFL=0.5)
    if precision != FP64:
        g = Channel(case.x, case.y, case.z, precision=precision, **case.kwargs())
    rng = np.random.default_rng(17)
    for comp in range(3):
        f = []
        for c, a in enumerate(field):
            a = rng.uniform(1.0, 2.0, a.shape) * (1e4 if c == comp else 1e3) * rng.choice([-1.0, 1.0], a.shape)
            f.append(np.asfortranarray(a.astype(np.float32).astype(np.float64)))
        shape = f[comp].shape
        last = (shape[0] - 1, shape[1] - 2 if comp != 1 else shape[1] - 1, shape[2] - 2 if comp != 2 else shape[2] - 1)
        for where in [(1, 1, 1), last, tuple(rng.integers(1, s - 1) for s in shape)]:
            f[comp][where] = 4096.0
            f[comp][tuple(rng.integers(1, s - 1) for s in shape)] = np.inf
            for q in (o, g):
                q.set_state(*f)
            assert g.compute_dt() == o.compute_dt()
        f[comp][2, 2, 2] = 0.0
        for q in (o, g):
            q.set_state(*f)
        assert g.compute_dt() == o.compute_dt()
