"""Whole-field reads just below and just above the size at which the threaded copy
begins, where its threads hold two or three chunks and one of them the partial
last; two channels reading at once, one of which finds the slots in use."""
import threading

import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, FP64, P, U, V, W, Channel
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu

LEAST, CHUNK = 16 << 20, 2 << 20  # of the threaded copy


# copies: every byte as the field was set
@pytest.mark.parametrize("n, threaded", [((130, 121, 130), False), ((130, 123, 130), True)])
def test_fields_on_either_side_of_the_limit(gpu, n, threaded):
    case, _ = cases.small_case(*n, seed=5)
    chans = [Channel(case.x, case.y, case.z, precision=q, **case.kwargs()) for q in (FP64, FP32_BULK)]
    rng = np.random.default_rng(11)
    want = []
    for g in chans:
        f = {w: np.asfortranarray(rng.standard_normal(g.shape(w)).astype(np.float32).astype(np.float64))
             for w in (U, V, W, P)}
        for w, a in f.items():
            assert (a.nbytes >= LEAST) == threaded and abs(a.nbytes - LEAST) < CHUNK and a.nbytes % CHUNK != 0
            g.set_field(w, a)
        want.append(f)
    seen = [None] * len(chans)

    def read(q):
        seen[q] = [{w: chans[q].get_field(w) for w in (U, V, W, P)} for _ in range(3)]

    ts = [threading.Thread(target=read, args=(q,)) for q in range(len(chans))]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for got, f in zip(seen, want):
        for one in got:
            for w, a in f.items():
                assert np.array_equal(one[w], a)
    [g.close() for g in chans]


# a read right after an asynchronous run returns the run's result, and channels
# made and closed meanwhile in another thread do not disturb it
def test_read_behind_a_run(gpu):
    case, field = cases.small_case(130, 123, 130, seed=6)
    small, small_field = cases.small_case(18, 9, 10, seed=1)
    got = []
    for beside in (False, True):
        g = Channel(case.x, case.y, case.z, **case.kwargs())
        g.set_state(*field)
        g.apply_boundary_conditions()
        g.compute_projection_step()
        g.set_scalars(dt=0.0, t=0.0, dPdx=case.dPdx, Qflow_x_0=g.compute_mean_mass_flow_U())
        g.run_steps(20)
        out = []
        t = threading.Thread(target=lambda: out.append(g.get_field(U)))
        t.start()
        while beside and t.is_alive():
            h = Channel(small.x, small.y, small.z, **small.kwargs())
            h.set_state(*small_field)
            h.close()
        t.join()
        got.append(out[0])
        g.close()
    assert np.isfinite(got[0]).all() and np.array_equal(*got)
