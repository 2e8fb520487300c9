"""Whole-field reads at the edge of the threaded copy's range: fields just below
and above it, a last chunk that is partial, several threads at once (one of them
finds the slots in use), and channels that come and go."""
import threading

import numpy as np
import pytest

from channel_rl_amd import FP32_BULK, FP64, P, U, V, W, Channel
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


# copies: every byte as the field was set, NU_T-sized boxes of 15.8, 16.3 and 33 MB
@pytest.mark.parametrize("n", [(130, 115, 130), (130, 119, 130), (194, 109, 194)])
def test_large_fields_return_as_set(gpu, n):
    case, _ = cases.small_case(*n, seed=5)
    chans = [Channel(case.x, case.y, case.z, precision=q, **case.kwargs()) for q in (FP64, FP32_BULK)]
    rng = np.random.default_rng(11)
    want = []
    for g in chans:
        f = {w: np.asfortranarray(rng.standard_normal(g.shape(w)).astype(np.float32).astype(np.float64))
             for w in (U, V, W, P)}
        for w, a in f.items():
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
