"""Whole-field reads into device memory, which the runtime's copy takes: fields
below and above the threaded copy's least size, every byte as set."""
import ctypes

import numpy as np
import pytest
import torch

from channel_rl_amd import U, Channel, load_library
from test_gpu_parity import cases

pytestmark = pytest.mark.gpu


# the threaded copy begins at 16 MiB
@pytest.mark.parametrize("n, large", [((34, 17, 34), False), ((130, 123, 130), True)])
def test_field_into_device_memory(gpu, n, large):
    case, _ = cases.small_case(*n, seed=5)
    g = Channel(case.x, case.y, case.z, **case.kwargs())
    a = np.asfortranarray(np.random.default_rng(2).standard_normal(g.shape(U)))
    assert (a.nbytes >= 16 << 20) == large
    g.set_field(U, a)
    t = torch.zeros(a.size, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert load_library().chan_get_field(g._h, U, ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))) == 0
    assert np.array_equal(t.cpu().numpy(), a.ravel(order="K"))
    g.close()
