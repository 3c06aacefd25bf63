"""The segment store that a forward run fills for the backward pass counts all
of its buffers against its limit of 4 GiB: with 65 million SRD cells the
collisions of an 11-step segment take 5 GB beside 40 beads, so the run leaves
the store to the backward pass.  The gradient is the one of segments that are
kept (FP64 sums of the same terms, grouped by segment: 1e-12)."""
import ctypes

import adjoint_case as case
import numpy as np
import pytest
import torch

from nwamd.abi import DeviceArray

pytestmark = pytest.mark.gpu

GAP, STEPS = 10, 11


def gradient(lib, K):
    p, e, s = case.srd_system()
    g, L = (8000, 8200), 12.0
    s.gridSize.x, s.gridSize.y, s.numCells = *g, g[0] * g[1]
    s.cellSize.x, s.cellSize.y = L / g[0], L / g[1]
    lib.setSolventParameters(ctypes.byref(s))
    pos, vel, zero, w, wv = case.srd_initial_state()
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    lib.nwRngSetSeed(case.SEED, case.OFFSET)
    d = [DeviceArray.from_numpy(lib, a) for a in (pos, vel, zero, zero, zero)]
    shifts = np.zeros((STEPS // GAP + 1) * 3, np.float32)
    free = torch.cuda.mem_get_info()[0]
    lib.nwAdjointForwardSrd(*[x.p for x in d], p.numFilaments, s.numParticles, case.DT, GAP,
                            shifts.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), STEPS, K)
    lib.threadSync()
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    taken = free - torch.cuda.mem_get_info()[0]
    dW, dWv = DeviceArray.from_numpy(lib, w), DeviceArray.from_numpy(lib, wv)
    out = (ctypes.c_double * 4)()
    lib.nwAdjointBackward(dW.p, dWv.p, out)
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    return np.array(out), taken


def test_store_counts_its_collisions(nwlib):
    whole, taken = gradient(nwlib, STEPS)
    assert taken < 4 << 30, taken
    kept, _ = gradient(nwlib, 4)
    assert np.abs(whole[:3]).min() > 0
    np.testing.assert_allclose(whole, kept, rtol=1e-12)
