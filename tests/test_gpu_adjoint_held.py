"""The forward run leaves its last segment for the backward pass: the gradient
for whole and ragged last segments, with the caller's arrays overwritten
between the two, and again for a second backward pass, against one segment a
step (FP64 sums of the same terms, grouped by segment: 1e-12)."""
import ctypes

import adjoint_case as case
import numpy as np
import pytest

from nwamd.abi import DeviceArray

pytestmark = pytest.mark.gpu


def gradients(lib, srd, steps, K):
    if srd:
        p, e, s = case.srd_system()
        lib.setSolventParameters(ctypes.byref(s))
        pos, vel, zero, w, wv = case.srd_initial_state()
    else:
        p, e = case.system()
        pos, vel, zero, w = case.initial_state()
        wv = np.zeros_like(w)
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    lib.nwRngSetSeed(case.SEED, case.OFFSET)
    d = [DeviceArray.from_numpy(lib, a) for a in (pos, vel, zero, zero, zero)]
    ptr = [x.p for x in d]
    if srd:
        sh = np.ascontiguousarray(case.srd_shifts(steps).reshape(-1))
        lib.nwAdjointForwardSrd(*ptr, p.numFilaments, s.numParticles, case.DT, case.SRD_GAP,
                                sh.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), steps, K)
    else:
        lib.nwAdjointForward(*ptr, p.numFilaments, case.DT, case.THETA[3], case.KT / case.DT, 1, steps, K)
    for x, a in zip(d, (pos, vel, zero, zero, zero)):
        x.upload(np.zeros_like(a))
    dW, dWv = DeviceArray.from_numpy(lib, w), DeviceArray.from_numpy(lib, wv)
    out = []
    for _ in range(2):
        g = (ctypes.c_double * 4)()
        lib.nwAdjointBackward(dW.p, dWv.p, g)
        out.append(np.array(g))
    return out


@pytest.mark.parametrize("srd", [False, True])
@pytest.mark.parametrize("K", [2, 7, 12, 24, 40])
def test_held_segment(nwlib, srd, K):
    ref = gradients(nwlib, srd, 24, 1)[0]
    assert np.abs(ref).max() > 0
    for g in gradients(nwlib, srd, 24, K):
        np.testing.assert_allclose(g, ref, rtol=1e-12)
