"""A batch's launches do not depend on what was last asked of a case on its own."""
import ctypes as C

import numpy as np
import pytest

import astr_amd as A
from astr_amd import hip

pytestmark = pytest.mark.gpu


def x_gradients(f):
    """The device's x gradients of u, v, w and T (behind the five fields of
    qrhs: nine velocity gradients, x first, then three of T)."""
    lay = A.Layout()
    assert A.lib().astr_hip_field_info(f.h, C.byref(lay)) == 0
    f.sync()
    out = np.empty((4, lay.field_stride))
    base = C.cast(lay.qrhs, C.c_void_p).value
    for row, fld in enumerate((0, 1, 2, 9)):
        src = C.c_void_p(base + 8 * lay.field_stride * (5 + fld))
        assert hip.rt().hipMemcpy(out[row].ctypes.data_as(C.c_void_p), src, 8 * lay.field_stride, 2) == 0
    return out[:, :lay.plane * f.shape[0]].reshape(4, f.shape[0], lay.plane)[:, :, :lay.pitch * f.shape[1]].reshape(
        (4,) + f.shape[:2] + (lay.pitch,))[..., :f.shape[2]]


def test_gradcal_before_a_batch_leaves_its_passes_alone():
    """gradcal makes a case's stress pass store the x gradients; the passes of
    a batch created afterwards do not (four fields written per stage): the
    stored gradients stay those of the state before the batch's steps."""
    flows = [A.Flow(A.tgv_config(n, deltat=2e-3)) for n in (24, 33)]
    for k, f in enumerate(flows):
        f.init_tgv(1e-2, k)
        dvel, dtmp = f.gradcal()
        got = x_gradients(f)
        assert np.array_equal(got[:3], dvel[:3]) and np.array_equal(got[3], dtmp[0])
    before = [x_gradients(f) for f in flows]
    b = A.Batch(flows)
    b.rk3(1)
    for f, g in zip(flows, before):
        assert np.array_equal(x_gradients(f), g)
    b.close()
