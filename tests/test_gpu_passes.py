"""The forms a pass takes by its tile count (one component per workgroup below
a limit, a whole tile above it) and the stress pass that computes the x
gradients itself, against the oracle on both sides of each limit.

Tolerances, as for the passes elsewhere: 1e-12 relative max-norm per variable
(momentum as one vector), 1e-9 for histories."""
import numpy as np
import pytest

import astr_amd as A
from fields import periodic_field
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-12
# (launch shape, dims): with the one-line (8) and two-line (7) shapes the y
# passes have these tiles: 128 | 136 (gradients that form the pressure), 320 |
# 324 (flux derivative), 384 | 390 (gradients), 512 | 513 (filter sweep)
SIDES = [(7, (15, 13, 15)), (7, (15, 13, 16)), (8, (15, 13, 19)), (8, (17, 13, 17)), (8, (15, 13, 23)),
         (8, (25, 13, 14)), (8, (15, 13, 31)), (8, (18, 13, 26)), (8, (40, 37, 0)), (7, (40, 37, 0))]


def relmax(a, b):
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(b).max(), 1e-300))


def state_err(a, b):
    return max(relmax(a[0], b[0]), relmax(a[1:4], b[1:4]), relmax(a[4], b[4]))


def force(f, shape):
    for prog in range(len(A.PASS_NAMES)):
        for d in range(3 if f.cfg.km > 0 else 2):
            f.set_pass_config(prog, d, shape, 2)


@pytest.mark.parametrize("shape,dims", SIDES)
def test_miniapp_on_both_sides_of_the_limits(shape, dims):
    s = O.OracleState(O.tgv_cfg(*dims, dt=1e-3))
    s.tgv_init(1e-3, 5)
    s.set_q(s.q.copy())
    f = A.Flow(A.tgv_config(*dims, deltat=1e-3))
    force(f, shape)
    f.upload(s.q.copy())
    got = f.rhscal()
    s.rhscal()
    for m in range(5):
        if m == 3 and dims[2] == 0:
            continue
        assert relmax(got[m], s.qrhs[m]) < TOL, m
    dvel, dtmp = f.gradcal()
    for m in range(9):
        assert relmax(dvel[m], s.dvel[m]) < TOL or np.abs(dvel[m]).max() < 1e-300, m
    ke, en, di = f.rk3(2, dissipation=True)
    ke0, en0 = s.rk3(2)
    assert state_err(f.download(), s.q) < TOL
    assert relmax(ke, ke0) < 1e-9 and relmax(en, en0) < 1e-9


@pytest.mark.parametrize("shape,dims", SIDES)
def test_main_on_both_sides_of_the_limits(shape, dims):
    s = O.MainState(O.tgv_cfg(*dims, dt=1e-3, suth_dim=110.3))
    q = periodic_field(A.main_config(*dims), 3)
    s.set_q(q.copy())
    f = A.Flow(A.main_config(*dims, deltat=1e-3))
    force(f, shape)
    f.upload(q)
    ke, en, di = f.rk3(2, dissipation=True)
    ke0, en0, di0 = s.rk3(2)
    qd, prd = f.download(prims=True)
    qo, pro = s.get()
    assert state_err(qd, qo) < TOL
    assert relmax(prd, pro) < TOL
    assert relmax(ke, ke0) < 1e-9 and relmax(en, en0) < 1e-9 and relmax(di, di0) < 1e-9


@pytest.mark.parametrize("main", [False, True])
@pytest.mark.parametrize("dims", [(40, 36, 28), (48, 40, 0)])
def test_x_gradients_of_the_stress_pass_have_the_gradient_pass_bits(main, dims):
    """The gradients the stress pass stores (both x passes on one launch
    shape) equal those of the x gradient pass on that shape bit for bit."""
    out = []
    for other in (8, 7):
        f = A.Flow((A.main_config if main else A.tgv_config)(*dims, deltat=1e-3))
        f.upload(periodic_field(f.cfg, 4))
        f.set_pass_config(0, 0, 8, 1)       # the x gradient pass
        f.set_pass_config(3, 0, other, 1)   # the stress pass
        out.append(f.gradcal())
    (dv, dt), (dv1, dt1) = out
    assert np.array_equal(dv, dv1) and np.array_equal(dt, dt1)
