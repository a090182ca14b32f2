"""The launch shapes a case gets without tuning, on both sides of the lengths
and line counts where they change, against the oracle: the filter sweeps alone
(1e-13 of each variable's maximum, sums of eleven terms) and a step (1e-12)."""
import numpy as np
import pytest

import astr_amd as A
from fields import periodic_field
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def err(a, b):
    return max(float(np.abs(a[m] - b[m]).max() / np.abs(b[m]).max()) for m in (slice(0, 1), slice(1, 4), slice(4, 5)))


# n = 137 | 138 and 313 | 314 with 8192 lines or more (137 x 91 x 90 along x) or 1024 or more
# and 3-D cases of fewer than 1024 lines along a direction
@pytest.mark.parametrize("dims", [(12, 12, 12), (30, 31, 30), (153, 12, 14), (154, 12, 14), (12, 73, 74), (80, 24, 24), (80, 25, 24), (137, 91, 90), (138, 91, 90), (137, 90, 88), (40, 137, 200), (36, 200, 137), (313, 40, 36),
                                  (314, 40, 36), (30, 314, 36), (32, 34, 314), (314, 30, 0), (400, 30, 0)])
def test_filter_and_step_on_default_shapes(dims):
    s = O.OracleState(O.tgv_cfg(*dims, dt=2e-4))
    q = periodic_field(A.tgv_config(*dims), 5)
    s.set_q(q.copy())
    f = A.Flow(A.tgv_config(*dims, deltat=2e-4))
    f.upload(q)
    f.filterq()
    s.filterq()
    assert err(f.download(), s.q) < 1e-13
    f.upload(q)
    s.set_q(q.copy())
    f.rk3(1, stats=False)
    s.rk3(1)
    assert err(f.download(), s.q) < 1e-12
