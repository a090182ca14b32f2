"""The two forms of a stage's start that a launch selection decides between: the
stress pass computing the x gradients itself (its shape and the x gradient
pass's alike), and a separate x gradient pass (shapes that differ), each against
the oracle (1e-12 relative max-norm per variable, momentum as one vector)."""
import numpy as np
import pytest

import astr_amd as A
from fields import periodic_field
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("main", [True, False])
@pytest.mark.parametrize("dims", [(24, 20, 16), (33, 28, 0)])
def test_both_forms_match_the_oracle(main, dims, own):
    q = periodic_field(A.tgv_config(*dims), 6)
    s = O.MainState(O.tgv_cfg(*dims, dt=1e-3, suth_dim=110.3)) if main else O.OracleState(O.tgv_cfg(*dims, dt=1e-3))
    s.set_q(q.copy())
    f = A.Flow((A.main_config if main else A.tgv_config)(*dims, deltat=1e-3))
    f.set_pass_config(3, 0, 2, 1)
    f.set_pass_config(0, 0, 2 if own else 4, 1)
    f.upload(q)
    f.profile_begin(400)
    f.rk3(2, stats=False)
    launched = f.profile_end()
    assert (("gc_first", "x") in launched) == (not own)
    s.rk3(2)
    got, want = f.download(), s.get()[0] if main else s.q
    for m in (slice(0, 1), slice(1, 4), slice(4, 5)):
        assert np.abs(got[m] - want[m]).max() <= 1e-12 * np.abs(want[m]).max()
