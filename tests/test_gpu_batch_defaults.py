"""Batches of cases nobody tuned: the launch shapes follow the lines of all cases
together.  On both sides of that rule's limit (1024 lines along a direction),
with cases whose selection was set among them, against the same cases stepped
alone (1e-13 of each variable's maximum, 1e-12 for the histories, as for
batches elsewhere)."""
import numpy as np
import pytest

import astr_amd as A
from test_gpu_batch import check_equal

pytestmark = pytest.mark.gpu


def cases(n, dims):
    out = []
    for k in range(n):
        f = A.Flow(A.vortex_config(*dims))
        f.init_vortex(4.0 + 0.1 * k)
        out.append(f)
    return out


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("n,dims,chosen", [(15, (66, 67), 0), (16, (64, 63), 0), (7, (150, 149), 3), (4, (270, 260), 1)])
def test_untuned_batch_equals_single_cases(n, dims, chosen, graph):
    flows, alone = cases(n, dims), cases(n, dims)
    for f in flows[:chosen]:
        for prog in (2, 3, 5, 6):
            for d in range(2):
                f.set_pass_config(prog, d, 3, 1)
    before = [f.pass_configs() for f in flows]
    b = A.Batch(flows)
    ke, en = b.rk3(3, graph=graph)
    single = [f.rk3(3) for f in alone]
    check_equal(flows, alone)
    for k, (ke0, en0) in enumerate(single):
        assert np.abs(ke[k] / ke0 - 1.0).max() < 1e-12 and np.abs(en[k] / en0 - 1.0).max() < 1e-12
    assert [f.pass_configs() for f in flows] == before  # a case's own selection stays
    assert b.info()["groups"] == (4 if chosen == 0 else 8)
    b.close()


def test_batch_of_a_mixed_size_keeps_each_case(n=9):
    mk = lambda: [A.Flow(A.tgv_config(24 + 3 * k, deltat=2e-3)) for k in range(n)] + cases(6, (80, 70))  # noqa: E731
    flows, alone = mk(), mk()
    for f, g in zip(flows, alone):
        if f.cfg.km:
            f.init_tgv(1e-3, 5)
            g.init_tgv(1e-3, 5)
    b = A.Batch(flows)
    b.rk3(2, stats=False)
    for g in alone:
        g.rk3(2, stats=False)
    check_equal(flows, alone)
    b.close()


@pytest.mark.parametrize("sides,groups", [((64, 100, 73, 150), 4), ((64, 100, 73, 154), 4), ((40, 73, 66, 50), 4)])
def test_cases_of_several_lengths_share_each_launch(sides, groups):
    """Nobody chose a shape: cases of different lengths stay one group per slot."""
    flows, alone = [[A.Flow(A.vortex_config(n)) for n in sides for _ in range(4)] for _ in range(2)]
    for f in flows + alone:
        f.init_vortex()
    b = A.Batch(flows)
    assert b.info()["groups"] == groups
    b.rk3(2, stats=False)
    for f in alone:
        f.rk3(2, stats=False)
    check_equal(flows, alone)
    b.close()
