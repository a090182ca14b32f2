"""The 16-lane reactor team's right-hand side, Jacobian, factorisation and solve
on their own, against the numpy restatement along an ignition: the base
mechanism, orders that are not whole numbers, irreversible reactions, and 38
reactions (a third reaction per lane).  Nine states: a last wavefront with one
team.

Tolerances, those of the one-thread kernel's comparison: f to 1e-12 and every
Jacobian column to 1e-10 of their norms (rate constants good to 1e-13, sums
that cancel by up to a few hundred).  The solution of (I - gh J) x = f against
numpy's of the device's own J and f: the matrix, with T scaled by 1e4, has a
condition number of up to about 1e4 at the gh used, so 1e-10 of the largest
mass fraction's component and of the temperature's."""
import numpy as np
import pytest

from astr_amd import chem as AC
from oracle import chem as OC
from test_chem import _trajectory
from test_gpu_chem_forms import MECH, _repeated, variant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("times,form", [(1, (False, False, False)), (1, (False, True, False)), (1, (False, False, True)),
                                        (2, (False, False, False)), (2, (False, True, True))])
def test_team_against_the_restatement(tmp_path, times, form):
    p, Ys = _trajectory(OC.Mechanism(MECH), times=(1e-6, 5e-6, 1e-5, 2e-5, 3e-5, 4e-5, 5e-5, 7e-5, 1e-4))
    Ys = np.abs(Ys)
    path = _repeated(tmp_path, times, variant(tmp_path, *form))
    gm, om = AC.Mechanism(path), OC.Mechanism(path)
    assert gm.nr == 19 * times
    gh = 1e-7
    f, J, x = gm.reactor_team_eval(np.full(len(Ys), p), Ys, gh)
    for i, y in enumerate(Ys):
        f0, J0 = om.reactor_rhs(y, p), om.reactor_jacobian(y, p)
        assert np.abs(f[i] - f0).max() <= 1e-12 * np.abs(f0).max(), i
        for j in range(y.size):
            assert np.abs(J[i][:, j] - J0[:, j]).max() <= 1e-10 * np.abs(J0[:, j]).max(), (i, j)
        x0 = np.linalg.solve(np.eye(y.size) - gh * J[i], f[i])
        assert abs(x[i, 0] - x0[0]) <= 1e-10 * abs(x0[0]), i
        assert np.abs(x[i, 1:] - x0[1:]).max() <= 1e-10 * np.abs(x0[1:]).max(), i
