"""The cell kernels' instances (9 species or any count up to 16; mass-action
products of unit terms or general orders) against the numpy restatement, on
mechanisms derived from the 9-species one: without N2, with orders that are
not whole numbers, with irreversible reactions.

Tolerance: a rate constant's exponent sums terms of up to about 100, each
rounded to 1e-16 of itself, so a rate is good to about 1e-13 of itself; the
species' net rates are compared to 1e-12 of the species' largest rate, cp and
h (sums of five or six terms) to 1e-13."""
import os

import numpy as np
import pytest

from astr_amd import chem as AC
from oracle import chem as OC

MECH = os.path.join(os.path.dirname(__file__), "golden", "Jachimowski88_H2-9-19.xml")


def variant(tmp_path, drop_n2, orders, irreversible):
    x = open(MECH).read()
    if drop_n2:
        a = x.index("<speciesArray")
        b = x.index("</speciesArray>", a)
        x = x[:a] + x[a:b].replace(" N2", "") + x[b:]
    if orders:
        assert "<reactants>O:2.0</reactants>" in x and "<reactants>H2:1 OH:1.0</reactants>" in x
        x = x.replace("<reactants>O:2.0</reactants>", "<reactants>O:1.5</reactants>")
        x = x.replace("<reactants>H2:1 OH:1.0</reactants>", "<reactants>H2:0.5 OH:1.0</reactants>")
    if irreversible:
        assert x.count('reversible="yes"') > 2
        x = x.replace('reversible="yes"', 'reversible="no"', 2)
    p = tmp_path / "mech.xml"
    p.write_text(x)
    return str(p)


FORMS = [(False, False, False), (True, False, False), (False, True, True), (True, True, False), (True, False, True)]


@pytest.mark.parametrize("form", FORMS)
def test_variants_differ_from_the_base(tmp_path, form):
    m, base = OC.Mechanism(variant(tmp_path, *form)), OC.Mechanism(MECH)
    assert len(m.names) == 9 - form[0] and m.nr == 19
    assert any(v not in (1.0, 2.0) for r in m.rx for _, v in r["reac"]) == form[1]
    assert sum(not r["rev"] for r in m.rx) == sum(not r["rev"] for r in base.rx) + 2 * form[2]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 5000])
@pytest.mark.parametrize("form", FORMS)
def test_gpu_rates_of_every_instance(tmp_path, form, n):
    path = variant(tmp_path, *form)
    gm, om = AC.Mechanism(path), OC.Mechanism(path)
    T, p, Y = AC.sample_cells(om.names, om.W, n, 29) if not form[0] else _cells_without_n2(om, n)
    wd, h, cp, hk = gm.rates(T, p, Y, species_h=True)
    wd0, h0, cp0, hk0 = om.rates(T, p, Y)
    big = np.abs(om.rates(T, p, Y, parts=True)[4]).max()  # the largest gross rate, kmol/m^3/s
    for k in range(om.ns):
        den = max(np.abs(wd0[k]).max(), 0.1 * big * om.W[k]) if n < 5000 else np.abs(wd0[k]).max()
        assert np.abs(wd[k] - wd0[k]).max() <= 1e-12 * den, om.names[k]
    assert np.abs(h - h0).max() <= 1e-13 * np.abs(hk0).max()
    assert np.abs(hk - hk0).max() <= 1e-13 * np.abs(hk0).max()
    assert np.abs(cp / cp0 - 1).max() < 1e-13


def _cells_without_n2(om, n):
    rng = np.random.default_rng(31)
    Y = rng.uniform(0.0, 1.0, (om.ns, n)) ** 3
    return rng.uniform(400.0, 2800.0, n), rng.uniform(0.5, 5.0, n) * 101325.0, Y / Y.sum(axis=0)


@pytest.mark.gpu
@pytest.mark.parametrize("orders", [False, True])
def test_gpu_a_cell_without_a_finite_rate_leaves_the_others_alone(tmp_path, orders):
    """NaN in one cell's H2O2 spoils that cell's reactions with H2O2 and the
    three-body ones, not N2's rate (zero: it takes part in none) and no bit of
    the wavefront's other cells; a cell so cold that its exponents leave the
    range of the plain exponential does not change its neighbours either."""
    gm = AC.Mechanism(variant(tmp_path, False, orders, False))
    ix = {s: k for k, s in enumerate(gm.names)}
    T, p, Y = AC.sample_cells(gm.names, gm.W, 130, 37)
    wd, h, cp = gm.rates(T, p, Y)
    T2, Y2 = T.copy(), Y.copy()
    Y2[ix["H2O2"], 70] = np.nan
    T2[5] = 40.0
    wd2, h2, cp2 = gm.rates(T2, p, Y2)
    keep = np.ones(130, bool)
    keep[[5, 70]] = False
    assert np.array_equal(wd2[:, keep], wd[:, keep])
    assert np.array_equal(h2[keep], h[keep]) and np.array_equal(cp2[keep], cp[keep])
    assert wd2[ix["N2"], 70] == 0.0 and np.isnan(wd2[ix["H2O2"], 70])


def _repeated(tmp_path, times, base):
    """The mechanism with its reactions repeated (with a pre-exponential
    factor divided by the count, the same chemistry): 19 * times records."""
    x = open(base).read()
    a, b = x.index("<reaction "), x.rindex("</reaction>") + len("</reaction>")
    import re
    body = re.sub(r"(<A[^>]*>)([^<]+)(</A>)", lambda m: m[1] + repr(float(m[2]) / times) + m[3], x[a:b])
    p = tmp_path / "many.xml"
    p.write_text(x[:a] + "\n".join([body] * times) + x[b:])
    return str(p)


@pytest.mark.gpu
@pytest.mark.parametrize("times,form", [(2, (False, False, False)), (1, (False, True, True)), (2, (False, True, False)),
                                        (1, (False, False, True))])
def test_gpu_reactor_team_on_derived_mechanisms(tmp_path, times, form):
    """A team's third reaction per lane (38 reactions), general orders and
    irreversible reactions: ignitions by the team and by the one-thread kernel
    agree to the integrator's tolerance, in about the same number of steps (a
    wrong Jacobian costs steps).  Nine reactors: a last wavefront with one."""
    gm = AC.Mechanism(_repeated(tmp_path, times, variant(tmp_path, *form)))
    assert gm.nr == 19 * times
    ix = {s: k for k, s in enumerate(gm.names)}
    rng = np.random.default_rng(41)
    reqs = []
    for _ in range(9):
        X = np.zeros(gm.ns)
        X[ix["H2"]], X[ix["O2"]], X[ix["N2"]] = 2.0 * rng.uniform(0.5, 2.0), 1.0, 3.76
        reqs.append((rng.uniform(1050.0, 1400.0), rng.uniform(1.0, 10.0) * 101325.0, X * gm.W / (X * gm.W).sum()))
    out = {}
    for lanes in (1, 16):
        pool = AC.ReactorPool(gm, 10, rtol=1e-6, atol=1e-12, lanes=lanes)
        for k, (T0, p, Y) in enumerate(reqs):
            pool.set(k, T0, p, Y, 2e-4)
        st = pool.run(max_tries=500)
        assert np.all(st[:9] == AC.ReactorPool.DONE) and st[9] == AC.ReactorPool.FREE
        out[lanes] = [pool.get(k) for k in range(9)]
        pool.close()
    for a, b in zip(out[1], out[16]):
        assert a[0] == b[0] and a[3] > 5
        assert abs(b[1] / a[1] - 1.0) < 1e-5
        assert np.abs(b[2] - a[2]).max() < 1e-6
        assert abs(a[3] - b[3]) <= max(2, a[3] // 20)
