"""The viscous flux must not cost the right-hand side of the convective flux's
accuracy.  Each flux derivative is taken of the difference of the two; formed
from a rounded convective flux, the difference rounds a second time at that
flux's size (the viscous flux is 1e-3 of it), and the right-hand side's error
grows by a fifth to a quarter, as a double against an extended-precision
restatement of the line operators shows.  Formed by one fused operation it
rounds once, as the convective flux alone does.

Measure: the RMS distance from the same right-hand side in extended precision,
with the viscous flux (Re 1600) over that without (Re 1e30), at Mach 1, where
pressure, kinetic energy and momentum fluxes are all of order one.  The viscous
part's own error is 1e-3 of the convective one's.  The RMS over 16 000 points
or more of errors that are correlated over a few points is good to about 1%;
the bound, 1.05, leaves five of those."""
import numpy as np
import pytest

import astr_amd as A
from fields import periodic_field

LD = np.longdouble


def derivative(f, axis):
    """df_compact of lines with periodic halo (derivative.F90:63-306), not
    divided by the spacing: explicit 6th-order rows at -1 and n+1, compact ones
    between."""
    f = np.moveaxis(f, axis, 0)
    n = f.shape[0] - 1
    ext = np.concatenate([f[n - 5:n], f, f[1:6]])  # rows -5 .. n+5
    row = lambda s: ext[4 + s:n + 7 + s]  # rows -1 .. n+1, shifted by s  # noqa: E731
    b = LD(7) / 9 * (row(1) - row(-1)) + LD(1) / 36 * (row(2) - row(-2))
    for r in (0, n + 2):
        e = lambda s: ext[r + 4 + s]  # noqa: E731
        b[r] = LD(3) / 4 * (e(1) - e(-1)) - LD(3) / 20 * (e(2) - e(-2)) + LD(1) / 60 * (e(3) - e(-3))
    # x(r-1)/3 + x(r) + x(r+1)/3 = b(r) between the end rows, x = b at them
    a, c = LD(1) / 3, np.zeros(n + 3, LD)
    for r in range(1, n + 2):
        m = 1 - a * c[r - 1]
        c[r] = a / m
        b[r] = (b[r] - a * b[r - 1]) / m
    for r in range(n + 1, 0, -1):
        b[r] -= c[r] * b[r + 1]
    return np.moveaxis(b[1:n + 2], 0, axis)


def rhs_extended(cfg, q, viscous):
    """rhscal (tgvsolver.F90:450-787) of q in extended precision."""
    nd = 3 if cfg.km > 0 else 2
    inv = [LD(cfg.im) / LD(cfg.lx), LD(cfg.jm) / LD(cfg.ly), LD(max(cfg.km, 1)) / LD(cfg.lz)]
    q = q.astype(LD)
    g1 = LD(cfg.gamma) - 1
    u = [q[1 + m] / q[0] for m in range(3)]
    p = g1 * (q[4] - (q[1] * u[0] + q[2] * u[1] + q[3] * u[2]) / 2)
    T = p / q[0] * LD(cfg.gamma) * LD(cfg.mach) ** 2
    D = lambda f, d: derivative(f, 2 - d) * inv[d]  # noqa: E731
    zero = np.zeros_like(p)
    out = [zero.copy() for _ in range(5)]
    if viscous:
        g = [[D(u[m], d) if d < nd else zero for d in range(3)] for m in range(3)]
        gt = [D(T, d) if d < nd else zero for d in range(3)]
        s = LD(cfg.sutherland) / LD(cfg.ref_tem)
        mu = T * np.sqrt(T) * (1 + s) / (T + s) / LD(cfg.reynolds)
        k = mu / LD(cfg.prandtl) / (g1 * LD(cfg.mach) ** 2)
        div = (g[0][0] + g[1][1] + g[2][2]) / 3
        sg = [[mu * (g[a][b] + g[b][a]) - (2 * mu * div if a == b else 0) for b in range(3)] for a in range(3)]
    for d in range(nd):
        for m in range(5):
            f = -(q[4] + p) * u[d] if m == 4 else -q[m] * u[d] - (p if m == d + 1 else 0)
            if viscous and 0 < m < 4:
                f = f + sg[d][m - 1]
            if viscous and m == 4:
                f = f + k * gt[d] + sg[d][0] * u[0] + sg[d][1] * u[1] + sg[d][2] * u[2]
            out[m] += D(f, d)
    return np.array(out)


def test_extended_derivative_is_sixth_order():
    err = []
    for n in (32, 64):
        x = LD(2) * LD(np.pi) * np.arange(n + 1) / n
        f = np.sin(x)[None, :, None] * np.ones((2, 1, 3), LD)
        err.append(float(np.abs(derivative(f, 1) * (n / (2 * LD(np.pi))) - np.cos(x)[None, :, None]).max()))
    assert err[1] < 3e-9 and err[0] / err[1] > 40


def per_point_metrics(f):
    """The uniform grid's metrics but for one entry at one point, off the
    diagonal and large enough for the passes to read metrics at every point; it
    reaches the three lines through the point."""
    n, l = (f.cfg.im, f.cfg.jm, f.cfg.km), (f.cfg.lx, f.cfg.ly, f.cfg.lz)
    dxi = np.zeros((3, 3) + f.shape)
    for d in range(3 if f.cfg.km else 2):
        dxi[d, d] = n[d] / l[d]
    dxi[0, 1, 0, 0, 0] = 1e-6
    f.set_metrics(np.full(f.shape, jacobian(f.cfg)), dxi)


def off_origin(a):
    """Without the planes through the first point."""
    return a[:, 1:, 1:, 1:] if a.shape[1] > 1 else a[:, :, 1:, 1:]


def jacobian(cfg):
    return cfg.lx / cfg.im * (cfg.ly / cfg.jm) * (cfg.lz / cfg.km if cfg.km else 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["miniapp", "main", "per-point metrics"])
@pytest.mark.parametrize("dims", [(28, 27, 24), (41, 26, 33), (150, 131, 0)])
def test_viscous_flux_adds_no_rounding_at_the_convective_size(path, dims):
    make = A.tgv_config if path == "miniapp" else A.main_config
    err = {}
    for re in (1600.0, 1e30):
        f = A.Flow(make(*dims, mach=1.0, reynolds=re))
        if path == "per-point metrics":
            per_point_metrics(f)
        q = periodic_field(f.cfg, 8)
        f.upload(q)
        got = f.rhscal()
        want = rhs_extended(f.cfg, q, re < 1e20)
        if path != "miniapp":  # the main path's right-hand side carries the Jacobian
            got = got / jacobian(f.cfg)
        got, want = off_origin(got), off_origin(want)
        assert float(np.abs(got - want).max() / np.abs(want).max()) < 1e-12
        err[re] = np.sqrt(((got - want).astype(float) ** 2).mean(axis=(1, 2, 3)))
        f.close()
    ratio = err[1600.0] / np.maximum(err[1e30], 1e-300)
    for m in (1, 2, 3, 4):
        if m == 3 and dims[2] == 0:
            continue
        assert ratio[m] < 1.05, (m, ratio)


def rhs_double_apart(cfg, q):
    """The convective right-hand side's momenta in double as the reference forms
    them: primitives, products and sums rounded one after the other, each
    flux differentiated on its own (here in extended precision)."""
    nd = 3 if cfg.km > 0 else 2
    u = [q[1 + m] / q[0] for m in range(3)]
    p = (q[4] - 0.5 * q[0] * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])) / (1.0 / (cfg.gamma - 1.0))
    n, l = (cfg.im, cfg.jm, cfg.km), (cfg.lx, cfg.ly, cfg.lz)
    out = np.zeros((3,) + p.shape, LD)
    for d in range(nd):
        for m in range(3):
            f = q[1 + m] * u[d] + p if m == d else q[1 + m] * u[d]
            out[m] -= derivative(f.astype(LD), 2 - d) * (LD(n[d]) / LD(l[d]))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("main", [False, True])
@pytest.mark.parametrize("mach", [0.5, 1.0])
@pytest.mark.parametrize("dims", [(28, 27, 24), (150, 131, 0)])
def test_momentum_is_as_exact_as_the_parts_apart(main, mach, dims):
    """Where p is of the momentum flux's size, the momenta's error, that of
    the line solves included, stays below the error that the rounded primitives
    and fluxes of the reference's order alone leave."""
    f = A.Flow((A.main_config if main else A.tgv_config)(*dims, mach=mach))
    q = periodic_field(f.cfg, 8)
    f.upload(q)
    got = f.rhscal()[1:4] / (jacobian(f.cfg) if main else 1.0)
    want = rhs_extended(f.cfg, q, True)[1:4]
    plain = rhs_double_apart(f.cfg, q) - rhs_extended(f.cfg, q, False)[1:4]
    rms = lambda e: np.sqrt((e.astype(float) ** 2).mean(axis=(1, 2, 3)))  # noqa: E731
    for m in range(3 if dims[2] else 2):
        assert rms(got - want)[m] <= rms(plain)[m], (m, rms(got - want), rms(plain))


@pytest.mark.gpu
@pytest.mark.parametrize("main", [False, True])
@pytest.mark.parametrize("dims", [(28, 27, 24), (150, 131, 0)])
def test_pressures_far_from_the_reference_state(main, dims):
    """The convective right-hand side does not depend on the configuration's
    Mach number, nor may its error: a state whose pressures are a hundredth of
    the reference pressure 1/(gamma Ma^2) of Mach 0.1, against the same state
    under Mach 1, whose reference pressure it has."""
    make = A.main_config if main else A.tgv_config
    err = []
    for mach in (1.0, 0.1):
        f = A.Flow(make(*dims, mach=mach, reynolds=1e30))
        q = periodic_field(make(*dims, mach=1.0), 8)
        f.upload(q)
        got = f.rhscal()
        if main:
            got = got / jacobian(f.cfg)
        want = rhs_extended(f.cfg, q, False)
        err.append(np.sqrt(((got - want).astype(float) ** 2).mean(axis=(1, 2, 3))))
        f.close()
    for m in (1, 2, 3):
        if m == 3 and dims[2] == 0:
            continue
        assert err[1][m] < 1.05 * err[0][m], (m, err)


@pytest.mark.gpu
@pytest.mark.parametrize("main", [False, True])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_a_point_that_is_not_finite_reaches_its_planes_only(main, value):
    """A point whose energy is not finite spoils the gradients along the three
    lines through it and the fluxes along the lines that cross those: the three
    planes through it.  Every other point keeps its bits, also where the point
    is the first of a tile of lines."""
    f = A.Flow((A.main_config if main else A.tgv_config)(28, 27, 24))
    q = periodic_field(f.cfg, 8)
    f.upload(q)
    want = f.rhscal()
    q[4, 8, 0, 0] = value
    f.upload(q)
    got = f.rhscal()
    keep = np.ones(q[0].shape, bool)
    keep[8], keep[:, 0], keep[:, :, 0] = False, False, False
    assert np.array_equal(got[:, keep], want[:, keep])
    assert not np.isfinite(got[4, 8, 0, 0])
