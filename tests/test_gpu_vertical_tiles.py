"""The column operators where their tiles end: levels either side of each
16-row tile, truncations whose orders do not fill a wavefront's 16 or a
block's 128, against the FP64 oracle.

Tolerance: three chained fp32 products of up to 65 terms, each at most
sqrt(65) half-ulps (6e-8) of its result: 3 sqrt(65) 6e-8 = 1.5e-6, rounded up
to 2e-6 of the largest value.
"""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import hip_transform
from oracle import semi_implicit as osi
from oracle.sht import OracleTransform, red_spectrum

pytestmark = pytest.mark.gpu

TOL = 2e-6


def _close(got, want):
    for g, w in zip(got, want):
        g = g.detach().cpu().numpy()
        assert np.max(np.abs(g - w)) < TOL * np.max(np.abs(w))
        t1 = g.shape[-1]
        assert not (g * np.triu(np.ones((t1, t1)), 1)).any()
        assert not g[..., 0].imag.any()


@pytest.mark.parametrize("trunc,nlev", [(3, 1), (14, 15), (15, 16), (16, 17), (21, 31), (30, 32),
                                        (33, 47), (31, 48), (20, 63), (130, 9), (127, 5)])
def test_levels_and_orders_at_the_edges_of_tiles(trunc, nlev):
    from arwen_spectral import semi_implicit as si

    o = OracleTransform.create(trunc, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    f32 = lambda a: np.asarray(a, dtype=np.float32)  # noqa: E731
    c64 = lambda a: np.asarray(a).astype(np.complex64)  # noqa: E731
    b, c, m, modal = osi.synthetic_operator(nlev, seed=nlev)
    k2 = f32(si.wave_operator(t))
    # the half maps' modes come from the FP64 operator (rounded first, its null
    # mode turns into a growing one)
    maps = [f32(x) for x in osi.symmetric_half_maps(modal, osi.x_modes(b, c), k2, 1500.0, 0.6)]
    b, c, m = f32(b), f32(c), f32(m)
    d = c64(o.project(red_spectrum(trunc, (nlev,), seed=1, scale=1e-5)))
    th = c64(o.project(red_spectrum(trunc, (nlev,), seed=2, scale=10.0)))
    ps = c64(o.project(red_spectrum(trunc, (), seed=3, scale=1e-2)))
    d[:, 0, 0], th[:, 0, 0], ps[0, 0] = 1e-6, 250.0, 0.3
    inv = f32(osi.helmholtz_inverse(modal, k2, 900.0, 1.0))
    _close(si.vertical_solve_shifted(t, d, th, ps, b, c, inv, k2, 900.0),
           osi.solve_shifted(o, d, th, ps, b, c, inv, k2, np.float32(900.0)))
    inv = f32(osi.helmholtz_inverse(modal, k2, 600.0, 0.6))
    _close(si.vertical_apply(t, d, th, ps, b, c, m, inv, k2, 600.0, 0.6),
           osi.apply(o, d, th, ps, b, c, m, inv, k2, np.float32(600.0), 0.6))
    _close(si.vertical_linear_tendencies(t, d, th, ps, b, c, k2, 0.7),
           osi.linear_tendencies(o, d, th, ps, b, c, k2, np.float32(0.7)))
    _close(si.vertical_half_apply(t, d, th, ps, b, c, *maps, k2),
           osi.half_apply(o, d, th, ps, b, c, maps, k2))


@pytest.mark.parametrize("trunc,nlev", [(33, 17), (38, 6), (60, 40), (30, 64)])
def test_half_map_error_is_that_of_two_sums(trunc, nlev):
    """x' = P_x x + Q_x (C D) with the two products summed apart and added
    once, in fp32 on the host: the device's rms error against FP64 is no more
    than that of the same sums.  Both are rms over thousands of rounded values
    of one distribution, so they agree to a few per cent; one accumulation
    through both products is at least sqrt(2) off.  Line: 1.2."""
    from arwen_spectral import semi_implicit as si

    o = OracleTransform.create(trunc, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    f32 = lambda a: np.asarray(a, dtype=np.float32)  # noqa: E731
    b, c, _, modal = osi.synthetic_operator(nlev, seed=nlev)
    k2 = f32(si.wave_operator(t))
    maps = [f32(x) for x in osi.symmetric_half_maps(modal, osi.x_modes(b, c), k2, 1500.0, 0.6)]
    b, c = f32(b), f32(c)
    d, th, ps = (o.project(red_spectrum(trunc, lead, seed=s, scale=a)).astype(np.complex64)
                 for lead, s, a in (((nlev,), 1, 1e-5), ((nlev,), 2, 10.0), ((), 3, 1e-2)))

    def dot(a, x):  # (n, i, j) by (j, n, m), a term at a time
        acc = np.zeros((a.shape[1], *x.shape[1:]), dtype=np.complex64)
        for j in range(a.shape[2]):
            term = a[:, :, j].T[:, :, None].astype(np.float64) * x[j].astype(np.complex128)
            acc = (acc + term).astype(np.complex64)  # one rounding of each part: an fma
        return acc

    every = np.broadcast_to(c, (trunc + 1, *c.shape))
    x = np.concatenate([th, ps[None]])
    host = dot(maps[2], x) + dot(maps[3], dot(every, d))
    want = osi.half_apply(o, d, th, ps, b, c, maps, k2)
    got = si.vertical_half_apply(t, d, th, ps, b, c, *maps, k2)
    rms = lambda e: float(np.sqrt(np.mean(np.abs(e) ** 2)))  # noqa: E731
    keep = np.tril(np.ones((trunc + 1, trunc + 1)))
    keep[0, 0] = 0  # passed through
    for g, h, w in zip(got[1:], (host[:-1], host[-1]), want[1:]):
        g = g.detach().cpu().numpy().astype(np.complex128)
        assert rms((g - w) * keep) < 1.2 * rms((h - w) * keep)


@pytest.mark.parametrize("nlev", [1, 4, 5, 15, 16, 18, 33])
def test_an_infinite_value_stays_infinite(nlev):
    """Matrices of one sign: +inf in one level of one column makes +inf of every
    output it reaches, not NaN, and touches no other column.  (The solve weighs
    the old divergence with 0 in x': 0 inf is NaN there.)"""
    from arwen_spectral import semi_implicit as si

    trunc, at = 6, (3, 1)
    o = OracleTransform.create(trunc, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    rng = np.random.default_rng(nlev)
    pos = lambda *shape: rng.uniform(0.5, 1.0, shape).astype(np.float32)  # noqa: E731
    k2, n1 = pos(trunc + 1), trunc + 1
    b, c, m, inv = pos(nlev, nlev + 1), pos(nlev + 1, nlev), -pos(nlev, nlev), pos(n1, nlev, nlev)
    maps = [pos(n1, nlev, nlev), pos(n1, nlev, nlev), pos(n1, nlev + 1, nlev + 1),
            pos(n1, nlev + 1, nlev + 1)]
    d, th, ps = (o.project(red_spectrum(trunc, lead, seed=s)).astype(np.complex64)
                 for lead, s in (((nlev,), 1), ((nlev,), 2), ((), 3)))
    calls = {
        "solve": lambda d, th: si.vertical_solve_shifted(t, d, th, ps, b, c, inv, k2, 2.0),
        "apply": lambda d, th: si.vertical_apply(t, d, th, ps, b, c, m, inv, k2, 2.0, 0.6),
        "tendencies": lambda d, th: si.vertical_linear_tendencies(t, d, th, ps, b, c, k2, 0.7),
        "half": lambda d, th: si.vertical_half_apply(t, d, th, ps, b, c, *maps, k2)}
    for name, call in calls.items():
        plain = [x.cpu().numpy() for x in call(d, th)]
        for which in (0, 1):
            args = [d.copy(), th.copy()]
            args[which].real[0, at[0], at[1]] = np.inf
            for k, (got, was) in enumerate(zip((x.cpu().numpy() for x in call(*args)), plain)):
                # tendencies: divergence from x alone, x from divergence alone
                reached = name != "tendencies" or (k == 0) == (which == 1)
                column = got.real[..., at[0], at[1]]
                if name == "solve" and which == 0 and k:
                    assert np.isnan(column).all()
                else:
                    assert np.isposinf(column).all() if reached else np.isfinite(column).all(), \
                        (name, which, k)
                got.real[..., at[0], at[1]] = was.real[..., at[0], at[1]]
                assert np.array_equal(got, was), (name, k)
