"""The point sampler where its tiles end: points and fields either side of a
tile, orders of every remainder of four degrees, one part and several, against
the FP64 oracle; and a point's bits must not depend on the tile it fell in.

Tolerance: FP64 sums of at most T^2/2 products of a three-term recurrence,
1e-12 of the largest value; the float32 sampler sums one order's T+1 fp32
terms, (T+1) 6e-8 at most, 2e-6 with T <= 33.
"""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import hip_transform
from oracle import sampling as osamp
from oracle.sht import OracleTransform, red_spectrum

pytestmark = pytest.mark.gpu

TOL = {"float64": 1e-12, "float32": 2e-6}


def _points(n):
    rng = np.random.default_rng(n)
    return rng.uniform(-89.0, 89.0, n), rng.uniform(0.0, 360.0, n)


def _fields(T, count, seed):
    return red_spectrum(T, (count,), seed=seed).astype(np.complex64)


@pytest.mark.parametrize("T,count,points", [(1, 1, 1), (2, 3, 15), (3, 8, 16), (6, 9, 17),
                                            (21, 5, 33), (31, 16, 65), (32, 17, 130), (33, 41, 97)])
@pytest.mark.parametrize("precision", list(TOL))
def test_tiles_match_the_oracle(T, count, points, precision):
    from arwen_spectral import sampling

    o = OracleTransform.create(T)
    t = hip_transform(o, "float32")
    lat, lon = _points(points)
    c, d = _fields(T, count, 1), _fields(T, count, 2)
    c128, d128 = c.astype(np.complex128), d.astype(np.complex128)

    def close(got, want):
        assert np.max(np.abs(got - want)) < TOL[precision] * np.max(np.abs(want))

    close(sampling.sample_scalar(t, c, lat, lon, precision=precision),
          osamp.sample_scalar(o, c128, lat, lon))
    for got, want in zip(sampling.sample_gradient(t, c, lat, lon, precision=precision),
                         osamp.sample_gradient(o, c128, lat, lon)):
        close(got, want)
    # psi and chi are formed in fp32 from vorticity and divergence (one
    # rounding of each coefficient) before the FP64 sums
    for got, want in zip(sampling.sample_wind(t, c, d, lat, lon, precision=precision),
                         osamp.sample_wind(o, c128, d128, lat, lon)):
        assert np.max(np.abs(got - want)) < 2e-6 * np.max(np.abs(want))


@pytest.mark.parametrize("kind", ["scalar", "gradient", "wind"])
@pytest.mark.parametrize("precision", list(TOL))
def test_a_points_bits_do_not_depend_on_its_tile(kind, precision):
    from arwen_spectral import sampling

    o = OracleTransform.create(63, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    lat, lon = _points(9000)
    c = _fields(63, 40, 3)
    fn = {"scalar": sampling.sample_scalar, "gradient": sampling.sample_gradient,
          "wind": sampling.sample_wind}[kind]

    def call(fields, s):
        args = (fields, fields[::-1].copy()) if kind == "wind" else (fields,)
        out = fn(t, *args, lat[s], lon[s], precision=precision)
        return out if isinstance(out, tuple) else (out,)

    whole = call(c, slice(None))
    for s in (slice(0, 1), slice(5, 40), slice(100, 1700)):
        for w, got in zip(whole, call(c, s)):
            assert np.array_equal(w[:, s], got)
    if kind != "wind":  # fewer fields: other column tiles
        for w, got in zip(whole, call(c[3:20].copy(), slice(None))):
            assert np.array_equal(w[3:20], got)


@pytest.mark.parametrize("T,points", [(127, 2033), (127, 3000), (127, 4064), (63, 4081), (63, 8160),
                                      (21, 16369), (21, 32736)])
@pytest.mark.parametrize("precision", list(TOL))
def test_two_to_five_column_tiles_of_one_point_tile(T, points, precision):
    """The ranges of points where a wavefront holds one point tile and several
    column tiles, with several parts and with one (T21): the oracle's values
    at some points, every output the bits of an 8-field call's, and nothing
    written beside the outputs and the workspace.

    Tolerance: float64 as above (T^2 / 2 roundings of 1.1e-16 are 9e-13 at
    T127); float32 (T + 1) 6e-8."""
    import ctypes

    import torch

    from arwen_spectral import _native

    o = OracleTransform.create(T, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    lib, dev = _native.load(), t.backend.device()
    lat, lon = _points(points)
    la, lo = np.deg2rad(lat), np.deg2rad(lon)
    pts = [torch.from_numpy(x).to(dev) for x in (np.sin(la), np.cos(la), lo)]
    fields = torch.from_numpy(_fields(T, 33, 5)).to(dev)
    pad, code = 4096, 0 if precision == "float64" else 1
    vp = lambda x: ctypes.c_void_p(x.data_ptr())  # noqa: E731

    def call(c):
        n = c.shape[0]
        nbytes = int(lib.arwen_sht_sample_workspace_bytes(t.plan_handle, n, 0, points))
        out = torch.full((n * points + 2 * pad,), 7.5, dtype=torch.float64, device=dev)
        work = torch.full((nbytes + 16 * pad,), 0x5A, dtype=torch.uint8, device=dev)
        _native.check(lib.arwen_sht_sample(
            t.plan_handle, vp(c), None, n, *map(vp, pts), points, 0, code, vp(work[8 * pad:]),
            nbytes, vp(out[pad:]), None, t.backend.stream()))
        assert (out[:pad] == 7.5).all() and (out[-pad:] == 7.5).all()
        assert (work[:8 * pad] == 0x5A).all() and (work[-8 * pad:] == 0x5A).all()
        return out[pad:-pad].reshape(n, points)

    tiles = torch.cat([call(fields[k:k + 8]) for k in range(0, 33, 8)])
    some = np.linspace(0, points - 1, 64).astype(int)
    want = osamp.sample_scalar(o, fields.cpu().numpy().astype(np.complex128), lat[some], lon[some])
    tol = TOL[precision] if precision == "float64" else (T + 1) * 6e-8
    assert np.max(np.abs(tiles[:, some].cpu().numpy() - want)) < tol * np.max(np.abs(want))
    for count in (17, 24, 25, 32, 33):
        assert torch.equal(call(fields[:count]), tiles[:count]), count


@pytest.mark.parametrize("T,points,count", [(127, 16400, 3), (127, 16321, 8), (127, 4100, 20),
                                            (31, 33000, 17), (21, 131080, 1)])
@pytest.mark.parametrize("kind", ["gradient", "wind"])
@pytest.mark.parametrize("precision", list(TOL))
def test_derivatives_at_many_points(T, points, count, kind, precision):
    """Four point tiles of one column tile (orders of every remainder, points of
    the last block missing), and a last column tile alone: the oracle's values
    at some points, the last ones among them, and the bits of a few points
    alone.  Tolerances as above; winds carry the fp32 rounding of psi and chi."""
    from arwen_spectral import sampling

    o = OracleTransform.create(T, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    lat, lon = _points(points)
    n = (count + 1) // 2 if kind == "wind" else count
    fields = [_fields(T, n, 5), _fields(T, n, 6)][:2 if kind == "wind" else 1]
    fn = {"gradient": (sampling.sample_gradient, osamp.sample_gradient),
          "wind": (sampling.sample_wind, osamp.sample_wind)}[kind]
    some = np.r_[0:16, points - 40:points]
    got = fn[0](t, *fields, lat, lon, precision=precision)
    want = fn[1](o, *(f.astype(np.complex128) for f in fields), lat[some], lon[some])
    few = fn[0](t, *fields, lat[some], lon[some], precision=precision)
    tol = max(TOL[precision], (T + 1) * 6e-8 if precision == "float32" else 0.0,
              2e-6 if kind == "wind" else 0.0)
    for g, w, f in zip(got, want, few):
        assert np.max(np.abs(g[:, some] - w)) < tol * np.max(np.abs(w))
        assert np.array_equal(g[:, some], f)
