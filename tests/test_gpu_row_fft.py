"""The longitude FFTs of rows that are not 64 L points long, on the device
against the FP64 oracle: every radix of the passes alone and combined, primes
in the first and in a later pass, the shortest row, and rows so long that
fewer of them share a block.

Tolerance: an output of a radix-R pass is a sum of R rounded products, whose
fp32 rounding grows as sqrt(R) half-ulps; 6e-8 (10 + 2 sqrt(R)) of the
field's maximum, R the largest prime factor, leaves the few passes of the
rest and the fp32 Legendre sums their own 6e-7.
"""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import hip_transform, rel_err
from oracle.sht import OracleTransform, red_spectrum

pytestmark = pytest.mark.gpu

# nlon: 2 and 4 points per order; radices 2..16; primes 17 (first pass), 19
# with 17 (a later prime pass), 23, 89, 257; 1334 = 2 23 29 and 1602 run four
# and 3072 two rows per block
LENGTHS = [4, 6, 10, 14, 18, 22, 26, 30, 34, 36, 40, 44, 66, 84, 100, 144, 150, 162, 182, 190,
           220, 224, 240, 322, 338, 514, 576, 646, 1024, 1152, 1334, 1602, 3072]


def _tol(n):
    largest = max(p for p in range(2, n + 1) if n % p == 0 and all(p % q for q in range(2, p)))
    return 6e-8 * (10 + 2 * np.sqrt(largest))


def _case(nlon):
    T = min(nlon // 2 - 1, 40)
    nlat = T + 1 + (nlon // 2) % 2  # odd and even latitude counts
    return OracleTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0)


@pytest.mark.parametrize("nlon", LENGTHS)
def test_scalar_and_waist_rows(nlon):
    import torch

    o = _case(nlon)
    t = hip_transform(o, "float32")
    c = red_spectrum(o.truncation, (3,), seed=nlon)
    g = o.inverse(c)
    tol = _tol(nlon)
    assert rel_err(t.inverse(c), g) < tol
    g32 = g.astype(np.float32)
    want = o.forward(g32.astype(np.float64))
    assert rel_err(t.forward(g32), want) < tol
    w = t.fourier_waist(g32)
    assert rel_err(w.values, o.fourier_waist(g32.astype(np.float64))) < tol
    banded = t.open_waist((3,), bands=2)
    for r0, r1 in reversed(banded.edges):
        banded.fill_band(r0, r1, g32[..., r0:r1, :])
    assert torch.equal(banded.close().values, w.values)  # a row depends on itself alone
    assert rel_err(t.waist_to_grid(t.contract_to_waist(c)), g) < 2 * tol


@pytest.mark.parametrize("nlon", [66, 182, 322, 1152, 1334])
def test_vector_components_fold_one_at_a_time(nlon):
    from arwen_spectral import VorticityDivergenceOperator

    o = _case(nlon)
    t = hip_transform(o, "float32")
    v = VorticityDivergenceOperator(t)
    z, d = (red_spectrum(o.truncation, (2,), seed=s) for s in (nlon, nlon + 1))
    gu, gv = o.wind_from_vordiv(z, d)
    u32, v32 = gu.astype(np.float32), gv.astype(np.float32)
    # vorticity and divergence weight a wind's rounding by about T (their
    # degrees' derivative) relative to their own maximum
    tol = _tol(nlon) * max(1.0, o.truncation / 4)
    for got, want in zip(v.vordiv_from_wind(u32, v32),
                         o.vordiv_from_wind(u32.astype(np.float64), v32.astype(np.float64))):
        assert rel_err(got, want) < tol


@pytest.mark.parametrize("nlon,fields", [(144, 40), (576, 40), (144, 3), (640, 90), (1602, 90),
                                         (704, 150), (1152, 90), (3072, 3), (5120, 2)])
def test_eight_four_two_and_one_rows_per_block(nlon, fields):
    """32 row pairs of as many fields as take 8, 8, 8, 4, 4, 2, 2, 2 and 1 rows per
    block.  Tolerances as above."""
    from arwen_spectral import VorticityDivergenceOperator

    o = OracleTransform.create(18, nlat=63, nlon=nlon, dealias_factor=1.0)
    t = hip_transform(o, "float32")
    tol = _tol(nlon)
    c, z, d = (red_spectrum(18, (fields,), seed=s) for s in (nlon, nlon + 1, nlon + 2))
    g = o.inverse(c)
    g32 = g.astype(np.float32)
    assert rel_err(t.inverse(c), g) < tol
    assert rel_err(t.forward(g32), o.forward(g32.astype(np.float64))) < tol
    v = VorticityDivergenceOperator(t)
    want = o.wind_from_vordiv(z, d)
    for got, w in zip(v.wind_from_vordiv(z, d), want):
        assert rel_err(got, w) < tol
    u32, v32 = (w.astype(np.float32) for w in want)
    for got, w in zip(v.vordiv_from_wind(u32, v32),
                      o.vordiv_from_wind(u32.astype(np.float64), v32.astype(np.float64))):
        assert rel_err(got, w) < tol * 18 / 4
