"""Single operations on a few fields (contracted straight from and to the
boundary layout) against the same operation as a batch job (the grouped GEMM):
equal bits, either side of the field counts where the path changes, at the
edges of its tiles: orders that do not fill an m-tile, one and several
k-chunks, an odd latitude count, 8 and 9 fields (column groups).  The grouped
path itself is held to the FP64 oracle elsewhere.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _red(torch, T, count, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.view_as_complex(torch.randn(count, T + 1, T + 1, 2, device="cuda", generator=g))
    return x.contiguous()  # above the triangle and Im(m = 0) as they come


@pytest.mark.parametrize("precision", ["float32", "bf16x6", "bf16x3"])
@pytest.mark.parametrize("T,nlat,nlon,counts", [
    (1, 2, 4, (1,)), (4, 7, 16, (1, 9)), (21, 33, 66, (8, 72, 73)), (63, 64, 128, (1, 9, 36, 37)),
    (64, 65, 192, (2, 9, 13)), (127, 128, 256, (1, 12, 18, 19)), (130, 140, 320, (3, 4, 8, 9)),
    (255, 256, 512, (1, 2, 4, 5)), (383, 384, 768, (1, 2, 3))])
def test_few_fields_have_the_grouped_bits(T, nlat, nlon, counts, precision):
    import torch

    from arwen_spectral import SphericalHarmonicTransform, TransformBatch

    t = SphericalHarmonicTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0,
                                          precision=precision)
    for n in counts:
        c = _red(torch, T, n, T + n)
        f = torch.randn(n, nlat, nlon, device="cuda")
        goff = torch.linspace(-1.0, 2.0, n, device="cuda")
        coff = torch.complex(goff, torch.zeros_like(goff)) + 0.5
        grids = [torch.empty(n, nlat, nlon, device="cuda") for _ in range(9)]
        specs = [torch.empty_like(c) for _ in range(2)]
        TransformBatch([
            ("inverse", t, c, grids[0]), ("inverse", t, c, grids[1], {"coeff_offset": coff}),
            ("zonal", t, c, grids[2]), ("meridional", t, c, grids[3]),
            ("gradient", t, c, (grids[4], grids[5])),
            ("inverse_gradient", t, c, tuple(grids[6:9])),
            ("forward", t, f, specs[0]),
            ("forward", t, f, specs[1], {"grid_offset": goff, "coeff_offset": coff})]).run()
        got = [t.inverse(c), t.inverse_about(c, coff), t.inverse_zonal_derivative(c),
               t.inverse_meridional_derivative(c), *t.gradient(c), *t.inverse_with_gradient(c),
               t.forward(f), t.forward_about(f, goff, coff)]
        for k, (a, b) in enumerate(zip(got, grids + specs)):
            assert torch.equal(a, b), f"T{T} {n} fields, result {k}"
        # the waist's head and tail take the same contraction
        w = t.contract_to_waist(c)
        assert np.isfinite(w.values.abs().sum().item())
        assert (t.waist_to_grid(w) - got[0]).abs().max() <= 2e-6 * got[0].abs().max()


@pytest.mark.parametrize("precision", ["float32", "bf16x6", "bf16x3"])
@pytest.mark.parametrize("T,nlat,nlon,counts", [
    (30, 31, 64, (1, 16)), (127, 128, 256, (16, 17)), (160, 170, 486, (6, 9)),
    (191, 192, 384, (1, 3, 4, 9, 10)), (255, 257, 514, (3,))])
def test_few_field_analysis_row_tiles(T, nlat, nlon, counts, precision):
    """Two and four row tiles per wavefront, the last block partly past the
    degrees (tiles not a multiple of four), both sides of the field counts."""
    import torch

    from arwen_spectral import SphericalHarmonicTransform, TransformBatch

    t = SphericalHarmonicTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0,
                                          precision=precision)
    for n in counts:
        f = torch.randn(n, nlat, nlon, device="cuda")
        out = torch.full((n, T + 1, T + 1), 7.0, device="cuda", dtype=torch.complex64)
        TransformBatch([("forward", t, f, out)]).run()
        assert torch.equal(t.forward(f), out), f"T{T} {n} fields"


@pytest.mark.parametrize("precision", ["float32", "bf16x6", "bf16x3"])
@pytest.mark.parametrize("T,nlat,nlon,counts", [(21, 33, 66, (1, 9, 72)), (64, 65, 192, (2, 13)),
                                                (127, 128, 256, (1, 12, 18, 19))])
def test_inverse_laplacian_has_the_grouped_bits(T, nlat, nlon, counts, precision):
    """The C entry point's inverse Laplacian flag on a single synthesis (few
    fields) against the batch job's."""
    import ctypes

    import torch

    from arwen_spectral import SphericalHarmonicTransform, TransformBatch, _native

    t = SphericalHarmonicTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0,
                                          precision=precision)
    lib, vp = _native.load(), lambda x: ctypes.c_void_p(x.data_ptr())
    for n in counts:
        c = _red(torch, T, n, T + n)
        want, got = (torch.empty(n, nlat, nlon, device="cuda") for _ in range(2))
        TransformBatch([("inverse", t, c, want, {"inverse_laplacian": True})]).run()
        _native.check(lib.arwen_sht_synthesis_about(t.plan_handle, vp(c), vp(got), n, None,
                                                    _native.JOB_INVLAP, t.backend.stream()))
        assert torch.equal(got, want), f"T{T} {n} fields"


def test_a_later_single_operation_is_checked_like_the_first():
    """The batch kept for an operation takes every call's buffers and flags:
    what the first call refuses, the next one refuses too."""
    import ctypes

    import torch

    from arwen_spectral import SphericalHarmonicTransform, _native

    t = SphericalHarmonicTransform.create(21, dealias_factor=1.0)
    lib = _native.load()
    c = _red(torch, 21, 2, 1)
    out = torch.empty(2, *t.grid.shape, device="cuda")
    off = torch.ones(2, dtype=torch.complex64, device="cuda")
    vp, s = lambda x: ctypes.c_void_p(x.data_ptr()), t.backend.stream()
    call = lib.arwen_sht_synthesis_about
    for _ in range(2):
        assert call(t.plan_handle, vp(c), vp(out), 2, None, 0, s) == _native.OK
        assert call(t.plan_handle, None, vp(out), 2, None, 0, s) == _native.EINVAL
        assert call(t.plan_handle, vp(c), None, 2, None, 0, s) == _native.EINVAL
        assert call(t.plan_handle, vp(c), vp(out), 2, None, 4, s) == _native.EINVAL
        assert call(t.plan_handle, vp(c), vp(out), 2, vp(off), _native.JOB_INVLAP,
                    s) == _native.EINVAL
        assert call(t.plan_handle, vp(c), vp(out), 2, vp(off), _native.JOB_EXP, s) == _native.OK
    torch.cuda.synchronize()
