"""The grouped GEMM's work queues: the same bits whatever the number of
workgroups an operation's items are dealt to (queues of one, two, three and
many items, workgroups without one), at the edges of the step lists: panels of
one trip, two segments, lists of more than 256 entries.
"""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _batch(torch, T, nlat, nlon, n, precision):
    from arwen_spectral import SphericalHarmonicTransform, TransformBatch

    t = SphericalHarmonicTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0,
                                          precision=precision)
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n)
    spec = lambda: torch.view_as_complex(  # noqa: E731
        torch.randn(n, T + 1, T + 1, 2, device="cuda", generator=g))
    grid = lambda: torch.randn(n, nlat, nlon, device="cuda", generator=g)  # noqa: E731
    outs = [torch.empty_like(grid()) for _ in range(5)] + [torch.empty_like(spec()) for _ in range(3)]
    b = TransformBatch([
        ("wind", t, (spec(), spec()), (outs[0], outs[1])), ("inverse", t, spec(), outs[2]),
        ("gradient", t, spec(), (outs[3], outs[4])),
        ("vordiv", t, (grid(), grid()), (outs[5], outs[6])), ("forward", t, grid(), outs[7])])
    return b, outs


@pytest.mark.parametrize("precision", ["float32", "bf16x6", "bf16x3"])
@pytest.mark.parametrize("T,nlat,nlon,n", [
    (2, 3, 8, 1), (21, 33, 66, 7), (63, 66, 128, 50), (130, 131, 320, 9), (30, 1030, 64, 3)])
def test_results_do_not_depend_on_the_queues(T, nlat, nlon, n, precision):
    import torch

    b, outs = _batch(torch, T, nlat, nlon, n, precision)
    b.run()
    ref = [o.clone() for o in outs]
    for cols, grid in ((32, 8), (32, 1), (32, 24), (32, 64), (64, 0), (64, 16), (32, 4096)):
        b.set_config(cols=(cols, cols), grid=(grid, grid))
        for o in outs:
            o.zero_()
        b.run()
        for k, (a, r) in enumerate(zip(outs, ref)):
            assert torch.equal(a, r), f"{cols} columns, grid {grid}, result {k}"


def test_lists_of_more_than_256_entries():
    """nlat 1030: the FP32 vector analysis lists 2 x 17 x 4 = 136 steps, the
    split modes (one segment above the FP64 orders) at most 68; the two agree
    to the FP32 error of a derivative, T eps sqrt(nlat) < 1e-4 of the largest."""
    import torch

    b32, o32 = _batch(torch, 30, 1030, 64, 3, "float32")
    b6, o6 = _batch(torch, 30, 1030, 64, 3, "bf16x6")
    for grid in (0, 8):
        b32.set_config(grid=(grid, grid))
        b32.run()
        b6.run()
        for a, r in zip(o32, o6):
            assert (a - r).abs().max() <= 1e-4 * r.abs().max()
