"""Frames of every size class of the launch spread: small frames give each wave a few
pixels (down to four in the stage kernels, one in the segment traces), larger ones 64.
The spread changes which wave a pixel is in and nothing else: a frame equals, bit for bit
and in every row and column, the one that a batch of one pass renders with 64 pixels a
wave, and its middle rows, whose neighbours the oracle has traced too, are the oracle's."""
import numpy as np
import pytest

from gpu_common import say, small_scene
from oracle.binding import Oracle
from volumetricrestirrelease_amd import abi
from volumetricrestirrelease_amd.volumetric_restir import VolumetricReSTIR, VolumetricReSTIRBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1, 1), (17, 3), (64, 63), (129, 127), (255, 257), (400, 330), (600, 450)])
def test_frame_of_any_spread_matches_the_oracle(width, height):
    import torch
    say(f"case: {width}x{height} frame against the oracle's rows")
    spec = small_scene(res=32, width=width, height=height, maxBounces=2, initialM=4, spatialReuseRounds=1,
                       spatialSampleCount=3)
    g = VolumetricReSTIR()
    g.setScene(spec)
    out = torch.zeros((height, width, 4), device="cuda")
    g.execute(out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()[..., :3].astype(np.float64)
    # rows whose spatial neighbours (10 px) the oracle has traced too
    y0 = max(0, height // 2 - 24)
    y1 = min(height, y0 + 48)
    o = Oracle()
    o.set_scene(spec)
    ref = o.execute(width, height, y0, y1, 8)[..., :3].astype(np.float64)
    lo = 0 if y0 == 0 else y0 + 11
    hi = height if y1 == height else y1 - 11
    a, b = got[lo:hi].reshape(-1, 3), ref[lo:hi].reshape(-1, 3) if ref.shape[0] == height else \
        ref[lo - y0:hi - y0].reshape(-1, 3)
    rel = np.abs(a - b) / np.maximum(np.maximum(np.abs(a), np.abs(b)), 1e-6)
    frac = float((rel.max(axis=1) <= 1e-3).mean())
    say(f"   pixels within 1e-3: {frac:.4f}")
    # the bar of whole uninjected frames (comparisons that rounding flips on single pixels)
    assert frac >= 0.97


@pytest.mark.parametrize("width,height", [(1, 1), (1, 200), (17, 3), (37, 1), (64, 63), (100, 61), (129, 127), (255, 257),
                                          (390, 333), (513, 509), (600, 450)])
def test_frame_of_any_spread_equals_the_unspread_one(width, height):
    """Widths and heights that leave remainders of the 16-wide tiles and of their 16, 8, 4, 2
    and 1 rows; the images start as NaN. (A batch runs TraceRays in one kernel: so does the
    pass alone here.)"""
    import torch
    say(f"case: {width}x{height} frame alone against a batch of one")
    spec = small_scene(res=32, width=width, height=height, maxBounces=3, initialM=3, spatialReuseRounds=1,
                       spatialSampleCount=3)
    imgs = []
    for batch in (False, True):
        g = VolumetricReSTIR()
        g.setScene(spec)
        assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_SPLIT_TRACE, 0) == 0
        out = torch.full((height, width, 4), float("nan"), device="cuda")
        if batch:
            b = VolumetricReSTIRBatch([g])
            b.execute([out])
        else:
            g.execute(out)
        torch.cuda.synchronize()
        imgs.append(out.cpu().numpy())
        if batch:
            b.close()
    assert np.isfinite(imgs[0]).all() and np.isfinite(imgs[1]).all()
    assert np.array_equal(imgs[0], imgs[1])


@pytest.mark.parametrize("points", [1, 7, 700, 5000])
def test_lattice_of_any_spread_gives_the_same_points(points):
    """A lattice of 1 to 5000 points in as many chunks as reach the next size class: chunk 0
    holds the same values whatever the launch's total."""
    import torch
    say(f"case: path-traced lattice, {points} points, 1 chunk against many")
    spec = small_scene(res=32, width=points, height=1 if points < 100 else 8, maxBounces=3)
    g = VolumetricReSTIR()
    g.setScene(spec)
    g.prepare_frame(spec.width, spec.height)
    g.end_frame()
    lh, lw = g.latticeShape(spec.width, spec.height, 1)
    one = torch.zeros((1, lh, lw, 4), device="cuda")
    many = torch.zeros((40, lh, lw, 4), device="cuda")
    g.referenceLattice(spec.width, spec.height, 1, 4, 77, one)
    g.referenceLattice(spec.width, spec.height, 1, 4, 77, many)
    torch.cuda.synchronize()
    assert torch.isfinite(many).all()
    assert torch.equal(one[0], many[0])
