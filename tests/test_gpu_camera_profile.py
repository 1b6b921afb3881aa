"""Camera-ray profiles: the split stages look the transmittance of a pixel's camera
ray up in a row of running optical depths (made once per frame) where the one-kernel
stages march the ray again for every evaluation. Both take the same march samples, so
frames agree to float summation order where the lookup can go wrong: samples before a
block's offset entry (2 x 2 x 2 blocks at mip 0, where the 0.01 offset spans several
steps), steps shorter than the 128-samples-per-brick cap, depths within rounding of a
step (a distant camera), a camera inside the volume (rows that start at the camera),
nearest filtering, rows of pixels that miss the grid, and every path length."""
import numpy as np
import pytest

from gpu_common import rel, say, small_scene
from volumetricrestirrelease_amd import abi
from volumetricrestirrelease_amd.volumetric_restir import VolumetricReSTIR

pytestmark = pytest.mark.gpu

CASES = {
    "blocks_mip0": dict(res=256, fp16=True, spatialVisibilityMipLevel=0, spatialLightingMipLevel=0, maxBounces=3),
    "short_steps": dict(res=64, spatialVisibilityTStepScale=0.03, maxBounces=2),
    "long_steps": dict(res=64, spatialVisibilityTStepScale=7.0, maxBounces=2),
    "nearest": dict(res=128, spatialVisibilityUseLinearSampler=0, maxBounces=1),
    "mixed_mips": dict(res=128, spatialVisibilityMipLevel=2, spatialLightingMipLevel=0, maxBounces=4),
    "no_talbot": dict(res=64, spatialMISMethod=0, temporalMISMethod=0, maxBounces=2),
    "far_camera": dict(res=64, posW=(20.0, 30.0, 180.0), fovY=0.02, maxBounces=2),
    "inside": dict(res=128, posW=(0.1, 0.05, 0.2), fovY=1.2, maxBounces=3),
    "odd_size": dict(res=96, width=37, height=19, maxBounces=2),
}


def scene(name):
    c = dict(CASES[name])
    pos, fov = c.pop("posW", None), c.pop("fovY", None)
    spec = small_scene(**{**dict(width=64, height=48, initialM=4, spatialReuseRounds=2, spatialSampleCount=4), **c})
    if pos:
        spec.camera.update(posW=pos, fovY=fov)
    spec.orbit_degrees_per_frame = 2.0
    return spec


def passes(spec):
    """The pass without rows and with them: the budget is the only difference."""
    out = []
    for budget in (0, 16384):
        g = VolumetricReSTIR()
        g.setScene(spec)
        assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_PROFILE_MB, budget) == 0
        out.append(g)
    return out


@pytest.mark.parametrize("name", list(CASES))
def test_looked_up_transmittances_are_the_marched_ones_ray_by_ray(name):
    """TraceRays draws its sample without the rows and weighs it with the camera ray's
    transmittance up to it: the reservoirs of every pixel hold the same sample, and p_y,
    proportional to that transmittance, the same value (both forms add a ray's samples one
    after the other in single precision; a few ulp where the compiler fuses differently)."""
    import torch
    from volumetricrestirrelease_amd.volumetric_restir import RESERVOIR_DTYPE
    say(f"case: TraceRays' reservoirs with and without rows, {name}")
    spec = scene(name)
    n = spec.width * spec.height
    both = passes(spec)
    rays = 0
    for f in range(4):
        got = []
        for g in both:
            g.resetHistory()
            g.setCamera(spec, f)
            g.prepare_frame(spec.width, spec.height)
            g.run_stage(abi.STAGE_GENERATE_FEATURES)
            g.run_stage(abi.STAGE_TRACE_RAYS)
            torch.cuda.synchronize()
            got.append(g.read(abi.BUF_RESERVOIRS0, 36 * n).view(RESERVOIR_DTYPE))
            g.end_frame()
        a, b = got
        for k in ("M", "depth", "lightID", "sampledPixel"):
            assert np.array_equal(a[k], b[k]), (f, k)
        for k in ("p_y", "runningSum"):
            assert rel(a[k], b[k]).max() <= 2e-6, (f, k, rel(a[k], b[k]).max())
        rays += int((a["p_y"] > 0).sum())
    say(f"   {rays} pixels with a sample")
    assert rays > n // 8


@pytest.mark.parametrize("name", list(CASES))
def test_profiled_camera_rays_match_marched_ones(name):
    import torch
    say(f"case: camera-ray profiles against marched camera rays, {name}: {CASES[name]}")
    spec = scene(name)
    frames = []
    for split in (0, 2):
        g = VolumetricReSTIR()
        g.setScene(spec)
        assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_SPLIT_REUSE, split) == 0
        out = torch.zeros((spec.height, spec.width, 4), device="cuda")
        got = []
        for f in range(3):
            g.setCamera(spec, f)
            g.execute(out)
            torch.cuda.synchronize()
            got.append(out.cpu().numpy().copy())
        frames.append(got)
    for f in range(3):
        a, b = frames[0][f][..., :3].reshape(-1, 3), frames[1][f][..., :3].reshape(-1, 3)
        assert np.isfinite(b).all() and a.mean() > 0
        frac = float((rel(a, b).max(axis=1) <= 1e-4).mean())
        say(f"   frame {f}: pixels equal within 1e-4: {frac:.5f}")
        # an ulp of a transmittance changes a resampling draw on at most a pixel or two
        assert frac >= 0.999
