"""The segment traces ray by ray: every ray that a split stage recorded, marched alone by
the tracking primitive, has the transmittance the trace wrote, for TraceRays' shadow rays
and for the spatial stage's camera and lighting rays, on grids where the sample counts of
the march are decided by rounding most often (many voxels a side, steps of a fraction of a
voxel), for both formats and filters and for rays of one and of two grids.

Both take the same samples at the same positions. A transmittance is exp(-tau) of n
samples' sum: another order of the sum moves tau by at most n 2^-24 of itself and by about
sqrt(n) 2^-24 where roundings are independent, so Tr by about 0.37 sqrt(n) 2^-24: 1.7e-6 for
n = 6000 (a tenth of a voxel along a 256^3 grid's diagonal; measured 1.9e-6), the bar is ten
times that. One sample too many or too few, or one in another voxel, is 1e-4 and more."""
import numpy as np
import pytest

from gpu_common import say, small_scene
from volumetricrestirrelease_amd import abi, scenes
from volumetricrestirrelease_amd.volumetric_restir import VolumetricReSTIR

pytestmark = pytest.mark.gpu

RAY = np.dtype([("o", "<f4", 3), ("tMax", "<f4"), ("d", "<f4", 3), ("kind", "<i4")])


def field(res, seed):
    """A smooth cloud on the GPU, zero over most of the cube, up to 1 inside."""
    import torch
    import torch.nn.functional as F
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    f = torch.zeros((res, res, res), device="cuda")
    for n, w in ((5, 1.0), (12, 0.5)):
        f += w * F.interpolate(torch.rand((1, 1, n, n, n), generator=g, device="cuda"), size=(res,) * 3,
                               mode="trilinear", align_corners=False)[0, 0]
    return ((f - 0.85) * 3.0).clamp_(0.0, 1.0).contiguous()


def pass_on(res, fp16, **params):
    spec = small_scene(res=8, width=112, height=80, fp16=fp16)
    spec.density, spec.dims, spec.num_mips = None, (res, res, res), 3
    spec.index_to_world = scenes.unit_cube_transform(res)
    spec.params.update(dict(maxBounces=3, initialM=8, spatialReuseRounds=1, spatialSampleCount=5))
    spec.params.update(params)
    g = VolumetricReSTIR()
    d = field(res, res)
    g.setSceneStreamed(spec, d)
    return g, spec


def check(g, spec, slots, options, what):
    """options[kind] = (mip, linear, tStepScale)"""
    import torch
    torch.cuda.synchronize()
    n = spec.width * spec.height
    counts = g.read(abi.BUF_RAY_COUNTS, 4 * n).view(np.int32)
    rays = g.read(abi.BUF_RAYS, n * slots * 32).view(RAY).reshape(n, slots)
    trs = g.read(abi.BUF_RAY_TRANSMITTANCES, n * slots * 4).view(np.float32).reshape(slots, n)
    assert counts.max() <= slots
    pix, slot = np.nonzero(np.arange(slots)[None, :] < counts[:, None])
    r, tr = rays[pix, slot], trs[slot, pix]
    assert len(r) > 4000
    worst = 0.0
    for kind, (mip, linear, step) in options.items():
        k = r["kind"] == kind
        if not k.any():
            continue
        inp = np.zeros((int(k.sum()), 8), np.float32)
        inp[:, :3], inp[:, 3:6], inp[:, 6] = r["o"][k], r["d"][k], r["tMax"][k]
        out = torch.zeros((len(inp), 8), device="cuda")
        g.track(abi.TRACK_TR_RAY_MARCHING, mip, linear, step, 1, torch.from_numpy(inp).cuda(),
                torch.zeros((len(inp), 3), dtype=torch.int32, device="cuda"), out)
        torch.cuda.synchronize()
        want = out[:, 0].cpu().numpy().astype(np.float64)
        e = np.abs(want - tr[k])
        worst = max(worst, float(e.max()))
        say(f"   {what}, kind {kind}: {len(inp)} rays, {np.mean((want > 0.01) & (want < 0.99)):.2f} of them partly "
            f"through, largest difference {e.max():.2e}")
        assert e.max() <= 2e-5, (what, kind, int((e > 2e-5).sum()))
    return worst


@pytest.mark.parametrize("res,fp16,mip,step,linear", [(512, True, 0, 0.25, 1), (512, True, 0, 1.0, 0),
                                                      (512, False, 1, 0.25, 1), (256, True, 0, 0.1, 1),
                                                      (128, False, 0, 3.0, 1), (128, True, 2, 20.0, 0)])
def test_traced_rays_of_one_grid_match_marched_ones(res, fp16, mip, step, linear):
    say(f"case: {res}^3 {'fp16' if fp16 else 'fp32'}, mip {mip}, steps x {step}, {'tri' if linear else 'nearest'}")
    g, spec = pass_on(res, fp16, initialLightingMipLevel=mip, initialLightingTStepScale=step,
                      initialLightingUseLinearSampler=linear, spatialVisibilityMipLevel=mip,
                      spatialLightingMipLevel=mip, spatialVisibilityTStepScale=step,
                      spatialLightingTStepScale=0.8 * step, spatialVisibilityUseLinearSampler=linear,
                      spatialLightingUseLinearSampler=linear)
    # the camera rays too are traced, not looked up
    assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_PROFILE_MB, 0) == 0
    run(g, spec, {1: (mip, linear, step)}, {0: (mip, linear, step), 1: (mip, linear, 0.8 * step)})


def test_traced_rays_of_two_grids_match_marched_ones():
    say("case: 256^3, camera rays on mip 0 trilinear, lighting rays on mip 1 nearest")
    g, spec = pass_on(256, True, initialLightingMipLevel=1, initialLightingTStepScale=0.5, spatialVisibilityMipLevel=0,
                      spatialLightingMipLevel=1, spatialVisibilityTStepScale=0.25, spatialLightingTStepScale=0.5,
                      spatialLightingUseLinearSampler=0)
    assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_PROFILE_MB, 0) == 0
    run(g, spec, {1: (1, 1, 0.5)}, {0: (0, 1, 0.25), 1: (1, 0, 0.5)})


def run(g, spec, trace, spatial):
    M, b, K = spec.params["initialM"], spec.params["maxBounces"], spec.params["spatialSampleCount"]
    g.setCamera(spec, 0)
    g.prepare_frame(spec.width, spec.height)
    g.run_stage(abi.STAGE_GENERATE_FEATURES)
    g.run_stage(abi.STAGE_TRACE_RAYS)
    stash = 3 * M + 4 * ((M + 3) // 4) + 7 * M * (b - 1) + (M * (b + 1) + 31) // 32
    check(g, spec, max(M * b, stash), trace, "TraceRays")
    g.run_stage(abi.STAGE_TEMPORAL_REUSE)
    g.run_stage(abi.STAGE_SPATIAL_REUSE)
    check(g, spec, K * (K - 1) * (b + 1), spatial, "SpatialReuse")


def test_grid_of_more_blocks_than_the_march_takes():
    """4096 x 2176 x 512 voxels at mip 0: 2176 blocks of 128^3, past the block mask of the
    march of one grid; a sparse field, in fp32. A voxel is 0.2 world units, so the walks'
    0.01 offset stays far below one (where it spans bricks, as it would on a unit cube, the
    hierarchical walk of this trace and the one of the tracking primitive end differently at
    the corners of empty blocks)."""
    import torch
    say("case: 4096 x 2176 x 512, mip 0, rays of the general segment trace")
    nx, ny, nz = 4096, 2176, 512
    spec = small_scene(res=8, width=160, height=112)
    spec.density, spec.dims, spec.num_mips = None, (nz, ny, nx), 1
    m = np.zeros(16, np.float32)
    m[0] = m[5] = m[10] = 0.2
    m[15], m[12], m[13], m[14] = 1.0, -0.1 * nx, -0.1 * ny, -0.1 * nz
    spec.index_to_world = m
    spec.params.update(maxBounces=3, initialM=8, spatialReuseRounds=1, spatialSampleCount=4, initialBaseMipLevel=0,
                       initialLightingMipLevel=0, temporalReprojectionMipLevel=0, spatialVisibilityMipLevel=0,
                       spatialLightingMipLevel=0, initialLightingTStepScale=1.0)
    size = 0.1 * nx  # world units of the unit cube's half side
    spec.camera.update(posW=tuple(size * x for x in spec.camera["posW"]), farZ=1000.0 * size)
    spec.lights = [(tuple(size * x for x in pos), inten) for pos, inten in spec.lights]
    spec.density_scale = 1.0 / size
    d = torch.zeros((nz, ny, nx), device="cuda")
    g0 = torch.Generator(device="cuda")
    g0.manual_seed(5)
    for _ in range(90):  # boxes of smooth density all over the grid
        z, y, x = (int(torch.randint(0, s - 256, (1,), generator=g0, device="cuda")) for s in (nz, ny, nx))
        box = torch.rand((1, 1, 4, 4, 4), generator=g0, device="cuda")
        d[z:z + 256, y:y + 256, x:x + 256] = torch.nn.functional.interpolate(box, size=(256,) * 3, mode="trilinear")[0, 0]
    g = VolumetricReSTIR()
    g.setSceneStreamed(spec, d)
    del d
    assert abi.load_library().vrestir_set_tuning(g.h, abi.TUNE_PROFILE_MB, 0) == 0
    run(g, spec, {1: (0, 1, 1.0)}, {0: (0, 1, 1.0), 1: (0, 1, 1.0)})
