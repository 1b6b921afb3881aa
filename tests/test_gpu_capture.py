"""Stages captured into a HIP graph and replayed between eager frames: every replay gives
what the captured stages gave, whatever frames ran in between, and eager stages after a
capture do not count on what the capture only recorded."""
import numpy as np
import pytest

from gpu_common import say, small_scene
from volumetricrestirrelease_amd import abi
from volumetricrestirrelease_amd.volumetric_restir import VolumetricReSTIR

pytestmark = pytest.mark.gpu


def make():
    spec = small_scene(res=64, width=96, height=64, maxBounces=2, initialM=4, spatialReuseRounds=1, spatialSampleCount=3)
    spec.orbit_degrees_per_frame = 25.0
    g = VolumetricReSTIR()
    g.setScene(spec)
    return g, spec


def begin(g, spec, frame):
    g.resetHistory()
    g.setCamera(spec, frame)
    g.prepare_frame(spec.width, spec.height)


def reservoirs(g, spec):
    import torch
    torch.cuda.synchronize()
    return g.read(abi.BUF_RESERVOIRS0, spec.width * spec.height * 36)


def eager(frame):
    """TraceRays' reservoirs of a frame of its own handle."""
    g, spec = make()
    begin(g, spec, frame)
    g.run_stage(abi.STAGE_GENERATE_FEATURES)
    g.run_stage(abi.STAGE_TRACE_RAYS)
    return reservoirs(g, spec)


@pytest.mark.parametrize("from_features", [True, False])
def test_replays_of_captured_stages_between_other_frames(from_features):
    """GenerateFeatures and TraceRays, or TraceRays alone, of frame 0 captured; eager frames
    of other cameras run between the replays."""
    import torch
    say(f"case: capture of {'GenerateFeatures and TraceRays' if from_features else 'TraceRays'}, 3 replays")
    want = eager(0)
    g, spec = make()
    out = torch.zeros((spec.height, spec.width, 4), device="cuda")
    g.setCamera(spec, 0)
    g.execute(out)  # allocates
    s = torch.cuda.Stream()
    begin(g, spec, 0)
    if not from_features:
        g.run_stage(abi.STAGE_GENERATE_FEATURES, stream=s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        if from_features:
            g.run_stage(abi.STAGE_GENERATE_FEATURES, stream=s)
        g.run_stage(abi.STAGE_TRACE_RAYS, stream=s)
    g.end_frame()
    for k in range(3):
        with torch.cuda.stream(s):
            graph.replay()
        assert np.array_equal(reservoirs(g, spec), want), k
        g.setCamera(spec, k + 3)
        g.execute(out)
        torch.cuda.synchronize()
        assert not np.array_equal(reservoirs(g, spec), want)


def test_eager_stage_after_captured_features():
    """TraceRays run eagerly after a capture that recorded GenerateFeatures: the rows that
    the capture has not made yet (its graph has not run) are made first."""
    import torch
    say("case: capture of GenerateFeatures only, then eager TraceRays on the same stream")
    want = eager(7)
    g, spec = make()
    out = torch.zeros((spec.height, spec.width, 4), device="cuda")
    g.setCamera(spec, 0)
    g.execute(out)
    s = torch.cuda.Stream()
    begin(g, spec, 7)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        g.run_stage(abi.STAGE_GENERATE_FEATURES, stream=s)
    g.run_stage(abi.STAGE_TRACE_RAYS, stream=s)
    assert np.array_equal(reservoirs(g, spec), want)
