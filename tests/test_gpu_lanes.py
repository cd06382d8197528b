"""Contexts of several streams made after other contexts came and went (GPU):
each lane's stream may be replaced while the context is made, and every frame
still has the single-stream results, eager and replayed."""
import numpy as np
import pytest

from lidar_amd import native as N
from lidar_amd import synth

pytestmark = pytest.mark.gpu

KEYS = ("seg_labels", "obstacle_index", "cluster_labels", "hull_offsets", "hull_indices")


def _context(frames, streams):
    return N.Context(max_frames=len(frames), max_points=max(f.n for f in frames), max_height=64, max_width=2048,
                     streams=streams)


@pytest.mark.parametrize("streams", [2, 4, 8])
def test_lanes_after_other_contexts(streams):
    frames = [synth.workload_c3(i) for i in range(9)]
    ins = [(f.x, f.y, f.z, f.ring) for f in frames]
    cfgs = [N.segmenter_config(image_height=f.height, image_width=f.width, elevation_up_deg=f.fov_up_deg,
                               elevation_down_deg=f.fov_down_deg) for f in frames]
    _context(frames[:1], 1).close()
    with _context(frames, 1) as one:
        want = one.process(ins, cfgs)
        _context(frames[:3], 3).close()
        for _ in range(2):
            with _context(frames, streams) as many:
                assert N.lib().lp_context_stream(many.h)
                for use_graph in (False, True, True):
                    print(f"{streams} streams, graph {use_graph}", flush=True)
                    for a, b in zip(want, many.process(ins, cfgs, use_graph=use_graph)):
                        assert a["status"] == 0 and b["status"] == 0
                        for k in KEYS:
                            assert np.array_equal(a[k], b[k]), k
