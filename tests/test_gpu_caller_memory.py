"""Clouds on the GPU in any layout, outputs in page-locked or pageable memory (GPU).

Staging gathers device clouds with one kernel and the outputs are written by
one; every layout and kind of memory gives what host arrays give.
"""
import ctypes

import numpy as np
import pytest
import torch

from lidar_amd import native as N
from lidar_amd import synth

pytestmark = pytest.mark.gpu

LAYOUTS = ["soa", "soa_odd_address", "records_32", "records_19", "no_ring"]


def device_cloud(f, layout, keep):
    c = N.Cloud()
    c.num_points, c.on_device = f.n, 1
    if layout.startswith("records"):
        size = int(layout.split("_")[1])
        rec = np.zeros((f.n, size), np.uint8)
        for k, a in enumerate((f.x, f.y, f.z)):
            rec[:, 4 * k + 1:4 * k + 5] = a.view(np.uint8).reshape(-1, 4)
        rec[:, 15:17] = f.ring.view(np.uint8).reshape(-1, 2)
        t = torch.from_numpy(rec).cuda()
        keep.append(t)
        c.x, c.y, c.z, c.ring = (t.data_ptr() + o for o in (1, 5, 9, 15))
        c.xyz_stride = c.ring_stride = size
        return c
    odd = 1 if layout == "soa_odd_address" else 0
    ptr = []
    for a in (f.x, f.y, f.z, f.ring):
        t = torch.zeros(a.nbytes + 8, dtype=torch.uint8, device="cuda")
        t[odd:odd + a.nbytes] = torch.from_numpy(a.view(np.uint8)).cuda()
        keep.append(t)
        ptr.append(t.data_ptr() + odd)
    c.x, c.y, c.z = ptr[:3]
    c.ring = None if layout == "no_ring" else ptr[3]
    c.xyz_stride, c.ring_stride = 4, 2
    return c


def output_arrays(n, pinned, odd):
    """(FrameOutputs, arrays): arrays start `odd` elements into their memory."""
    out, arrays = N.FrameOutputs(), {}
    for name, dtype, count in (("seg_labels", torch.int32, n), ("obstacle_index", torch.int32, n),
                               ("cluster_labels", torch.int32, n), ("hull_offsets", torch.int32, n + 1),
                               ("hull_indices", torch.int32, n), ("noise_labels", torch.uint8, n),
                               ("ground_index", torch.int32, n), ("unknown_index", torch.int32, n),
                               ("boxes", torch.float64, 10 * n)):
        t = torch.zeros(count + odd, dtype=dtype, pin_memory=pinned)[odd:]
        setattr(out, name, t.data_ptr())
        arrays[name] = t.numpy()
    out.hull_capacity = n
    return out, arrays


@pytest.mark.parametrize("streams", [1, 3])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_device_clouds_and_output_memory(layout, streams):
    frames = [synth.make_frame(height=32, width=512 + 131 * k, fov_up=10.67, fov_down=-30.67, layout=1, rain=60,
                               seed=40 + k) for k in range(19)]  # more than one staging launch
    cfgs = [N.segmenter_config(image_height=f.height, image_width=f.width, elevation_up_deg=f.fov_up_deg,
                               elevation_down_deg=f.fov_down_deg) for f in frames]
    B = len(frames)
    most = max(f.n for f in frames)
    with N.Context(max_frames=B, max_points=most, max_height=32, max_width=4096, streams=streams) as ctx:
        ctx.set_noise_filter(N.noise_config())
        ctx.set_oriented_boxes(True)
        ctx.set_label_clouds(True)
        host = [(f.x, f.y, f.z, None if layout == "no_ring" else f.ring) for f in frames]
        ref = ctx.process(host, cfgs)
        keep = []
        clouds = (N.Cloud * B)(*[device_cloud(f, layout, keep) for f in frames])
        carr = (N.SegmenterConfig * B)(*cfgs)
        ccfg = N.clusterer_config()
        torch.cuda.synchronize()
        L = N.lib()
        for pinned, odd in ((True, 0), (True, 1), (False, 0)):
            outs = (N.FrameOutputs * B)()
            arrays, res = [], (N.FrameResult * B)()
            for k, f in enumerate(frames):
                # Every other frame the other kind of memory.
                outs[k], a = output_arrays(f.n, pinned if k % 2 else not pinned, odd)
                arrays.append(a)
            N.check(L.lp_batch_stage(ctx.h, carr, B, ctypes.byref(ccfg), B, clouds))
            N.check(L.lp_batch_run(ctx.h, 1))
            N.check(L.lp_batch_fetch(ctx.h, outs, res))
            for k, r in enumerate(ref):
                a, K, V = arrays[k], r["num_clusters"], len(r["hull_indices"])
                assert res[k].num_points == r["num_points"] and res[k].num_clusters == K
                assert np.array_equal(a["noise_labels"], r["noise_labels"])
                assert np.array_equal(a["seg_labels"][:r["num_points"]].view(np.uint32), r["seg_labels"])
                for name in ("obstacle_index", "cluster_labels", "ground_index", "unknown_index"):
                    assert np.array_equal(a[name][:len(r[name])], r[name]), name
                    assert not a[name][len(r[name]):].any(), name
                assert np.array_equal(a["hull_offsets"][:K + 1], r["hull_offsets"])
                assert np.array_equal(a["hull_indices"][:V], r["hull_indices"])
                boxes = a["boxes"].reshape(-1, 10)
                assert all(np.array_equal(boxes[q, :8], r["boxes"][q]["corners"].reshape(-1)) for q in range(K))
                assert not boxes[K:].any()


def test_hull_capacity_is_checked_and_later_outputs_stay():
    f = synth.make_frame(height=32, width=1024, fov_up=10.67, fov_down=-30.67, layout=1, seed=5)
    cfg = N.segmenter_config(image_height=f.height, image_width=f.width, elevation_up_deg=f.fov_up_deg,
                             elevation_down_deg=f.fov_down_deg)
    with N.Context(max_frames=1, max_points=f.n, max_height=32, max_width=1024) as ctx:
        ctx.set_oriented_boxes(True)
        ref = ctx.process([(f.x, f.y, f.z, f.ring)], cfg)[0]
        for capacity in (len(ref["hull_indices"]) - 1, 1, 0, -1):
            out, a = output_arrays(f.n, True, 0)
            out.hull_capacity = capacity
            res = N.FrameResult()
            assert N.lib().lp_batch_fetch(ctx.h, ctypes.byref(out), ctypes.byref(res)) == N.ERR_CAPACITY
            assert res.status == N.ERR_CAPACITY
            assert np.array_equal(a["cluster_labels"][:len(ref["cluster_labels"])], ref["cluster_labels"])
            assert not a["hull_indices"].any() and not a["boxes"].any()
