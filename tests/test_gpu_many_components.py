"""Clusters of clouds with very many components (GPU, against the oracle): on
both sides of the number of obstacles up to which one workgroup ranks them, of
the roots it takes a turn and of the sizes it sums a turn."""
import numpy as np
import pytest

from lidar_amd import native as N

pytestmark = pytest.mark.gpu

FINE = dict(voxel_grid_range_resolution_m=0.1, voxel_grid_azimuth_resolution_deg=0.1,
            voxel_grid_elevation_resolution_deg=0.2)


def _scatter(n):
    """Points anywhere around the sensor: in fine voxels most are alone."""
    rng = np.random.default_rng(n)
    az, dist = rng.uniform(0, 2 * np.pi, n), rng.uniform(3, 95, n)
    return tuple(np.ascontiguousarray(a, np.float32)
                 for a in (dist * np.cos(az), dist * np.sin(az), rng.uniform(-3, 6, n) * dist / 40))


@pytest.mark.parametrize("min_size", [1, 2])
@pytest.mark.parametrize("n", [8191, 8193, 70000, 262143, 262144, 262145, 400001])
def test_cloud(oracle, n, min_size):
    cloud = _scatter(n)
    kw = dict(FINE, min_cluster_size=min_size)
    so, want = oracle.cluster(*cloud, oracle.cluster_config(**kw), max_voxels=n)
    print(f"{n} points, {want.max() + 1} clusters", flush=True)
    with N.Context(max_points=n, max_voxels=n) as ctx:
        st, got = ctx.cluster(*cloud, N.clusterer_config(**kw))
    assert so == 0 and st == 0
    assert np.array_equal(got, want)


def _pixels(height, width, points):
    """A point above the ground in each of `points` pixels, at any range."""
    rng = np.random.default_rng(points)
    p = rng.permutation(height * width)[:points]
    az, dist = 2 * np.pi * (p % width + 0.5) / width, rng.uniform(12, 95, points)
    return tuple(np.ascontiguousarray(a, t) for a, t in
                 ((dist * np.cos(az), np.float32), (dist * np.sin(az), np.float32),
                  (rng.uniform(-1, 2.2, points), np.float32), (p // width, np.uint16)))


def _expected(oracle, cloud, sc, kw):
    """Labels and hulls from the oracle's single objects."""
    st, seg, _ = oracle.segment(*cloud, cfg=oracle.seg_config(**sc))
    obs = np.flatnonzero(seg == 2)
    so, lab = oracle.cluster(*(a[obs] for a in cloud[:3]), oracle.cluster_config(**kw), max_voxels=1 << 19)
    assert st == 0 and so == 0
    members = np.argsort(lab, kind="stable")[(lab < 0).sum():]
    sizes = np.bincount(lab[lab >= 0])
    x, y = (a[obs].astype(np.float64) for a in cloud[:2])
    hulls, first = [], 0
    for n in sizes:
        m = members[first:first + n]
        hulls.append(np.arange(n) if n < 3 else oracle.convex_hull(x[m], y[m]))
        first += n
    return dict(seg_labels=seg, cluster_labels=lab, num_clusters=len(sizes),
                hull_offsets=np.cumsum([0] + [len(h) for h in hulls]),
                hull_indices=np.concatenate(hulls) if hulls else np.zeros(0, np.int32))


# 128x2048 pixels are as many obstacles as one workgroup ranks.
@pytest.mark.parametrize("width", [2048, 2049])
def test_frames(oracle, width):
    sc = dict(image_height=128, image_width=width, road_maximum_slope_m_per_m=0.0)
    frames = [_pixels(128, width, n) for n in (8000, 20000, 128 * width, 40)]
    x, y, z, ring = frames[3]
    frames[3] = (x, y, np.full_like(z, -1.73), ring)  # ground only: no obstacles
    kw = dict(FINE, min_cluster_size=1)
    want = [_expected(oracle, f, sc, kw) for f in frames]
    clusters = [w["num_clusters"] for w in want]
    print(f"clusters {clusters}", flush=True)
    assert clusters[0] < 8192 < clusters[1] < 2 * clusters[1] < clusters[2] and clusters[3] == 0
    with N.Context(max_frames=4, max_points=128 * width, max_height=128, max_width=width, max_voxels=1 << 19) as ctx:
        for graph in (False, True, True):
            outs = ctx.process(frames, N.segmenter_config(**sc), N.clusterer_config(**kw), use_graph=graph)
            for k, (out, w) in enumerate(zip(outs, want)):
                assert out["status"] == 0
                for key, value in w.items():
                    assert np.array_equal(out[key], value), (k, key)
