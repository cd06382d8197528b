"""Hulls of clusters with so many candidates that several workgroups take them
through the rounds (GPU, against the oracle)."""
import numpy as np
import pytest

from lidar_amd import native as N

pytestmark = pytest.mark.gpu


def _ring(rng, n, noise, dtype=np.float64):
    """Points about a circle: of each chunk of them many are hull vertices."""
    a, r = rng.uniform(0, 2 * np.pi, n), 30 + rng.normal(0, noise, n)
    return tuple(v.astype(dtype).astype(np.float64) for v in (r * np.cos(a), r * np.sin(a)))


def _check(oracle, lists):
    with N.Context(max_points=max(sum(len(x) for x, _ in lists), 64)) as ctx:
        st, hulls = ctx.convex_hulls(lists)
    assert st == 0
    for (x, y), h in zip(lists, hulls):
        r = oracle.convex_hull(x, y)
        assert np.array_equal(np.stack([x[h], y[h]], 1), np.stack([x[r], y[r]], 1))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("noise,sizes", [(0.02, (4096, 12300, 12700, 20000, 26000)), (0.1, (4096, 22000, 23000, 50000))])
def test_list_sizes(oracle, noise, sizes, dtype):
    """Candidates of one workgroup, of four and of more, among small lists."""
    rng = np.random.default_rng(int(1000 * noise))
    lists = [_ring(rng, 7, 1.0)]
    for n in sizes:
        lists += [_ring(rng, n, noise, dtype), _ring(rng, 300, 0.0, dtype), _ring(rng, 5, 1.0)]
    print(f"noise {noise} {dtype.__name__}", flush=True)
    _check(oracle, lists)


def test_capacity(oracle):
    """Every point a vertex: as many as the last workgroup holds, and one more."""
    rng = np.random.default_rng(4)
    _check(oracle, [_ring(rng, 4096, 0.0)])
    with N.Context(max_points=20000) as ctx:
        for n in (4097, 6144, 6145, 20000):
            st, _ = ctx.convex_hulls([_ring(rng, n, 0.0)])
            assert st == N.ERR_CAPACITY
        x, y = _ring(rng, 3000, 0.003)
        st, hulls = ctx.convex_hulls([(x, y)])  # and the context goes on
        assert st == 0 and np.array_equal(x[hulls[0]], x[oracle.convex_hull(x, y)])


def _wall(seed, columns, noise):
    """One cluster: a wall about the sensor, its points in any order."""
    rng = np.random.default_rng(seed)
    p = rng.permutation(64 * columns)
    az, row = 2 * np.pi * (p % columns + 0.5) / 2048, p // columns
    dist = 20 + rng.normal(0, noise, len(p))
    return tuple(np.ascontiguousarray(a, t) for a, t in
                 ((dist * np.cos(az), np.float32), (dist * np.sin(az), np.float32), (-1.2 + row / 20, np.float32),
                  (row, np.uint16)))


# 16 frames and more take smaller workgroups.
@pytest.mark.parametrize("frames", [1, 3, 16])
def test_walls(oracle, frames):
    sc = dict(image_height=64, image_width=2048, road_maximum_slope_m_per_m=0.0)
    different = [_wall(k, columns, noise) for k, (columns, noise) in
                 enumerate([(1434, 0.02), (600, 0.003), (1945, 0.1)][:frames])]
    want = [oracle.process_frame(*f, scfg=oracle.seg_config(**sc)) for f in different]
    print(f"{frames} frames, hulls of {[len(w['hull_indices']) for w in want]}", flush=True)
    with N.Context(max_frames=frames, max_points=64 * 1945) as ctx:
        ctx.set_oriented_boxes(True)
        outs = ctx.process([different[k % len(different)] for k in range(frames)], N.segmenter_config(**sc))
    for k, (out, w) in enumerate((o, want[k % len(different)]) for k, o in enumerate(outs)):
        cloud = different[k % len(different)]
        obs = out["obstacle_index"]
        assert out["status"] == 0 and w["status"] == 0 and out["num_clusters"] == w["num_clusters"]
        assert np.array_equal(out["cluster_labels"], w["cluster_labels"])
        assert np.array_equal(out["hull_offsets"], w["hull_offsets"])
        for c in range(w["num_clusters"]):
            members = obs[w["cluster_labels"] == c]
            got, ref = (members[o["hull_indices"][w["hull_offsets"][c]:w["hull_offsets"][c + 1]]] for o in (out, w))
            assert np.array_equal(cloud[0][got], cloud[0][ref]) and np.array_equal(cloud[1][got], cloud[1][ref])
        assert out["boxes"][0]["is_valid"]
