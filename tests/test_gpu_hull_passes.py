"""Hull ranks of more clusters than the launch takes at once (GPU): a workgroup
goes through several runs of clusters, of small ones only and of small ones
with some that the whole workgroup takes, in any order.  Against the oracle."""
import numpy as np
import pytest

from lidar_amd import native as N

pytestmark = pytest.mark.gpu

LISTS_AT_ONCE = 256 * 16  # workgroups x wavefronts of the launch for standalone lists


def _small(rng):
    n = int(rng.integers(1, 8))
    return rng.normal(0, 3, n), rng.normal(0, 1, n)


def _large(rng):
    """More hull vertices than a wavefront takes."""
    a = rng.uniform(0, 2 * np.pi, int(rng.integers(70, 90)))
    return 50 * np.cos(a), 50 * np.sin(a)


@pytest.mark.parametrize("order", ["small first", "large first", "alternating", "mixed"])
def test_list_runs(oracle, order):
    """Three passes of the launch and a little: the runs of 16 lists that have
    large ones, one to three each at any place, differ from pass to pass."""
    rng = np.random.default_rng(len(order))
    count = 3 * LISTS_AT_ONCE + 37
    lists = [_small(rng) for _ in range(count)]
    for first in range(0, count, 16):
        turn, run = first // LISTS_AT_ONCE, first // 16
        large = {"small first": turn == 1, "large first": turn != 1, "alternating": (turn + run) % 2 == 0,
                 "mixed": rng.random() < 0.5}[order]
        for k in rng.choice(16, int(rng.integers(1, 4)), replace=False) if large else ():
            if first + k < count:
                lists[first + k] = _large(rng)
    print(f"{count} lists, {order}", flush=True)
    with N.Context(max_points=1 << 19) as ctx:
        st, hulls = ctx.convex_hulls(lists)
    assert st == 0
    for (x, y), h in zip(lists, hulls):
        assert np.array_equal(h, oracle.convex_hull(x, y))


@pytest.mark.parametrize("count", [64, 4096])
def test_as_many_lists_as_points(count):
    """One-point lists that fill the context: there is one offset more than
    points."""
    rng = np.random.default_rng(count)
    with N.Context(max_points=count) as ctx:
        for lists in (count, count - 1, count):
            st, hulls = ctx.convex_hulls([rng.normal(0, 9, (2, 1)) for _ in range(lists)])
            assert st == 0 and all(np.array_equal(h, [0]) for h in hulls)


def _frame(seed, posts):
    """Lone points all around, each a cluster of its own or of a few, and eight
    arcs of 72 columns, every point of which is a hull vertex.  An arc's first
    point comes anywhere in the input, so its cluster has any place."""
    rng = np.random.default_rng(seed)
    col = rng.permutation(1024 * 24)[:posts]
    az = [2 * np.pi * (col % 1024 + 0.5) / 1024]
    dist = [rng.uniform(25, 80, posts)]
    z = [rng.uniform(0, 2, posts)]
    row = [8 + col // 1024]
    key = [rng.uniform(0, 1, posts)]
    for k in range(8):
        az.append(2 * np.pi * (k * 120 + 5 + np.arange(72)) / 1024)
        dist.append(np.full(72, rng.uniform(15, 20)))
        z.append(np.full(72, 1.0))
        row.append(np.full(72, 1 + k % 4))
        key.append(rng.uniform(rng.uniform(0, 1), 1, 72))
    az, dist, z, row, key = (np.concatenate(a) for a in (az, dist, z, row, key))
    order = np.argsort(key)
    return tuple(np.ascontiguousarray(a[order], t) for a, t in
                 ((dist * np.cos(az), np.float32), (dist * np.sin(az), np.float32), (z, np.float32), (row, np.uint16)))


# Frames of one lane, lone points, and the clusters per frame the launch takes
# at once: workgroups per frame x wavefronts of each.
@pytest.mark.parametrize("frames,posts,at_once", [(15, 2600, 68 * 16), (16, 2600, 128 * 8), (64, 700, 32 * 8),
                                                  (128, 500, 16 * 8)])
def test_frame_runs(oracle, frames, posts, at_once):
    sc = dict(image_height=32, image_width=1024, road_maximum_slope_m_per_m=0.0)
    different = [_frame(100 * frames + k, posts + 40 * k) for k in range(3)]
    want = [oracle.process_frame(*f, scfg=oracle.seg_config(**sc), ccfg=oracle.cluster_config(min_cluster_size=1))
            for f in different]
    for w in want:
        vertices = np.diff(w["hull_offsets"])
        assert w["status"] == 0 and len(vertices) > at_once and (vertices > 64).sum() > 4
    print(f"{frames} frames of {[len(np.diff(w['hull_offsets'])) for w in want]} clusters", flush=True)
    with N.Context(max_frames=frames, max_points=4096, max_height=32, max_width=1024) as ctx:
        outs = ctx.process([different[k % 3] for k in range(frames)], N.segmenter_config(**sc),
                           N.clusterer_config(min_cluster_size=1))
    for k, out in enumerate(outs):
        w = want[k % 3]
        assert out["status"] == 0
        for key in ("cluster_labels", "hull_offsets", "hull_indices"):
            assert np.array_equal(out[key], w[key]), (k, key)
