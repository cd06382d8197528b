"""Hulls at the edges of what one wavefront, one workgroup and one run of
clusters take (GPU, against the oracle's chain): points per chunk, chunks per
cluster, hull vertices per list, lists per frame."""
import numpy as np
import pytest

from lidar_amd import native as N

pytestmark = pytest.mark.gpu


def _blob(rng, n):
    return (rng.normal(0, 3, n).astype(np.float32).astype(np.float64),
            rng.normal(0, 1, n).astype(np.float32).astype(np.float64))


def _circle(rng, n):
    a = rng.uniform(0, 2 * np.pi, n)
    return 50 * np.cos(a), 50 * np.sin(a)


def _check(oracle, lists, max_points=200000):
    with N.Context(max_points=max_points) as ctx:
        st, hulls = ctx.convex_hulls(lists)
    assert st == 0
    for (x, y), h in zip(lists, hulls):
        r = oracle.convex_hull(x, y)
        assert np.array_equal(np.stack([x[h], y[h]], 1), np.stack([x[r], y[r]], 1))


@pytest.mark.parametrize("kind", [_blob, _circle])
@pytest.mark.parametrize("n", [1, 2, 3, 64, 65, 255, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4000])
def test_list_sizes(oracle, kind, n):
    """A list of n points between small ones; on the circle every point is a
    vertex, so more than a chunk of them is left after the rounds."""
    rng = np.random.default_rng(n)
    print(f"{kind.__name__} {n}", flush=True)
    _check(oracle, [_blob(rng, 5), kind(rng, n), _blob(rng, 9)])


@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 255, 256, 257, 513, 4095, 4097, 9001])
def test_list_counts(oracle, count):
    """Many lists, among them neighbours that a whole workgroup takes and one
    at either end."""
    rng = np.random.default_rng(count)
    lists = [_blob(rng, int(n)) for n in rng.integers(1, 12, count)]
    for k in (0, count // 2, count // 2 + 1, count - 1):
        if k < count:
            lists[k] = _blob(rng, 1500) if k % 2 else _circle(rng, 200)
    print(f"{count} lists", flush=True)
    _check(oracle, lists)


@pytest.mark.parametrize("frames", [15, 16, 17])
def test_frames_per_batch(frames):
    """Batches on both sides of the number of frames from which the hull
    stage takes smaller workgroups: each frame's hulls as it has them alone."""
    from lidar_amd import synth
    fs = [synth.make_frame(height=32, width=700 + 40 * (k % 5), fov_up=10.67, fov_down=-30.67, layout=1, seed=60 + k)
          for k in range(frames)]
    cfgs = [N.segmenter_config(image_height=f.height, image_width=f.width, elevation_up_deg=f.fov_up_deg,
                               elevation_down_deg=f.fov_down_deg) for f in fs]
    ins = [(f.x, f.y, f.z, f.ring) for f in fs]
    dims = dict(max_points=max(f.n for f in fs), max_height=32, max_width=1024)
    print(f"{frames} frames", flush=True)
    with N.Context(max_frames=frames, **dims) as all_, N.Context(max_frames=1, **dims) as one:
        for k, got in enumerate(all_.process(ins, cfgs)):
            want = one.process(ins[k:k + 1], cfgs[k:k + 1])[0]
            assert got["status"] == 0 and want["status"] == 0
            for key in ("cluster_labels", "hull_offsets", "hull_indices"):
                assert np.array_equal(got[key], want[key]), key
