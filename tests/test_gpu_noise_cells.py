"""The noise filter's grid passes at the edges of their steps (GPU, against
the definition): cells of 1 to a few thousand points in shuffled order, so the
input-order pass decides little, neighbour counts around the tests of a step,
and radii from one cell to the whole frame."""
import numpy as np
import pytest

from lidar_amd import native as N

pytestmark = pytest.mark.gpu


def _cloud(rng, scale):
    parts = []
    for k, n in enumerate([1, 2, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 79, 80, 81, 127, 129, 255, 257, 1000, 2500]):
        cell = np.array([12 + 2.0 * (k % 6), -7 + 3.0 * (k // 6), 1.0 * (k % 3)]) * [scale, scale, 1.0]
        parts.append(np.floor(cell) + rng.uniform(0.02, 0.98, (n, 3)))
    parts.append(rng.uniform(-40 * scale, 40 * scale, (900, 3)) * [1, 1, 0.1])
    p = np.concatenate(parts).astype(np.float32)
    return p[rng.permutation(len(p))]


@pytest.mark.parametrize("k", [1, 2, 4, 9, 17, 70, 300])
@pytest.mark.parametrize("radius,scale", [(0.05, 1.0), (0.3, 1.0), (0.9, 1.0), (1.6, 2.0), (2.7, 2.0), (3.5, 1.0)])
def test_cells_and_radii(oracle, k, radius, scale):
    p = _cloud(np.random.default_rng(17), scale)
    x, y, z = (np.ascontiguousarray(p[:, a]) for a in range(3))
    kw = dict(min_neighbours=k, min_search_radius_m=radius)
    print(f"{len(x)} points, {k} neighbours within {radius} m", flush=True)
    with N.Context(max_points=8192) as c:
        st, lab = c.remove_noise(x, y, z, N.noise_config(**kw))
    assert st == 0
    ref, _ = oracle.noise_definition(x, y, z, oracle.noise_config(**kw))
    assert np.array_equal(lab, ref)
    assert 0 < lab.sum() or k == 1


@pytest.mark.parametrize("n", [1023, 1024, 1025, 2048, 2049, 5000])
def test_kept_points_per_tile(n):
    """The kept points of frames around a compaction tile: counts that add up
    and, in input order, exactly the points labelled VALID."""
    from lidar_amd import synth
    f = synth.make_frame(height=32, width=512, fov_up=10.67, fov_down=-30.67, layout=1, rain=400, seed=5)
    ins = [tuple(a[:n] for a in (f.x, f.y, f.z, f.ring))]
    cfg = N.segmenter_config(image_height=32, image_width=512, elevation_up_deg=f.fov_up_deg,
                             elevation_down_deg=f.fov_down_deg)
    print(f"{n} points", flush=True)
    with N.Context(max_points=n, max_height=32, max_width=512) as with_filter, \
            N.Context(max_points=n, max_height=32, max_width=512) as plain:
        with_filter.set_noise_filter(N.noise_config())
        got = with_filter.process(ins, cfg)[0]
        valid = got["noise_labels"] == 0
        want = plain.process([tuple(np.ascontiguousarray(a[valid]) for a in ins[0])], cfg)[0]
    assert got["status"] == 0 and want["status"] == 0
    assert len(got["seg_labels"]) == int(valid.sum()) < n
    for key in ("seg_labels", "obstacle_index", "cluster_labels", "hull_indices"):
        assert np.array_equal(got[key], want[key]), key
