"""Boxes of hulls whose edges give areas that agree in float (GPU, against the
oracle's sequential rule): straight sides of rectangles with points rounded to
float, and regular polygons, whose every edge gives the same area."""
import numpy as np
import pytest

from lidar_amd import native as N

from tests.test_gpu_noise_boxes import box_equal

pytestmark = pytest.mark.gpu


def side_hull(oracle, rng, points, bulge, where):
    """Hull of points along a rectangle's sides, which bend outward by `bulge`."""
    w, h = rng.uniform(4, 60), rng.uniform(2, 20)
    side, t = rng.integers(0, 4, points), rng.uniform(-1, 1, points)
    out = 1 + bulge * (1 - t * t)
    x = np.where(side < 2, t * w, np.where(side == 2, -w, w) * out)
    y = np.where(side < 2, np.where(side == 0, -h, h) * out, t * h)
    a = rng.uniform(0, np.pi)
    px = (where + x * np.cos(a) - y * np.sin(a)).astype(np.float32).astype(np.float64)
    py = (x * np.sin(a) + y * np.cos(a) - where).astype(np.float32).astype(np.float64)
    k = oracle.convex_hull(px, py)
    return px[k], py[k]


def polygons(oracle, bulge, where):
    rng = np.random.default_rng(8)
    out = [side_hull(oracle, rng, points, bulge, where) for points in (12, 40, 90, 200, 600, 1000, 1000)]
    for n in (8, 60, 64, 66, 130, 258, 700):
        t = np.arange(n) * (2 * np.pi / n)
        out.append((where + 9.0 * np.cos(t), 9.0 * np.sin(t)))
    fits = lambda x, y: 3 <= len(x) <= 1024 and len(oracle.antipodal_pairs(x, y)) <= (128 if len(x) <= 64 else 2048)
    return [(x, y) for x, y in out if fits(x, y)]


@pytest.mark.parametrize("where", [0.0, 50.0])
@pytest.mark.parametrize("bulge", [0.0, 1e-7, 1e-5, 1e-4])
def test_boxes_of_equal_areas(oracle, bulge, where):
    polys = polygons(oracle, bulge, where)
    refs = [oracle.obb_rotating_calipers(x, y) for x, y in polys]
    print(f"bulge {bulge}, at {where}: {[len(x) for x, _ in polys]} vertices", flush=True)
    assert len(polys) >= 8
    with N.Context(max_frames=1, max_points=32768) as ctx:
        st, boxes = ctx.oriented_boxes(polys)
    assert st == 0
    for (x, _), got, ref in zip(polys, boxes, refs):
        assert box_equal(got, ref), len(x)
