"""Parallel antipodal walk of the oriented boxes vs the oracle's serial one (GPU).

Sizes at the edges of the kernel's groups (64 vertices per wavefront, 256
threads per workgroup, 1024 vertices in all) and polygons whose walk the
parallel form must hand back to the serial one: rounded ties, repeated
vertices, clockwise and collinear input.
"""
import numpy as np
import pytest

from lidar_amd import native as N

from tests.test_gpu_noise_boxes import box_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with N.Context(max_frames=1, max_points=262144) as c:
        yield c


def polygon(kind, n, rng):
    t = (np.arange(n) + rng.uniform(0.05, 0.9, n)) * (2 * np.pi / n)
    if kind == "regular":
        t = np.arange(n) * (2 * np.pi / n)
    x, y = 4.0 * np.cos(t), 1.5 * np.sin(t)
    if kind == "clockwise":
        x, y = x[::-1], y[::-1]
    if kind == "repeated":
        x[n // 2], y[n // 2] = x[n // 2 - 1], y[n // 2 - 1]
    if kind == "grid":
        x, y = np.floor(4 * x) / 4, np.floor(4 * y) / 4
    if kind == "collinear":
        y = 0.0 * y
    if kind == "float":
        x, y = (30.0 + x).astype(np.float32).astype(np.float64), (y - 12.0).astype(np.float32).astype(np.float64)
    return np.ascontiguousarray(x), np.ascontiguousarray(y)


@pytest.mark.parametrize("kind", ["convex", "regular", "float", "clockwise", "repeated", "grid", "collinear"])
def test_boxes_equal_the_serial_walk(ctx, oracle, kind):
    rng = np.random.default_rng(3)
    polys, refs = [], []
    for n in (3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 255, 256, 257, 511, 1023, 1024):
        x, y = polygon(kind, n, rng)
        if len(oracle.antipodal_pairs(x, y)) <= (128 if n <= 64 else 2048):
            polys.append((x, y))
            refs.append(oracle.obb_rotating_calipers(x, y))
    assert len(polys) >= 10
    st, boxes = ctx.oriented_boxes(polys)
    assert st == 0
    for (x, _), got, ref in zip(polys, boxes, refs):
        assert box_equal(got, ref), (kind, len(x))
    st, boxes = ctx.oriented_boxes(polys * 40)  # more polygons than one row of 256
    assert st == 0 and all(box_equal(g, r) for g, r in zip(boxes, refs * 40))
