"""Large-error node correction on the GPU at the edges of its work split (two nodes a
wave, eight a workgroup): node counts around them, windows at the image's corners and
one pixel outside, and pixels that tie for nearest -- whole windows, or every second
pixel -- where the first in the oracle's order wins.  Against the oracle as the planted
frame is: the same nodes, values within 1e-5."""
import numpy as np
import pytest

from test_gpu_node_correction import compare
from test_oracle_node_correction import CX, CY, F, H, INIT, W, W2C, camera_point, m12, rigid, world_of_camera

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 65])
def test_sizes_and_ties(n):
    rng = np.random.default_rng(n)
    pixels = [(2, 2), (W - 3, H - 3), (W - 3, 2), (2, H - 3), (1, 10), (W - 2, 10), (14, 10)]
    live = np.zeros((n, 4), np.float32)
    prev = np.zeros((H, W, 4), np.float32)
    for k in range(n):
        u, v = pixels[k % len(pixels)]
        c = camera_point(u, v)
        live[k] = np.append(world_of_camera(c), 1.0)
        for y in range(max(0, v - 2), min(H, v + 3)):
            for x in range(max(0, u - 2), min(W, u + 3)):
                prev[y, x, :3] = c + (0.0 if (x + y) % 2 or u == 14 else 0.002)  # ties
    prev[:, :, 3] = 1.0
    guided = np.array([m12(rigid(np.radians(rng.uniform(-1, 1, 3)), rng.uniform(-0.003, 0.003, 3))) for _ in range(H * W)],
                      np.float32).reshape(H, W, 12)
    views = [dict(intrinsic=[F, F, CX, CY], initial_camera_se3=m12(INIT), world2camera=m12(W2C), previous_vertex=prev,
                  guided_se3=guided, guided_valid=(rng.random((H, W)) < 0.8).astype(np.uint8))]
    knn = np.repeat(np.arange(n, dtype=np.uint16)[:, None], 4, 1)
    weight = np.tile(np.array([1, 0, 0, 0], np.float32), (n, 1))
    identity = np.tile(np.array([0, 0, 0, 1, 0, 0, 0, 0], np.float32), (n, 1))
    nodes = dict(error=np.full(n, 1.0, np.float32), live=live, se3=identity, knn=knn, weight=weight)
    surfels = dict(vertex=live.copy(), normal=np.tile(np.array([0, 0, -1, 0], np.float32), (n, 1)), knn=knn, weight=weight)
    compare(views, W, H, nodes, surfels, min_corrected=min(n, 1))
