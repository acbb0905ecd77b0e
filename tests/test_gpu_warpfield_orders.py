"""Node graph and skinning on the GPU around the node count where a node's lanes change
(8192: a wave and 16 lanes in the graph, 16 lanes and one in the skinning) and the tiles
of 1024 nodes, with nodes in no order, on a line that comes nearer (every node enters
the slots) and on one that goes away; coincident nodes and nodes that are not finite.
Indices bit for bit against the oracle, weights within 1e-6 of it."""
import numpy as np
import pytest

from multiviewdynrecon_amd import warpfield as wf
from test_gpu_warpfield import dev, host
from test_oracle_warpfield import cloud, oracle_graph, oracle_skin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["none", "nearer", "away"])
@pytest.mark.parametrize("n", [3, 17, 1023, 1024, 1025, 1031, 2048, 2053, 6144, 6145, 8191, 8192, 8193, 8201, 9217, 12288, 12291])
def test_orders(n, order):
    rng = np.random.default_rng(n)
    nodes, pts = cloud(rng, n), cloud(rng, 131)
    if order != "none":
        nodes[:, :3] *= 1e-3
        nodes[:, 0] = np.linspace(0, 1, n) if order == "nearer" else np.linspace(1, 0, n)
        pts[:, 0] += 2.0
    nodes[n // 2] = nodes[0]
    nodes[n // 3, 1] = np.nan
    nodes[n // 5, :3] = np.inf
    np.testing.assert_array_equal(host(wf.BuildNodesGraph(dev(nodes))).view(np.uint16), oracle_graph(nodes))
    vk, vw, nk, nw = (host(t) for t in wf.PerformSkinning(dev(pts), dev(nodes), 0.5))
    k_ref, w_ref = oracle_skin(np.concatenate([pts, nodes]), nodes, 0.5)
    np.testing.assert_array_equal(np.concatenate([vk.view(np.uint16), nk.view(np.uint16)]), k_ref)
    np.testing.assert_allclose(np.concatenate([vw, nw]), w_ref, rtol=1e-6, atol=1e-7)
