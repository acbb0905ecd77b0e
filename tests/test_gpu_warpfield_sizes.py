"""Node graph and skinning on the GPU where their work split changes: fewer nodes
than result slots, boxes of 8 nodes (below, exactly, one past), batches of 64 boxes
(512 nodes), passes of 4096 nodes, vertex counts that leave waves and workgroups
part full, nodes in spatial order and in none, equal and coincident points, a vertex
out of reach, one that is not a number and nodes that are not finite.  Indices bit
for bit against the oracle; weights within 1e-6 of it (the device's expf against the
host's, each within an ulp or two, and four of them normalised)."""
import numpy as np
import pytest

from multiviewdynrecon_amd import warpfield as wf
from test_gpu_warpfield import dev, host
from test_oracle_warpfield import cloud, oracle_graph, oracle_skin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, vertices, ordered", [
    (1, 1, False), (3, 63, False), (7, 64, True), (8, 65, False), (9, 511, True), (15, 512, False), (17, 513, True),
    (511, 700, True), (512, 700, False), (513, 1025, True), (521, 300, False), (4095, 2000, True), (4097, 2000, False),
    (8203, 600, True),
])
def test_sizes(n, vertices, ordered):
    rng = np.random.default_rng(n)
    nodes, pts = cloud(rng, n), cloud(rng, vertices)
    if ordered:
        nodes, pts = (a[np.lexsort(np.floor(a[:, :3] * 20).T)] for a in (nodes, pts))
    if n > 8:
        nodes[n // 2] = nodes[0]           # coincident nodes
        nodes[n - 1, :3] = np.inf
        nodes[n // 3, 1] = np.nan
    if vertices > 4:
        pts[1] = pts[0]
        pts[2, :3] = nodes[0, :3]          # on a node
        pts[3, :3] = 2e3                   # beyond the slots' first distance
        pts[vertices // 2, 0] = np.nan
    np.testing.assert_array_equal(host(wf.BuildNodesGraph(dev(nodes))).view(np.uint16), oracle_graph(nodes))
    vk, vw, nk, nw = (host(t) for t in wf.PerformSkinning(dev(pts), dev(nodes), 0.5))
    k_ref, w_ref = oracle_skin(np.concatenate([pts, nodes]), nodes, 0.5)
    np.testing.assert_array_equal(np.concatenate([vk.view(np.uint16), nk.view(np.uint16)]), k_ref)
    np.testing.assert_allclose(np.concatenate([vw, nw]), w_ref, rtol=1e-6, atol=1e-7)
