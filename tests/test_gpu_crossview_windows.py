"""Cross-view search windows on the GPU: inside the image and over its border, one tap
wide, a wave's lanes or more wide; sparse and dense edges.  Bit-exact against the
oracle (whole numbers)."""
import pytest

from multiviewdynrecon_amd.crossview import CrossViewEdgeCorrespondence, crossview_input, default_config
from test_gpu_crossview_handle import lists
from test_gpu_crossview_sizes import frame
from test_oracle_crossview import oracle_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edges", [400, None])
@pytest.mark.parametrize("radius, step", [(0, 1), (3, 7), (5, 2), (6, 1), (9, 3)])
def test_windows(radius, step, edges):
    W, H = 61, 47
    cv = frame(21 + radius, 2 if edges is None else 3, W, H, edges)
    cfg = default_config(max_width=W, max_height=H, search_radius=radius, search_step=step)
    h = CrossViewEdgeCorrespondence(cfg)
    ci, keep = crossview_input(cv, device="cuda")
    h.SetCrossViewMatchingInput(ci)
    h.FindCrossViewEdgeMatchedPairs()
    assert lists(h) == oracle_lists(cv, cfg)


@pytest.mark.parametrize("radius, step", [(31, 1), (32, 1), (40, 1), (63, 2)])
def test_wide_windows(radius, step):
    W, H = 140, 131
    cv = frame(31 + radius, 2, W, H, 250)
    cfg = default_config(max_width=W, max_height=H, search_radius=radius, search_step=step, max_distance2=1e-3)
    h = CrossViewEdgeCorrespondence(cfg)
    ci, keep = crossview_input(cv, device="cuda")
    h.SetCrossViewMatchingInput(ci)
    h.FindCrossViewEdgeMatchedPairs()
    want = oracle_lists(cv, cfg)
    assert lists(h) == want and len(want[0]) > 0


@pytest.mark.parametrize("spare", [255, 256, 257])
@pytest.mark.parametrize("step", [1, 2])
def test_mostly_edges(step, spare):
    """Either side of 7/8 edge pixels, where threads take over from waves."""
    W, H = 32, 32
    cv = frame(7, 2, W, H, None)
    for view, n in zip(cv.views, (spare // 2, spare - spare // 2)):
        view.maps["edge_mask"].reshape(-1)[n:2 * n] = 0
    assert sum(int((v.maps["edge_mask"] == 1).sum()) for v in cv.views) == 2 * W * H - spare
    cfg = default_config(max_width=W, max_height=H, search_radius=4, search_step=step)
    h = CrossViewEdgeCorrespondence(cfg)
    ci, keep = crossview_input(cv, device="cuda")
    h.SetCrossViewMatchingInput(ci)
    h.FindCrossViewEdgeMatchedPairs()
    assert lists(h) == oracle_lists(cv, cfg)
