"""What a cross-view object keeps from one call to the next."""
import pytest
import torch

from multiviewdynrecon_amd.crossview import CrossViewEdgeCorrespondence, crossview_input, default_config
from test_gpu_crossview_sizes import frame
from test_oracle_crossview import oracle_lists

pytestmark = pytest.mark.gpu


def lists(h):
    got = [h.GetCrossViewMatchingCorrPairs(), h.GetCrossViewMatchingUniqueCorrPairs(), h.GetCrossViewBackTracingCorrPairs()]
    return [[tuple(int(x) for x in r) for r in lst] for lst in got]


def test_first_call_on_a_stream_beside_a_busy_null_stream():
    """A new object's edge counter is clear for a call on a stream that does not wait
    for the null stream, where creation clears it."""
    W, H = 48, 40
    cv = frame(5, 3, W, H, 300)
    cfg = default_config(max_width=W, max_height=H)
    want = oracle_lists(cv, cfg)
    ci, keep = crossview_input(cv, device="cuda")
    a = torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(50):
        a = torch.nn.functional.normalize(a @ a)
    h = CrossViewEdgeCorrespondence(cfg)
    h.SetCrossViewMatchingInput(ci)
    h.FindCrossViewEdgeMatchedPairs(stream=side.cuda_stream)
    side.synchronize()
    assert lists(h) == want
