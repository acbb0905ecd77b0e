"""Large-error node correction on the GPU at node counts around its four nodes a wave
and sixteen a workgroup, ties and image corners as in the sizes test."""
import pytest

import test_gpu_node_correction_sizes as sizes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 5, 15, 16, 17, 31, 33])
def test_sizes_and_ties(n):
    sizes.test_sizes_and_ties(n)
