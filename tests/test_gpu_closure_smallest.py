"""The closure's kernels on the smallest grid, 8^3: fewer tiles than workgroups
in the convolutions, two slots of weight gradients.  Reference and tolerances
are those of the other sizes."""
import pytest

import test_gpu_closure_sizes as sizes

pytestmark = pytest.mark.gpu


def test_network_of_the_smallest_grid_matches_fp64():
    sizes.test_network_matches_fp64(8)
