"""LBVH at the sizes where the segment tree's launches change (subtrees of
1024 leaves, ten levels a launch) and with long ranges of equal codes, whose
node searches leave the code window of a workgroup."""
from __future__ import annotations

import pytest

from test_gpu_grid import test_lbvh_nodes_and_boxes_match_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,n", [("random", 3), ("random", 255), ("random", 256),
                                    ("random", 257), ("random", 1023), ("random", 1024),
                                    ("random", 1025), ("random", 2049), ("duplicates", 1537),
                                    ("identical", 1025), ("identical", 5000),
                                    ("random", 1 << 20), ("random", (1 << 20) + 1)])
def test_edges(case, n):
    check(case, n)
