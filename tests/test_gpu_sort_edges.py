"""The grid's sort at the sizes where its launch plan changes: one workgroup
for every digit, tiles that add up their own digit offsets, tiles behind a
row scan; cell counts give 1 to 3 digit passes, even and uneven."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_grid import check_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 64, 65, 1023, 1024, 1025, 2048, 2049, 4097, 8191, 8192, 8193,
                               10241, 131071, 131072, 131073])
@pytest.mark.parametrize("dims", [(4, 4, 4), (40, 30, 50), (130, 130, 130)])
def test_sort_plans_match_oracle(n, dims):
    rng = np.random.default_rng(n + dims[0])
    cell = 1.0 / dims[0]
    x = rng.uniform(-0.01, 1.01, (n, 3)).astype(np.float32)
    x[: n // 4] = x[0]  # long runs of one key
    check_grid(x, (0.0, 0.0, 0.0), dims, cell, f"{n} {dims}")
