"""
How far separators are merged upwards, by the rows (``csrc/analysis.cpp``, ``default_merge_rows``): fronts of
up to 256 columns in all up to 524,288 rows, 128 up to 1,048,576 and none beyond. Every index the sweeps and
their two task lists form from such plans is in range (``hg_plan_validate``).
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import heat_oracle as ho
from ordito_amd import analysis, creation


@pytest.mark.parametrize("shape,widest", [((1024, 512), 256), ((1021, 514), 128), ((1049, 1001), 0)])
def test_merged_fronts_keep_to_their_tier(shape, widest):
    v, f = creation.torus(*shape, 1.0, 0.3, 0.1, 3)
    pattern = ho.operator_pattern(len(v), f)
    plan = analysis.analyse(pattern.indptr, pattern.indices, v, validate=True)
    kids = np.diff(plan.arrays["child_ptr"])
    # Bisection gives a separator two children; a front of more took theirs in.
    merged = plan.arrays["ncol"][kids > 2]
    if widest:
        assert len(merged) > 100 and widest / 2 < merged.max() <= widest
    else:
        assert len(merged) == 0
