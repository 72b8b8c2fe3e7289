"""c8_rows' rows of sixteen heads (launches of more than 256 rows of eight
heads, above eight heads): head counts that leave a row or a group of eight
part full, both load policies, masked entries, and padded launches re-planned
into partitions, whose states and tickets count rows of eight heads.  Bit-exact
with the oracle on the launch's plan."""
import sys

import numpy as np
import pytest

from tests import workloads
from tests.device_cases import joint_flags, run_hip, run_oracle
from tests.test_gpu_chunk import padded

pytestmark = pytest.mark.gpu

CASES = [
    # name, ratio, queries, lengths, heads, index mode, padding tokens
    ("nine_heads", 4, [140], [2600], 9, "uniform", 0),            # one head in a row's second group
    ("three_groups", 4, [70, 21], [4600, 150], 20, "holes", 2),   # a row of sixteen and one of four
    ("full_rows", 4, [33], [5000], 64, "mixed", 0),
    ("decode", 4, [1] * 70, list(range(700, 700 + 70 * 61, 61)), 32, "uniform", 0),   # streamed loads, 70 requests
    ("window_only", 1, [45], [300], 48, "uniform", 1),
    ("replanned", 4, [3, 5], [6000, 900], 20, "dups", 100),       # 24 live rows: several partitions each
    ("replanned_streamed", 4, [1] * 9, [5000 + 7 * b for b in range(9)], 16, "uniform", 140),
]


@pytest.mark.parametrize("name,ratio,queries,lengths,heads,mode,pad", CASES, ids=[c[0] for c in CASES])
def test_wide_rows_match_oracle(name, ratio, queries, lengths, heads, mode, pad):
    print(f"[wide rows] {name}", file=sys.stderr, flush=True)
    case = workloads.make_case(92, ratio, queries, lengths, heads=heads, index_mode=mode)
    launch = case
    if pad:
        launch = padded(case, pad)
        if ratio == 4:
            filler = np.full((pad,) + case["cmp_indices"].shape[1:], -1, np.int32)
            launch["cmp_indices"] = np.concatenate([case["cmp_indices"], filler])
    assert launch["q"].shape[0] * ((heads + 7) // 8) > 256
    out, lse, op = run_hip(launch, splits=1)
    plan = op.device_splits()
    assert (plan > 1) == name.startswith("replanned")
    live = int(case["cu_q"][-1])
    assert not out[live:].any() and not lse[live:].any(), "padding rows are not zero"
    assert op.workspace is None or not op.workspace.any(), "merge tickets must return to zero"
    ref, ref_lse, _ = run_oracle(case, plan, joint=joint_flags(launch, 1))
    diff = out[:live] != ref
    assert not diff.any(), f"{int(diff.sum())} BF16 mismatches"
    np.testing.assert_allclose(lse[:live], ref_lse, rtol=0, atol=2e-6)
