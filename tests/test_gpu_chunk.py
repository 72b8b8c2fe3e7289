"""Prefill-shaped C128 and window-only launches (c8_chunk: one query row per
wave, eight neighbouring rows of a work-group sharing their KV tiles): how the
octets of rows meet requests, padding, joint rows, head groups and unreadable
pages.  Bit-exact with the oracle on the launch's plan; every launch here is
one that kernel takes (1025-2048 window-only rows or more than 768 C128 rows,
16 query tokens per request on average)."""
import sys

import numpy as np
import pytest

from tests import workloads
from tests.device_cases import joint_flags, query_subcase, run_hip, run_oracle

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def padded(case, pad):
    """The case at a graph's capacity: `pad` NaN query rows of an empty request."""
    live = int(case["cu_q"][-1])
    nan = np.full((pad,) + case["q"].shape[1:], 0x7FC0, np.uint16)
    out = dict(case, q=np.concatenate([case["q"], nan]),
               cu_q=np.concatenate([case["cu_q"], [live + pad]]).astype(np.int32),
               seq_lens=np.concatenate([case["seq_lens"], [0]]).astype(np.int32))
    for name in ("ori", "cmp"):
        if out[name] is not None:
            out[name].table = np.concatenate([out[name].table, out[name].table[:1]])
    return out


CASES = [
    # name, ratio, queries, lengths, heads, padding rows
    ("one_request", 1, [1041], [1041], 8, 0),                    # positions from 0 on, a last octet of one row
    ("pairs", 1, [1041, 1007], [1500, 1030], 8, 0),              # 256 octets, one of two requests
    ("pairs_c128", 128, [1041, 1007], [17600, 18000], 8, 0),     # the same, tiles of both in turn
    ("joint_straddle", 128, [1041, 1007], [3000, 9000], 8, 0),   # joint rows: one request after the other
    ("joint_edges", 128, [800], [16900], 8, 0),                  # rows of 127 to 132 compressed rows
    ("tails", 128, [403, 5, 399], [20000, 300, 17000], 8, 3),    # requests that start inside octets
    ("crowded", 1, [1020, 1, 1, 2, 1, 1023], [1100, 9, 700, 2, 131, 1200], 8, 0),   # several in one octet
    ("many_requests", 1, [17] * 70, list(range(17, 17 + 70 * 9, 9)), 8, 5),         # more than one wave's metadata
    ("keyless", 1, [700, 4, 400], [698, 1, 800], 8, 0),          # negative positions
    ("head_groups", 128, [300, 101], [17000, 2500], 20, 2),      # three groups of eight, the last of four
    ("four_heads", 1, [600, 500], [700, 2000], 4, 1),
    ("replanned", 128, [30, 9], [20000, 700], 8, 900),           # few live rows: several partitions each
    ("padded_joint", 128, [60, 9], [3000, 700], 8, 900),
]


@pytest.mark.parametrize("name,ratio,queries,lengths,heads,pad", CASES, ids=[c[0] for c in CASES])
def test_chunk_launch_matches_oracle(name, ratio, queries, lengths, heads, pad):
    from npu_sparse_attn_sharedkv_int8 import c8_attention
    say(f"[chunk] {name}")
    case = workloads.make_case(90, ratio, queries, lengths, heads=heads)
    launch = padded(case, pad) if pad else case
    rows = launch["q"].shape[0] * ((heads + 7) // 8)
    assert (1024 < rows <= 2048 if ratio == 1 else rows > 768) and launch["q"].shape[0] >= 16 * len(launch["seq_lens"])
    out, lse, op = run_hip(launch, splits=1)
    plan, joint = op.device_splits(), joint_flags(launch, 1)
    assert (plan > 1) == (name == "replanned")
    live = int(case["cu_q"][-1])
    assert not out[live:].any() and not lse[live:].any(), "padding rows are not zero"
    dead = c8_attention.keyless_tokens(case["cu_q"], case["seq_lens"], live)
    keep = [t for t in range(live) if not dead[t]]
    assert not out[[t for t in range(live) if dead[t]]].any(), "keyless rows are not zero"
    # The launch's own requests where the oracle takes them, else one request per row.
    sub = case if len(keep) == live else query_subcase(case, keep)
    ref, ref_lse, _ = run_oracle(sub, plan, joint=joint)
    diff = out[keep] != ref
    assert not diff.any(), f"{int(diff.sum())} BF16 mismatches, rows {sorted(set(np.argwhere(diff)[:, 0]))[:8]}"
    np.testing.assert_allclose(lse[keep], ref_lse, rtol=0, atol=2e-6)


@pytest.mark.parametrize("ratio,queries,length,before", [(1, 1097, 1300, 3), (128, 900, 17300, 13), (128, 2, 17000, 1200)])
def test_tokens_before_the_first_request(ratio, queries, length, before):
    """One request that starts at token `before`, inside an octet or short: its
    rows are computed and the tokens of no request are zero."""
    case = workloads.make_case(96, ratio, [queries], [length])
    nan = np.full((before,) + case["q"].shape[1:], 0x7FC0, np.uint16)
    launch = dict(case, q=np.concatenate([nan, case["q"]]), cu_q=case["cu_q"] + np.int32([before, before]))
    assert launch["cu_q"].dtype == np.int32
    say(f"[chunk] {before} tokens before the first request, ratio {ratio}")
    out, lse, op = run_hip(launch, splits=1)
    assert not out[:before].any() and not lse[:before].any()
    ref, ref_lse, _ = run_oracle(case, 1, joint=joint_flags(launch, 1))
    assert (out[before:] == ref).all()
    np.testing.assert_allclose(lse[before:], ref_lse, rtol=0, atol=2e-6)


ROUNDS = [   # more than 256 octets: a work-group takes several, one after the other
    ("partial", 1, [2601], [2601], 8, 0),                                # a last round of 70 octets, the last of one row
    ("partial_c128", 128, [2100], [17600], 8, 0),
    ("three", 1, [4300], [5000], 8, 0),
    ("three_c128", 128, [4300], [9000], 8, 0),
    ("joint_boundary", 128, [2200], [17200], 8, 0),                      # joint rows first, rows of two tiles after them
    ("tails", 128, [1003, 900, 203], [17000, 3000, 9100], 8, 0),         # taken by the last round's idle work-groups
    ("full_pairs", 1, [1501, 1302, 1293], [1600, 4000, 1293], 8, 0),     # 512 octets, none idle: two requests at once
    ("full_pairs_c128", 128, [1501, 1302, 1293], [17600, 3000, 9000], 8, 0),
    ("mixed", 128, [1000] + [1] * 20 + [1203], [17000] + list(range(200, 200 + 20 * 900, 900)) + [2500], 8, 0),
    ("head_groups", 128, [700, 201], [17000, 2500], 20, 0),              # 2703 rows of three groups
    ("padded", 1, [2500, 301], [2600, 900], 8, 800),
]


@pytest.mark.parametrize("name,ratio,queries,lengths,heads,pad", ROUNDS, ids=[c[0] for c in ROUNDS])
def test_several_rounds_match_oracle(name, ratio, queries, lengths, heads, pad):
    say(f"[chunk] rounds: {name}")
    case = workloads.make_case(97, ratio, queries, lengths, heads=heads)
    launch = padded(case, pad) if pad else case
    live = int(case["cu_q"][-1])
    groups = (heads + 7) // 8
    assert live * groups > (2560 if ratio == 1 else 2048) and launch["q"].shape[0] >= 16 * len(launch["seq_lens"])
    out, lse, op = run_hip(launch, splits=1)
    assert op.device_splits() == 1
    assert not out[live:].any() and not lse[live:].any(), "padding rows are not zero"
    ref, ref_lse, _ = run_oracle(case, 1, joint=joint_flags(launch, 1))
    diff = out[:live] != ref
    assert not diff.any(), f"{int(diff.sum())} BF16 mismatches, rows {sorted(set(np.argwhere(diff)[:, 0]))[:8]}"
    np.testing.assert_allclose(lse[:live], ref_lse, rtol=0, atol=2e-6)


@pytest.mark.parametrize("ratio", [1, 128])
def test_unreadable_pages_of_the_first_round(ratio):
    """Masked window rows in a work-group's first octet and none in its second."""
    case = workloads.make_case(98, ratio, [2900], [3100])
    case["ori"].table[0, 20] = case["ori"].pages + 3   # logical rows 640-671: query rows 440-598
    say(f"[chunk] unreadable pages of the first round, ratio {ratio}")
    out, lse, op = run_hip(case, splits=1)
    rows = list(range(430, 720, 2))   # octets 55-74 of XCD 1, and 77-89, the second of its work-groups
    ref, ref_lse, few = run_hip(query_subcase(case, rows), splits=1)
    assert (out[rows] == ref).all() and (lse[rows] == ref_lse).all()


@pytest.mark.parametrize("ratio", [1, 128])
def test_unreadable_pages_equal_the_general_path(ratio):
    """Block-table entries past the pool (window) and negative ones
    (compressed): the rows on them are masked, as in a launch of a few of the
    same rows (c8_attention)."""
    case = workloads.make_case(91, ratio, [1100], [18400 if ratio == 128 else 1300])
    table = case["ori"].table
    table[0, [table.shape[1] - 2, table.shape[1] - 9]] = case["ori"].pages + 3
    if ratio == 128:
        case["cmp"].table[0, [1, 4]] = -1
    say(f"[chunk] unreadable pages, ratio {ratio}")
    out, lse, op = run_hip(case, splits=1)
    rows = list(range(3, 1100, 13)) + list(range(1092, 1100))
    ref, ref_lse, few = run_hip(query_subcase(case, rows), splits=1)
    assert (out[rows] == ref).all() and (lse[rows] == ref_lse).all()
