"""Launches that the capacity or the average request sends to c8_chunk and whose
live rows another kernel takes in less time: few live rows in a graph's prefill
capacity, and a full prefill chunk with many one-token requests beside it.
c8_chunk runs such rows whole, as c8_attention would, bit-exact with the oracle
and in about their time."""
import sys

import numpy as np
import pytest

from tests import workloads
from tests.device_cases import DeviceCase, joint_flags, query_subcase, run_hip, run_oracle
from tests.test_gpu_chunk import padded

pytestmark = pytest.mark.gpu

CASES = [
    # name, ratio, queries, lengths, heads, padding rows
    ("two_passes", 128, [300, 9], [17000, 700], 8, 900),           # 309 rows over 256 work-groups
    ("most_rows", 128, [768], [16900], 8, 300),                    # the last count that takes whole rows
    ("octets", 128, [769], [16900], 8, 300),                       # and the first that takes octets
    ("joint", 128, [290, 40], [3000, 700], 8, 900),                # every row joint, two passes
    ("head_groups", 128, [150, 40], [17000, 2500], 20, 400),       # 570 rows of three groups
    ("many_requests", 128, [4] * 210, list(range(300, 300 + 210 * 90, 90)), 8, 2600),   # 840 rows, four a request
    ("window", 1, [300, 9], [17000, 700], 8, 1300),                # some work-group of an XCD with one row of its two
    ("window_one_row", 1, [1], [50], 8, 1300),
    ("window_passes", 1, [600, 300], [900, 4000], 8, 400),         # 900 rows over 512 half work-groups
    ("window_keyless", 1, [200, 4, 90], [198, 1, 300], 8, 1300),   # negative positions
    ("window_groups", 1, [100, 33], [3000, 50], 20, 700),          # rows of sixteen heads and of four
    ("window_four_heads", 1, [61], [2000], 4, 1300),
    ("window_mixed", 1, [1] * 64 + [1984], list(range(90, 90 + 64 * 40, 40)) + [2500], 8, 0),   # 56 tails of 256 octets
    ("mixed", 128, [1] * 20 + [801] + [2] * 10, list(range(200, 200 + 20 * 900, 900)) + [17100] + [16500, 40] * 5, 8, 3),
    ("mixed_groups", 128, [600] + [1] * 30, [16900] + list(range(100, 100 + 30 * 700, 700)), 16, 0),   # two rows a token
    ("window_mixed_groups", 1, [901] + [1] * 40, [1300] + list(range(1, 1 + 40 * 50, 50)), 16, 2),
]


@pytest.mark.parametrize("name,ratio,queries,lengths,heads,pad", CASES, ids=[c[0] for c in CASES])
def test_padded_launch_matches_oracle(name, ratio, queries, lengths, heads, pad):
    from npu_sparse_attn_sharedkv_int8 import c8_attention
    print(f"[padded] {name}", file=sys.stderr, flush=True)
    case = workloads.make_case(93, ratio, queries, lengths, heads=heads)
    launch = padded(case, pad) if pad else case
    rows, live = launch["q"].shape[0] * ((heads + 7) // 8), int(case["cu_q"][-1])
    assert (rows > 1024 if ratio == 1 else rows > 768) and launch["q"].shape[0] >= 16 * len(launch["seq_lens"])
    out, lse, op = run_hip(launch, splits=1)
    assert op.device_splits() == 1
    assert not out[live:].any() and not lse[live:].any(), "padding rows are not zero"
    dead = c8_attention.keyless_tokens(case["cu_q"], case["seq_lens"], live)
    keep = [t for t in range(live) if not dead[t]]
    assert not out[[t for t in range(live) if dead[t]]].any(), "keyless rows are not zero"
    sub = case if len(keep) == live else query_subcase(case, keep)
    ref, ref_lse, _ = run_oracle(sub, 1, joint=joint_flags(launch, 1))
    diff = out[keep] != ref
    assert not diff.any(), f"{int(diff.sum())} BF16 mismatches, rows {sorted(set(np.argwhere(diff)[:, 0]))[:8]}"
    np.testing.assert_allclose(lse[keep], ref_lse, rtol=0, atol=2e-6)


def microseconds(call, calls=50, rounds=7):
    import torch
    for _ in range(5):
        call()
    times = []
    for _ in range(rounds):
        first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        first.record()
        for _ in range(calls):
            call()
        last.record()
        torch.cuda.synchronize()
        times.append(first.elapsed_time(last) * 1000 / calls)
    return sorted(times)[rounds // 2]


@pytest.mark.parametrize("ratio,live,length", [(128, 40, 6000), (128, 200, 32768), (128, 200, 131072),
                                               (1, 40, 8192), (1, 512, 8192)])
def test_padded_launch_takes_the_time_of_its_live_rows(ratio, live, length):
    """A launch of 2048 query tokens with `live` live ones takes no more than
    1.5 times an eager launch of those and a fill of the padding's outputs
    together (measured: 0.9-1.2 times; an octet of eight rows on each of a few
    work-groups took 1.7-3 times)."""
    import torch
    from npu_sparse_attn_sharedkv_int8 import PreparedAttention, SharedKVCase
    capacity = 2048
    made = DeviceCase(94, ratio, [live], [length])
    eager = PreparedAttention(made.dev, made.ori_scale, made.cmp_scale)
    d = made.dev
    q = torch.cat([d.q, d.q.new_zeros((capacity - live,) + d.q.shape[1:])])
    both = lambda table: None if table is None else torch.cat([table, table])
    whole = SharedKVCase(q=q, ori=d.ori, ori_block_table=both(d.ori_block_table),
                         cu_q=torch.tensor([0, live, live], dtype=torch.int32, device="cuda"),
                         seq_lens=torch.tensor([length, 0], dtype=torch.int32, device="cuda"), sink=d.sink, cmp=d.cmp,
                         cmp_block_table=both(d.cmp_block_table), cmp_indices=None, ratio=ratio, window=d.window,
                         softmax_scale=d.softmax_scale)
    op = PreparedAttention(whole, made.ori_scale, made.cmp_scale)
    assert op.splits == 1
    fill = torch.empty_like(op.out[live:])
    took, alone, zero = microseconds(op.run), microseconds(eager.run), microseconds(fill.zero_)
    print(f"[padded] ratio {ratio}, {live} of {capacity} at {length}: {took:.1f} us, eager {alone:.1f}, fill {zero:.1f}",
          file=sys.stderr, flush=True)
    assert took <= 1.5 * (alone + zero)


def test_chunk_with_decode_requests_takes_the_time_of_its_parts():
    """2048 window-only tokens, 64 of them requests of one token: octets would
    need a second round for those (1.18 times the two parts' own launches, here
    0.98)."""
    from npu_sparse_attn_sharedkv_int8 import PreparedAttention
    parts = [([1] * 64, list(range(1000, 1000 + 64 * 400, 400))), ([1984], [32768])]
    whole = tuple(parts[0][i] + parts[1][i] for i in range(2))
    times = []
    for queries, lengths in (whole, *parts):
        made = DeviceCase(95, 1, queries, lengths)
        op = PreparedAttention(made.dev, made.ori_scale, made.cmp_scale)
        times.append(microseconds(op.run))
    print(f"[padded] mixed: {times[0]:.1f} us, its parts {times[1]:.1f} and {times[2]:.1f}", file=sys.stderr, flush=True)
    assert times[0] <= 1.1 * (times[1] + times[2])
