"""The output division at numerators so small (below 2^-102) that a quotient
corrected by its FMA residual is no longer correctly rounded: every kernel that
divides, bit-exact with the oracle, which divides.

Q is zero, so that every key has weight 1 and a head's denominator is the row's
number of keys and its sink's exponential.  The V codes are 1 and the compressed
ones 0, so that the numerator is the number of window keys times the channel's
scale, and the scales are ones for which the residual form, evaluated here,
gives another BF16 value than the division for some head of the first row."""
import sys

import numpy as np
import pytest

from tests import workloads
from tests.device_cases import joint_flags, run_hip, run_oracle

pytestmark = pytest.mark.gpu

F32 = np.float32


def by_residual(num, den):
    """num / den from the rounded reciprocal, its product and the FMA residual."""
    r = (F32(1) / den).astype(F32)
    q = (num * r).astype(F32)
    wide = np.float64
    e = (wide(num) - wide(q) * wide(den)).astype(F32)     # exact in FP64, rounded as the FMA does
    return (wide(q) + wide(e) * wide(r)).astype(F32)


def numerator(window_keys, scale):
    """The kernels' FP32 value: P and V codes x channel scale x 1/127."""
    return F32(127 * window_keys) * scale * F32(1 / 127)


def bits(x):
    return workloads.bf16_bits(x.astype(F32))


def sensitive_scales(rng, window_keys, dens, share=64):
    """512 channel scales, at least `share` of which tell the two quotients
    apart at one of the denominators: numerators near the middle between two
    BF16 results."""
    found, spare = [], None
    for _ in range(40):
        n = 1 << 18
        den = rng.choice(dens, n)
        result = ((bits(2.0 ** rng.uniform(-137, -120, n)).astype(np.uint32) << 16) | 0x8000).view(F32)
        near = (result.astype(np.float64) * den / window_keys).astype(F32).view(np.int32) + rng.integers(-4, 5, n)
        scale = near.astype(np.int32).view(F32)
        num = numerator(window_keys, scale)
        hit = bits(by_residual(num, den)) != bits(num / den)
        found.extend(scale[hit])
        spare = scale
        if len(found) >= workloads.DIM:
            break
    assert len(found) >= share
    return np.concatenate([np.array(found, F32), spare])[:workloads.DIM]


CASES = [
    # name, ratio, requests, tokens of each, length, heads, partitions
    ("one_row_a_work_group", 1, 7, 1, 1, 8, 1),
    ("rows", 1, 300, 1, 1, 8, 1),                    # c8_rows
    ("rows_of_sixteen", 1, 150, 1, 1, 16, 1),
    ("rows_c4", 4, 3, 100, 700, 8, 1),
    ("octets", 1, 1, 1100, 1100, 8, 1),              # c8_chunk
    ("octets_c128", 128, 1, 800, 800, 8, 1),
    ("two_partitions", 4, 1, 3, 1500, 8, 2),
    ("nine_partitions", 4, 1, 3, 4500, 8, 9),
    ("grouped", 4, 1, 8, 4500, 8, 3),
]


@pytest.mark.parametrize("name,ratio,requests,tokens,length,heads,splits", CASES, ids=[c[0] for c in CASES])
def test_tiny_numerators(name, ratio, requests, tokens, length, heads, splits):
    rng = np.random.default_rng(99)
    case = workloads.make_case(99, ratio, [tokens] * requests, [length] * requests, heads=heads)
    case["q"][:] = 0
    case["sink"][:] = -3 - np.arange(heads) * F32(0.21)
    position = length - tokens
    window_keys = min(position + 1, 128)
    listed = {1: 0, 4: min((position + 1) // 4, 1024), 128: (position + 1) // 128}[ratio]
    dens = np.exp(case["sink"].astype(np.float64)).astype(F32) + F32(window_keys) + F32(listed)
    scale = sensitive_scales(rng, window_keys, dens)
    case["ori"].pool[:] = 1
    case["ori"].scale[:] = scale
    if case["cmp"] is not None:
        case["cmp"].pool[:] = 0
    print(f"[division] {name}", file=sys.stderr, flush=True)
    group = 2 if name == "grouped" else None
    out, lse, op = run_hip(case, splits=splits, query_group=group)
    ref, ref_lse, _ = run_oracle(case, op.device_splits(), joint=joint_flags(case, splits), query_group=group or 1,
                                 tile=op.tile_size if group else 128)
    # The oracle's first row holds these quotients, and the residual form's are others.
    num = numerator(window_keys, scale)
    assert (ref[0] == bits(num / dens[:, None])).all()
    assert (ref[0] != bits(by_residual(num, dens[:, None]))).sum() >= 64
    assert (out == ref).all()
    np.testing.assert_allclose(lse, ref_lse, rtol=0, atol=2e-6)
