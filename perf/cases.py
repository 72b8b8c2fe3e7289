"""Performance cases of the shared-KV INT8 path: what a serving program has it do.

A case is a dict of plain values.  prepare() makes the inputs on the GPU from
a seed and the operator that a serving program keeps (PreparedAttention or
PreparedCacheWrite); run() is one pass through it; exact() is the same
attention in 64 bits in plain torch.

Attention cases
  ratio 1, 4 or 128        window-only, C4 top-k or C128 layer
  batch, q_lo, q_hi        requests, and the query tokens of each (spread over
                           q_lo .. q_hi): 1-4 in decode (main and draft
                           tokens), hundreds to thousands in a prefill chunk
  ctx_lo, ctx_hi           sequence lengths, new tokens included, spread evenly
  capacity                 query tokens of the launch when it is replayed at a
                           graph's capacity (0: the live tokens); the requests
                           past `batch` are empty (capacity_batch in all)
  heads                    8 per GPU under tensor parallelism; 16 to 64 where
                           attention is sharded less or not at all
  topk, sorted             C4 list length, and whether it comes in index or in
                           score order
  draft                    the original rows as explicit physical slots (the
                           draft layer's lists) in place of the window
  lse                      whether the log-sum-exp is asked for too
  layers                   16 KiB pages that share one page stride (the layers
                           of a serving pool; 38 of them at 622592 bytes)
Writer cases
  rows, pages, layers, int64, paired, skipped (share of rows with slot -1)
"""
import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
for _p in (ROOT, ROOT / "ascend-int8-attention_amd"):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

from npu_sparse_attn_sharedkv_int8 import PreparedAttention, PreparedCacheWrite, SharedKVCase  # noqa: E402

DIM, BLOCK, WINDOW = 512, 32, 128
PAGE = BLOCK * DIM
DEVICE = "cuda"
DRAFT_SLOTS = 256
MOST_TOKENS = 2048               # query tokens of a prefill launch at eight heads
MOST_DECODE = 700                # and of a decode launch
MOST_PAGES = 131072              # compressed pages of the largest pool


def attention(name, ratio, batch, q, ctx, *, heads=8, topk=1024, in_order=True, lse=False, draft=False, capacity=0,
              capacity_batch=0, layers=38):
    return dict(name=name, kind="attention", ratio=ratio, batch=batch, q_lo=q[0], q_hi=q[1], ctx_lo=ctx[0],
                ctx_hi=ctx[1], heads=heads, topk=topk if ratio == 4 else 0, sorted=in_order, lse=lse, draft=draft,
                capacity=capacity, capacity_batch=capacity_batch, layers=layers)


def listed():
    return [
        # A lone request's decode step on a C128 layer with a short context: the smallest call.
        attention("c128_decode_1x1", 128, 1, (1, 1), (4096, 4096)),
        # The same on a C4 layer (window and 1024 of 4096 compressed rows), with its LSE.
        attention("c4_decode_1x1", 4, 1, (1, 1), (16384, 16384), lse=True),
        # A batch of 32 requests with a main and a draft token each, mixed contexts: ordinary decode.
        attention("c4_decode_32x2", 4, 32, (2, 2), (2048, 65536)),
        # Long-context decode on a C128 layer: every compressed row of 64 requests.
        attention("c128_decode_64x1", 128, 64, (1, 1), (65536, 131072)),
        # A large decode batch on a C4 layer, lists in score order.
        attention("c4_decode_256x2", 4, 256, (2, 2), (2048, 65536), in_order=False, layers=3),
        # A draft layer's window-only step replayed at a graph's capacity of 48 requests, 31 of them live.
        attention("draft_decode_31of48", 1, 31, (2, 2), (1500, 65536), draft=True, capacity=96, capacity_batch=48),
        # Chunked prefill on a C4 layer: 2048 new tokens on a 30720-token prefix.
        attention("c4_prefill_2048", 4, 1, (2048, 2048), (32768, 32768)),
        # A ragged prefill batch on a C128 layer.
        attention("c128_prefill_ragged", 128, 3, (301, 1023), (9001, 50001)),
        # A window-only layer's prefill chunks.
        attention("window_prefill_ragged", 1, 2, (777, 1271), (2500, 32768)),
        # Sixteen heads per GPU (128 heads on eight GPUs): a C4 prefill chunk.
        attention("c4_prefill_16_heads", 4, 1, (1024, 1024), (16384, 16384), heads=16),
        # All 64 heads on one GPU (data-parallel attention): C4 decode.
        attention("c4_decode_64_heads", 4, 32, (1, 1), (8192, 65536), heads=64, lse=True),
        # One step's incremental cache write of a prefill chunk.
        dict(name="cache_write_4096", kind="write", rows=4096, pages=1024, layers=38, int64=False, paired=False,
             skipped=0.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a decode step, a prefill chunk, a wide-head launch, a
    draft layer's step or a cache write of sizes spread over the same ranges."""
    family = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "heads", "draft", "write"])
    if family == "write":
        rows = _log(rng, 1, 8192)
        return dict(kind="write", rows=rows, pages=max(4, rows // BLOCK * rng.choice([2, 4]) + rng.randint(0, 7)),
                    layers=rng.choice([1, 3, 38]), int64=rng.random() < 0.5, paired=rng.random() < 0.5,
                    skipped=rng.choice([0.0, 0.0, 0.1]))
    ratio = 1 if family == "draft" else rng.choice([4, 4, 128] if family == "heads" else [4, 4, 4, 128, 128, 1])
    heads = rng.choice([16, 16, 32, 64]) if family == "heads" else rng.choice([8, 8, 8, 4])
    in_order, lse = rng.random() < 0.6, rng.random() < 0.3
    topk = rng.choice([1024, 1024, 1024, 512]) if ratio == 4 else 0
    capacity = capacity_batch = 0
    if family == "prefill" or (family == "heads" and rng.random() < 0.4):
        batch = rng.randint(1, 4)
        total = _log(rng, 180, MOST_TOKENS * 8 // max(8, heads))
        q_hi = max(1, total // batch)
        q_lo = max(1, q_hi - rng.randint(0, q_hi // 2))
        ctx_lo = q_hi + _log(rng, 1, 30000)
        ctx_hi = min(ctx_lo + _log(rng, 1, 30000), 65536)
        ctx_hi = max(ctx_lo, ctx_hi)
        layers = rng.choice([1, 3, 38])
    else:
        q_lo = q_hi = rng.choice([1, 2, 2, 3, 4])
        ctx_lo = _log(rng, 200, 65536)
        ctx_hi = min(131072, int(ctx_lo * rng.uniform(1.0, 8.0)))
        per_request = max(1, ctx_hi // 4 // BLOCK)
        batch = _log(rng, 1, max(1, min(256, MOST_DECODE // (q_hi * max(1, heads // 8)), MOST_PAGES // per_request)))
        layers = rng.choice([1, 3]) if batch * per_request > 4096 else rng.choice([1, 3, 38])
        if family != "heads" and rng.random() < 0.25:
            capacity_batch = batch + rng.randint(1, batch + 3)
            capacity = capacity_batch * q_hi
    return {k: v for k, v in attention("", ratio, batch, (q_lo, q_hi), (ctx_lo, ctx_hi), heads=heads, topk=topk,
                                       in_order=in_order, lse=lse, draft=family == "draft", capacity=capacity,
                                       capacity_batch=capacity_batch, layers=layers).items() if k != "name"}


def _spread(lo, hi, n, shift):
    """n whole numbers spread over lo .. hi (both met from two on), in a mixed order."""
    if n == 1:
        return [hi]
    ends = [lo + (hi - lo) * i // (n - 1) for i in range(n)]
    step = next(s for s in range(max(1, int(n * 0.618)), 2 * n + 2) if math.gcd(s, n) == 1)
    return [ends[(shift + i * step) % n] for i in range(n)]


def requests(case):
    """(query tokens, sequence lengths) of the live requests."""
    queries = _spread(case["q_lo"], case["q_hi"], case["batch"], 0)
    lengths = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"], case["batch"] // 3)
    return queries, [max(n, q) for q, n in zip(queries, lengths)]


def work(case):
    """Each cache row that some query of its sequence lists, Q, the lists, the
    table entries and the scales read once, outputs written once; one
    multiplication and addition per query, key, head and channel, in Q K and
    in P V."""
    if case["kind"] == "write":
        live = case["rows"] * (1 - case["skipped"])
        slot = (8 if case["int64"] else 4) * (2 if case["paired"] else 1)
        return {"bytes": live * 3 * DIM + case["rows"] * slot + 4 * DIM, "flops": 0}
    queries, lengths = requests(case)
    tokens = max(case["capacity"], sum(queries))
    rows = entries = keys = 0.0
    for q, n in zip(queries, lengths):
        positions = range(n - q, n)
        window = n - max(0, n - q + 1 - WINDOW)
        rows += window
        entries += window / BLOCK + 1
        listed_rows = unseen = 0.0
        if case["ratio"] == 128:
            listed_rows = n // 128
            keys += sum((p + 1) // 128 for p in positions)
        elif case["ratio"] == 4:
            unseen = 1.0
            for p in positions:
                count = (p + 1) // 4
                take = min(count, case["topk"])
                keys += take
                unseen *= 1 - take / count if count else 1
            listed_rows = n // 4 * (1 - unseen)
        rows += listed_rows
        entries += min(listed_rows, n / max(1, case["ratio"]) / BLOCK)
        keys += sum(min(n if case["draft"] else p + 1, WINDOW + (n - 1 - p if case["draft"] else 0)) for p in positions)
    lists = tokens * (case["topk"] + (DRAFT_SLOTS if case["draft"] else 0)) * 4
    q_out = tokens * case["heads"] * (DIM * 4 + (4 if case["lse"] else 0))
    return {"bytes": rows * DIM + entries * 4 + lists + q_out + DIM * 8, "flops": 4.0 * keys * case["heads"] * DIM}


def tolerance(case):
    """Cache codes are whole numbers: exact.  Attention quantises Q and the
    softmax weights to INT8 against maxima that depend on how a list is cut
    into tiles and partitions, and gives BF16: four times what 1, 2, 3 and 5
    partitions of the same launches differ by.  Up to eight heads the codes
    carry a residual (0.0007 of the norm, 0.016 at one value); above eight
    they do not (0.015, and more than one at single values)."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": 0.0028, "max": 0.064} if case["heads"] <= 8 else {"rel": 0.03, "max": 0.99}


def _pool(gen, pages, layers):
    """A pool of `pages` pages holding INT8 codes as calibrated scales give
    them (about normal, absmax below 127 / 1.1) at a stride of `layers` pages,
    its view of one layer and the layer's FP32 scales (16 outlier channels)."""
    stride = layers * PAGE
    flat = torch.zeros(pages * stride, dtype=torch.int8, device=DEVICE)
    blocks = flat.view(pages, stride)
    step = 4096
    for p in range(0, pages, step):
        n = min(step, pages - p)
        x = torch.randn((n, PAGE), generator=gen, device=DEVICE)
        blocks[p:p + n, :PAGE] = (x * 25.0).round_().clamp_(-127, 127).to(torch.int8)
    scale = (0.9 + 0.2 * torch.rand(DIM, generator=gen, device=DEVICE)) * (1.1 * 4.6 / 127)
    outliers = torch.randperm(DIM, generator=gen, device=DEVICE)[:16]
    scale[outliers] *= 8
    return flat.as_strided((pages, BLOCK, 1, DIM), (stride, DIM, DIM, 1)), scale


def _paged(gen, touched, width, layers, spare):
    """A pool and block table for requests that touch the logical pages
    touched[b] = (first, end): shuffled physical pages, a quarter more than
    needed, and `spare` empty requests in the table."""
    total = sum(end - first for first, end in touched)
    pages = max(1, math.ceil(1.25 * total))
    physical = torch.randperm(pages, generator=gen, device=DEVICE).to(torch.int32)
    table = torch.zeros((len(touched) + spare, max(1, width)), dtype=torch.int32, device=DEVICE)
    at = 0
    for b, (first, end) in enumerate(touched):
        table[b, first:end] = physical[at:at + end - first]
        at += end - first
    view, scale = _pool(gen, pages, layers)
    return view, table, scale


def _top_lists(gen, counts, topk, in_order):
    """Per query, topk distinct rows below its count (all of them and -1 past
    them where it has fewer), in index or random order."""
    most = int(counts.max())
    width = max(topk, most)
    out = torch.empty((len(counts), topk), dtype=torch.int32, device=DEVICE)
    step = max(1, (1 << 24) // width)
    for t in range(0, len(counts), step):
        c = counts[t:t + step, None]
        x = torch.rand((len(c), width), generator=gen, device=DEVICE)
        x = torch.where(torch.arange(width, device=DEVICE) < c, x, -1.0)
        score, ids = torch.topk(x, topk, dim=1)
        ids = torch.where(score >= 0, ids, width)
        if in_order:
            ids = ids.sort(dim=1).values
        out[t:t + step] = torch.where(ids < width, ids, -1)
    return out.view(len(counts), 1, topk)


def inputs(case, seed):
    """The SharedKVCase, its scales and the queries' positions and requests."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    queries, lengths = requests(case)
    live = sum(queries)
    tokens = max(case["capacity"], live)
    spare = max(0, case["capacity_batch"] - case["batch"])
    cu = [0]
    for q in queries:
        cu.append(cu[-1] + q)
    cu += [live] * spare
    owner = torch.repeat_interleave(torch.arange(len(queries)), torch.tensor(queries))
    position = torch.cat([torch.arange(n - q, n) for q, n in zip(queries, lengths)])
    q = torch.randn((tokens, case["heads"], DIM), generator=gen, device=DEVICE).bfloat16()
    ori_pages = [(max(0, n - k + 1 - WINDOW) // BLOCK, (n + BLOCK - 1) // BLOCK) for k, n in zip(queries, lengths)]
    ori, ori_table, ori_scale = _paged(gen, ori_pages, (max(lengths) + BLOCK - 1) // BLOCK, case["layers"], spare)
    ratio = case["ratio"]
    cmp = cmp_table = cmp_scale = lists = slots = None
    if ratio != 1:
        rows = [n // ratio for n in lengths]
        width = (max(rows) + BLOCK - 1) // BLOCK
        cmp, cmp_table, cmp_scale = _paged(gen, [(0, (r + BLOCK - 1) // BLOCK) for r in rows], width, case["layers"],
                                           spare)
    if ratio == 4:
        counts = torch.zeros(tokens, dtype=torch.int64)
        counts[:live] = (position + 1) // 4
        lists = _top_lists(gen, counts.to(DEVICE), case["topk"], case["sorted"])
    if case["draft"]:
        last = torch.tensor(lengths)[owner] - 1
        first = (position + 1 - WINDOW).clamp(min=0)
        row = first[:, None] + torch.arange(DRAFT_SLOTS)[None, :]
        there = row <= last[:, None]
        row = torch.where(there, row, last[:, None]).to(DEVICE)
        place = ori_table[owner.to(DEVICE)[:, None], row // BLOCK] * BLOCK + (row % BLOCK).int()
        slots = torch.full((tokens, 1, DRAFT_SLOTS), -1, dtype=torch.int32, device=DEVICE)
        slots[:live, 0] = torch.where(there.to(DEVICE), place, -1)
    as_int = dict(dtype=torch.int32, device=DEVICE)
    made = SharedKVCase(q=q, ori=ori, ori_block_table=ori_table, cu_q=torch.tensor(cu, **as_int),
                        seq_lens=torch.tensor(lengths + [0] * spare, **as_int),
                        sink=torch.linspace(-2, 2, case["heads"], device=DEVICE), cmp=cmp, cmp_block_table=cmp_table,
                        cmp_indices=lists, ratio=ratio, window=WINDOW, softmax_scale=1 / math.sqrt(DIM),
                        ori_indices=slots)
    return made, ori_scale, cmp_scale, position.to(DEVICE), owner.to(DEVICE)


def prepare(case, seed):
    if case["kind"] == "write":
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        cache, scale = _pool(gen, case["pages"], case["layers"])
        updates = (torch.randn((case["rows"], DIM), generator=gen, device=DEVICE) * (scale * 25.0)).bfloat16()
        slots = torch.randperm(case["pages"] * BLOCK, generator=gen, device=DEVICE)[:case["rows"]]
        skip = torch.rand(case["rows"], generator=gen, device=DEVICE) < case["skipped"]
        if case["paired"]:
            slots = torch.stack([slots // BLOCK, slots % BLOCK], 1)
            slots[skip] = -1
        else:
            slots = torch.where(skip, -1, slots)
        slots = slots.to(torch.int64 if case["int64"] else torch.int32)
        return PreparedCacheWrite(cache, updates, slots, (1.0 / scale.double()).float())
    made, ori_scale, cmp_scale, _, _ = inputs(case, seed)
    return PreparedAttention(made, ori_scale, cmp_scale, return_lse=case["lse"])


def run(state):
    out = state.run()
    if isinstance(state, PreparedAttention) and state.lse is not None:
        return {"out": out, "lse": state.lse}
    return {"out": out}


def exact(case, seed):
    """Softmax attention over the dequantised rows with the sink in the
    denominator, in 64 bits; padding queries are zero."""
    if case["kind"] == "write":
        return None
    made, ori_scale, cmp_scale, position, owner = inputs(case, seed)
    tokens, heads = made.q.shape[:2]
    out = torch.zeros((tokens, heads, DIM), dtype=torch.float64, device=DEVICE)
    lse = torch.zeros((tokens, heads), dtype=torch.float64, device=DEVICE)
    ratio = case["ratio"]
    most = int((position.max() + 1) // ratio) if ratio == 128 else 0
    live = len(position)
    sink = made.sink.double()[None, :, None]
    for t in range(0, live, 32):
        at, who = position[t:t + 32, None], owner[t:t + 32, None]
        if case["draft"]:
            slot = made.ori_indices[t:t + 32, 0][:len(at)].long()
            kinds = [(made.ori, ori_scale, slot >= 0, slot.clamp(min=0))]
        else:
            row = at + 1 - WINDOW + torch.arange(WINDOW, device=DEVICE)
            kinds = [(made.ori, ori_scale, row >= 0, _slots(made.ori_block_table, who, row.clamp(min=0)))]
        if ratio != 1:
            if ratio == 4:
                row = made.cmp_indices[t:t + 32, 0][:len(at)].long()
            else:
                row = torch.arange(most, device=DEVICE)[None, :].expand(len(at), most)
            there = (row >= 0) & (row < (at + 1) // ratio)
            kinds.append((made.cmp, cmp_scale, there, _slots(made.cmp_block_table, who, row.clamp(min=0))))
        rows = torch.cat([pool[slot // BLOCK, slot % BLOCK, 0].double() * scale.double()
                          for pool, scale, _, slot in kinds], 1)
        there = torch.cat([k[2] for k in kinds], 1)[:, None, :]
        q = made.q[t:t + 32][:len(at)].double()
        score = torch.matmul(q, rows.transpose(1, 2).contiguous()) * made.softmax_scale
        score = torch.where(there, score, -math.inf)
        score = torch.cat([sink.expand(len(at), heads, 1), score], 2)
        lse[t:t + len(at)] = torch.logsumexp(score, 2)
        out[t:t + len(at)] = torch.matmul(torch.softmax(score, 2)[:, :, 1:].contiguous(), rows)
    return {"out": out, "lse": lse} if case["lse"] else {"out": out}


def _slots(table, who, row):
    """Physical row of logical row `row` of request `who`."""
    page = (row // BLOCK).clamp(max=table.shape[1] - 1)
    return table[who, page].long() * BLOCK + row % BLOCK
