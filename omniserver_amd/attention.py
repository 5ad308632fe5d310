"""Host side of the pool attention kernels (decode split-K and packed causal prefill).

``prefill_attention_pool`` is the varlen causal attention of the packed prefill
(omniserve/cache/kv_prealloc.py:181-203) over K/V already written to the pool: the host
cuts every segment into query blocks of consecutive tokens and picks a kernel by the number
of workgroups and the longest context (``prefill_plan``):

* omni_prefill_attention_rows, nearly everywhere: a workgroup takes one KV head's (token,
  query head) rows of a block in 32-row tiles, (rows, key groups) = (128, 1), (128, 2),
  (64, 4) or (32, 8): fewer rows per workgroup and more key groups the fewer rows there are;
* omni_prefill_attention_split (<= 16-token blocks, one (block, query head) item per
  workgroup, its key tiles split over four waves) for the shortest contexts, where the rows
  kernel's longer start and merge show;
* omni_prefill_attention (one wave per item) and its split form, whose accesses ask for no
  alignment, for what the rows kernel does not take: more than 32 query heads per KV head,
  a scale that is not a positive normal fp32, operands off a 16-byte boundary.

MI355X, 12 heads / 2 KV heads, us per launch, rows (128, 1) / (128, 2) / (64, 4) / (32, 8),
then the best of the per-wave, split and shared-tile kernels: one 4096-token prompt 86.8 /
69.4 / 90.3 / 123.7, 193; 1 x 2048 43.2 / 34.9 / 29.1 / 42.8, 98.5; 1 x 1024 24.1 / 20.5 /
16.1 / 17.8, 31.7; 1 x 512 14.7 / 13.4 / 10.9 / 9.3, 13.8; 1 x 256 9.8 / 10.0 / 8.5 / 7.5,
6.5; 2 x 2048 54.8 / 39.7 / 56.5 / 81.8, 105; 4 x 1024 33.5 / 33.5 / 40.4 / 60.0, 59; 8 x 512
22.6 / 24.4 / 32.8 / 48.7, 37; 16 x 256 16.6 / 20.0 / 28.4 / 43.8, 26; 64 x 64 11.6 / 16.9 /
24.7 / 40.4, 12.7; 4 x 256 10.2 / 10.3 / 8.8 / 13.3, 12.4; 16 x 24 6.5 / 7.7 / 6.8 / 6.7, 4.5;
a 256-token chunk at 1792 keys 42.4 / 33.9 / 25.9 / 19.3, 22.5; a 1024-token chunk at 3000
keys 78.3 / 61.0 / 46.4 / 56.1, 107; 32 single tokens at 2048 keys 40.8 / 33.1 / 27.1 / 21.0,
42.
"""

from __future__ import annotations

import operator
from array import array

import torch

from ._lib import call, lib, ptr, stream

QBLOCK = 16
# blocks of the shared-tile entry points, kept for callers of the C header alone
QBLOCK_GQA = 32
# the rows kernel's most query heads per KV head
ROWS_MAX_GROUP = 32
# (block, head) items per CU up to which the split kernel, not the per-wave one, runs
SPLIT_ITEMS_PER_CU = 4


_CUS = {}


def num_cus(device) -> int:
    if device not in _CUS:
        _CUS[device] = torch.cuda.get_device_properties(device).multi_processor_count
    return _CUS[device]


def query_blocks(seg_lengths, device, block: int = QBLOCK) -> torch.Tensor:
    """int32 [nqb, 2] (first token, count) covering every segment in blocks of <= block.  On a
    new batch this is part of the first layer's call, so the table is filled natively, straight
    into the staging buffer."""
    device = torch.device(device)
    most = sum(seg_lengths) // block + len(seg_lengths)
    host = torch.empty(most, 2, dtype=torch.int32, pin_memory=device.type == "cuda")
    lens = array("i", seg_lengths)
    n = lib().omni_query_blocks(lens.buffer_info()[0], len(lens), block, host.data_ptr(), most)
    if n < 0:
        raise ValueError(f"segments {list(seg_lengths)} in blocks of {block}")
    return host[:n].to(device, non_blocking=True)


def _blocks_fit(seg_lengths, tokens: int, block: int, most: int) -> bool:
    """Whether blocks of at most block tokens cover the segments (tokens in all) in at most
    most of them; counted only where the sum and number of segments leave it open."""
    if -(-tokens // block) > most:
        return False
    if tokens // block + len(seg_lengths) <= most:
        return True
    return sum([-(-L // block) for L in seg_lengths]) <= most


def prefill_plan(seg_lengths, starts, nh: int, nkv: int, cus: int) -> tuple:
    """(entry point, tokens per query block, extra arguments) for segments of seg_lengths
    tokens appended at starts, in 16-byte aligned tensors (see the module docstring for what
    each form measures)."""
    group = nh // nkv
    if group > ROWS_MAX_GROUP:
        return fallback_plan(seg_lengths, nh, cus)
    tokens = sum(seg_lengths)
    keys = max(map(operator.add, starts, seg_lengths), default=0)
    items_fit = lambda most: _blocks_fit(seg_lengths, tokens, QBLOCK, most // nh)
    wgs_fit = lambda rows, most: _blocks_fit(seg_lengths, tokens, rows // group, most // nkv)
    # Short contexts: the split kernel starts and merges in 1-2.5 us less until its items queue
    # or its four waves' key steps add up, sooner for blocks of few rows, of which the rows
    # kernel wastes less.  Us, split / rows, 12 / 2 heads: 16 tokens at 64 keys 4.2 / 6.3, 320
    # 7.2 / 8.4, 600 9.4 / 9.9, 800 11.6 / 11.5; one token at 64 4.5 / 5.2, 256 6.3 / 6.0, 420
    # 8.4 / 7.6; 256 tokens at 600 9.8 / 10.2; without grouping (16 / 16) 128 at 420 8.5 / 9.3,
    # 600 11.4 / 10.5.  Two rounds of items: 8 x 64 4.8 / 6.6, 4 x 128 6.3 / 6.9, 4 x 128 at 320
    # 10.4 / 8.7; 32 single tokens at 64 4.8 / 5.3, 80 6.0 / 5.6.  Three: 8 x 100 8.9 / 7.2.
    full = max(seg_lengths, default=0) * group >= 32
    if ((keys <= (320 if not full else 640 if group > 1 else 448) and items_fit(cus))
            or (keys <= (128 if full else 64) and items_fit(2 * cus))):
        return ("omni_prefill_attention_split", QBLOCK, ())
    # Rows to spare for every CU only in 128s: fewer rows per workgroup while those still fit
    # one round of the CUs, with the keys dealt to as many groups as the waves allow.  A long
    # context takes 64 rows also where they are more than one round but 128 would leave CUs
    # idle: the last blocks' chain of key tiles is what counts (1 x 2048: 29.1 against 34.9).
    if wgs_fit(32, cus):
        form = (32, 8)
    elif wgs_fit(64, cus) or (keys >= 1024 and wgs_fit(128, cus - 1)):
        form = (64, 4)
    elif keys > 1024 and wgs_fit(128, 4 * cus - 1):
        form = (128, 2)      # 2 x 2048: 39.7 against 54.8 us in one group
    else:
        form = (128, 1)      # short chains, or workgroups enough: 8 x 512 22.6 against 24.4
    return ("omni_prefill_attention_rows", form[0] // group, form)


def fallback_plan(seg_lengths, nh: int, cus: int) -> tuple:
    """The kernels that take any head grouping, scale sign and operand alignment."""
    split = _blocks_fit(seg_lengths, sum(seg_lengths), QBLOCK, SPLIT_ITEMS_PER_CU * cus // nh)
    return ("omni_prefill_attention_split" if split else "omni_prefill_attention", QBLOCK, ())


def prefill_attention_pool(writer, q: torch.Tensor, layer_idx: int, scale: float,
                           out: torch.Tensor, q_stride: int | None = None) -> torch.Tensor:
    """Causal attention of the writer's packed tokens over their pool rows."""
    pool = writer.pool
    nh = pool.n_heads
    plans = getattr(writer, "_attn_plan", None)
    if plans is None:
        plans = writer._attn_plan = {}
    qp, op = q.data_ptr(), out.data_ptr()
    # also a scale that fp32 does not hold as a normal number, which the rows kernel refuses
    plain = bool((qp | op) & 15) or not scale >= 2.0 ** -126
    plan = plans.get(plain)
    if plan is None:
        cus = num_cus(q.device)
        if plain:
            fn, block, extra = fallback_plan(writer.seg, nh, cus)
        else:
            fn, block, extra = prefill_plan(writer.seg, writer.starts, nh, pool.n_kv_heads, cus)
        plan = plans[plain] = (fn, query_blocks(writer.seg, q.device, block), extra)
    fn, qb, extra = plan
    call(fn, qp, q_stride or q.stride(0), ptr(pool.k[layer_idx]),
         ptr(pool.v[layer_idx]), pool.max_batch, pool.max_len, ptr(writer.token_slot),
         ptr(writer.kv_len), ptr(qb), qb.shape[0], op, nh * pool.head_dim, nh,
         pool.n_kv_heads, pool.head_dim, float(scale), *extra, stream())
    return out
