"""GPU parity of the full-attention prefill for few query rows (32 rows shared
by the four waves of a block; FlashPrefillFullKernel + PrefillMergeKernel,
kernels/flash_attention_prefill.mojo:117-248) against the oracle's
token-partitioned route, within 1e-2 (one bf16 spacing where |x| >= 2): key
counts around the tile (16) and iteration (64, 128) edges, blocks of one to all
live rows, tokens decoding beside a chunk, page sizes down to one tile, kv head
counts that do and do not divide the XCDs.  The cache rows past each sequence's
last key hold NaN: nothing may read a value from them."""
import numpy as np
import pytest

import oracle
from inferno_amd import attention as A
from inferno_amd.kv import FULL, AttentionPlan, KVRunTable
from tests.gpu_util import announce, empty_dev, from_dev, to_dev
from tests.helpers import assert_bar, compare_bf16, make_prefill_case, seeded_bf16

pytestmark = pytest.mark.gpu

EDGES = ([0, 14, 15, 47, 62, 63, 64, 126, 127, 128, 200, 255], [2, 1, 2, 17, 1, 1, 16, 1, 33, 1, 5, 3])
# 40 sequences of one to three tokens: more blocks than CUs at 8 kv heads.
MANY = ([(37 * i) % 290 for i in range(40)], [1 + i % 3 for i in range(40)])
MIXED = ([700, 31, 530, 1], [90, 1, 1, 1])
# Enough rows for whole query blocks (64 tokens on two waves per row group).
BLOCKS = ([0, 63, 130, 14, 200], [64, 65, 70, 50, 1])
LONG = ([0, 63, 330], [700, 65, 300])


@pytest.mark.parametrize("head_dim,nkv,page_len,shape", [
    (256, 8, 64, EDGES), (256, 8, 16, EDGES), (256, 8, 1024, MIXED), (256, 1, 64, MIXED),
    (256, 3, 32, EDGES), (256, 8, 64, MANY), (256, 8, 16, MANY), (512, 2, 64, EDGES),
    (512, 2, 16, MIXED), (512, 3, 1024, EDGES), (512, 1, 64, MANY), (256, 32, 16, BLOCKS),
    (256, 32, 1024, BLOCKS), (256, 8, 64, LONG)])
def test_prefill_few_rows(head_dim, nkv, page_len, shape):
    announce(f"few-row prefill d={head_dim} kv={nkv} page={page_len} runs={len(shape[0])}")
    prefix, new = shape
    nq = nkv * (2 if head_dim == 256 else 8)
    kvs = nkv * head_dim
    case = make_prefill_case(head_dim + nkv + page_len, prefix, new, page_len=page_len)
    n = sum(new)
    q = seeded_bf16(n * nq * head_dim, 1)
    k, v = (seeded_bf16(case.cache_rows * kvs, s).reshape(-1, kvs) for s in (2, 3))
    used = np.zeros(case.cache_rows, dtype=bool)
    for pages, p, m in zip(case.pages, prefix, new):
        rows = np.concatenate([np.arange(page_len) + g * page_len for g in pages])[:p + m]
        used[rows] = True
    k_dev, v_dev = k.copy(), v.copy()
    k_dev[~used] = 0x7FC0
    v_dev[~used] = 0x7FC0
    table = KVRunTable()
    for r in case.runs:
        table.begin_run(int(r[0]), int(r[1]))
        for j in range(int(r[3])):
            table.add_base_row(int(case.base_rows[int(r[2]) + j]))
    plan = AttentionPlan(table, n, kind=FULL, window=0, cache_size=page_len, page_len=page_len,
                         cache_rows=case.cache_rows, cap=4, kv_row_bytes=kvs * 2)
    assert plan.summary.mode == 2 and int(plan.info[14]) > 0
    out = empty_dev(n * nq * head_dim, np.uint16)
    partials, ps = A.partials_buffer(plan, nq, head_dim)
    A.attention_bf16(plan, to_dev(q), to_dev(k_dev), to_dev(v_dev), out, partials, ps, num_q=nq,
                     num_kv=nkv, head_dim=head_dim, kv_stride=kvs)
    ref = oracle.attention(FULL, case.runs, case.base_rows, q, k.ravel(), v.ravel(), num_q=nq,
                           num_kv=nkv, head_dim=head_dim, kv_stride=kvs, window=0,
                           cache_size=page_len, page_len=page_len, seq_len=n, cap=4, threads=16)
    assert_bar(compare_bf16(from_dev(out, np.uint16), ref), "few-row prefill")
