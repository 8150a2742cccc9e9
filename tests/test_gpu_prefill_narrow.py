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
from tests.helpers import (ROUTE_NARROW_PAIRS, ROUTE_NARROW_TILES, ROUTE_PAIR, ROUTE_WIDE,
                           assert_bar, bf16_route, bf16_to_f32, compare_bf16, make_prefill_case,
                           seeded_bf16)

pytestmark = pytest.mark.gpu

EDGES = ([0, 14, 15, 47, 62, 63, 64, 126, 127, 128, 200, 255], [2, 1, 2, 17, 1, 1, 16, 1, 33, 1, 5, 3])
# 40 sequences of one to three tokens: more blocks than CUs at 8 kv heads.
MANY = ([(37 * i) % 290 for i in range(40)], [1 + i % 3 for i in range(40)])
MIXED = ([700, 31, 530, 1], [90, 1, 1, 1])
# Enough rows for whole query blocks (64 tokens on two waves per row group).
BLOCKS = ([0, 63, 130, 14, 200], [64, 65, 70, 50, 1])
LONG = ([0, 63, 330], [700, 65, 300])


def _check(head_dim, nkv, page_len, shape, label, gap=0, scale=None, kernel=None):
    """gap: elements between a cache row's heads and the next row.  scale: of the
    queries.  kernel: the one that the plan has to take."""
    prefix, new = shape
    nq = nkv * (2 if head_dim == 256 else 8)
    width = nkv * head_dim
    kvs = width + gap
    case = make_prefill_case(head_dim + nkv + page_len, prefix, new, page_len=page_len)
    n = sum(new)
    q = seeded_bf16(n * nq * head_dim, 1)
    if scale:
        q = oracle.f32_to_bf16((bf16_to_f32(q) * np.float32(scale)).ravel())
    k, v = (seeded_bf16(case.cache_rows * kvs, s).reshape(-1, kvs) for s in (2, 3))
    used = np.zeros(case.cache_rows, dtype=bool)
    for pages, p, m in zip(case.pages, prefix, new):
        rows = np.concatenate([np.arange(page_len) + g * page_len for g in pages])[:p + m]
        used[rows] = True
    k_dev, v_dev = k.copy(), v.copy()
    for x in (k_dev, v_dev):
        x[~used] = 0x7FC0
        x[:, width:] = 0x7FC0
    table = KVRunTable()
    for r in case.runs:
        table.begin_run(int(r[0]), int(r[1]))
        for j in range(int(r[3])):
            table.add_base_row(int(case.base_rows[int(r[2]) + j]))
    plan = AttentionPlan(table, n, kind=FULL, window=0, cache_size=page_len, page_len=page_len,
                         cache_rows=case.cache_rows, cap=4, kv_row_bytes=kvs * 2)
    assert plan.summary.mode == 2 and int(plan.info[14]) > 0
    if kernel is not None:
        assert bf16_route(plan, nq, nkv, head_dim, kvs)[0] == kernel
    out = empty_dev(n * nq * head_dim, np.uint16)
    partials, ps = A.partials_buffer(plan, nq, head_dim)
    A.attention_bf16(plan, to_dev(q), to_dev(k_dev), to_dev(v_dev), out, partials, ps, num_q=nq,
                     num_kv=nkv, head_dim=head_dim, kv_stride=kvs)
    ref = oracle.attention(FULL, case.runs, case.base_rows, q, k.ravel(), v.ravel(), num_q=nq,
                           num_kv=nkv, head_dim=head_dim, kv_stride=kvs, window=0,
                           cache_size=page_len, page_len=page_len, seq_len=n, cap=4, threads=16)
    assert_bar(compare_bf16(from_dev(out, np.uint16), ref), label)


@pytest.mark.parametrize("head_dim,nkv,page_len,shape", [
    (256, 8, 64, EDGES), (256, 8, 16, EDGES), (256, 8, 1024, MIXED), (256, 1, 64, MIXED),
    (256, 3, 32, EDGES), (256, 8, 64, MANY), (256, 8, 16, MANY), (512, 2, 64, EDGES),
    (512, 2, 16, MIXED), (512, 3, 1024, EDGES), (512, 1, 64, MANY), (256, 32, 16, BLOCKS),
    (256, 32, 1024, BLOCKS), (256, 8, 64, LONG)])
def test_prefill_few_rows(head_dim, nkv, page_len, shape):
    announce(f"few-row prefill d={head_dim} kv={nkv} page={page_len} runs={len(shape[0])}")
    _check(head_dim, nkv, page_len, shape, "few-row prefill")


# More query blocks than a wave looks through at once (64), a chunk among them.
CROWD = ([(29 * i) % 90 for i in range(150)], [200 if i == 77 else 1 + i % 3 for i in range(150)])
TILED = ([400, 20, 900], [300, 130, 170])
WIDE = ([0, 900, 100], [400, 350, 400])
WIDE3 = ([0, 300, 150, 70], [300, 129, 240, 31])


@pytest.mark.parametrize("head_dim,nkv,page_len,shape,gap,scale,kernel", [
    (256, 8, 64, EDGES, 8, None, ROUTE_NARROW_PAIRS), (256, 8, 64, MIXED, 0, 1 / 16, ROUTE_NARROW_PAIRS),
    (256, 8, 32, MANY, 64, None, ROUTE_NARROW_TILES), (256, 8, 64, TILED, 0, 1 / 16, ROUTE_NARROW_TILES),
    (256, 8, 64, CROWD, 0, None, ROUTE_NARROW_TILES), (256, 1, 16, CROWD, 0, None, ROUTE_NARROW_PAIRS),
    (256, 8, 64, LONG, 8, None, ROUTE_PAIR), (256, 8, 64, LONG, 0, 1 / 16, ROUTE_PAIR),
    (512, 2, 64, EDGES, 8, None, ROUTE_NARROW_TILES), (512, 2, 64, MIXED, 0, 1 / 16, ROUTE_NARROW_TILES),
    (512, 1, 32, CROWD, 0, None, ROUTE_NARROW_TILES), (512, 3, 64, WIDE3, 0, None, ROUTE_WIDE),
    (512, 2, 1024, WIDE, 0, None, ROUTE_WIDE), (512, 2, 64, WIDE, 8, 1 / 16, ROUTE_WIDE)])
def test_prefill_kernels(head_dim, nkv, page_len, shape, gap, scale, kernel):
    """Each kernel that a full-attention plan over pages of 16 rows and more can take,
    by name: cache rows wider than their heads (the rest NaN), and queries scaled by
    1/16, whose attention spreads over many keys (most tiles without lo parts)."""
    label = f"kernel {kernel} d={head_dim} kv={nkv} page={page_len} runs={len(shape[0])}"
    announce(label)
    _check(head_dim, nkv, page_len, shape, label, gap=gap, scale=scale, kernel=kernel)
