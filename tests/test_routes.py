"""Which kernel a full-attention token plan or an o_proj batch takes, and with how many
workgroups (host rules; no GPU is touched)."""
import ctypes as C

import numpy as np
import pytest

from inferno_amd._lib import I64, P_I64, lib
from inferno_amd.kv import FULL, AttentionPlan, KVRunTable
from tests.helpers import (ROUTE_FULL, ROUTE_NARROW_PAIRS, ROUTE_NARROW_TILES, ROUTE_PAIR,
                           ROUTE_WIDE, bf16_route, make_prefill_case)


def token_plan(prefix, new, page_len=64, num_kv=8, head_dim=256):
    case = make_prefill_case(1, prefix, new, page_len=page_len)
    table = KVRunTable()
    for r in case.runs:
        table.begin_run(int(r[0]), int(r[1]))
        for j in range(int(r[3])):
            table.add_base_row(int(case.base_rows[int(r[2]) + j]))
    return AttentionPlan(table, sum(new), kind=FULL, window=0, cache_size=page_len,
                         page_len=page_len, cache_rows=case.cache_rows, cap=1,
                         kv_row_bytes=num_kv * head_dim * 2, device="cpu")


def live_blocks(new, num_kv, tokens):
    return num_kv * sum(-(-n // tokens) for n in new)


@pytest.mark.parametrize("head_dim,num_kv,gqa,tokens", [(256, 8, 2, 16), (256, 1, 2, 16),
                                                        (512, 2, 8, 4), (512, 1, 8, 4)])
def test_narrow_workgroups_are_those_with_tokens(head_dim, num_kv, gqa, tokens):
    """A workgroup without tokens looks for some through the whole plan: of many
    sequences of one token each, there may be none."""
    new = [1] * 500 + [32]
    plan = token_plan([30] * 501, new, num_kv=num_kv, head_dim=head_dim)
    kernel, blocks = bf16_route(plan, num_kv * gqa, num_kv, head_dim)
    assert kernel in (ROUTE_NARROW_TILES, ROUTE_NARROW_PAIRS)
    assert blocks == live_blocks(new, num_kv, tokens)


@pytest.mark.parametrize("head_dim,num_kv,gqa,tokens", [(256, 8, 2, 16), (512, 2, 8, 4)])
def test_narrow_workgroups_cover_every_token(head_dim, num_kv, gqa, tokens):
    rng = np.random.default_rng(head_dim)
    seen = 0
    for _ in range(60):
        n = int(rng.integers(1, 40))
        new = [int(x) for x in np.ceil(2.0 ** rng.uniform(0, 7, n))]
        kernel, blocks = bf16_route(token_plan([5] * n, new, num_kv=num_kv, head_dim=head_dim),
                                    num_kv * gqa, num_kv, head_dim)
        if kernel not in (ROUTE_NARROW_TILES, ROUTE_NARROW_PAIRS):
            continue
        seen += 1
        live = live_blocks(new, num_kv, tokens)
        # Every run may end in a partial block; no more than that is added.
        assert live <= blocks <= live + num_kv * n
    assert seen > 20


def test_a_tie_goes_to_the_query_blocks():
    plan = token_plan([25] * 300, [20] * 300, num_kv=1)
    assert bf16_route(plan, 2, 1, 256) == (ROUTE_PAIR, 0)


@pytest.mark.parametrize("top,block_size,blocks", [(0, 64, 1), (63, 64, 1), (64, 64, 2), (199, 128, 2),
                                                   (131071, 128, 1024)])
def test_index_waves_end_with_the_longest_context(top, block_size, blocks):
    """The scores' rows are padded to 16 blocks; the padding gets no waves."""
    plan = token_plan([0, top], [1, 1], page_len=128)
    fn = lib().ifr_internal_index_blocks
    fn.restype, fn.argtypes = C.c_int64, [P_I64, I64]
    assert fn(plan.info_ptr, block_size) == blocks
    assert lib().ifr_index_scores_bytes(plan.info_ptr, 4, block_size) == 2 * 4 * 4 * (-(-blocks // 16) * 16)


def gemm_plan(rows, cols, seq_len, workspace_bytes):
    fn = lib().ifr_internal_gemm_plan
    fn.restype, fn.argtypes = None, [I64, I64, I64, I64, P_I64]
    plan = (C.c_int64 * 3)()
    fn(rows, cols, seq_len, workspace_bytes, plan)
    return tuple(plan)


def test_the_gemm_tests_cover_every_tile_kernel():
    from tests.test_gpu_gemm import TILE_CASES

    for (seq, rows, cols), plan in TILE_CASES.items():
        bytes_ = lib().ifr_gemm_cols_workspace_bytes(rows, cols, seq)
        assert gemm_plan(rows, cols, seq, bytes_) == plan, (seq, rows, cols)
        assert bytes_ == (plan[2] * seq * rows * 4 if plan[2] > 1 else 0)
    shapes = [(64, 64), (128, 64), (128, 128), (192, 128), (256, 128)]
    assert {(m, n, s > 1) for m, n, s in TILE_CASES.values()} == {
        (m, n, split) for m, n in shapes for split in (False, True)}


@pytest.mark.parametrize("seq,cols,slices", [(1, 4096, 16), (16, 256, 1), (16, 4096, 16), (16, 4608, 9),
                                             (1, 8192, 16), (17, 4096, 8), (64, 8192, 16)])
def test_decode_batches_slice_k(seq, cols, slices):
    """Slices of 256 up to 16 tokens and k of 4,096 (joined in the workgroup, no
    workspace), of 512 past either."""
    assert gemm_plan(2816, cols, seq, 1 << 40) == (0, 0, slices)
    joined = seq <= 16 and cols <= 4096
    assert lib().ifr_gemm_cols_workspace_bytes(2816, cols, seq) == (0 if joined else slices * seq * 2816 * 4)


@pytest.mark.parametrize("page_len,kv_stride", [(8, None), (64, (1 << 25) + 8)])
def test_small_pages_and_wide_rows_take_the_query_blocks(page_len, kv_stride):
    """A tile that may leave its page, and row offsets past 32 bits, stay with the
    kernels that look every row up."""
    for new in ([1, 40], [700, 300]):
        plan = token_plan([100, 100], new, page_len=page_len)
        assert bf16_route(plan, 16, 8, 256, kv_stride) == (ROUTE_FULL, 0)
        assert bf16_route(plan, 16, 2, 512, kv_stride) == (ROUTE_WIDE, 0)
