"""GPU parity of the o_proj GEMM after the attention (dispatch_gemm_cols,
kernels/gemm.mojo:198-225) through the C ABI: bit-exact on integer-valued
operands (exact sums), and within one bf16 spacing of the oracle on random
operands (the MFMA and VDPBF16PS add the same exact products in different
orders), at the decode shapes (split contraction) and multi-tile batches."""
import numpy as np
import pytest

import oracle
from inferno_amd import attention as A
from tests.gpu_util import announce, empty_dev, from_dev, to_dev
from tests.helpers import bf16_to_f32, bf16_ulp, compare_bf16

pytestmark = pytest.mark.gpu


def _bf(x) -> np.ndarray:
    return oracle.f32_to_bf16(np.asarray(x, dtype=np.float32).ravel())


def _run(xb, wb, seq, rows, cols) -> np.ndarray:
    out = empty_dev(max(seq * rows, 1), np.uint16)
    ws = A.gemm_cols_workspace(rows, cols, seq)
    A.dispatch_gemm_cols(to_dev(xb), to_dev(wb), out, rows=rows, cols=cols, seq_len=seq,
                         workspace=ws)
    return from_dev(out, np.uint16)[:seq * rows].reshape(seq, rows)


@pytest.mark.parametrize("seq,rows,cols", [(1, 2816, 4096), (64, 2816, 4096), (20, 80, 1024),
                                           (40, 2816, 512), (5, 48, 256), (130, 320, 512),
                                           (200, 192, 4096), (3, 64, 8192), (16, 32, 384)])
def test_gemm_cols_matches_oracle(seq, rows, cols):
    announce(f"gemm_cols seq={seq} rows={rows} cols={cols}")
    rng = np.random.default_rng(seq * 7 + rows)
    xb = _bf(rng.standard_normal((seq, cols)) * 0.5)
    wb = _bf(rng.standard_normal((rows, cols)) * 0.02)
    got = _run(xb, wb, seq, rows, cols)
    want = oracle.gemm_cols(xb, wb, rows=rows, cols=cols)
    r = compare_bf16(got, want)
    assert r["n_fail"] == 0 and r["n_nan"] == 0, r
    # Tighter than the bar: one bf16 spacing, plus the f32 accumulation error
    # of either order (2^-22 of sum |x||w|), which is what remains where the
    # sum cancels to near zero and a spacing is tiny.  A dropped or repeated
    # product (|x w| ~ 1e-2) exceeds it.
    a = bf16_to_f32(got).astype(np.float64)
    b = bf16_to_f32(want).astype(np.float64)
    xf = np.abs(bf16_to_f32(xb).astype(np.float64).reshape(seq, cols))
    wf = np.abs(bf16_to_f32(wb).astype(np.float64).reshape(rows, cols))
    bound = bf16_ulp(b) * 1.0001 + 2.0 ** -22 * (xf @ wf.T)
    assert np.all(np.abs(a - b) <= bound), float(np.max(np.abs(a - b) - bound))


@pytest.mark.parametrize("seq,rows,cols", [(3, 64, 256), (64, 2816, 4096), (70, 80, 384)])
def test_gemm_cols_integer_operands_bit_exact(seq, rows, cols):
    announce(f"gemm_cols exact seq={seq} rows={rows} cols={cols}")
    rng = np.random.default_rng(rows + cols)
    x = rng.integers(-3, 4, (seq, cols))
    w = rng.integers(-3, 4, (rows, cols))
    got = _run(_bf(x), _bf(w), seq, rows, cols)
    want = oracle.gemm_cols(_bf(x), _bf(w), rows=rows, cols=cols)
    assert np.array_equal(got, want)


# Batches past the decode sizes and the plan each takes with its workspace: tile
# tokens, tile columns, k slices.  Every tile shape with and without slices; ragged
# last tiles in both directions; 2, 4, 6, 16, 64 and 128 chunks of the loop (three
# chunks deep); one to three bands of token tiles.  The plans themselves are checked
# without a GPU (test_routes.py).
TILE_CASES = {
    (65, 16, 128): (64, 64, 1), (127, 144, 256): (64, 64, 1), (129, 80, 384): (64, 64, 1),
    (193, 2816, 512): (64, 64, 1), (65, 272, 2048): (64, 64, 4),
    (500, 2816, 4096): (128, 64, 1), (65, 2816, 4096): (128, 64, 4),
    (769, 2816, 256): (128, 128, 1), (1933, 272, 4096): (128, 128, 4),
    (1537, 2816, 128): (192, 128, 1), (2000, 2816, 384): (192, 128, 1),
    (4099, 1040, 128): (192, 128, 1), (324, 2816, 8192): (192, 128, 4),
    (2137, 2816, 256): (256, 128, 1), (1175, 5376, 256): (256, 128, 1),
    (398, 2816, 8192): (256, 128, 4),
}


@pytest.mark.parametrize("seq,rows,cols", TILE_CASES)
def test_gemm_cols_tiles_bit_exact(seq, rows, cols):
    """Integer operands, so every sum is exact in any order."""
    announce(f"gemm_cols tiles seq={seq} rows={rows} cols={cols}")
    rng = np.random.default_rng(seq + rows + cols)
    x = rng.integers(-3, 4, (seq, cols)).astype(np.float32)
    w = rng.integers(-3, 4, (rows, cols)).astype(np.float32)
    got = _run(_bf(x), _bf(w), seq, rows, cols)
    # |sum| <= 9 * 8192: exact in f32, and one rounding to bf16 in the oracle's conversion.
    assert np.array_equal(got, oracle.f32_to_bf16((x @ w.T).ravel()).reshape(seq, rows))


@pytest.mark.parametrize("seq,rows,cols", [(1, 16, 256), (1, 2816, 4096), (15, 48, 512),
                                           (16, 2816, 8192), (1, 80, 8192), (11, 48, 4608),
                                           (7, 80, 1536), (17, 80, 4096)])
def test_gemm_cols_few_tokens_bit_exact(seq, rows, cols):
    """One to sixteen tokens and the first size past them: 1 to 16 slices of 256
    (joined in the workgroup) and, past k of 4,096 or 16 tokens, of 512."""
    test_gemm_cols_integer_operands_bit_exact(seq, rows, cols)


@pytest.mark.parametrize("seq,splits", [(400, 0), (400, 1), (400, 2), (400, 3.99), (400, 4),
                                        (321, 0), (200, 2), (200, 7)])
def test_gemm_cols_workspace_smaller_than_the_plan(seq, splits):
    """Room for that many splits' partials.  The plan takes four at these sizes; past
    320 tokens (more than 256 tiles of 64 x 64) none are needed, before that two.
    Integer operands, so every split count is exact."""
    rows, cols = 2816, 8192
    announce(f"gemm_cols workspace seq={seq} splits={splits}")
    rng = np.random.default_rng(seq)
    x = rng.integers(-3, 4, (seq, cols)).astype(np.float32)
    w = rng.integers(-3, 4, (rows, cols)).astype(np.float32)
    out = empty_dev(seq * rows, np.uint16)
    floats = int(splits * seq * rows)
    ws = to_dev(np.full(floats + 4096, 7.0, np.float32))  # the last 4,096 stay as they are
    A.dispatch_gemm_cols(to_dev(_bf(x)), to_dev(_bf(w)), out, rows=rows, cols=cols, seq_len=seq,
                         workspace=ws[:floats] if floats else None)
    assert np.array_equal(from_dev(out, np.uint16).reshape(seq, rows),
                          oracle.f32_to_bf16((x @ w.T).ravel()).reshape(seq, rows))
    assert np.all(from_dev(ws, np.float32)[floats:] == 7.0)


def test_gemm_cols_rejects_unsupported_shapes():
    from inferno_amd._lib import InfernoHipError

    x = empty_dev(64 * 512, np.uint16)
    w = empty_dev(64 * 512, np.uint16)
    out = empty_dev(64 * 64, np.uint16)
    with pytest.raises(InfernoHipError):
        A.dispatch_gemm_cols(x, w, out, rows=64, cols=200, seq_len=2)   # cols % 128
    with pytest.raises(InfernoHipError):
        A.dispatch_gemm_cols(x, w, out, rows=40, cols=128, seq_len=2)   # rows % 16
    assert A.gemm_cols_workspace(64, 512, 64) is not None  # this shape splits k
    with pytest.raises(InfernoHipError):
        A.dispatch_gemm_cols(x, w, out, rows=64, cols=512, seq_len=64)  # no workspace
    x, w, out = (empty_dev(n, np.uint16) for n in (65 * 8192, 64 * 8192, 65 * 64))
    with pytest.raises(InfernoHipError):
        A.dispatch_gemm_cols(x, w, out, rows=64, cols=8192, seq_len=16)
    with pytest.raises(InfernoHipError):
        A.dispatch_gemm_cols(x, w, out, rows=64, cols=8192, seq_len=65)  # nor past the decode sizes
