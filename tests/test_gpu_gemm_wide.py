"""The wide-tile Q4_K GEMM (128 rows x 64 tokens per workgroup) at its edges:
a last token group of 32, ragged rows and tokens, one super-block of K, and the
smallest grid it takes, against the oracle's per-token GEMV."""
import numpy as np
import pytest

from llm_core_amd import hip
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,T", [
    (8192, 256, 193),     # 4 groups, the last of one token (Tp % 64 == 32), one super-block
    (8100, 512, 209),     # a ragged last row tile, 17 tokens in the last group
    (16385, 256, 520),    # 129 row tiles, the last of one row; 5 wide tiles a CU against 9
    (8191, 512, 385),     # 2 wide tiles a CU against 4
    (32768, 256, 65),     # 2 against 3: wide up to 6 super-blocks,
    (8200, 1792, 257),    # the 128 x 32 tiles from 7
    (16385, 512, 97),
    (8191, 1024, 256),    # rows % 4 != 0: per-row stores
    (4096, 512, 512),     # exactly 256 workgroups
    (4224, 768, 491),     # 33 row tiles: XCD 0 has one more than the others
    (8320, 768, 385),     # 65 of them
])
def test_gemm_wide(ctx, rows, cols, T):
    W = hip.synth_weight(12, rows, cols, seed=rows + T)
    X = hip.synth_normal(T * cols, seed=7)
    xq = O.quantize_q8_0(X)
    y = ctx.alloc(T * rows * 4)
    ctx.write(y, np.full(T * rows, np.nan, np.float32))
    ctx.gemm_q4k_q8(y, ctx.upload(W), ctx.upload(xq), rows, T, cols, hip.row_bytes(12, cols))
    got = ctx.download(y, np.float32, T * rows).reshape(T, rows)
    assert np.isfinite(got).all()
    nb = cols // 32 * 36
    for t in sorted({t for t in (0, 1, 31, 32, 63, 64, T // 2, T - 1) if t < T}):
        want = O.gemv_q8(12, W, xq[t * nb:(t + 1) * nb], rows, cols).astype(np.float64)
        # fp32 sums of cols / 32 + cols / 256 terms in another order
        tol = (cols // 32 + cols // 256 + 8) * 2.0 ** -24 * np.abs(want).max() * 8
        assert np.max(np.abs(got[t] - want)) <= tol, (t, np.max(np.abs(got[t] - want)), tol)


@pytest.mark.parametrize("rows,cols,T", [
    (4096, 6144, 33),     # 8 ranges of 3 super-blocks, the shortest taken
    (1000, 10240, 70),    # ragged rows and tokens, 14 ranges, the last of one super-block
    (1024, 11008, 65),    # 8 row tiles x 2 groups, 43 super-blocks in 15 ranges
    (2048, 6144, 512),    # 128 tiles: 2 ranges of 12
    (24640, 512, 40),     # 193 tiles, one range
    (2560, 6144, 129),    # 20 row tiles: three on half the XCDs and two on the others, 3 ranges
    (4096, 2048, 300),    # 160 tiles, one range
    (2560, 11008, 48),    # the int8 kernel's 16 x 16 tiles are sooner done
])
def test_gemm_q6k_ranges(ctx, rows, cols, T):
    W = hip.synth_weight(14, rows, cols, seed=rows + T)
    if (rows * hip.row_bytes(14, cols)) % 16:
        pytest.skip("the last block does not end on a 16-byte boundary: the dot4 kernel")
    X = hip.synth_normal(T * cols, seed=9)
    xq = O.quantize_q8_0(X)
    y = ctx.alloc(T * rows * 4)
    ctx.write(y, np.full(T * rows, np.nan, np.float32))
    ctx.gemm_q6k_q8(y, ctx.upload(W), ctx.upload(xq), rows, T, cols, hip.row_bytes(14, cols))
    got = ctx.download(y, np.float32, T * rows).reshape(T, rows)
    assert np.isfinite(got).all()
    nb = cols // 32 * 36
    for t in sorted({t for t in (0, 31, 32, 63, T // 2, T - 1) if t < T}):
        want = O.gemv_q8(14, W, xq[t * nb:(t + 1) * nb], rows, cols).astype(np.float64)
        # fp32 sums of cols / 32 + cols / 256 terms in another order
        tol = (cols // 32 + cols // 256 + 8) * 2.0 ** -24 * np.abs(want).max() * 8
        assert np.max(np.abs(got[t] - want)) <= tol, (t, np.max(np.abs(got[t] - want)), tol)
