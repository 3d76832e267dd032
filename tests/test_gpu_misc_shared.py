"""The Q8_0 / Q5_0 / F16 GEMM with activations shared through LDS at its edges:
exactly 160 workgroups, ragged rows and tokens, one block, odd block counts (a
half-filled last stage, rows that start inside a dword) and W off a dword; and
the general kernel just below and at 16 tokens."""
import numpy as np
import pytest

from llm_core_amd._ffi import AXF_TYPE_F16, AXF_TYPE_Q5_0, AXF_TYPE_Q8_0, call
from oracle import oracle as O
from test_gpu_misc import blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [AXF_TYPE_Q8_0, AXF_TYPE_Q5_0, AXF_TYPE_F16])
@pytest.mark.parametrize("rows,cols,T,off", [
    (5120, 256, 128, 0),   # 80 x 2 workgroups, the fewest
    (5056, 256, 128, 0),   # 79 x 2: the general kernel
    (6144, 32, 100, 0),    # 96 x 2 workgroups, one block: K range 1 is empty
    (6082, 96, 65, 0),     # ragged rows, one token past a group, 3 blocks
    (12226, 160, 33, 0),   # 5 blocks, ragged rows and tokens
    (3072, 928, 250, 0),   # 29 blocks
    (4096, 1024, 192, 0),
    (6144, 96, 128, 2),    # Q5_0 rows that start off a dword keep the general kernel
    (1000, 1024, 16, 0),   # 16 tokens: the general kernel's 16-token wave tiles, K in 4 ranges,
    (1000, 288, 16, 0),    # in 2 (the second shorter),
    (37, 96, 16, 0),       # and whole
])
def test_shared_gemm(ctx, qtype, rows, cols, T, off):
    if off and qtype == AXF_TYPE_F16:
        off = 16
    rng = np.random.default_rng(rows + cols + T)
    if qtype == AXF_TYPE_F16:
        W = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float16)
    else:
        W = blocks(qtype, rows, cols, 5 + qtype)
    X = rng.standard_normal((T, cols)).astype(np.float32)
    rb = O.misc_row_bytes(qtype, cols)
    raw = np.concatenate([np.zeros(off, np.uint8), np.ascontiguousarray(W).view(np.uint8).ravel()])
    dW, dX = ctx.upload(raw), ctx.upload(X)
    y0 = rng.standard_normal((T, rows)).astype(np.float32)
    dY = ctx.upload(np.full(T * rows, np.nan, np.float32))
    call("axf_hip_gemm_misc_f32", ctx.handle, qtype, dY.ptr, dW.ptr + off, dX.ptr, rows, T, cols, rb, 0)
    got = ctx.download(dY, np.float32, T * rows).reshape(T, rows)
    byt = raw[off:].reshape(rows, rb)
    w = np.stack([O.dequant_row(qtype, byt[r], cols) for r in range(rows)]).astype(np.float64)
    want = X.astype(np.float64) @ w.T
    # a split activation is within 2^-23 of its row's largest value at most, and each
    # output a chain of up to 32 + cols / 32 fp32 roundings of sums of |w||x|
    bound = (2.0 ** -22 + (32 + cols / 32) * 2.0 ** -24) * (np.abs(X).astype(np.float64) @ np.abs(w.T))
    bound += 2.0 ** -23 * np.abs(X).max(1, keepdims=True) * np.abs(w).sum(1)[None]
    assert (np.abs(got - want) <= bound).all()
    ctx.write(dY, y0)
    call("axf_hip_gemm_misc_f32", ctx.handle, qtype, dY.ptr, dW.ptr + off, dX.ptr, rows, T, cols, rb, 1)
    acc = ctx.download(dY, np.float32, T * rows).reshape(T, rows)
    assert np.array_equal(acc, y0 + got)
    for b in (dW, dX, dY):
        b.free()
