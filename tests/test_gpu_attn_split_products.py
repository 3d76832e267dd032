"""Prefill attention by split fp16 products (64-row workgroups) at its edges:
group sizes that do not divide 64, ragged tokens, K and V of any scale, and
values its scales do not cover, which take the fp32 kernel's arithmetic."""
import numpy as np
import pytest

from llm_core_amd._ffi import call
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def attend(ctx, q, kc, vc, pos0, H, KVH, hd, cos_t, sin_t, path=0):
    T = q.shape[0]
    bufs = [ctx.upload(x) for x in (q, kc, vc, cos_t, sin_t)]
    do, dq8 = ctx.alloc(T * H * hd * 4), ctx.alloc(T * H * hd // 32 * 36)
    ctx.write(do, np.full(T * H * hd, 7e7, np.float32))
    call("axf_hip_attn_prefill", ctx.handle, do.ptr, dq8.ptr, bufs[0].ptr, H * hd, None, bufs[1].ptr,
         bufs[2].ptr, pos0, T, H, KVH, hd, bufs[3].ptr, bufs[4].ptr, path)
    got = ctx.download(do, np.float32, T * H * hd).reshape(T, H * hd)
    q8 = ctx.download(dq8, np.uint8, T * H * hd // 32 * 36).reshape(T, -1)
    for b in bufs + [do, dq8]:
        b.free()
    return got, q8


@pytest.mark.parametrize("H,KVH,T,pos0,kscale,vscale", [
    (24, 24, 512, 384, 1.0, 1.0),     # 192 workgroups, as many rounds either way: the 16-row kernel
    (24, 24, 512, 768, 1.0, 1.0),     # the same, its first mean position (1024)
    (32, 32, 400, 440, 1.0, 1.0),     # fewer rounds, their first mean position (640)
    (64, 8, 190, 930, 1.0, 1.0),      # 8 heads per kv head, 8 tokens per workgroup, past 1024
    (172, 172, 66, 1100, 1.0, 1.0),   # two rounds either way, the second group's rows hardly used
    (28, 4, 440, 500, 1.0, 1.0),      # 7 heads per kv head: 9 tokens (63 rows), the last group ragged
    (64, 8, 190, 700, 1.0, 1.0),
    (40, 40, 300, 1000, 3e-5, 1e9),   # small K (uniform weights), large V
    (40, 40, 300, 1000, 40.0, 1e-8),  # one key takes nearly all of each row
])
def test_split_products_match_oracle(ctx, H, KVH, T, pos0, kscale, vscale):
    hd, n = 128, pos0 + T
    rng = np.random.default_rng(H + T)
    q = rng.standard_normal((T, H * hd)).astype(np.float32)
    kc = (rng.standard_normal(n * KVH * hd) * kscale).astype(np.float32)
    vc = (rng.standard_normal(n * KVH * hd) * vscale).astype(np.float32)
    cos_t, sin_t = O.rope_table(hd, 10000.0, n)
    got, q8 = attend(ctx, q, kc, vc, pos0, H, KVH, hd, cos_t, sin_t)
    k64, v64 = kc.reshape(n, KVH, hd).astype(np.float64), vc.reshape(n, KVH, hd).astype(np.float64)
    for t in (0, 1, 8, 9, 63, T // 2, T - 2, T - 1):
        qt = O.rope(q[t], pos0 + t, H, hd, cos_t, sin_t).reshape(H, hd).astype(np.float64)
        seen = pos0 + t + 1
        for h in range(0, H, 5):
            k, v = k64[:seen, h // (H // KVH)], v64[:seen, h // (H // KVH)]
            s = k @ qt[h] / np.sqrt(hd)
            w = np.exp(s - s.max())
            w /= w.sum()
            err = np.abs(got[t, h * hd:(h + 1) * hd] - w @ v)
            # a score carries 2^-22 of |q||k| / sqrt(hd) at most (split products and fp32
            # sums), the weighted sum a few roundings of sum w |v|
            smax = np.linalg.norm(qt[h]) * np.linalg.norm(k, axis=1).max() / np.sqrt(hd)
            tol = (32 * 2.0 ** -24 + 2.0 ** -22 * smax) * (w @ np.abs(v))
            assert (err <= tol).all(), (t, h, float((err / tol).max()))
        assert np.array_equal(q8[t], O.quantize_q8_0(got[t]))


@pytest.mark.parametrize("H,KVH", [(32, 32), (64, 16)])
def test_split_products_out_of_range(ctx, H, KVH):
    """Infinities, NaN and magnitudes past the scales, at keys that start a row group, a
    tile or neither: the rows that see them as the 16-row fp32 kernel leaves them (which
    calls of 128 tokens take, in the same row groups), the others as ever."""
    hd, T, pos0 = 128, 512, 512
    n, G = pos0 + T, H // KVH
    rng = np.random.default_rng(8)
    q = rng.standard_normal((T, H, hd)).astype(np.float32)
    kc = rng.standard_normal((n, KVH, hd)).astype(np.float32)
    vc = rng.standard_normal((n, KVH, hd)).astype(np.float32)
    kc[600, 3] *= 1e15
    vc[700, 4, 5] = np.inf
    vc[800, 5, 6] = np.nan
    vc[:, 6] *= 1e-30
    kc[900, 7] = -np.inf
    vc[816, 8, 6] = np.nan
    kc[811, 9, 3] = np.nan
    vc[827, 10] = np.nan
    q[299, 11 * G, 7] = np.nan
    vc[1023, 12, 127] = -np.inf
    vc[100, 13, 64] = np.nan  # every row sees it
    q = q.reshape(T, H * hd)
    cos_t, sin_t = O.rope_table(hd, 10000.0, n)
    got, _ = attend(ctx, q, kc.ravel(), vc.ravel(), pos0, H, KVH, hd, cos_t, sin_t)
    ref = np.concatenate([attend(ctx, q[t:t + 128], kc.ravel(), vc.ravel(), pos0 + t, H, KVH, hd,
                                 cos_t, sin_t)[0] for t in range(0, T, 128)])
    got, ref = got.reshape(T, H, hd), ref.reshape(T, H, hd)
    for h in range(H):
        same = np.isnan(got[:, h]) == np.isnan(ref[:, h])
        assert same.all(), (h, "first row", int(np.argmin(same.all(1))))
        fine = np.isfinite(ref[:, h])
        assert np.array_equal(np.isfinite(got[:, h]), fine), h
        if h // G not in (4, 5, 7, 8, 9, 10, 11, 12, 13):
            assert fine.all(), h
        if fine.any():
            scale = np.abs(ref[:, h][fine]).max()
            assert np.max(np.abs(got[:, h][fine] - ref[:, h][fine])) <= 1e-5 * scale, h


@pytest.mark.parametrize("H,KVH,std", [
    (32, 32, 1e3), (32, 32, 3e3), (32, 32, 6e3), (32, 32, 2e4), (128, 16, 5e4), (32, 32, 1e6),
])
def test_split_products_large_scores(ctx, H, KVH, std):
    """q.k / sqrt(hd) from 1e6 to 1e12 with every operand well inside the scales: the
    softmax is one key's, and the row that key's V."""
    hd, T, pos0 = 128, 512, 512
    n, G = pos0 + T, H // KVH
    rng = np.random.default_rng(int(std))
    q = (rng.standard_normal((T, H * hd)) * std).astype(np.float32)
    kc = (rng.standard_normal((n, KVH, hd)) * std).astype(np.float32)
    vc = rng.standard_normal((n, KVH, hd)).astype(np.float32)
    cos_t, sin_t = O.rope_table(hd, 10000.0, n)
    got, _ = attend(ctx, q, kc.ravel(), vc.ravel(), pos0, H, KVH, hd, cos_t, sin_t)
    assert np.isfinite(got).all()
    got = got.reshape(T, H, hd)
    clear = 0
    for t in range(0, T, 3):
        qt = O.rope(q[t], pos0 + t, H, hd, cos_t, sin_t).reshape(H, hd).astype(np.float64)
        seen = pos0 + t + 1
        for h in (t % H, (7 * t + 5) % H):
            k = kc[:seen, h // G].astype(np.float64)
            s = k @ qt[h] / np.sqrt(hd)
            best, second = np.argsort(s)[:-3:-1]
            # a score's error: 128 fp32 products and sums, and the scaling's rounding
            err = 2.0 ** -24 * 130 * np.linalg.norm(qt[h]) * np.linalg.norm(k, axis=1).max() / np.sqrt(hd)
            # with the two best further apart than both errors and ln(seen * 2^24) the
            # others' weights are under one rounding of the sum
            if s[best] - s[second] < 2 * err + np.log(seen * 2.0 ** 24):
                continue
            clear += 1
            v = vc[best, h // G]
            assert np.abs(got[t, h] - v).max() <= 4 * 2.0 ** -24 * np.abs(v).max(), (t, h)
    assert clear > 50


def test_cache_past_32_bit_offsets(ctx):
    """A layer's K (and V) of over 4 GiB: 272 KV heads and nearly 32768 positions, rows
    that repeat every 241 positions (no divisor of a wrapped offset's distance)."""
    H, hd, T, pos0, period = 272, 128, 64, 32700, 241
    n = pos0 + T
    rng = np.random.default_rng(3)
    kb, vb = (rng.standard_normal((period, H, hd), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((T, H * hd), dtype=np.float32)
    row = H * hd * 4
    caches = []
    for b in (kb, vb):
        c = ctx.alloc(n * row)
        ctx.write(c, b)
        for i in range(period, n, period):
            ctx.copy(c.at(i * row), c, min(period, n - i) * row)
        caches.append(c)
    dq, cos, sin = (ctx.upload(x) for x in (q, np.ones((n, hd // 2), np.float32),
                                            np.zeros((n, hd // 2), np.float32)))
    do = ctx.upload(np.full(T * H * hd, np.nan, np.float32))
    call("axf_hip_attn_prefill", ctx.handle, do.ptr, None, dq.ptr, H * hd, None, caches[0].ptr,
         caches[1].ptr, pos0, T, H, H, hd, cos.ptr, sin.ptr, 0)
    got = ctx.download(do, np.float32, T * H * hd).reshape(T, H, hd)
    for b in caches + [dq, cos, sin, do]:
        b.free()
    for h in (0, 100, 271):
        for t in (0, 40, T - 1):
            seen = pos0 + t + 1
            times = np.bincount(np.arange(seen) % period, minlength=period)
            qt = q[t].reshape(H, hd)[h].astype(np.float64)
            k, v = kb[:, h].astype(np.float64), vb[:, h].astype(np.float64)
            s = k @ qt / np.sqrt(hd)
            w = np.exp(s - s.max()) * times
            w /= w.sum()
            # as above, and the weights' sum of `seen` terms
            smax = np.linalg.norm(qt) * np.linalg.norm(k, axis=1).max() / np.sqrt(hd)
            tol = ((32 + seen / 64) * 2.0 ** -24 + 2.0 ** -22 * smax) * (w @ np.abs(v))
            assert (np.abs(got[t, h] - w @ v) <= tol).all(), (t, h)


@pytest.mark.parametrize("H,KVH", [(32, 32), (64, 16)])
@pytest.mark.parametrize("kind", ["q rows", "k keys", "v channels", "v keys", "v later key", "qkv"])
def test_split_products_mixed_magnitudes(ctx, H, KVH, kind):
    """Rows, keys and channels of very different size next to each other: every output as
    near to 64 bits as fp32 sums of its own terms, whatever the largest beside them."""
    hd, T, pos0 = 128, 512, 512
    n, G = pos0 + T, H // KVH
    rng = np.random.default_rng(len(kind) + H)
    q = rng.standard_normal((T, H, hd)).astype(np.float32)
    kc = rng.standard_normal((n, KVH, hd)).astype(np.float32)
    vc = rng.standard_normal((n, KVH, hd)).astype(np.float32)

    def powers(lo, hi, *shape):
        return np.exp2(rng.integers(lo, hi + 1, shape)).astype(np.float32)

    if kind in ("q rows", "qkv"):  # up to scores of 2^16
        q *= powers(-14, 12, T, H, 1)
    if kind in ("k keys", "qkv"):
        kc *= powers(-30, 3, n, KVH, 1)
    if kind in ("v channels", "qkv"):
        vc *= powers(-26, 0, 1, KVH, hd)
    if kind == "v keys":
        vc *= powers(-13, 13, n, KVH, 1)
    if kind == "v later key":  # earlier rows of its tile give it no weight
        vc[700] *= 2.0 ** 24
        vc[813, :, 1::2] *= 2.0 ** 24
    q = q.reshape(T, H * hd)
    cos_t, sin_t = O.rope_table(hd, 10000.0, n)
    got, _ = attend(ctx, q, kc.ravel(), vc.ravel(), pos0, H, KVH, hd, cos_t, sin_t)
    got = got.reshape(T, H, hd)
    worst = 0.0
    for t in sorted({*range(0, T, 23), 186, 187, 188, 288, 299, 300, 301, 302}):
        qt = O.rope(q[t], pos0 + t, H, hd, cos_t, sin_t).reshape(H, hd).astype(np.float64)
        seen = pos0 + t + 1
        for h in range(t % 3, H, 3):
            k, v = kc[:seen, h // G].astype(np.float64), vc[:seen, h // G].astype(np.float64)
            s = k @ qt[h] / np.sqrt(hd)
            w = np.exp(s - s.max())
            w /= w.sum()
            # a score is off by 3 * 2^-22 of sum |q||k| / sqrt(hd) at most (the parts' last
            # bits 2^-23 each, l * l 2^-22, RoPE and the sums 2^-22), which moves the output
            # by that much of its weight times |v - out|; the weights and the sum of p v take
            # a few roundings each
            out = w @ v
            ds = 3 * 2.0 ** -22 * (np.abs(k) @ np.abs(qt[h])) / np.sqrt(hd) + 2.0 ** -22 * np.abs(s - s.max())
            # (the weights and V keep 2^-50 of their largest whatever their size)
            tol = (w * ds) @ np.abs(v - out) + 48 * 2.0 ** -24 * (w @ np.abs(v))
            tol += 2.0 ** -50 * (np.abs(v).sum(0) + np.abs(v).max())
            ratio = float((np.abs(got[t, h] - out) / tol).max())
            worst = max(worst, ratio)
            assert ratio <= 1, (t, h, ratio)
    print(kind, "largest error over its bound:", round(worst, 3))
