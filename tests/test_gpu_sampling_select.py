"""The sampler's threshold selection (k <= 64, penalty windows <= 1024) at the
edges of its range, against the oracle's penalty and sample()."""
import numpy as np
import pytest

from llm_core_amd import hip
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LOWEST = np.float32(np.finfo(np.float32).min)


def logits_of(kind, n, rng):
    if kind == "ascending":  # each thread's share of a chunk is the worst mix of ranks
        return np.sort(rng.standard_normal(n)).astype(np.float32)
    if kind == "blocked":  # every large value with one thread (stride 256) of each chunk
        x = rng.standard_normal(n).astype(np.float32)
        x[7::256] += 20.0
        return x
    if kind == "equal":
        return np.full(n, 0.25, np.float32)
    x = rng.standard_normal(n).astype(np.float32) * 3
    x[rng.random(n) < 0.5] = -np.inf
    x[rng.random(n) < 0.3] = LOWEST
    x[rng.integers(0, n, 80)] = 2.5
    return x


@pytest.mark.parametrize("n", [1, 63, 4095, 4096, 4097, 32003])
@pytest.mark.parametrize("kind", ["ascending", "blocked", "equal", "lowest"])
def test_select_matches_oracle(ctx, n, kind):
    rng = np.random.default_rng(n)
    for k in (1, 2, 40, 63, 64, 65):
        for last_n in (1, 64, 1024, 1025):
            x = logits_of(kind, n, rng)
            hist = rng.integers(0, n, 1100).astype(np.int32)
            hist[-3:] = hist[-900]  # an id of the window more than once
            r = float(rng.random(dtype=np.float32))
            d = ctx.upload(x)
            tok = ctx.sample(d, n, 0.8, k, 0.95, 1.1, last_n, hist, r)
            pen = O.rep_penalty(x, hist, last_n, 1.1)
            np.testing.assert_array_equal(ctx.download(d, np.float32, n), pen)
            want, margin = O.sample(pen, k, 0.95, 0.8, r)
            # a decision as near as 2k ulps of a cumulative probability may fall either
            # way (expf on the device and in glibc differ by an ulp)
            assert tok == want or margin < 1e-5 + 2 * k * 2.0 ** -23, (k, last_n, tok, want, margin)
            d.free()


def test_select_equals_sort_path(ctx):
    """The same draws through the selection (window 1024) and the sorts (1025, which the
    history is too short to tell apart): one token for one."""
    rng = np.random.default_rng(3)
    for n in (1000, 32000, 151936):
        for trial in range(24):
            x = (rng.standard_normal(n) * 2.5).astype(np.float32)
            hist = rng.integers(0, n, 90).astype(np.int32)
            k, p, r = int(rng.integers(1, 65)), float(rng.choice([0.5, 0.9, 1.0])), float(rng.random())
            toks = []
            for last_n in (1024, 1025):
                d = ctx.upload(x)
                toks.append(ctx.sample(d, n, 0.7, k, p, 1.2, last_n, hist, r))
                d.free()
            assert toks[0] == toks[1], (n, trial, k, p, r, toks)
