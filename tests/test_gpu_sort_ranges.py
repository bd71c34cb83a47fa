"""The device depth sort (ptl_debug_depth_sort) against the oracle's libstdc++
introsort restatement where its launches differ: ranges on both sides of the 8192
elements that one workgroup finishes when the ranges are few, the same sizes among
more ranges than compute units (2048 elements then), tiles of 4096 carried over by
look-back, and keys that exhaust the recursion limit (heapsorted ranges)."""
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def killer(n):
    """Keys that put the smallest two of what is left where the median of three
    looks, so that ranges shrink slowly and the recursion limit runs out."""
    a = np.zeros(n, np.int64)
    idx = list(range(n))
    lo = 0
    while len(idx) > 3:  # the two smallest left go where the median is looked for
        f, m = 1, len(idx) // 2
        a[idx[f]], a[idx[m]] = lo, lo + 1
        lo += 2
        first = idx[0]
        rest = [x for k, x in enumerate(idx) if k not in (0, f, m)]
        idx = [first] + rest
    for x in idx:
        a[x] = lo
        lo += 1
    return a


PATTERNS = {
    "depths": lambda rng, n: rng.integers(0, 70, n),
    "equal": lambda rng, n: np.full(n, 3),
    "two": lambda rng, n: rng.integers(0, 2, n),
    "distinct": lambda rng, n: rng.permutation(n),
    "organ": lambda rng, n: np.minimum(np.arange(n), n - 1 - np.arange(n)),
    "killer": lambda rng, n: killer(n),
}
SIZES = [16, 17, 33, 1023, 1024, 1025, 4096, 4097, 8191, 8192, 8193, 8209, 16384, 20000]


@pytest.mark.parametrize("fill", [0, 300], ids=["few", "many"])
@pytest.mark.parametrize("pattern", sorted(PATTERNS))
def test_gpu_depth_sort_ranges(gpu_ctx, pattern, fill):
    rng = np.random.default_rng(len(pattern) + fill)
    sizes = [n for n in SIZES if pattern != "killer" or n <= 8209] + [int(x) for x in rng.integers(1, 40, fill)]
    keys = np.concatenate([PATTERNS[pattern](rng, n).astype(np.int32) for n in sizes])
    bounds = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    print("depth sort", pattern, len(sizes), "ranges", file=sys.stderr, flush=True)
    got = gpu_ctx.depth_sort(keys, bounds)
    for p in range(len(sizes)):
        b, e = int(bounds[p]), int(bounds[p + 1])
        assert np.array_equal(got[b:e], oracle.introsort(keys[b:e]) + b), f"range {p} (size {e - b})"
