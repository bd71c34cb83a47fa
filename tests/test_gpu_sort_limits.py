"""The device depth sort on both sides of its rule for the ranges that one workgroup
finishes (8192 elements, or 2048 past 4M elements in programs of under 1M, or with more
programs than compute units): against the oracle's libstdc++ introsort restatement."""
import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
M = 1 << 20


@pytest.mark.parametrize("sizes", [[4 * M], [4 * M + 1], [2 * M, 2 * M - 9, 9], [2 * M, 2 * M, 1], [M] * 5,
                                   [M] * 4 + [M - 4], [700_001] * 6 + [8192, 8193, 2048, 2049, 17], [60_000] * 70 + [9000]],
                         ids=lambda s: f"{len(s)}x{s[0]}")
def test_gpu_depth_sort_limits(gpu_ctx, sizes):
    rng = np.random.default_rng(len(sizes) + sizes[0])
    keys = np.concatenate([rng.integers(0, 70 if n > 10_000 else n, n) for n in sizes]).astype(np.int32)
    bounds = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    print("depth sort of", len(sizes), "ranges,", keys.shape[0], "elements", file=sys.stderr, flush=True)
    got = gpu_ctx.depth_sort(keys, bounds)
    for p in range(len(sizes)):
        b, e = int(bounds[p]), int(bounds[p + 1])
        assert np.array_equal(got[b:e], oracle.introsort(keys[b:e]) + b), f"range {p} (size {e - b})"
