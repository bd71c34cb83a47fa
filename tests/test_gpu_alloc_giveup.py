"""A lockstep that gives up waiting for its walk (forced: one walk workgroup more than
there is), in each of the lockstep's kernels: every kernel ends, the allocation is done
again one kernel after the other, and the output equals the oracle's."""
import sys

import numpy as np
import pytest

import oracle
from ptilopsis_amd import parse_source, workloads as W

pytestmark = pytest.mark.gpu
OUT = ("words", "func_ids", "func_starts", "func_ends", "func_sizes")


def program(nf):
    targets = np.random.default_rng(nf).integers(8, 40, nf).astype(np.uint32)
    targets[[0, 8 * (nf // 16), nf - 1]] = 600  # many chunks of the walk's rows
    return parse_source(W.program_source(0x61FE + nf, nf, targets)[0])


# one group; one wave of one row of lanes, of four; a workgroup of up to 4 and 15
# slots, of three slots a wave; states in device memory, 4 and 8 functions a thread
@pytest.mark.parametrize("nf", [5, 100, 400, 800, 4000, 10_000, 30_000, 40_000])
def test_gpu_lockstep_gives_up_and_is_redone(gpu_ctx, nf):
    t = program(nf)
    want = oracle.compile_tree(t)
    before = int(gpu_ctx.dump("ra_redos")[0])
    print("forced give-up,", nf, "functions,", t.n, "nodes", file=sys.stderr, flush=True)
    try:
        for on, redos in ((2, 1), (1, 1)):
            gpu_ctx.set_overlap(on)
            got = gpu_ctx.compile(t)
            assert int(gpu_ctx.dump("ra_redos")[0]) - before == redos
            for k in OUT:
                assert np.array_equal(np.asarray(got[k]), np.asarray(want[k])), (nf, on, k)
    finally:
        gpu_ctx.set_overlap(1)


def test_gpu_batch_gives_up_and_is_redone(gpu_ctx):
    trees = [program(nf) for nf in (3, 5, 100, 400, 800, 4000)]
    print("forced give-up, a batch of", len(trees), "programs", file=sys.stderr, flush=True)
    before = int(gpu_ctx.dump("ra_redos")[0])
    try:
        gpu_ctx.set_overlap(2)
        got = gpu_ctx.compile_batch(trees)
    finally:
        gpu_ctx.set_overlap(1)
    assert int(gpu_ctx.dump("ra_redos")[0]) - before == 1
    for t, r in zip(trees, got):
        want = oracle.compile_tree(t)
        for k in OUT:
            assert np.array_equal(np.asarray(r[k]), np.asarray(want[k])), k
