"""Register allocation's walks at the sizes where their launch changes: programs
around one group of 8 functions (k_ra_lane0_one), around 16 and 64 groups (the
lockstep in one wave, one row of lanes or four) and 256, 960 and 2880 groups (a
workgroup of one slot of 64 groups a wave or three), alone with walk and lockstep
overlapped and not, and together in one batch; and operands defined more words
back than the walks' LDS rings hold.  Every output equals
the oracle's."""
import sys

import numpy as np
import pytest

import oracle
from ptilopsis_amd import parse_source, workloads as W

pytestmark = pytest.mark.gpu
OUT = ("words", "func_ids", "func_starts", "func_ends", "func_sizes")
COUNTS = (1, 7, 8, 9, 16, 17, 127, 128, 129, 136, 137, 511, 512, 513, 520)


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def assert_same(gpu, ref, what):
    for k in OUT:
        assert np.array_equal(np.asarray(gpu[k]), np.asarray(ref[k])), (what, k)


def program(nf):
    return parse_source(W.program_source(0xA110 + nf, nf, min_stmts=1, max_stmts=9)[0])


@pytest.mark.parametrize("nf", COUNTS)
def test_gpu_alloc_function_counts(gpu_ctx, nf):
    t = program(nf)
    want = oracle.compile_tree(t)
    try:
        for on in (1, 0):
            say("allocation,", nf, "functions, overlap", on)
            gpu_ctx.set_overlap(on)
            assert_same(gpu_ctx.compile(t), want, (nf, on))
    finally:
        gpu_ctx.set_overlap(1)


@pytest.mark.parametrize("nf", [2048, 2049, 7680, 7681, 23040, 23041])
def test_gpu_alloc_group_classes(gpu_ctx, nf):
    # a few long functions among short ones, so that slots empty and are packed
    rng = np.random.default_rng(nf)
    targets = np.where(rng.random(nf) < 0.02, 1500, 60).astype(np.uint32)
    targets[[0, 8 * (nf // 16)]] = 4000
    t = parse_source(W.program_source(0xA110 + nf, nf, targets)[0])
    want = oracle.compile_tree(t)
    try:
        for on in (1, 0):
            say("allocation,", nf, "functions,", t.n, "nodes, overlap", on)
            gpu_ctx.set_overlap(on)
            assert_same(gpu_ctx.compile(t), want, (nf, on))
    finally:
        gpu_ctx.set_overlap(1)


def test_gpu_alloc_function_counts_batch(gpu_ctx):
    trees = [program(nf) for nf in COUNTS]
    say("allocation, one batch of", len(trees), "programs")
    for nf, t, r in zip(COUNTS, trees, gpu_ctx.compile_batch(trees)):
        assert_same(r, oracle.compile_tree(t), nf)


@pytest.mark.parametrize("nf", [0, 9, 70])
def test_gpu_alloc_far_operands(gpu_ctx, nf):
    # wide balanced expressions: an operand's word is thousands of words back
    base = dict(W.STRESS, min_args=2, max_args=4)
    t = W.stress_program(0xFA4, 16000) if nf == 0 else parse_source(
        W.program_source(0xFA4 + nf, nf, base=base, min_stmts=1, max_stmts=2, max_nest=1)[0])
    o = oracle.Oracle(t)
    o.run(4)
    far = 0
    for name in ("rs1", "rs2"):
        a = o.get(name).astype(np.int64)
        d = np.arange(a.shape[0]) - (a - 64)
        far += int(((a > 63) & (a < 1 << 31) & (d > 255)).sum())
    o.close()
    assert far > 0
    say("allocation, far operands", far, "in", t.n, "nodes")
    assert_same(gpu_ctx.compile(t), oracle.compile_tree(t), nf)


@pytest.mark.parametrize("where", ["first", "middle", "last"])
@pytest.mark.parametrize("nf", [9, 24, 130, 512])
def test_gpu_alloc_one_function_left(gpu_ctx, nf, where):
    # one lane-0 function far longer than the others, in the first, a middle or
    # the last group: the lockstep in one wave ends on it alone, from steps on
    # both sides of a block
    groups = (nf + 7) // 8
    g = {"first": 0, "middle": groups // 2, "last": groups - 1}[where]
    for k in range(3):
        rng = np.random.default_rng(97 * nf + k)
        targets = rng.integers(20, 300, nf).astype(np.uint32)
        targets[8 * g] = 2500
        t = parse_source(W.program_source(0xA1100 + 8 * nf + k, nf, targets)[0])
        say("allocation, one long function,", nf, where, k)
        assert_same(gpu_ctx.compile(t), oracle.compile_tree(t), (nf, where, k))
