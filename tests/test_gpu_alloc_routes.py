"""Programs with calls of many arguments, in which an operand names a word of another
function: where that word defines its register the allocation is k_ra_serial's, and
where it does not (a register that is never set reads as x0 in any order) it stays
with the walks and the lockstep.  The oracle's words after optimize say which kind a
program is; outputs equal the oracle's either way."""
import re
import sys

import numpy as np
import pytest

import oracle
from ptilopsis_amd import parse_source, workloads as W

pytestmark = pytest.mark.gpu
OUT = ("words", "func_ids", "func_starts", "func_ends", "func_sizes")
# arguments of a function, functions, seed: reads of registers that nothing defines
UNSET = [(6, 16, 3, 15), (6, 16, 8, 12), (6, 16, 12, 148), (7, 11, 8, 65), (7, 11, 20, 117), (10, 16, 12, 39),
         (10, 16, 20, 86)]
SET = [(7, 16, 12, 3), (12, 16, 12, 5)]  # reads of registers that another function defines


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def source(lo, hi, nf, k):
    return W.program_source(0xABC00 + k, nf, np.full(nf, 300, np.uint32), dict(W.BASE, min_args=lo, max_args=hi))[0]


def foreign_reads(tree):
    """Operands naming a word outside the part of their function up to themselves:
    how many of them name a word that does not define its register, and how many do."""
    o = oracle.Oracle(tree)
    o.run(4)
    rd, rs1, rs2, starts = (o.get(k).astype(np.int64) for k in ("rd", "rs1", "rs2", "func_starts"))
    o.close()
    i = np.arange(rd.shape[0])
    first = starts[np.searchsorted(starts, i, side="right") - 1]
    assert not ((rd > 63) & (rd != i + 64)).any()
    v = np.concatenate([np.where((a > 63) & ((a - 64 < first) | (a - 64 > i)), a - 64, -1) for a in (rs1, rs2)])
    v = v[v >= 0]
    return int((rd[v] != v + 64).sum()), int((rd[v] == v + 64).sum())


def compiled(ctx, tree):
    ctx.profile(True)
    try:
        return ctx.compile(tree), ctx.kernel_times()
    finally:
        ctx.profile(False)


def assert_same(gpu, ref, what):
    for k in OUT:
        assert np.array_equal(np.asarray(gpu[k]), np.asarray(ref[k])), (what, k)


@pytest.mark.parametrize("more", [0, 600], ids=["alone", "with 600 functions"])
@pytest.mark.parametrize("case", UNSET)
def test_gpu_unset_register_reads_keep_the_walks(gpu_ctx, case, more):
    src = source(*case)
    if more:  # past 64 groups: the lockstep in a workgroup
        filler = W.program_source(0xABC, more, min_stmts=1, max_stmts=3)[0]
        src += re.sub(r"\bf(\d+)\b", r"g\1", filler)
    t = parse_source(src)
    unset, defined = foreign_reads(t)
    assert unset > 0 and defined == 0
    say("reads of registers never set:", unset, case, t.n, "nodes")
    r, names = compiled(gpu_ctx, t)
    assert "k_ra_walk" in names and "k_ra_serial" not in names
    assert_same(r, oracle.compile_tree(t), (case, more))


@pytest.mark.parametrize("case", SET)
def test_gpu_reads_of_another_functions_register_are_serial(gpu_ctx, case):
    t = parse_source(source(*case))
    assert foreign_reads(t)[1] > 0
    say("reads of another function's register", case, t.n, "nodes")
    r, names = compiled(gpu_ctx, t)
    assert "k_ra_serial" in names
    assert_same(r, oracle.compile_tree(t), case)


@pytest.mark.parametrize("small", [0, 1])
def test_gpu_both_kinds_in_a_batch(gpu_ctx, small):
    trees = [parse_source(source(*c)) for c in UNSET + SET]
    old = [gpu_ctx.tune_get("small_programs", b) for b in range(4)]
    for b in range(4):
        gpu_ctx.tune_set("small_programs", b, small)
    say("batch of", len(trees), "programs with reads of other functions' words, small", small)
    try:
        for c, t, r in zip(UNSET + SET, trees, gpu_ctx.compile_batch(trees)):
            assert_same(r, oracle.compile_tree(t), (c, small))
    finally:
        for b in range(4):
            gpu_ctx.tune_set("small_programs", b, old[b])
