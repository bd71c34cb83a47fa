"""Operands defined further back than each allocation kernel's LDS ring holds, so that
their states are read back from device memory: the wave-a-function walk (16384 words,
read back from 16320), the one-group lockstep (4096, read back from 4032), the walk of
64 functions a wave and the lockstep in one wave and in a workgroup (248), marked ones
among them.  Every output equals the oracle's."""
import sys

import numpy as np
import pytest

import oracle
from ptilopsis_amd import parse_source

pytestmark = pytest.mark.gpu
OUT = ("words", "func_ids", "func_starts", "func_ends", "func_sizes")
SPINE = 10


def wide(v, lit, leaves, ops, k=0):
    if leaves == 1:
        return lit if k % 7 == 3 else v
    h = leaves // 2
    return f"({wide(v, lit, h, ops, 2 * k + 1)} {ops[k % len(ops)]} {wide(v, lit, leaves - h, ops, 2 * k + 2)})"


def far_function(name, leaves, typ="int", n=2):
    """n statements v op (v op (... wide expression)): the outer operands' words are
    about 3 * leaves words and more before the words that use them."""
    v, lit = ("v0", "7") if typ == "int" else ("v0", "1.5")
    ops = "+-*"
    body = ""
    for s in range(n):
        e = wide(v, lit, leaves, ops[s:] + ops[:s])
        for k in range(SPINE):
            e = f"({v} {ops[(k + s) % 3]} {e})"
        body += f"  v0 = {e};\n"
    return f"function {name}(v0 : {typ}) : {typ} {{\n{body}  return v0;\n}}\n"


def small_function(name, k):
    return f"function {name}(v0 : int) : int {{\n  v0 = (v0 + (v0 * {k % 100 + 1}));\n  return v0;\n}}\n"


def program(nf, far):
    """nf functions; far: {function: (leaves, type)}, the others small."""
    return parse_source("".join(far_function(f"f{k}", *far[k]) if k in far else small_function(f"f{k}", k)
                                for k in range(nf)))


def distances(tree):
    """Per function, how many words back its operands' words are."""
    o = oracle.Oracle(tree)
    o.run(4)
    rs1, rs2, starts = (o.get(k).astype(np.int64) for k in ("rs1", "rs2", "func_starts"))
    o.close()
    i = np.arange(rs1.shape[0])
    f = np.searchsorted(starts, i, side="right") - 1
    out = [[] for _ in range(starts.shape[0])]
    for a in (rs1, rs2):
        m = (a > 63) & (i - (a - 64) > 200)
        for k, d in zip(f[m], (i - (a - 64))[m]):
            out[k].append(int(d))
    return [np.array(x, np.int64) for x in out]


def swapped_reads(ref, f):
    """Arithmetic words of function f whose first operand is read through t0 or ft5,
    the registers of swapped operands, among the last SPINE before its return."""
    w = ref["words"][ref["func_starts"][f]:ref["func_ends"][f]].astype(np.int64)
    w = w[((w & 0x7F) == 0x33) | ((w & 0x7F) == 0x3B) | ((w & 0x7F) == 0x53)]
    return int((((w[-SPINE - 4:] >> 15) & 31) == 5).sum())


def check(ctx, tree, what):
    ref = oracle.compile_tree(tree)
    try:
        for on in (1, 0):
            print("allocation, far operands,", what, tree.n, "nodes, overlap", on, file=sys.stderr, flush=True)
            ctx.set_overlap(on)
            got = ctx.compile(tree)
            for k in OUT:
                assert np.array_equal(np.asarray(got[k]), np.asarray(ref[k])), (what, on, k)
    finally:
        ctx.set_overlap(1)
    return ref


@pytest.mark.parametrize("typ", ["int", "float"])
def test_gpu_far_operands_one_group(gpu_ctx, typ):
    # 0 is k_ra_lane0_one's, the others have a wave of the walk each
    t = program(8, {k: (5600 + 37 * k, typ) for k in range(8)})
    d = distances(t)
    assert all((d[k] >= 16384).sum() >= 2 * SPINE for k in range(8))
    ref = check(gpu_ctx, t, typ)
    assert swapped_reads(ref, 0) > 0


@pytest.mark.parametrize("leaves", [1330, 1337, 1344, 1351, 1358, 1365, 5430, 5437, 5444, 5451, 5458])
def test_gpu_far_operands_at_the_rings_ends(gpu_ctx, leaves):
    # distances on both sides of 4032 and 4096, of 16320 and 16384
    t = program(3, {0: (leaves, "int"), 1: (leaves, "int"), 2: (leaves - 6, "int")})
    lo, hi = (4032, 4096) if leaves < 4000 else (16320, 16384)
    assert all(((x > lo - 64) & (x < hi + 64)).sum() >= SPINE for x in distances(t))
    check(gpu_ctx, t, leaves)


@pytest.mark.parametrize("nf", [24, 130, 600, 7700])
def test_gpu_far_operands_of_more_groups(gpu_ctx, nf):
    # lane-0 functions (one far longer than the others) and walked ones with far
    # operands: the lockstep in one wave (24, 130 functions) and in a workgroup
    far = {0: (300, "int"), 8: (2500, "int"), 16: (700, "float"), 1: (900, "int"), 9: (400, "float"),
           8 * (nf // 16): (600, "int"), 8 * ((nf - 1) // 8): (500, "float"), nf - 2: (350, "int")}
    t = program(nf, far)
    d = distances(t)
    assert all((d[k] >= 248).sum() >= 2 * SPINE for k in far)
    ref = check(gpu_ctx, t, nf)
    assert sum(swapped_reads(ref, k) for k in far if k % 8 == 0) > 0
