"""ptl_compile_noalloc allocates no pinned host memory: on a context that has compiled
nothing before, the pinned staging buffers are the same size after the call, for an
ordinary program and for one of as many functions as its node limit allows."""
import sys

import pytest

from ptilopsis_amd import abi, parse_source, workloads as W
from ptilopsis_amd.generator import Context
from test_zz_no_alloc import LIMIT, DevTree, assert_same, compile_noalloc, hip  # noqa: F401 (hip: a fixture)

pytestmark = pytest.mark.gpu


def tiny_functions():
    """Functions that return nothing, up to 1000 nodes below the limit."""
    one = parse_source("function f0() : void { }").n
    two = parse_source("function f0() : void { }\nfunction f1() : void { }").n
    return parse_source("\n".join(f"function f{k}() : void {{ }}" for k in range((LIMIT - 1000 - one) // (two - one))))


@pytest.mark.parametrize("which", ["240k", "tiny functions"])
def test_gpu_noalloc_pins_nothing(gpu_ctx, hip, which):  # noqa: F811
    t = W.program_of_size(0x5EED0A11, 240_000) if which == "240k" else tiny_functions()
    assert LIMIT - 30_000 < t.n <= LIMIT
    want = gpu_ctx.compile(t)
    print("noalloc on a new context:", which, t.n, "nodes,", want["n_funcs"], "functions", file=sys.stderr, flush=True)
    ctx = Context(0)
    try:
        before = ctx.dump("pinned").tolist()
        s, _, got = compile_noalloc(hip, ctx, DevTree(hip, t), want["n_words"], want["n_funcs"])
        assert s == abi.PTL_OK, abi.ERRORS.get(s, s)
        assert ctx.dump("pinned").tolist() == before
        assert_same(got, want, which)
    finally:
        ctx.close()
