"""Two workers' batches of programs whose waiting locksteps take half a compute unit and
more each: every result is the one compiled alone, and no lockstep gives up waiting."""
import sys

import numpy as np
import pytest

from ptilopsis_amd import parse_source, workloads as W
from ptilopsis_amd.generator import Server

pytestmark = pytest.mark.gpu
OUT = ("words", "func_ids", "func_starts", "func_ends", "func_sizes")


def test_gpu_serve_large_programs_do_not_starve(gpu_ctx):
    one = lambda k, nf: parse_source(W.program_source(0x5E40 + k, nf, np.full(nf, 20, np.uint32))[0])
    trees = [one(k, 520 + 40 * (k % 4)) for k in range(48)] + [one(k, 2100) for k in range(48, 72)]
    alone = [gpu_ctx.compile(t) for t in trees]
    print("serving", len(trees), "programs,", sum(t.n for t in trees), "nodes", file=sys.stderr, flush=True)
    srv = Server(0, max_batch=18, workers=2)
    try:
        for _ in range(3):
            tickets = [srv.submit(t) for t in trees]
            for p, k in enumerate(tickets):
                r = srv.wait(k)[0]
                assert all(np.array_equal(r[o], alone[p][o]) for o in OUT), p
        assert srv.redos() == 0
    finally:
        srv.close()
    assert gpu_ctx.dump("ra_redos").size == 1
