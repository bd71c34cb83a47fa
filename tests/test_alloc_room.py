"""The lockstep workgroups that wait for a walk leave the walks a compute unit: planned
for several contexts that compile at the same time, on the host alone."""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_SO = os.path.join(ROOT, "ptilopsis_amd", "libptl_hip.so")
# programs and functions of each, of every launch class
MIX = [(512, 5), (512, 60), (96, 300), (64, 700), (64, 4000), (8, 10_000), (4, 40_000)]
BATCHES = {"a few": [(10, 5), (10, 60)], "one group": [(4096, 5)], "small": [(1024, 40)], "65 groups": [(64, 520)],
           "257 groups": [(64, 2056)], "one large": [(1, 20_000)], "all": MIX}


@pytest.mark.parametrize("contexts", [1, 2, 8])
@pytest.mark.parametrize("batch", sorted(BATCHES))
def test_waiting_locksteps_of_all_contexts_leave_room(batch, contexts):
    if not os.path.exists(HIP_SO):
        pytest.skip("libptl_hip.so not built (run __graft_entry__.build())")
    from ptilopsis_amd import abi
    lib = abi.bind(C.CDLL(HIP_SO))
    per = np.concatenate([np.full(n, f, np.int64) for n, f in BATCHES[batch]])
    funcs = np.concatenate([[0], np.cumsum(per)]).astype(np.uint32)
    sizes = np.random.default_rng(1).integers(3, 400, funcs[-1]).astype(np.uint32)
    room = np.zeros(contexts)
    assert lib.ptl_debug_ra_room(sizes.ctypes.data, funcs.ctypes.data, per.shape[0], contexts, 256,
                                 room.ctypes.data) == 0
    assert room[0] > 0 and room.sum() < 255, room
    if batch in ("a few", "one large"):  # what fits for all waits for all
        assert (room == room[0]).all()
