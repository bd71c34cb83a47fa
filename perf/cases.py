"""The framework's own workloads as timed passes through its public entry points.

A case names a path and its sizes; prepare() makes its programs from a seed with
the seeded generator and front end (ptilopsis_amd.workloads), run() takes them
through the library once.  Outputs are instruction words, function tables,
DepthTree arrays and text: whole numbers and bytes throughout, so exact() has
no 64-bit value to give and results are compared for equality.

Paths (`path`):
  compile   Context.compile: one program's DepthTree in host arrays, words and
            function table back in host arrays -- what the reference's caller does
            per source file
  resident  one program kept in HBM, its words left in HBM (the plain pipeline of
            the benchmark)
  batch     many programs kept in HBM, compiled in one pass, words left in HBM (the
            batched pipeline of the benchmark); `shape` "base" has sizes log-normal
            around 8k nodes within [1k, 1M], "stress" wide expressions and deeply
            nested statements
  records   Context.compile_arena: a forest of parser records in host arrays, built
            into trees and compiled, results back in host arrays
  tree      Context.tree_build: one program's parser records to DepthTree arrays
  noalloc   ptl_compile_noalloc: device arrays in, the caller's device buffers out
  text      a resident compile and its text, formatted on the device: `form` "asm"
            (to_asm) or "listing" (print's coloured disassembly)
  serve     Server: a burst of requests submitted together and each waited for
"""
from __future__ import annotations

import ctypes as C
import math
import os
import random
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from ptilopsis_amd import abi, workloads as W
from ptilopsis_amd.generator import Context, PtlError, Server
from ptilopsis_amd.native import Arena, parse_arena, parse_source

_LISTED = [
    # the serving stream's smallest program: one short function, host arrays in and out
    dict(name="compile_200", path="compile", nodes=200),
    # the serving stream's median program
    dict(name="compile_4k", path="compile", nodes=4_000),
    # one source file of the single_50k configuration's size
    dict(name="compile_50k", path="compile", nodes=50_000),
    # an ordinary file compiled between device buffers by a caller that may not allocate
    dict(name="noalloc_13k", path="noalloc", nodes=13_337),
    # a large program whose tree stays in HBM
    dict(name="resident_1m", path="resident", nodes=1_000_000, functions=1_250),
    # the benchmark's large_16m configuration, the largest single program
    dict(name="resident_16m", path="resident", nodes=16_000_000, functions=20_000),
    # a quarter of the batch_4096 configuration
    dict(name="batch_1024", path="batch", shape="base", programs=1024, nodes=8_000),
    # a sixteenth of the stress_1024 configuration
    dict(name="stress_64", path="batch", shape="stress", programs=64, nodes=64_000),
    # a build of 60 files, handed over as the parser left them
    dict(name="records_60", path="records", programs=60, nodes=4_000),
    # tree construction alone, for a caller that keeps the DepthTree
    dict(name="tree_2m", path="tree", nodes=2_000_000, functions=2_500),
    # assembly output of one ordinary file
    dict(name="asm_50k", path="text", form="asm", nodes=50_000),
    # the serving stream: 60 requests in the queue at once
    dict(name="serve_60", path="serve", programs=60, nodes=4_000),
]


def listed():
    return [dict(c) for c in _LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    path = rng.choice(["compile", "compile", "resident", "batch", "stress", "records", "tree", "noalloc", "text",
                       "text", "serve"])
    if path == "compile":
        return dict(path=path, nodes=_log(rng, 200, 1_000_000))
    if path == "resident":
        n = _log(rng, 20_000, 8_000_000)
        return dict(path=path, nodes=n, functions=max(9, n // _log(rng, 400, 2_000)))
    if path == "batch":
        return dict(path=path, shape="base", programs=_log(rng, 2, 1000), nodes=8_000)
    if path == "stress":
        return dict(path="batch", shape="stress", programs=_log(rng, 1, 60), nodes=_log(rng, 16_000, 64_000))
    if path in ("records", "serve"):
        return dict(path=path, programs=_log(rng, 1, 60), nodes=_log(rng, 1_000, 16_000))
    if path == "tree":
        n = _log(rng, 300, 2_000_000)
        return dict(path=path, nodes=n, functions=max(1, n // _log(rng, 400, 2_000)))
    if path == "noalloc":
        return dict(path=path, nodes=_log(rng, 300, 200_000))
    return dict(path=path, form=rng.choice(["asm", "listing"]), nodes=_log(rng, 200, 500_000))


# what a program using the library keeps for its lifetime: one context (its
# resident slots shared out to the states alive) and one server
_ctx = None
_server = None
_free_slots = list(range(63, -1, -1))


def _context() -> Context:
    global _ctx
    if _ctx is None:
        _ctx = Context(0)
    return _ctx


class _Resident:
    """A resident slot, given back with the state that holds it."""

    def __init__(self):
        self.slot = _free_slots.pop()

    def __del__(self):
        _free_slots.append(self.slot)


class _Words:
    """The device words of the context's last compile, for torch.as_tensor."""

    def __init__(self, ptr: int, n: int):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), version=2)


def _source(case: dict, seed: int, nodes: int) -> str:
    if "functions" in case:
        return W.sized_source(seed, nodes, case["functions"])
    return W.source_of_size(seed, nodes)


def _sizes(case: dict):
    """Program sizes of a case with several; the seed changes the programs, not how
    large they are."""
    n, at = case["programs"], case["programs"] * 1_000_003 + case["nodes"]
    if case["path"] == "batch":
        return W.request_sizes(n, at, case["nodes"], 1.5, 1_000, 1_000_000)
    # the serving stream's spread (sigma 2.0), its clip scaled down so that a burst
    # stays a burst of requests and not one large program
    return W.request_sizes(n, at, case["nodes"], 2.0, 200, 256_000)


def _nodes(case: dict) -> int:
    """About how many nodes a case's programs have together."""
    if "programs" not in case:
        return case["nodes"]
    if case.get("shape") == "stress":
        return case["programs"] * case["nodes"]
    return int(_sizes(case).sum())


def _programs(one, n: int) -> list:
    """one(0..n-1); the generator and the front end run outside the interpreter lock."""
    if n == 1:
        return [one(0)]
    with ThreadPoolExecutor(min(16, n, os.cpu_count() or 1)) as ex:
        return list(ex.map(one, range(n)))


def _room(case: dict) -> int:
    """Nodes (and words, which are somewhat fewer) that a buffer for a case's results
    holds: a generated program's size is near its target, a small one's less so."""
    return _nodes(case) * 3 // 2 + 4096 * case.get("programs", 1)


def prepare(case: dict, seed: int) -> dict:
    """The programs, where the path keeps them, and the caller's buffers for the
    results, whose unused ends stay zero."""
    path = case["path"]
    room = _room(case)
    base = (seed + 1) << 20
    s = dict(path=path, ctx=_context())
    if path in ("compile", "resident", "text", "noalloc"):
        tree = parse_source(_source(case, base, case["nodes"]))
        if path == "compile":
            s["tree"] = tree
        elif path == "noalloc":
            s["n"], s["max_depth"] = tree.n, tree.max_depth
            s["in"] = [torch.from_numpy(np.ascontiguousarray(a).view(np.uint8)).cuda() for a in tree.arrays()]
            s["out"] = torch.zeros(room, dtype=torch.int32, device="cuda")
            s["funcs"] = [torch.zeros(room // 8, dtype=torch.int32, device="cuda") for _ in range(4)]
        else:
            s["form"] = case.get("form")
            s["res"] = _Resident()
            s["ctx"].upload(s["res"].slot, tree)
    elif path == "batch":
        if case["shape"] == "stress":
            trees = _programs(lambda p: W.stress_program(base + p, case["nodes"]), case["programs"])
        else:
            sizes = _sizes(case)
            trees = _programs(lambda p: W.program_of_size(base + p, int(sizes[p])), case["programs"])
        s["res"] = _Resident()
        s["n"] = len(trees)
        s["ctx"].upload_batch(s["res"].slot, trees)
    elif path == "serve":
        sizes = _sizes(case)
        s["trees"] = _programs(lambda p: W.program_of_size(base + p, int(sizes[p])), case["programs"])
        global _server
        if _server is None:
            _server = Server(0)
    elif path == "records":
        sizes = _sizes(case)
        s["arena"] = Arena.concat(_programs(lambda p: parse_arena(W.source_of_size(base + p, int(sizes[p]))),
                                            case["programs"]))
    elif path == "tree":
        s["arena"] = parse_arena(_source(case, base, case["nodes"]))
    else:
        raise ValueError(path)
    if path in ("resident", "batch"):
        s["out"] = torch.zeros(room, dtype=torch.int32, device="cuda")
    elif path == "text":
        s["out"] = np.zeros(room * (32 if s["form"] == "asm" else 240), np.uint8)
    elif path == "tree":
        s["out"] = [np.zeros(room, t) for t in (np.uint8, np.uint8, np.int32, np.int32, np.int32, np.uint32)]
    elif path != "noalloc":
        s["out"] = np.zeros(room, np.int32)
    return s


_FUNCS = ("func_ids", "func_starts", "func_ends", "func_sizes")


def _gather(out, results: list) -> list:
    """The programs' words one after the other in the caller's buffer, and their
    function tables."""
    at = 0
    for r in results:
        w = r["words"]
        out[at:at + w.shape[0]] = w.view(np.int32)
        at += w.shape[0]
    tabs = [[r[k].view(np.int32) for r in results] for k in _FUNCS]
    return [out, np.array([r["n_words"] for r in results]), [np.concatenate(t) for t in tabs]]


def _take(s: dict, n: int):
    """The words of the context's last compile moved into the caller's buffer on the
    device; the context's next call may overwrite them, so the copy is waited for."""
    ctx = s["ctx"]
    s["out"][:n].copy_(torch.as_tensor(_Words(ctx.lib.ptl_result_device(ctx.h), n), device="cuda"))
    torch.cuda.current_stream().synchronize()
    return s["out"]


def run(s: dict):
    path, ctx = s["path"], s["ctx"]
    if path == "compile":
        return _gather(s["out"], [ctx.compile(s["tree"])])
    if path == "resident":
        r = ctx.compile_resident(s["res"].slot, copy_out=False)
        return [_take(s, r["n_words"]), r["n_words"], r["n_funcs"], r["W0"], r["W1"]]
    if path == "batch":
        out = (abi.PtlResult * s["n"])()
        st = ctx.lib.ptl_compile_resident_batch(ctx.h, s["res"].slot, 0, out)
        if st != abi.PTL_OK:
            raise PtlError(st)
        v = np.frombuffer(out, np.int64).reshape(s["n"], -1)[:, abi.PtlResult.n_words.offset // 8].copy()
        return [_take(s, int(v.sum())), v]
    if path == "noalloc":
        a = abi.PtlAst(*[t.data_ptr() for t in s["in"]], s["n"], s["max_depth"])
        r = abi.PtlResult()
        st = ctx.lib.ptl_compile_noalloc(ctx.h, C.byref(a), s["out"].data_ptr(), s["out"].shape[0],
                                         *[f.data_ptr() for f in s["funcs"]], s["funcs"][0].shape[0], C.byref(r))
        if st != abi.PTL_OK:
            raise PtlError(st)
        return [s["out"], r.n_words, s["funcs"], r.n_funcs]
    if path == "records":
        return _gather(s["out"], ctx.compile_arena(s["arena"]))
    if path == "tree":
        t = ctx.tree_build(s["arena"])[0]
        for o, a in zip(s["out"], t.arrays()):
            o[:t.n] = a
        return s["out"][:5] + [s["out"][5].view(np.int32), t.n]
    if path == "text":
        ctx.compile_resident(s["res"].slot, copy_out=False)
        txt = np.frombuffer(ctx.result_asm(0) if s["form"] == "asm" else ctx.result_listing(0), np.uint8)
        s["out"][:txt.shape[0]] = txt
        return [s["out"], txt.shape[0]]
    tickets = [_server.submit(t) for t in s["trees"]]
    return _gather(s["out"], [_server.wait(t)[0] for t in tickets])


def work(case: dict) -> dict:
    """Bytes in and out of one pass: 18 per node of a tree (two types, parent,
    depth, child index, data), 18 per record and its one kid entry of 4 before
    construction, 4 per word (about 0.95 words a node), 16 per function table row
    (about 800 nodes a function), about 18 per line of assembly and 200 per line of
    listing."""
    path, n = case["path"], _nodes(case)
    out = 4 * 0.95 * n + 16 * (n / 800 + 1)
    if path == "tree":
        return dict(bytes=(18 + 18) * n, flops=0)
    if path == "records":
        return dict(bytes=(18 + 18) * n + out, flops=0)
    if path == "text":
        return dict(bytes=18 * n + (18 if case["form"] == "asm" else 200) * 0.95 * n, flops=0)
    return dict(bytes=18 * n + out, flops=0)


def exact(case: dict, seed: int):
    return None
