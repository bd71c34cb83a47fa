// MI355X (gfx950) implementation of the reference's data-parallel RISC-V code
// generator: rv_generator_avx with one thread (src/codegen/rv_generator_avx.cpp),
// stage for stage, bit-exact.
//
// Every stage is integer gather/scatter/scan work bound by HBM bandwidth; no
// stage is a dense contraction.  Arrays are structure-of-arrays in HBM; u8 for
// node and data types, u32 elsewhere.  Stages and where their semantics come from:
//
//   preprocess   k_pre12 (passes 1+2, :126-266), k_pre3 (pass 3, :270-305)
//   isn_cnt      k_scan<CountOp> (count :315-369 + exclusive scan :374-392),
//                k_cnt_fix (:398-447), function table (:451-515)
//   isn_gen      k_gen_regs (parent-slot propagation) then k_gen_owner /
//                k_gen_write (:584-886).  The reference walks depth levels
//                bottom-up, but every parent slot has one writer and is read
//                only by its parent, so both passes run over all nodes at once;
//                word slots written by more than one node go to the writer the
//                reference writes last: the shallowest node, then the later one
//                in the reference's depth sort (its libstdc++ std::sort order,
//                reproduced exactly by the introsort kernels below).
//   optimize     k_opt_init + k_opt_iter (:891-1016), a chaotic in-place
//                iteration of the same monotone operator; it reaches the same
//                greatest fixpoint as the reference's two-copy iteration.
//   regalloc     k_ra_walk (functions not in lane 0 of an 8-function group:
//                independent), k_ra_lane0_wave / k_ra_lane0 (lane-0 functions in
//                step lockstep: they share the first 64-entry region of the
//                reference's register_state snapshot, :1290-1354), k_ra_serial (exact
//                in-order walk for programs where a function names a register that
//                another defines), then counts, scan, emit (:1422-1697), function table
//                fix and frame words (:1714-1811).
//   fix_jumps    size + scan + fused move/encode/postprocess (:1853-1993, 1995-2011).
//
// Batches: P programs concatenated node-wise run through the same kernels.
// Each element finds its program by binary search in the program tables (node,
// word and function bases); isn_gen computes in the program's own word indices
// (register numbers are ORed with them) and then offsets virtual registers and
// jump targets by the program's word base, so every program's words are
// exactly those of its own compile, back to back.
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <chrono>
#include <string>
#include <vector>
#include <algorithm>
#include <future>
#include <mutex>
#include <type_traits>

#include "rv_spec.h"
#include "../../include/ptl.h"

#define DEV __device__ __forceinline__

// ---------------------------------------------------------------- constants
__constant__ uint32_t c_word[RV_NTYPES * 4 * 6];
__constant__ uint32_t c_bits[RV_NTYPES * 4 * 6];
__constant__ uint8_t c_dense[256];
__constant__ uint8_t c_pareas[44];

DEV uint32_t spec_i(uint32_t ty, uint32_t o, uint32_t rt) { return ((uint32_t)c_dense[ty] * 4u + o) * 6u + rt; }
DEV uint32_t size_of(uint32_t ty, uint32_t rt) { return (c_bits[spec_i(ty, 0, rt)] >> 19) & 7u; }

// error flags raised by kernels (bit set in ctx->d_flags)
// EF_XCONFLICT: some program has a word in none of the forms the allocation
// walks take (ra_op); those programs are allocated by k_ra_serial.
// EF_WAIT: the allocation lockstep gave up waiting for the concurrent walk's rows.
enum : uint32_t { EF_OOB = 1, EF_CALLPATH = 4, EF_XCONFLICT = 32, EF_WAIT = 64 };

// ------------------------------------------------------------------ helpers
// Workgroup barrier that orders LDS only: global loads and stores stay in
// flight across it.  Correct where every global location a thread reads was
// last written by that same thread (program order covers it) or before the
// kernel started, and where global atomics are read only by later kernels.
DEV void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Program of element i given the programs' bases (last p with base[p] <= i).
DEV uint32_t prog_of(const uint32_t *base, uint32_t P, uint32_t i) {
    uint32_t lo = 0, hi = P;
    while (hi - lo > 1) { const uint32_t m = (lo + hi) >> 1; if (base[m] <= i) lo = m; else hi = m; }
    return lo;
}

// The same where neighbouring lanes look up neighbouring elements (node- or
// word-parallel kernels): one search for the wave's first active lane, on a
// wave-uniform index, then each lane steps from there to its own program (the
// programs are long against a wave, so mostly no step).
DEV uint32_t prog_of_w(const uint32_t *base, uint32_t P, uint32_t i) {
    const uint32_t i0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)i);
    uint32_t p = prog_of(base, P, i0);
    while (p > 0 && base[p] > i) --p;
    while (p + 1 < P && base[p + 1] <= i) ++p;
    return p;
}

DEV uint32_t ffz_gcc(uint64_t v) {
    // include/utils.hpp:25-45 as compiled by GCC: __builtin_ffs(int) of ~val sees 32 bits.
    uint32_t low = (uint32_t)(~v);
    return low == 0 ? 64u : (uint32_t)__builtin_ctz(low);
}

template <typename T>
__global__ void k_fill(T *p, uint64_t n, T v) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// Several fills in one launch (a launch takes longer than most of them): words of
// 256-byte aligned ranges, four a thread and step.
struct ClearRange { uint32_t *p; uint64_t n; uint32_t v; };
struct ClearList { ClearRange r[8]; uint32_t count; };
__global__ __launch_bounds__(256) void k_clear(ClearList L, uint64_t quads) {
    const uint64_t stride = (uint64_t)gridDim.x * 256u;
    for (uint64_t i = blockIdx.x * (uint64_t)256 + threadIdx.x; i < quads; i += stride) {
        uint64_t q = i;
        for (uint32_t k = 0; k < L.count; ++k) {
            const uint64_t nq = (L.r[k].n + 3u) / 4u;
            if (q >= nq) { q -= nq; continue; }
            uint32_t *p = L.r[k].p + 4u * q;
            const uint32_t v = L.r[k].v, m = (uint32_t)min((uint64_t)4, L.r[k].n - 4u * q);
            if (m == 4u && (reinterpret_cast<uint64_t>(p) & 15u) == 0u) *reinterpret_cast<uint4 *>(p) = make_uint4(v, v, v, v);
            else for (uint32_t y = 0; y < m; ++y) p[y] = v;
            break;
        }
    }
}

// Words from different places, then two arrays of n, to consecutive (pinned host) words.
struct GatherList { const uint32_t *p[8]; uint32_t count; };
__global__ void k_gather(GatherList g, const uint32_t *a, const uint32_t *b, uint32_t n, uint32_t *dst) {
    if (threadIdx.x < g.count) dst[threadIdx.x] = *g.p[threadIdx.x];
    for (uint32_t i = threadIdx.x; i < 2u * n; i += blockDim.x) dst[g.count + i] = i < n ? a[i] : b[i - n];
}
// The words and the four function arrays of a small result, likewise.
__global__ __launch_bounds__(256) void k_gather_result(const uint32_t *words, uint32_t nw, const uint32_t *f0,
                                                       const uint32_t *f1, const uint32_t *f2, const uint32_t *f3,
                                                       uint32_t nf, uint32_t *dst) {
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < nw + 4u * nf; i += gridDim.x * 256u) {
        uint32_t k = i, v;
        if (k < nw) v = words[k];
        else {
            k -= nw;
            v = k < nf ? f0[k] : k < 2u * nf ? f1[k - nf] : k < 3u * nf ? f2[k - 2u * nf] : f3[k - 3u * nf];
        }
        dst[i] = v;
    }
}

// A plain streaming copy (16 B per thread and step, grid-stride), for the
// measured HBM bandwidth the stages are reported against.
__global__ __launch_bounds__(256) void k_copy16(const uint4 *a, uint4 *b, uint64_t n) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += stride) b[i] = a[i];
}

static inline uint32_t grid_for(uint64_t n, uint32_t block) {
    uint64_t g = (n + block - 1) / block;
    if (g == 0) g = 1;
    return (uint32_t)std::min<uint64_t>(g, 0x7FFFFFFFull);
}

// ------------------------------------------------------- reduce-then-scan
// Exclusive u32 scan over n elements in three launches with no inter-block
// waiting: per-tile sums, one workgroup scanning the tile sums, then each tile
// rescans its elements with its offset.  A tile is 256 threads x 16 items.
// Elements are produced striped (element k*256 + t by thread t, so every load
// of Op::value is coalesced) and, for the rescan, transposed through LDS so
// that each thread owns 16 consecutive elements, which a wave64 shuffle scan
// and LDS combine.  Op::value(i) produces element i, Op::emit(i, exclusive,
// value) consumes the result.
constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 16;
constexpr uint64_t SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

DEV uint32_t wave_incl_scan(uint32_t x, uint32_t lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(x, d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
    return x;
}

DEV uint32_t wave_sum(uint32_t x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

template <class Op>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(Op op, uint64_t n, uint32_t *tile_sums) {
    __shared__ uint32_t s_w[SCAN_BLOCK / 64];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        uint64_t i = base + (uint64_t)k * SCAN_BLOCK;
        if (i < n) sum += op.value(i);
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
#pragma unroll
        for (int w = 0; w < SCAN_BLOCK / 64; ++w) t += s_w[w];
        tile_sums[blockIdx.x] = t;
    }
}

// One workgroup: exclusive scan of the tile sums in place; the grand total to *total.
__global__ __launch_bounds__(1024) void k_scan_tiles(uint32_t *sums, uint32_t ntiles, uint32_t *total) {
    __shared__ uint32_t s_w[16];
    __shared__ uint32_t s_carry;
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    for (uint32_t b = 0; b < ntiles; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = i < ntiles ? sums[i] : 0u;
        const uint32_t x = wave_incl_scan(v, lane);
        if (lane == 63) s_w[wid] = x;
        __syncthreads();
        uint32_t pre = s_carry, all = 0;
        for (uint32_t w = 0; w < 16; ++w) { if (w < wid) pre += s_w[w]; all += s_w[w]; }
        if (i < ntiles) sums[i] = pre + x - v;
        __syncthreads();
        if (threadIdx.x == 0) s_carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0 && total) *total = s_carry;
}

// The rescan of one tile: v[k] = element base + k of this thread (base = tile
// start + 16 * thread), and the exclusive prefix of its first element.
template <class Op>
DEV uint32_t scan_tile(const Op &op, uint64_t n, const uint32_t *tile_pre, uint32_t *s_w, uint32_t *s_v,
                       uint32_t (&v)[SCAN_ITEMS]) {
    const uint64_t tb = (uint64_t)blockIdx.x * SCAN_TILE;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t e = (uint32_t)k * SCAN_BLOCK + threadIdx.x;
        s_v[e + e / 16u] = tb + e < n ? op.value(tb + e) : 0u;  // element e at e + e/16 (one pad word per 16)
    }
    __syncthreads();
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        v[k] = s_v[threadIdx.x * (SCAN_ITEMS + 1) + k];  // element t*16 + k
        sum += v[k];
    }
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(sum, lane);
    if (lane == 63) s_w[wid] = x;
    __syncthreads();
    uint32_t run = tile_pre[blockIdx.x] + x - sum;
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / 64; ++w) if ((uint32_t)w < wid) run += s_w[w];
    return run;
}

template <class Op>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_down(Op op, uint64_t n, const uint32_t *tile_pre) {
    __shared__ uint32_t s_w[SCAN_BLOCK / 64];
    __shared__ uint32_t s_v[SCAN_TILE + SCAN_TILE / 16];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint32_t run = scan_tile(op, n, tile_pre, s_w, s_v, v);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        uint64_t i = base + k;
        if (i < n) op.emit(i, run, v[k]);
        run += v[k];
    }
}

// ------------------------------------------------------- single-pass scan
// The same exclusive scan in one launch with decoupled look-back: each element
// is produced once.  A workgroup takes the next tile from a ticket counter, so
// tiles start in order and every tile it waits on is already running; it
// scans its tile as above, publishes the tile's aggregate, and wave 0 looks
// back over the published words of its predecessors 64 at a time, summing
// aggregates back to the nearest inclusive prefix (tile -1 counts as an
// inclusive 0) and waiting while a nearer word is unpublished.  It then
// publishes its own inclusive prefix and the tile emits.  Status word of a
// tile: value | flag << 32 (1 aggregate, 2 inclusive), all zero before the
// launch; the ticket counter is the word after the last tile's.  A status
// word carries its own value, so no other data is ordered by it: the stores
// and polls are relaxed device-scope atomics.
constexpr uint64_t SCAN_AGG = 1ull << 32, SCAN_INCL = 2ull << 32;

template <class Op>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_dlb(Op op, uint64_t n, unsigned long long *status,
                                                         uint32_t ntiles, uint32_t *total) {
    __shared__ uint32_t s_w[SCAN_BLOCK / 64];
    __shared__ uint32_t s_v[SCAN_TILE + SCAN_TILE / 16];
    __shared__ uint32_t s_tile, s_pre;
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_tile = atomicAdd(reinterpret_cast<uint32_t *>(status + ntiles), 1u);
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint64_t tb = (uint64_t)tile * SCAN_TILE;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t e = (uint32_t)k * SCAN_BLOCK + threadIdx.x;
        s_v[e + e / 16u] = tb + e < n ? op.value(tb + e) : 0u;  // element e at e + e/16 (one pad word per 16)
    }
    __syncthreads();
    uint32_t v[SCAN_ITEMS], sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        v[k] = s_v[threadIdx.x * (SCAN_ITEMS + 1) + k];  // element t*16 + k
        sum += v[k];
    }
    const uint32_t x = wave_incl_scan(sum, lane);
    if (lane == 63) s_w[wid] = x;
    __syncthreads();
    uint32_t agg = 0, run = x - sum;
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / 64; ++w) {
        agg += s_w[w];
        if ((uint32_t)w < wid) run += s_w[w];
    }
    if (wid == 0) {
        if (lane == 0)
            __hip_atomic_store(status + tile, (unsigned long long)agg | (tile == 0 ? SCAN_INCL : SCAN_AGG),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t pre = 0;
        int64_t j = (int64_t)tile - 1;  // nearest predecessor not yet summed (lane 0 reads it)
        while (j >= 0) {
            const int64_t idx = j - (int64_t)lane;
            const unsigned long long st =
                idx >= 0 ? __hip_atomic_load(status + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : SCAN_INCL;
            const uint64_t incl = __ballot((st >> 32) == 2u), none = __ballot((st >> 32) == 0u);
            const uint32_t stop = incl ? (uint32_t)__builtin_ctzll(incl) : 64u;
            if (none && (uint32_t)__builtin_ctzll(none) < stop) {  // a nearer tile has not published yet
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            pre += wave_sum(lane <= stop ? (uint32_t)st : 0u);
            if (incl) break;
            j -= 64;
        }
        if (lane == 0) {
            if (tile > 0)
                __hip_atomic_store(status + tile, (unsigned long long)(pre + agg) | SCAN_INCL, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            s_pre = pre;
            if (total && tile == ntiles - 1) *total = pre + agg;
        }
    }
    __syncthreads();
    run += s_pre;
    const uint64_t base = tb + (uint64_t)threadIdx.x * SCAN_ITEMS;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint64_t i = base + k;
        if (i < n) op.emit(i, run, v[k]);
        run += v[k];
    }
}

// ----------------------------------------------------------- device state
struct Dev {
    // inputs: P programs concatenated node-wise, parents global
    const uint8_t *pt, *prt;
    const int32_t *par, *depth, *cidx;
    const uint32_t *ndin;
    uint64_t n;
    uint32_t maxd;           // largest max depth of the programs
    uint32_t P;
    const uint32_t *pn;      // node base of each program (P+1)
    uint32_t *pw;            // word base of each program after isn_gen (P+1)
    uint32_t *pf;            // function base of each program (P+1)
    // preprocess / isn_cnt
    uint8_t *ty8, *rt8;
    uint32_t *nd;
    uint32_t *loc;
    uint32_t *decl;          // func_decl node indices, F
    uint32_t *fids, *fstarts, *fsizes, *fends;
    uint32_t F;
    // isn_gen
    uint32_t *regs;          // 3n
    uint32_t *rank;          // n (sorted position of each node)
    uint32_t *rinv;          // n (node at each sorted position), with rank
    uint64_t *owner;         // W0
    uint32_t W0;
    uint32_t *w0_instr, *w0_rd, *w0_rs1, *w0_rs2, *w0_jt;
    // optimize
    uint8_t *used, *sstore, *usedi;
    // regalloc
    uint4 *w0_f4;            // per word: rd, rs1, rs2, instruction (one 16-byte load)
    uint32_t *ops;           // per word: what the allocation walks need of it (ra_op)
    uint16_t *sym;           // per virtual register: assigned register | swapped << 8 | (lane-0 walks) the
                             // register it was defined in << 9
    uint32_t *cflag;         // per program: it is allocated by k_ra_serial
    uint32_t *ra_off;
    uint32_t W1;
    uint32_t *w1_instr, *w1_rd, *w1_rs1, *w1_rs2, *w1_jt;
    // fix_jumps
    uint32_t *fj_off;
    uint32_t W2;
    uint32_t *words;
    uint32_t *flags;
    uint32_t *counter;
};

// ================================================================ preprocess
DEV void classify(uint32_t &ty, uint32_t rt, uint32_t ci, uint32_t &nd) {
    if ((ty & 0xF0u) != 0xF0u) return;
    if (rt == DT_FLOAT || rt == DT_FLOAT_REF) {
        bool comp = (int32_t)nd > 7;
        uint32_t reg = ci - 8u;
        bool stk = (int32_t)reg > 7 && comp;
        bool asint = !stk && comp;
        if (stk) ty |= 2u;
        if (asint) ty |= 1u;
        if (stk) reg -= 8u;
        if (comp) nd = reg;
    } else {
        uint32_t id = nd, fa = ci - id;
        uint32_t reg = id + (fa - ((int32_t)fa > 7 ? 8u : 0u));
        uint32_t osm = ((int32_t)reg > 7 ? 0xFFFFFFFFu : 0u) & id;  // ANDed with the value (D9)
        ty |= osm & 2u;
        reg -= 8u & osm;
        nd = reg;
    }
}

// Passes 1 and 2.  Pass 2's stores are gated by "the 8-node vector holds a
// call-argument list" but not masked by it (:236-262): 8-lane groups of the
// wave64 ballot are exactly the reference's 8-node vectors.
__global__ __launch_bounds__(256) void k_pre12(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    uint32_t ty = 0, rt = 0, ci = 0, nd = 0;
    bool in = i < d.n;
    if (in) {
        ty = c_pareas[d.pt[i]]; rt = d.prt[i]; ci = (uint32_t)d.cidx[i]; nd = d.ndin[i];
        classify(ty, rt, ci, nd);
    }
    if (!in) return;
    // does the node's 8-node vector (counted from its program's first node)
    // hold a call argument list?
    const uint32_t prg = prog_of_w(d.pn, d.P, (uint32_t)i);
    const uint32_t v0 = d.pn[prg] + (((uint32_t)i - d.pn[prg]) & ~7u), v1 = min(v0 + 8u, d.pn[prg + 1]);
    bool block_has_list = false;
    for (uint32_t j = v0; j < v1; ++j) block_has_list |= c_pareas[d.pt[j]] == RV_CALL_ARGS;
    if (block_has_list && (uint32_t)i > d.pn[prg]) {
        uint64_t j = i - 1;
        uint32_t pty = c_pareas[d.pt[j]], prt = d.prt[j], pci = (uint32_t)d.cidx[j], pnd = d.ndin[j];
        classify(pty, prt, pci, pnd);
        if (pty == RV_CARG_STK) nd = pnd + 1u;
        else if (pty == RV_CARG && prt == DT_FLOAT) {
            int32_t ia = (int32_t)(pci - pnd) - 8;
            nd = (uint32_t)(ia > 0 ? ia : 0);
        }
    }
    d.ty8[i] = (uint8_t)ty;
    d.rt8[i] = (uint8_t)rt;
    d.nd[i] = nd;
}

// Pass 3 (:270-305): a FLOAT node marks its comparison-like parent FLOAT; the
// parent passes it on only if it sits in a later 8-node vector than the child
// (within one vector the scatter lands after the vector's load).
__global__ __launch_bounds__(256) void k_pre3(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.n || d.prt[i] != DT_FLOAT) return;
    const uint32_t b = d.pn[prog_of_w(d.pn, d.P, (uint32_t)i)];  // vectors count from the program's first node
    uint64_t cur = i;
    for (;;) {
        int32_t p = d.par[cur];
        if (p < 0) break;
        if ((d.ty8[p] & 0xE0u) != 0xE0u) break;
        d.rt8[p] = DT_FLOAT;
        if (((cur - b) >> 3) < (((uint64_t)p - b) >> 3)) cur = (uint64_t)p;
        else break;
    }
}

// ================================================================== isn_cnt
struct CountOp {
    Dev d;
    DEV uint32_t value(uint64_t i) const {
        uint32_t ty = d.ty8[i], rt = d.rt8[i];
        uint32_t s = size_of(ty, rt);
        if (ty == RV_CALL_ARGS) {
            s += 1;
            if (i > 0 && (d.ty8[i - 1] & 0xF4u) == 0xF4u) s += (uint32_t)d.cidx[i - 1] + 1u;
        }
        int32_t p = d.par[i];
        uint32_t pty = d.ty8[p != -1 ? (uint32_t)p : d.pn[prog_of(d.pn, d.P, (uint32_t)i)]];  // root: the program's node 0
        int32_t ci = d.cidx[i];
        bool ife = pty == RV_IF_ELSE;
        if (ci == 0 && (ife || pty == RV_IF)) s += 1;
        if (ci == 1 && (ife || pty == RV_WHILE)) s += 1;
        return s;
    }
    DEV void emit(uint64_t i, uint32_t excl, uint32_t) const { d.loc[i] = excl; }
};

// The counts alone (the generator's node_sizes member), for the debug print.
__global__ void k_node_sizes(Dev d, uint32_t *out) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i < d.n) out[i] = CountOp{d}.value(i);
}

// Location fix (:398-447).  A condition child moves its control-flow parent
// right after its own base words; call arguments then move to their slot in the
// argument list, which always wins over the first rule at one thread.
__global__ __launch_bounds__(256) void k_cnt_fix(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    int32_t p = d.par[i];
    uint32_t ty = d.ty8[i];
    uint32_t ci = (uint32_t)d.cidx[i];
    if (p > -1) {
        uint32_t pty = d.ty8[p];
        bool cond = ((pty & 0xD0u) == 0xD0u) && ci == (pty & 1u);
        if (cond && (pty & 0xF4u) != 0xF4u) d.loc[p] = d.loc[i] + size_of(ty, d.rt8[i]);
    }
    if ((ty & 0xF4u) == 0xF4u && p > -1) d.loc[i] = d.loc[p] + ci + 1u;
}

struct DeclOp {
    Dev d;
    DEV uint32_t value(uint64_t i) const { return d.ty8[i] == RV_FDECL ? 1u : 0u; }
    DEV void emit(uint64_t i, uint32_t excl, uint32_t v) const { if (v) d.decl[excl] = (uint32_t)i; }
};

// Every program's first position starts an insertion-sort leaf.
__global__ void k_prog_bounds(uint8_t *bound, const uint32_t *pn, uint32_t P) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < P) bound[pn[p]] = 1;
}

// Batched input: parents arrive local to their program's node range.
__global__ void k_globalize_parents(int32_t *par, uint64_t n, const uint32_t *pn, uint32_t P) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t p = par[i];
    if (p >= 0) par[i] = p + (int32_t)pn[prog_of_w(pn, P, (uint32_t)i)];
}

// Word base of every program: the exclusive count scan at its first node (the
// location fix does not move a program's first node); total at P.
__global__ void k_prog_words(Dev d, const uint32_t *total) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > d.P) return;
    d.pw[p] = p < d.P ? d.loc[d.pn[p]] : *total;
}

// Function base of every program: functions (decl nodes, in node order) before
// its first node.
__global__ void k_prog_funcs(Dev d, const uint32_t *F) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > d.P) return;
    const uint32_t b = p < d.P ? d.pn[p] : (uint32_t)d.n;
    uint32_t lo = 0, hi = *F;  // first decl index >= b
    while (lo < hi) { const uint32_t m = (lo + hi) >> 1; if (d.decl[m] < b) lo = m + 1; else hi = m; }
    d.pf[p] = lo;
}

// Function table (:451-515): ids = node data, starts = previous decl location + 6.
__global__ void k_functab(Dev d) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= d.F) return;
    uint32_t dn = d.decl[k];
    uint32_t off = 6u + d.loc[dn];
    const uint32_t prg = prog_of(d.pf, d.P, k);
    uint32_t prev = k > d.pf[prg] ? 6u + d.loc[d.decl[k - 1]] : d.pw[prg];
    d.fids[k] = d.nd[dn];
    d.fstarts[k] = prev;
    d.fsizes[k] = off - prev;
    d.fends[k] = off;
}

// =================================================================== isn_gen
struct Lane {
    bool has;
    int32_t pai;
    uint32_t dpv, loc, word, rd, rs1, rs2, jt, wb;
};

// The inputs of one node that all four of its lanes share, loaded once: its
// program (word base, function base and count), types, parent, parent type,
// child index, location and data.
struct GenNode {
    uint32_t nn, prg, wb, fb, Fp, wn, ty, rt, ci, loc, ndv, pty;
    int32_t par;
};

DEV GenNode gen_node(const Dev &d, uint32_t nn) {
    GenNode N;
    N.nn = nn;
    N.prg = prog_of_w(d.pn, d.P, nn);
    N.wb = d.pw[N.prg]; N.wn = d.pw[N.prg + 1] - N.wb;
    N.fb = d.pf[N.prg]; N.Fp = d.pf[N.prg + 1] - N.fb;
    N.ty = d.ty8[nn]; N.rt = d.rt8[nn];
    N.par = d.par[nn];
    N.pty = N.par != -1 ? d.ty8[N.par] : 0u;
    N.ci = (uint32_t)d.cidx[nn];
    N.loc = d.loc[nn];
    N.ndv = d.nd[nn];
    return N;
}

// One (node, offset) lane of the level loop body (:585-884), computed in the
// word indices of the node's own program (register numbers are ORed with word
// indices, :676-697, :842); L.loc is the global word slot.
DEV void gen_lane(const Dev &d, const GenNode &N, uint32_t o, bool full, Lane &L) {
    const uint32_t nn = N.nn, wb = N.wb, fb = N.fb, Fp = N.Fp, ty = N.ty, rt = N.rt;
    const uint32_t si = spec_i(ty, o, rt);
    const uint32_t b = c_bits[si];
    const bool has = b & 1u;
    const bool prop = has || o == 0;
    const int32_t par = prop ? N.par : 0;
    const bool nopar = par == -1;
    const bool lfp = !nopar && prop;
    const uint32_t pty = lfp ? N.pty : 0u;
    const uint32_t ci = lfp ? N.ci : 0u;
    const bool noncond = ((pty & 0xD0u) == 0xD0u) && !(ci == (pty & 1u));
    bool call = noncond;
    if ((nopar || !noncond) && prop) {
        uint32_t ct = (b >> 2) & 3u;
        if (ct == 1) call = true;
        if (ct == 2 && (int32_t)rt > 1) call = true;
    }
    L.has = has;
    L.pai = call ? (int32_t)((uint32_t)par * 3u + ci) : -1;
    const uint32_t iib = o + (prop ? N.loc - wb : 0u);
    uint32_t rd = 0;
    const uint32_t ndv = N.ndv;
    if (has) {
        uint32_t ct = (b >> 4) & 7u;
        if (ct == 3) rd |= 32u;
        if (ct == 4) rd |= 10u;
        if (ct == 1) rd |= ndv + 10u;
        if (ct == 2) rd |= ndv + 42u;
        bool hov = call || (ct == 0 && ((b >> 1) & 1u));
        if (hov) rd |= iib + 64u;
    }
    const bool use_rd = nopar || (!noncond && lfp);
    const uint32_t instr_no = iib + (noncond ? ((b >> 19) & 7u) : 0u);
    L.dpv = (use_rd ? rd : 0u) | (noncond ? instr_no : 0u);
    if (!full || !has) { L.rd = rd; return; }
    uint32_t iloc = iib;
    if (o == 1 && ty == RV_IF_ELSE) iloc = d.regs[(uint64_t)nn * 3 + 1];
    if (o == 1 && ty == RV_WHILE) iloc = d.regs[(uint64_t)nn * 3 + 2];
    const bool add2 = ty == RV_FDECL || (o > 1 && ty == RV_FDECL_DUMMY);
    const bool cal1 = o == 1 && ty == RV_CALL_ARGS;
    if (add2 || cal1) iloc += 2u;
    if (cal1 && nn > 0) {
        uint32_t ppt = d.ty8[nn - 1];
        if ((ppt & 0xF4u) == 0xF4u) iloc += (uint32_t)d.cidx[nn - 1];
    }
    uint32_t word = c_word[si];
    const uint32_t cc = (b >> 13) & 7u;
    const uint32_t nd4 = ndv * 4u;
    if (cc == 1) word |= ndv & 0xFFFFF000u;
    if (cc == 2) word |= (ndv & 0xFFFu) << 20;
    if (cc == 3) word |= (0u - (nd4 + 8u)) << 20;
    if (cc == 4) word |= nd4 << 20;
    if (cc == 5) word |= (0u - nd4) << 20;
    const uint32_t jc = (b >> 16) & 7u;
    uint32_t jt = 0;
    if (jc >= 1 && jc <= 5) jt = d.regs[(uint64_t)nn * 3 + 1 + (jc > 2 ? 1 : 0)] + ((jc & 1u) == 0 ? 1u : 0u);
    if (jc == 6) { if (ndv < Fp) jt |= d.fends[fb + ndv] - wb - 6u; else atomicOr(d.flags, EF_OOB); }
    if (jc == 7) { if (ndv < Fp) jt |= d.fstarts[fb + ndv] - wb; else atomicOr(d.flags, EF_OOB); }
    uint32_t rs[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        uint32_t oc = (b >> (7 + 3 * s)) & 7u;
        uint32_t arg = 0;
        if (oc == 1 || oc == 4 || oc == 5 || oc == 6) {
            uint64_t ri = (uint64_t)nn * 3;
            if (oc == 1) ri += s;
            if (oc == 4 || oc == 5) ri += 1;
            if (oc == 5) ri -= s;
            arg = d.regs[ri];
        }
        if (oc == 2) arg |= ndv + 10u;
        if (oc == 3) arg |= ndv + 42u;
        if (oc == 7) arg |= iib + 63u;
        rs[s] = arg;
    }
    L.loc = iloc + wb; L.word = word; L.rd = rd; L.rs1 = rs[0]; L.rs2 = rs[1]; L.jt = jt;
    L.wb = wb;
}

// Parent-slot propagation: the last propagating lane of a node wins the slot.
__global__ __launch_bounds__(256) void k_gen_regs(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    int32_t slot = -1; uint32_t val = 0;
    const GenNode N = gen_node(d, (uint32_t)i);
    for (uint32_t o = 0; o < 4; ++o) {
        Lane L;
        gen_lane(d, N, o, false, L);
        if (L.pai >= 0) { slot = L.pai; val = L.dpv; }
    }
    if (slot >= 0) {
        if ((uint64_t)slot < d.n * 3) d.regs[slot] = val;
        else atomicOr(d.flags, EF_OOB);
    }
}

DEV uint64_t owner_key(const Dev &d, uint32_t nn, uint32_t o, bool use_rank) {
    uint64_t level = (uint64_t)(d.maxd - (uint32_t)d.depth[nn]) + 1u;
    uint64_t r = use_rank ? d.rank[nn] : nn;
    return (level << 34) | (r << 2) | o;
}

__global__ __launch_bounds__(256) void k_gen_owner(Dev d, int use_rank) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    const GenNode N = gen_node(d, (uint32_t)i);
    const uint64_t k0 = owner_key(d, (uint32_t)i, 0, use_rank != 0);
    for (uint32_t o = 0; o < 4; ++o) {
        Lane L;
        gen_lane(d, N, o, true, L);
        if (!L.has) continue;
        if (L.loc >= d.W0) { atomicOr(d.flags, EF_OOB); continue; }
        atomicMax((unsigned long long *)&d.owner[L.loc], (unsigned long long)(k0 | o));
    }
}

// Counts slots won by one node but also written by another node of equal depth.
__global__ __launch_bounds__(256) void k_gen_ties(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.n) return;
    const GenNode N = gen_node(d, (uint32_t)i);
    const uint64_t k0 = owner_key(d, (uint32_t)i, 0, false);
    for (uint32_t o = 0; o < 4; ++o) {
        Lane L;
        gen_lane(d, N, o, true, L);
        if (!L.has || L.loc >= d.W0) continue;
        const uint64_t k = k0 | o;
        uint64_t w = d.owner[L.loc];
        if ((w >> 34) == (k >> 34) && ((w >> 2) & 0xFFFFFFFFull) != i) atomicAdd(d.counter, 1u);
    }
}

// The words of isn_gen, one thread per word slot (W0 + 1 of them, the last a
// zero pad): the slot's owner key names its writer, a node (through rinv when the
// keys hold sorted positions) and one of its lanes, whose word is computed
// again; a slot nobody writes is zero.  The five arrays are written in slot
// order, each slot once, so they need no clearing beforehand.
__global__ __launch_bounds__(256) void k_gen_write(Dev d, int use_rank) {
    const uint64_t w = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (w > d.W0) return;
    const uint64_t key = w < d.W0 ? d.owner[w] : 0ull;  // keys are >= 1 << 34
    uint32_t instr = 0, rd = 0, rs1 = 0, rs2 = 0, jt = 0;
    if (key != 0ull) {
        const uint32_t o = (uint32_t)key & 3u, r = (uint32_t)(key >> 2);
        const uint32_t nn = use_rank ? d.rinv[r] : r;
        const GenNode N = gen_node(d, nn);
        Lane L;
        gen_lane(d, N, o, true, L);
        if (!L.has || L.loc != w) atomicOr(d.flags, EF_OOB);
        const uint32_t wn = N.wn;
        if (d.P > 1 && (((int32_t)L.rd > 63 && L.rd - 64u >= wn) || ((int32_t)L.rs1 > 63 && L.rs1 - 64u >= wn) ||
                        ((int32_t)L.rs2 > 63 && L.rs2 - 64u >= wn)))
            atomicOr(d.flags, EF_OOB);
        instr = L.word;
        rd = (int32_t)L.rd > 63 ? L.rd + L.wb : L.rd;
        rs1 = (int32_t)L.rs1 > 63 ? L.rs1 + L.wb : L.rs1;
        rs2 = (int32_t)L.rs2 > 63 ? L.rs2 + L.wb : L.rs2;
        jt = L.jt + L.wb;
    }
    d.w0_instr[w] = instr; d.w0_rd[w] = rd; d.w0_rs1[w] = rs1; d.w0_rs2[w] = rs2; d.w0_jt[w] = jt;
}

// ------------------------------------------ libstdc++ introsort, reproduced
// std::sort over node ids with key depth (rv_generator_avx.cpp:539-541) is
// introsort: depth limit 2*floor(log2 n), median of (first+1, mid, last-1)
// moved to first, unguarded Hoare partition around it, ranges <= 16 left for a
// final insertion sort, heapsort where the limit runs out.  The k-th left stop
// (key >= pivot, scanning up from first+1) swaps with the k-th right stop
// (key <= pivot, scanning down from last-1) while they have not crossed, so one
// partition is a stream compaction of the stops and a search; all ranges of one
// recursion depth are partitioned together.  Each level works on the list of
// its ranges only (their positions concatenated: the level's active list,
// offsets in Seg::off, ranges in position order); ranges that are done leave it.
struct Seg { uint32_t first, last, limit, off; };

__global__ void k_sort_init(uint32_t *sidx, int32_t *skey, const int32_t *depth, uint64_t n) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    sidx[i] = (uint32_t)i; skey[i] = depth[i];
}

DEV void swap_pos(uint32_t *sidx, int32_t *skey, uint32_t a, uint32_t b) {
    uint32_t ti = sidx[a]; sidx[a] = sidx[b]; sidx[b] = ti;
    int32_t tk = skey[a]; skey[a] = skey[b]; skey[b] = tk;
}

// std::__move_median_to_first(first, first+1, mid, last-1); returns the pivot key.
DEV int32_t median_to_first(uint32_t first, uint32_t last, uint32_t *sidx, int32_t *skey) {
    uint32_t a = first + 1, b = first + (last - first) / 2, c = last - 1;
    int32_t ka = skey[a], kb = skey[b], kc = skey[c];
    uint32_t pick;
    if (ka < kb) { if (kb < kc) pick = b; else if (ka < kc) pick = c; else pick = a; }
    else if (ka < kc) pick = a;
    else if (kb < kc) pick = c;
    else pick = b;
    swap_pos(sidx, skey, first, pick);
    return skey[first];
}

// The first level: one range per program of more than 16 nodes.
// (A single one comes by value and is stored here.)
__global__ void k_sort_root(Seg *segs, uint32_t m, uint32_t *sidx, int32_t *skey, int32_t *pivot, Seg one) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= m) return;
    const Seg g = m == 1 ? one : segs[s];
    if (m == 1) segs[0] = one;
    pivot[s] = median_to_first(g.first, g.last, sidx, skey);
}

// Last range whose active offset is <= a.
DEV uint32_t seg_find(const Seg *segs, uint32_t m, uint32_t a) {
    uint32_t lo = 0, hi = m;
    while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (segs[mid].off <= a) lo = mid; else hi = mid; }
    return lo;
}

// Walks SCAN_ITEMS consecutive active indices from a0, tracking their range.
// Last range whose active offset is <= a, among ranges [lo, hi) (the answer
// is known to lie there).
DEV uint32_t seg_find_in(const Seg *segs, uint32_t lo, uint32_t hi, uint32_t a) {
    while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (segs[mid].off <= a) lo = mid; else hi = mid; }
    return lo;
}

// The ranges holding a workgroup's items [a_lo, a_hi]: one search per
// workgroup, so each thread then searches only this window.
// Called by every thread of the workgroup; items [a_lo, a_lo + span) clipped to A.
struct SegWindow { uint32_t lo, hi; };
DEV SegWindow seg_window(const Seg *segs, uint32_t m, uint32_t A, uint32_t a_lo, uint32_t span) {
    __shared__ uint32_t w[2];
    if (a_lo < A) {
        const uint32_t a_hi = min(A, a_lo + span) - 1;
        if (threadIdx.x == 0) w[0] = seg_find(segs, m, a_lo);
        if (threadIdx.x == 64) w[1] = seg_find(segs, m, a_hi);
    }
    __syncthreads();
    const SegWindow r{w[0], w[1] + 1};
    __syncthreads();
    return r;
}

struct SegWalk {
    const Seg *segs; uint32_t m, s, nxt; Seg g;
    DEV SegWalk(const Seg *sg, uint32_t mm, uint32_t a0) : segs(sg), m(mm) {
        s = seg_find(sg, mm, a0); g = sg[s]; nxt = s + 1 < mm ? sg[s + 1].off : 0xFFFFFFFFu;
    }
    DEV SegWalk(const Seg *sg, uint32_t mm, SegWindow wd, uint32_t a0) : segs(sg), m(mm) {
        s = seg_find_in(sg, wd.lo, wd.hi, a0); g = sg[s]; nxt = s + 1 < mm ? sg[s + 1].off : 0xFFFFFFFFu;
    }
    DEV void to(uint32_t a) {
        while (a >= nxt) { ++s; g = segs[s]; nxt = s + 1 < m ? segs[s + 1].off : 0xFFFFFFFFu; }
    }
    DEV uint32_t pos(uint32_t a) const { return g.first + (a - g.off); }
};

// Left/right stop flags of the element at pos of range g (pivot key p): the
// pivot itself, at first, takes part in neither.
DEV uint32_t stop_bits(const Seg &g, int32_t p, const int32_t *skey, uint32_t i) {
    if (i == g.first) return 0;
    const int32_t k = skey[i];
    return (!(k < p) ? 1u : 0u) | (!(p < k) ? 2u : 0u);
}

// Compaction of the stops: Lpos[k] / Rpos[k] = position of the k-th left / right
// stop of the level; base[s] = counts before range s, *total those of the level.
// One pass over the active list: tiles in ticket order, both counts carried by
// decoupled look-back as in k_scan_dlb, a status word each (the ticket counter is
// word 2 * cap), all zero before the launch.
// (Three launches, a reduction before and its scan between, took 17 us a level on
// 50k nodes and read the keys twice: 61 us a level of 16M.)
// The level kernels read the level's counts from the device (lv[0] active
// elements, lv[1] ranges) and are launched on grids sized for an upper bound
// of them; workgroups past the counts exit.
__global__ __launch_bounds__(SCAN_BLOCK) void k_sortlvl_scan(const Seg *segs, const uint32_t *lv,
                                                             const int32_t *pivot, const int32_t *skey,
                                                             unsigned long long *status, uint32_t cap, uint2 *total,
                                                             uint32_t *Lpos, uint32_t *Rpos, uint2 *base) {
    __shared__ uint32_t sL[SCAN_BLOCK / 64], sR[SCAN_BLOCK / 64], s_tile, pL, pR;
    const uint32_t A = lv[0], m = lv[1];
    if (blockIdx.x * (uint32_t)SCAN_TILE >= A) return;
    // the tile's stops, staged: its left and right stops are each one
    // contiguous range of Lpos / Rpos, written out coalesced at the end
    __shared__ uint32_t stL[SCAN_TILE], stR[SCAN_TILE];
    if (threadIdx.x == 0) s_tile = atomicAdd(reinterpret_cast<uint32_t *>(status + 2 * (uint64_t)cap), 1u);
    __syncthreads();
    const uint32_t tile = s_tile;
    const SegWindow wd = seg_window(segs, m, A, tile * (uint32_t)SCAN_TILE, (uint32_t)SCAN_TILE);
    const uint32_t a0 = tile * (uint32_t)SCAN_TILE + threadIdx.x * SCAN_ITEMS;
    uint32_t bits = 0, cl = 0, cr = 0;  // 2 bits per item
    if (a0 < A) {
        SegWalk w(segs, m, wd, a0);
        int32_t p = pivot[w.s];
        for (int k = 0; k < SCAN_ITEMS; ++k) {
            const uint32_t a = a0 + k;
            if (a >= A) break;
            const uint32_t s0 = w.s;
            w.to(a);
            if (w.s != s0) p = pivot[w.s];
            const uint32_t b = stop_bits(w.g, p, skey, w.pos(a));
            bits |= b << (2 * k);
            cl += b & 1u; cr += b >> 1;
        }
    }
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint32_t xl = wave_incl_scan(cl, lane), xr = wave_incl_scan(cr, lane);
    if (lane == 63) { sL[wid] = xl; sR[wid] = xr; }
    __syncthreads();
    uint32_t nL = 0, nR = 0;
    uint32_t rl = xl - cl, rr = xr - cr;  // offsets within the tile's ranges
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / 64; ++w) {
        if ((uint32_t)w < wid) { rl += sL[w]; rr += sR[w]; }
        nL += sL[w]; nR += sR[w];
    }
    if (wid == 0) {
        auto put = [&](uint32_t l, uint32_t r, uint64_t flag) {
            __hip_atomic_store(status + 2u * tile, (unsigned long long)l | flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(status + 2u * tile + 1u, (unsigned long long)r | flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        if (lane == 0) put(nL, nR, tile == 0 ? SCAN_INCL : SCAN_AGG);
        uint32_t l = 0, r = 0;
        for (int64_t j = (int64_t)tile - 1; j >= 0;) {  // nearest predecessor not yet summed (lane 0 reads it)
            const int64_t idx = j - (int64_t)lane;
            unsigned long long sl = SCAN_INCL, sr = SCAN_INCL;
            if (idx >= 0) {
                sl = __hip_atomic_load(status + 2 * idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sr = __hip_atomic_load(status + 2 * idx + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            // (a tile of which only one word is there, or is inclusive, is read again)
            const uint32_t fl = sl >> 32 == sr >> 32 ? (uint32_t)(sl >> 32) : 0u;
            const uint64_t incl = __ballot(fl == 2u), none = __ballot(fl == 0u);
            const uint32_t stop = incl ? (uint32_t)__builtin_ctzll(incl) : 64u;
            if (none && (uint32_t)__builtin_ctzll(none) < stop) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            l += wave_sum(lane <= stop ? (uint32_t)sl : 0u);
            r += wave_sum(lane <= stop ? (uint32_t)sr : 0u);
            if (incl) break;
            j -= 64;
        }
        if (lane == 0) {
            if (tile > 0) put(l + nL, r + nR, SCAN_INCL);
            pL = l; pR = r;
            if ((tile + 1u) * (uint64_t)SCAN_TILE >= A) *total = make_uint2(l + nL, r + nR);
        }
    }
    __syncthreads();
    const uint32_t tL = pL, tR = pR;
    if (a0 < A) {
        SegWalk w(segs, m, wd, a0);
        for (int k = 0; k < SCAN_ITEMS; ++k) {
            const uint32_t a = a0 + k;
            if (a >= A) break;
            w.to(a);
            const uint32_t i = w.pos(a);
            if (a == w.g.off) base[w.s] = make_uint2(tL + rl, tR + rr);
            const uint32_t b = (bits >> (2 * k)) & 3u;
            if (b & 1u) stL[rl++] = i;
            if (b & 2u) stR[rr++] = i;
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nL; k += SCAN_BLOCK) Lpos[tL + k] = stL[k];
    for (uint32_t k = threadIdx.x; k < nR; k += SCAN_BLOCK) Rpos[tR + k] = stR[k];
}

struct SegCut { uint32_t baseL, cntL, baseR, cntR, m, cut, uni, pad; };

// Ranges whose keys are all equal.  For them the introsort's moves do not
// depend on the keys: median-of-three picks the middle element (all three
// comparisons false: iter_swap(first, first + len/2)), the unguarded partition
// stops at every element and swaps first+1+k with last-1-k for k < (len-1)/2,
// and the cut falls at first+1+(len-1)/2; the final insertion sort moves none of
// them.  So each element's final place follows from its place alone.
// uniform_depth: partition levels until every subrange is <= 16 (the left
// child, 1+(len-1)/2, is never the smaller one).
DEV uint32_t uniform_depth(uint32_t len) {
    uint32_t dpt = 0;
    while (len > 16) { len = 1u + (len - 1u) / 2u; ++dpt; }
    return dpt;
}

// Final place of the element at pos of an all-equal range [a, b), whose first
// median swap has been made already.
DEV uint32_t uniform_final(uint32_t a, uint32_t b, uint32_t pos) {
    bool first = true;
    while (b - a > 16) {
        const uint32_t len = b - a;
        if (!first) { const uint32_t mid = a + len / 2; if (pos == a) pos = mid; else if (pos == mid) pos = a; }
        first = false;
        const uint32_t K = (len - 1) / 2;
        if ((pos >= a + 1 && pos < a + 1 + K) || (pos >= b - K && pos < b)) pos = a + b - pos;
        const uint32_t cut = a + 1 + K;
        if (pos >= cut) a = cut; else b = cut;
    }
    return pos;
}

__global__ void k_sort_search(const Seg *segs, const uint32_t *lv, const uint2 *base, const uint2 *total,
                              const uint32_t *Lpos, const uint32_t *Rpos, SegCut *cuts,
                              unsigned long long *qa_next) {
    const uint32_t m = lv[1];
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) *qa_next = 0ull;  // the counts that k_sort_plan adds to
    if (s >= m) return;
    uint32_t first = segs[s].first, last = segs[s].last;
    const uint2 b0 = base[s], b1 = s + 1 < m ? base[s + 1] : *total;
    uint32_t bL = b0.x, bR = b0.y, cL = b1.x - b0.x, cR = b1.y - b0.y;
    // m = largest k with L_k < R_k (1-based), L_k = Lpos[bL+k-1], R_k = Rpos[bR+cR-k]
    uint32_t lo = 0, hi = cL < cR ? cL : cR;
    while (lo < hi) {
        uint32_t mid = (lo + hi + 1) / 2;
        if (Lpos[bL + mid - 1] < Rpos[bR + cR - mid]) lo = mid; else hi = mid - 1;
    }
    uint32_t mm = lo;
    uint32_t cut = 0xFFFFFFFFu;
    if (mm + 1 <= cL) cut = Lpos[bL + mm];
    if (mm >= 1) { uint32_t r = Rpos[bR + cR - mm]; if (r < cut) cut = r; }
    if (cut <= first || cut >= last) cut = first + 1;  // unreachable after a median-of-three pivot
    // every element stopped on both sides: all keys equal the pivot
    const uint32_t len = last - first;
    if (cL == len - 1 && cR == len - 1 && uniform_depth(len) <= segs[s].limit) {
        cuts[s] = SegCut{bL, cL, bR, cR, 0, last, 1, 0};
        return;
    }
    cuts[s] = SegCut{bL, cL, bR, cR, mm, cut, 0, 0};
}

// The partition's swaps: pair k of a range (1-based) swaps its k-th left and
// k-th-from-the-end right stop; the index within the range is the pair number.
// A workgroup covers 256*SCAN_ITEMS active indices, consecutive lanes taking
// consecutive pairs (coalesced stop lists).
__global__ __launch_bounds__(256) void k_sort_swap(const Seg *segs, const uint32_t *lv, const SegCut *cuts,
                                                   const uint32_t *Lpos, const uint32_t *Rpos, uint32_t *sidx,
                                                   int32_t *skey, unsigned long long *status_next, uint32_t cap) {
    const uint32_t A = lv[0], m = lv[1];
    static_assert(256 * SCAN_ITEMS == SCAN_TILE, "a tile a workgroup");
    if (threadIdx.x == 0) {  // cleared for the next level's scan, of no more tiles
        status_next[2 * (uint64_t)blockIdx.x] = 0ull;
        status_next[2 * (uint64_t)blockIdx.x + 1] = 0ull;
        if (blockIdx.x == 0) status_next[2 * (uint64_t)cap] = 0ull;
    }
    if (blockIdx.x * 256u * SCAN_ITEMS >= A) return;
    const SegWindow wd = seg_window(segs, m, A, blockIdx.x * 256u * SCAN_ITEMS, 256u * SCAN_ITEMS);
    const uint32_t a0 = blockIdx.x * 256u * SCAN_ITEMS + threadIdx.x;
    if (a0 >= A) return;
    SegWalk w(segs, m, wd, a0);
    SegCut c = cuts[w.s];
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t a = a0 + 256u * k;
        if (a >= A) break;
        const uint32_t s0 = w.s;
        w.to(a);
        if (w.s != s0) c = cuts[w.s];
        const uint32_t kk = a - w.g.off + 1;
        if (kk <= c.m) swap_pos(sidx, skey, Lpos[c.baseL + kk - 1], Rpos[c.baseR + c.cntR - kk]);
    }
}

// Level counters.  qa[l & 1] = ranges << 32 | active elements of level l
// (each level's plan resets and fills the next one's); ue = all-equal ranges
// << 32 | their elements (accumulated); one 64-bit atomic per pair keeps a
// list's slots and offsets in the same order.
// nloc: ranges listed for k_sort_local; bad: a listed range of a size it does
// not take (never, by construction; the host reports it as an internal error).
struct SortCnt { unsigned long long qa[2], ue; uint32_t nheap, nloc, bad, pad; };

// Ranges of at most SORT_LOCAL (or SORT_LOCAL_FEW) elements finish in one workgroup's LDS
// (k_sort_local): k_sort_plan lists them (median already moved to first)
// instead of the next level.
constexpr uint32_t SORT_LOCAL = 2048, SORT_LOCAL_FEW = 8192;

DEV uint32_t block_excl_scan(uint32_t v, uint32_t *tmp /* 16 */, uint32_t &total) {
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(v, lane);
    if (lane == 63) tmp[wid] = x;
    __syncthreads();
    uint32_t pre = 0, all = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; ++w) { if (w < wid) pre += tmp[w]; all += tmp[w]; }
    __syncthreads();
    total = all;
    return pre + x - v;
}

// The children of every partitioned range (1024 ranges per workgroup): next
// level (with their active offsets), heapsort list, or leaves (marked in
// `bound`); all-equal ranges to the closed-form list (offsets in its own
// element order); then median-of-three for every new range of the next level.
// Workgroups take their slots of each list with one atomic, so the lists are
// in workgroup-arrival order; every consumer needs only that a list's slots and
// offsets agree.
__global__ __launch_bounds__(1024) void k_sort_plan(const Seg *segs, const SegCut *cuts, const uint32_t *lv,
                                                    Seg *next, int32_t *next_pivot, Seg *heap, Seg *uni,
                                                    Seg *loc, int32_t *loc_pivot,
                                                    unsigned long long *qa_next, SortCnt *cnt, uint8_t *bound,
                                                    uint32_t *sidx, int32_t *skey, uint32_t lcap) {
    __shared__ uint32_t tmp[16];
    __shared__ uint32_t base[6];
    const uint32_t m = lv[1];
    if (blockIdx.x * blockDim.x >= m) return;
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    Seg g{0, 0, 0, 0};
    SegCut ct{};
    if (s < m) { g = segs[s]; ct = cuts[s]; }
    const bool v = s < m, un = v && ct.uni;
    const uint32_t lim = g.limit - 1;
    const uint32_t c0 = ct.cut - g.first, c1 = g.last - ct.cut;
    const bool r0 = v && !un && c0 > 16 && lim > 0, r1 = v && !un && c1 > 16 && lim > 0;
    const bool n0 = r0 && c0 > lcap, n1 = r1 && c1 > lcap;    // next level
    const bool l0 = r0 && c0 <= lcap, l1 = r1 && c1 <= lcap;  // finished in LDS
    const bool h0b = v && !un && c0 > 16 && lim == 0, h1b = v && !un && c1 > 16 && lim == 0;
    uint32_t tq, ta, th, tu, te, tl;
    const uint32_t xl = block_excl_scan((l0 ? 1u : 0u) + (l1 ? 1u : 0u), tmp, tl);
    const uint32_t xq = block_excl_scan((n0 ? 1u : 0u) + (n1 ? 1u : 0u), tmp, tq);
    const uint32_t xa = block_excl_scan((n0 ? c0 : 0u) + (n1 ? c1 : 0u), tmp, ta);
    const uint32_t xh = block_excl_scan((h0b ? 1u : 0u) + (h1b ? 1u : 0u), tmp, th);
    const uint32_t xu = block_excl_scan(un ? 1u : 0u, tmp, tu);
    const uint32_t xe = block_excl_scan(un ? g.last - g.first : 0u, tmp, te);
    if (threadIdx.x == 0) {
        const unsigned long long qa = (tq | ta) ? atomicAdd(qa_next, ((unsigned long long)tq << 32) | ta) : 0ull;
        const unsigned long long ue = (tu | te) ? atomicAdd(&cnt->ue, ((unsigned long long)tu << 32) | te) : 0ull;
        base[0] = (uint32_t)(qa >> 32); base[1] = (uint32_t)qa;
        base[2] = th ? atomicAdd(&cnt->nheap, th) : 0u;
        base[3] = (uint32_t)(ue >> 32); base[4] = (uint32_t)ue;
        base[5] = tl ? atomicAdd(&cnt->nloc, tl) : 0u;
    }
    __syncthreads();
    if (!v) return;
    if (un) {
        uni[base[3] + xu] = Seg{g.first, g.last, g.limit, base[4] + xe};
        bound[g.first] = 2;
        return;
    }
    bound[ct.cut] = 1;
    uint32_t q = base[0] + xq, a = base[1] + xa, h = base[2] + xh;
    if (n0) { next[q] = Seg{g.first, ct.cut, lim, a}; next_pivot[q] = median_to_first(g.first, ct.cut, sidx, skey); ++q; a += c0; }
    if (n1) { next[q] = Seg{ct.cut, g.last, lim, a}; next_pivot[q] = median_to_first(ct.cut, g.last, sidx, skey); }
    uint32_t lq = base[5] + xl;
    if (l0) { loc[lq] = Seg{g.first, ct.cut, lim, 0}; loc_pivot[lq] = median_to_first(g.first, ct.cut, sidx, skey); ++lq; }
    if (l1) { loc[lq] = Seg{ct.cut, g.last, lim, 0}; loc_pivot[lq] = median_to_first(ct.cut, g.last, sidx, skey); }
    if (h0b) heap[h++] = Seg{g.first, ct.cut, 0, 0};
    if (h1b) heap[h++] = Seg{ct.cut, g.last, 0, 0};
}

// One listed range per workgroup, all its remaining levels in LDS: the same
// partitions as the level kernels above (stops, pairs, cut, all-equal ranges
// in closed form when their recursion fits the limit), the same outputs
// (boundaries in `bound`, entries of the heap and all-equal lists), its
// subranges kept in position order.  Each thread holds ppt consecutive positions.
template <uint32_t CAP, uint32_t NT>
__global__ __launch_bounds__(NT) void k_sort_local(const Seg *loc, const int32_t *loc_pivot, const SortCnt *cntr,
                                                   uint32_t *sidx, int32_t *skey, uint8_t *bound, Seg *heap,
                                                   Seg *uni, SortCnt *cnt) {
    constexpr uint32_t SUBS = CAP / 17 + 2;
    static_assert(CAP % NT == 0 && CAP / NT <= 16 && SUBS <= NT, "two bits of `bits` a position, a thread a subrange");
    __shared__ int32_t K[CAP];
    __shared__ uint32_t X[CAP];
    __shared__ uint16_t LP[CAP], RP[CAP];
    __shared__ uint16_t sf[2][SUBS], sl[2][SUBS];
    __shared__ uint8_t slim[2][SUBS];
    __shared__ int32_t spiv[2][SUBS];
    __shared__ uint16_t bL[SUBS + 1], bR[SUBS + 1], cts[SUBS];  // stops before a subrange; its cut
    __shared__ uint8_t unis[SUBS];
    __shared__ uint16_t uf[SUBS], ul[SUBS];  // all-equal ranges found
    __shared__ uint8_t ulim[SUBS];
    __shared__ uint32_t tmp[16], nnext, nuni;
    __shared__ unsigned long long ubase;
    if (blockIdx.x >= cntr->nloc) return;
    const uint32_t tid = threadIdx.x;
    const Seg g = loc[blockIdx.x];
    const uint32_t base = g.first, len = g.last - g.first;
    if (len > CAP || len < 17) { if (tid == 0) atomicOr(&cnt->bad, 1u); return; }
    for (uint32_t p = tid; p < len; p += NT) { K[p] = skey[base + p]; X[p] = sidx[base + p]; }
    if (tid == 0) {
        sf[0][0] = 0; sl[0][0] = (uint16_t)len; slim[0][0] = (uint8_t)g.limit; spiv[0][0] = loc_pivot[blockIdx.x];
        nuni = 0;
    }
    uint32_t cur = 0, nsub = 1;
    __syncthreads();
    const uint32_t ppt = (len + NT - 1) / NT, p0 = min(tid * ppt, len), pe = min(p0 + ppt, len);
    while (nsub > 0) {
        // stops of this thread's positions: subrange walk from the last one starting at or before p0
        uint32_t s0 = 0;
        {
            uint32_t lo = 0, hi = nsub;
            while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (sf[cur][mid] <= p0) lo = mid; else hi = mid; }
            s0 = lo;
        }
        uint32_t bits = 0, cl = 0, cr = 0;
        {
            uint32_t s = s0;
            for (uint32_t p = p0, k = 0; p < pe; ++p, k += 2) {
                while (s + 1 < nsub && sf[cur][s + 1] <= p) ++s;
                if (p < sf[cur][s] || p >= sl[cur][s] || p == sf[cur][s]) continue;
                const int32_t kk = K[p], pv = spiv[cur][s];
                const uint32_t b = (!(kk < pv) ? 1u : 0u) | (!(pv < kk) ? 2u : 0u);
                bits |= b << k;
                cl += b & 1u; cr += b >> 1;
            }
        }
        // both counts in one scan (each at most CAP, so 16 bits apiece)
        uint32_t tot2;
        const uint32_t x2 = block_excl_scan(cl | (cr << 16), tmp, tot2);
        uint32_t rl = x2 & 0xFFFFu, rr = x2 >> 16;
        const uint32_t rl0 = rl;
        {
            uint32_t s = s0;
            for (uint32_t p = p0, k = 0; p < pe; ++p, k += 2) {
                while (s + 1 < nsub && sf[cur][s + 1] <= p) ++s;
                if (p == sf[cur][s]) { bL[s] = (uint16_t)rl; bR[s] = (uint16_t)rr; cts[s] = (uint16_t)(p + 1); unis[s] = 0; }
                const uint32_t b = (bits >> k) & 3u;
                if (b & 1u) LP[rl++] = (uint16_t)p;
                if (b & 2u) RP[rr++] = (uint16_t)p;
            }
        }
        if (tid == 0) { bL[nsub] = (uint16_t)(tot2 & 0xFFFFu); bR[nsub] = (uint16_t)(tot2 >> 16); }
        __syncthreads();
        // Each pair's swap, by the thread holding its left stop.  The pairs with
        // L_k < R_k are the first ones, so each thread tells its own from the two
        // stops; the one at the first pair that is not (or the last left stop)
        // sets the cut, as k_sort_search.
        {
            uint32_t s = s0, r = rl0;
            for (uint32_t p = p0, k = 0; p < pe; ++p, k += 2) {
                while (s + 1 < nsub && sf[cur][s + 1] <= p) ++s;
                if (!((bits >> k) & 1u)) continue;
                const uint32_t f = sf[cur][s], l = sl[cur][s], b0 = bL[s], b1 = bR[s];
                const uint32_t cL = bL[s + 1] - b0, cR = bR[s + 1] - b1, kk = r++ - b0, n = l - f;
                if (cL == n - 1 && cR == n - 1 && uniform_depth(n) <= slim[cur][s]) {
                    if (kk == 0) { cts[s] = (uint16_t)l; unis[s] = 1; }
                    continue;
                }
                const uint32_t q = kk < cR ? RP[b1 + cR - 1u - kk] : 0u;          // right stop kk
                const uint32_t qp = kk - 1u < cR ? RP[b1 + cR - kk] : 0u;         // and kk - 1
                const bool pair = p < q;
                uint32_t cut = 0xFFFFFFFFu;
                if (pair) {
                    const int32_t tk = K[p]; K[p] = K[q]; K[q] = tk;
                    const uint32_t tx = X[p]; X[p] = X[q]; X[q] = tx;
                    if (kk == cL - 1u) cut = q;
                } else if (kk == 0u) {
                    cut = p;
                } else if (LP[b0 + kk - 1u] < qp) {
                    cut = min(p, qp);
                }
                if (cut > f && cut < l) cts[s] = (uint16_t)cut;  // (first + 1: unreachable after a median-of-three pivot)
            }
        }
        __syncthreads();
        // children (k_sort_plan): the next subranges in position order, each with
        // its median moved to first; up to 64 subranges by one wave
        const uint32_t nx = cur ^ 1u;
        const bool one = nsub <= 64u;
        if (!one || tid < 64u) {
            uint32_t nc = 0, f = 0, l = 0, cut = 0, lim = 0;
            bool c0n = false, c1n = false;
            if (tid < nsub) {
                f = sf[cur][tid]; l = sl[cur][tid]; cut = cts[tid];
                const uint32_t limit = slim[cur][tid];
                lim = limit - 1u;
                if (unis[tid]) {
                    const uint32_t u = atomicAdd(&nuni, 1u);
                    uf[u] = (uint16_t)f; ul[u] = (uint16_t)l; ulim[u] = (uint8_t)limit;
                    bound[base + f] = 2;
                } else {
                    bound[base + cut] = 1;
                    const uint32_t c0 = cut - f, c1 = l - cut;
                    c0n = c0 > 16 && lim > 0; c1n = c1 > 16 && lim > 0;
                    if (c0 > 16 && lim == 0) heap[atomicAdd(&cnt->nheap, 1u)] = Seg{base + f, base + cut, 0, 0};
                    if (c1 > 16 && lim == 0) heap[atomicAdd(&cnt->nheap, 1u)] = Seg{base + cut, base + l, 0, 0};
                    nc = (c0n ? 1u : 0u) + (c1n ? 1u : 0u);
                }
            }
            uint32_t tot, q;
            if (one) {
                const uint32_t x = wave_incl_scan(nc, tid);
                q = x - nc;
                tot = (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
            } else {
                q = block_excl_scan(nc, tmp, tot);
            }
            if (c0n) { sf[nx][q] = (uint16_t)f; sl[nx][q] = (uint16_t)cut; slim[nx][q] = (uint8_t)lim; spiv[nx][q] = median_to_first(f, cut, X, K); ++q; }
            if (c1n) { sf[nx][q] = (uint16_t)cut; sl[nx][q] = (uint16_t)l; slim[nx][q] = (uint8_t)lim; spiv[nx][q] = median_to_first(cut, l, X, K); }
            if (tid == 0) nnext = tot;
        }
        __syncthreads();
        cur = nx;
        nsub = nnext;
    }
    for (uint32_t p = tid; p < len; p += NT) { skey[base + p] = K[p]; sidx[base + p] = X[p]; }
    const uint32_t nu = nuni;
    if (nu > 0) {  // the all-equal ranges to their list (ranges << 32 | elements)
        uint32_t tot;
        const uint32_t o = block_excl_scan(tid < nu ? (uint32_t)(ul[tid] - uf[tid]) : 0u, tmp, tot);
        if (tid == 0) ubase = atomicAdd(&cnt->ue, ((unsigned long long)nu << 32) | tot);
        __syncthreads();
        if (tid < nu) uni[(uint32_t)(ubase >> 32) + tid] = Seg{base + uf[tid], base + ul[tid], ulim[tid], (uint32_t)ubase + o};
    }
}

// libstdc++ heap routines on one range, one thread (std::__make_heap,
// std::__adjust_heap, std::__push_heap, std::__sort_heap).
DEV void heap_adjust(uint32_t *si, int32_t *sk, uint32_t base, int64_t hole, int64_t len, uint32_t vi, int32_t vk) {
    const int64_t top = hole;
    int64_t child = hole;
    while (child < (len - 1) / 2) {
        child = 2 * (child + 1);
        if (sk[base + child] < sk[base + child - 1]) child--;
        si[base + hole] = si[base + child]; sk[base + hole] = sk[base + child];
        hole = child;
    }
    if ((len & 1) == 0 && child == (len - 2) / 2) {
        child = 2 * (child + 1);
        si[base + hole] = si[base + child - 1]; sk[base + hole] = sk[base + child - 1];
        hole = child - 1;
    }
    int64_t parent = (hole - 1) / 2;
    while (hole > top && sk[base + parent] < vk) {
        si[base + hole] = si[base + parent]; sk[base + hole] = sk[base + parent];
        hole = parent;
        parent = (hole - 1) / 2;
    }
    si[base + hole] = vi; sk[base + hole] = vk;
}

__global__ void k_sort_heap(const Seg *heap, const uint32_t *heap_cnt, uint32_t *si, int32_t *sk, uint8_t *bound) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= *heap_cnt) return;
    uint32_t base = heap[s].first;
    bound[base] = 2;
    int64_t len = heap[s].last - heap[s].first;
    if (len >= 2) {
        for (int64_t parent = (len - 2) / 2;; --parent) {
            heap_adjust(si, sk, base, parent, len, si[base + parent], sk[base + parent]);
            if (parent == 0) break;
        }
    }
    for (int64_t last = len; last > 1;) {
        --last;
        uint32_t vi = si[base + last]; int32_t vk = sk[base + last];
        si[base + last] = si[base]; sk[base + last] = sk[base];
        heap_adjust(si, sk, base, 0, last, vi, vk);
    }
}

// Leaves are the ranges between consecutive boundaries, marked in `bound` (1 at
// each range start, at most 16 elements, insertion-sorted; 2: an all-equal or a
// heapsorted range, in which nothing moves).  Insertion sort keeps equal keys in
// order, so an element's final place is the count of the leaf's elements before
// it in that order: a thread an element, the tile with 16 more on either side in
// LDS.  (A thread a leaf sorting it in memory, and a pass for the ranks: 25 + 6 us
// on 4k nodes.)
constexpr uint32_t LEAF = 16;
__global__ __launch_bounds__(256) void k_sort_leaves(const uint8_t *bound, uint64_t n, const uint32_t *si,
                                                     const int32_t *sk, uint32_t *rank, uint32_t *rinv) {
    __shared__ int32_t K[256 + 2 * LEAF];
    __shared__ uint8_t B[256 + 2 * LEAF];
    const uint64_t t0 = blockIdx.x * (uint64_t)256;
    for (uint32_t x = threadIdx.x; x < 256u + 2u * LEAF; x += 256u) {
        const uint64_t i = t0 + x;  // element i - LEAF
        const bool in = i >= LEAF && i - LEAF < n;
        K[x] = in ? sk[i - LEAF] : 0;
        B[x] = in ? bound[i - LEAF] : 1;
    }
    __syncthreads();
    const uint64_t i = t0 + threadIdx.x;
    if (i >= n) return;
    const uint32_t v = si[i], x = threadIdx.x + LEAF;
    uint32_t b = x, pos = x;
    while (!B[b] && x - b < LEAF - 1u) --b;
    if (B[b] == 1) {
        const int32_t k = K[x];
        pos = b;
        for (uint32_t y = b; y < x; ++y) pos += K[y] <= k ? 1u : 0u;
        for (uint32_t y = x + 1u; y < b + LEAF && !B[y]; ++y) pos += K[y] < k ? 1u : 0u;
    }
    const uint64_t q = t0 + pos - LEAF;
    rank[v] = (uint32_t)q;
    rinv[q] = v;
}

// Elements of all-equal ranges go to their closed-form places (after the
// plain ranks, which they overwrite).
__global__ void k_sort_rank_uniform(const Seg *uni, uint32_t nuni, uint32_t total, const uint32_t *si,
                                    uint32_t *rank, uint32_t *rinv) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total) return;
    // the range of the wave's first active element by one search on a
    // wave-uniform index, then each lane steps on to its own (a range has more
    // than 16 elements, so a wave spans at most five)
    uint32_t si0 = seg_find(uni, nuni, (uint32_t)__builtin_amdgcn_readfirstlane((int)e));
    while (si0 + 1 < nuni && uni[si0 + 1].off <= e) ++si0;
    const Seg g = uni[si0];
    const uint32_t p = g.first + (e - g.off);
    const uint32_t v = si[p], q = uniform_final(g.first, g.last, p);
    rank[v] = q;
    rinv[q] = v;  // (positions of an all-equal range are a permutation of it)
}

// ================================================================= optimize
__global__ __launch_bounds__(256) void k_opt_init(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.W0) return;
    int32_t a = (int32_t)(d.w0_rs1[i] - 64u), b = (int32_t)(d.w0_rs2[i] - 64u);
    uint32_t w = d.w0_instr[i] & 0x707Fu;
    bool st = w == 0x2023u || w == 0x2027u;
    if (a >= 0) { if ((uint32_t)a < d.W0) { d.used[a] = 1; if (st) d.sstore[a] = 1; } else atomicOr(d.flags, EF_OOB); }
    if (b >= 0) { if ((uint32_t)b < d.W0) { d.used[b] = 1; if (st) d.sstore[b] = 1; } else atomicOr(d.flags, EF_OOB); }
}

// One sweep: a word whose destination register is unused clears its sources
// (except sources of stores).  Repeated until a sweep changes nothing.  A
// word's sources are mostly the words just before it, so each workgroup
// repeats its own range of OPT_RANGE words until no word of the range lost its
// use; only chains crossing ranges need further sweeps.  `changed` is set by a
// clear of a word outside the clearing workgroup's range, by a word whose
// destination lies outside its range (its flag could change under it), or by a
// range that did not settle within its 64 rounds: a launch with none of these
// has every range settled on values no other workgroup changed, which is the
// fixpoint.  (Generated code names a word's own register as its destination,
// so the second case does not arise there.)
constexpr uint32_t OPT_RANGE = 256 * 8;

// The range's fields and its used/store flags are staged in LDS once; the
// rounds read them there (flags of other ranges from HBM).  A clear is written
// to both (flags only go from 1 to 0, so HBM never takes back a clear made by
// another workgroup); a clear another workgroup makes in this range during the
// launch is a cross clear, which asks for the next launch, where it is staged.
//
// The round's "some word of the range lost its use" flag is double-buffered by
// round parity.  Thread 0 clears local[(round + 1) & 1] at the top of the next
// round while slower waves may still be reading local[round & 1] after the
// round's last barrier; it can only come back to local[round & 1] (two rounds
// later) after every wave has passed the next round's first barrier, i.e.
// after every wave has read it.  With a single flag, a wave still to read it
// could see the next round's clear, leave the loop and drop its words from
// the later rounds, and the launch could then report a fixpoint early.
// Thread t sweeps its own 8 consecutive words, highest first, so a chain of
// words naming the word before (the usual shape) settles inside one sweep of
// its thread rather than one link per round; the range is kept in LDS
// transposed (word k at (k % 8) * 256 + k / 8), so that the threads' k-th words
// sit in consecutive banks.
DEV uint32_t opt_tp(uint32_t k) { return (k & 7u) * 256u + (k >> 3); }

__global__ __launch_bounds__(256) void k_opt_iter(Dev d, uint32_t *changed) {
    static_assert(OPT_RANGE == 256 * 8, "8 words per thread");
    __shared__ int local[2];
    __shared__ uint32_t s_rd[OPT_RANGE], s_r1[OPT_RANGE], s_r2[OPT_RANGE];
    __shared__ uint8_t s_used[OPT_RANGE], s_st[OPT_RANGE];
    const uint64_t b0 = (uint64_t)blockIdx.x * OPT_RANGE;
    const uint64_t b1 = b0 + OPT_RANGE < d.W0 ? b0 + OPT_RANGE : d.W0;
    const uint32_t nr = (uint32_t)(b1 - b0);
    const uint32_t t = threadIdx.x, k0 = 8u * t;
    if (k0 + 8u <= nr) {
        // this thread's 8 words with two 16-byte loads per field (b0 and k0 are multiples of 8)
        const uint4 *rd4 = reinterpret_cast<const uint4 *>(d.w0_rd + b0 + k0);
        const uint4 *r14 = reinterpret_cast<const uint4 *>(d.w0_rs1 + b0 + k0);
        const uint4 *r24 = reinterpret_cast<const uint4 *>(d.w0_rs2 + b0 + k0);
        const uint4 x0 = rd4[0], x1 = rd4[1], y0 = r14[0], y1 = r14[1], z0 = r24[0], z1 = r24[1];
        const uint2 u8 = *reinterpret_cast<const uint2 *>(d.used + b0 + k0);
        const uint2 s8 = *reinterpret_cast<const uint2 *>(d.sstore + b0 + k0);
        const uint32_t xr[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        const uint32_t yr[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
        const uint32_t zr[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t e = j * 256u + t;
            s_rd[e] = xr[j]; s_r1[e] = yr[j]; s_r2[e] = zr[j];
            s_used[e] = (uint8_t)((j < 4 ? u8.x : u8.y) >> (8u * (j & 3u)));
            s_st[e] = (uint8_t)((j < 4 ? s8.x : s8.y) >> (8u * (j & 3u)));
        }
    } else {
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t k = k0 + j;
            if (k >= nr) break;
            const uint32_t e = j * 256u + t;
            s_rd[e] = d.w0_rd[b0 + k]; s_r1[e] = d.w0_rs1[b0 + k]; s_r2[e] = d.w0_rs2[b0 + k];
            s_used[e] = d.used[b0 + k]; s_st[e] = d.sstore[b0 + k];
        }
    }
    auto used_of = [&](uint32_t x) -> bool { return (uint64_t)x - b0 < nr ? s_used[opt_tp(x - (uint32_t)b0)] != 0 : d.used[x] != 0; };
    auto store_of = [&](uint32_t x) -> bool { return (uint64_t)x - b0 < nr ? s_st[opt_tp(x - (uint32_t)b0)] != 0 : d.sstore[x] != 0; };
    bool cross = false;  // a clear outside the range, or a destination outside it
    bool settled = false;
    for (int round = 0; round < 64; ++round) {
        if (threadIdx.x == 0) local[round & 1] = 0;
        __syncthreads();
        bool loc = false;
        for (int32_t j = 7; j >= 0; --j) {
            const uint32_t k = k0 + (uint32_t)j;
            if (k >= nr) continue;
            const uint32_t e = (uint32_t)j * 256u + t;
            const uint32_t rd = s_rd[e];
            if (!((int32_t)rd > 63)) continue;
            const uint32_t v = rd - 64u;
            if (v >= d.W0) continue;
            cross |= (uint64_t)v - b0 >= nr;
            if (used_of(v)) continue;
            const int32_t a = (int32_t)(s_r1[e] - 64u), b = (int32_t)(s_r2[e] - 64u);
            if (a >= 0 && (uint32_t)a < d.W0 && !store_of((uint32_t)a) && used_of((uint32_t)a)) {
                const bool in = (uint64_t)(uint32_t)a - b0 < nr;
                if (in) s_used[opt_tp((uint32_t)a - (uint32_t)b0)] = 0;
                d.used[a] = 0;
                loc |= in; cross |= !in;
            }
            if (b >= 0 && (uint32_t)b < d.W0 && !store_of((uint32_t)b) && used_of((uint32_t)b)) {
                const bool in = (uint64_t)(uint32_t)b - b0 < nr;
                if (in) s_used[opt_tp((uint32_t)b - (uint32_t)b0)] = 0;
                d.used[b] = 0;
                loc |= in; cross |= !in;
            }
        }
        if (loc) local[round & 1] = 1;
        __syncthreads();
        if (!local[round & 1]) { settled = true; break; }
    }
    if (cross || (!settled && threadIdx.x == 0)) *changed = 1;
}

// ---- the allocation walks' view of a word -------------------------------
// A walk step of a function is a chain of dependent instructions, and the
// longest function's chain bounds the stage, so everything about a word that
// does not depend on the allocation is worked out here, for all words at once:
// where its operands' states are (the word that defines the register, as a
// distance back in the function), whether it takes a free register, the
// constant register it writes otherwise.  A step then reads one 4-byte op in
// place of the 16-byte word and its comparisons.
//   bits 0-7, 8-15  distance of the word defining rs1 / rs2 (0: no operand
//                   state, the register read is x0; a word that names its own
//                   register reads the cleared state, which is the same)
//   bits 16-21      register written when none is allocated (0: none)
//   OP_ALLOC        rd is the word's own register, a free integer register
//   OP_SELF         rd is the word's own register (float: always f5, see ffz_gcc)
//   OP_FP           an OP-FP word (its swapped operands go to f5 / f6)
//   OP_FAR1/2       rs1 / rs2 is defined more than OP_WINDOW words back: its
//                   state is read from HBM
//   OP_ZERO         an operand names the word's own register: its entry ends up 0
constexpr uint32_t OP_ROWS = 256;     // rows of the walks' LDS rings (a power of two)
constexpr uint32_t OP_WINDOW = 248;   // words back an operand's state is in LDS for sure (ring_low)
constexpr uint32_t OP_CONST = 16;     // shift of the constant register
constexpr uint32_t OP_ALLOC = 1u << 22, OP_SELF = 1u << 23, OP_FP = 1u << 24, OP_FAR1 = 1u << 25, OP_FAR2 = 1u << 26,
                   OP_ZERO = 1u << 27;

// Whether an operand of function f's word i that names word v, of another function
// or after i, reads the cleared state whatever the order of the walks: v is a word
// of f's program that does not define its register (a word that defines another
// one's is odd itself), or a later word of f itself (v > i), not yet defined.
DEV bool ra_never_set(const Dev &d, uint32_t f, uint32_t s, uint32_t i, uint32_t v) {
    const uint32_t p = prog_of(d.pf, d.P, f);
    if (v < d.pw[p] || v >= d.pw[p + 1]) return false;
    return d.w0_rd[v] != v + 64u || (v > i && v - s < d.fsizes[f]);
}

// The op of word i of function f, the words [s, s + size).  `odd` turns true for a
// word of another form: an operand naming a word of another function that defines
// its register (isn_gen ORs a word's own virtual register into physical argument
// registers, rv_generator_avx.cpp:676-697, :842, which for calls with many
// arguments can name one), or a destination other than the word's own register.
// The walks keep a register's state with the one thread that walks its function,
// in the order of that function's words; a program with an odd word is allocated by
// k_ra_serial in the reference's step and group order.  A register that nothing has
// defined yet reads as x0 in any order and its state stays cleared: no operand (a
// program of 20 functions and 7.2k words with one such read: walk and lockstep 0.45
// ms, k_ra_serial 2.54).
DEV uint32_t ra_op(const Dev &d, uint32_t f, uint32_t i, uint32_t s, uint32_t rd, uint32_t rs1, uint32_t rs2,
                   uint32_t ins, bool &odd) {
    const bool fp = (ins & 0x7Fu) == 0x53u;
    uint32_t op = fp ? OP_FP : 0u;
    const uint32_t rs[2] = {rs1, rs2};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if ((int32_t)rs[k] <= 63) continue;
        const uint32_t v = rs[k] - 64u;
        if (v >= d.W0) { atomicOr(d.flags, EF_OOB); odd = true; continue; }
        if (v < s || v > i) { odd = odd || !ra_never_set(d, f, s, i, v); continue; }
        const uint32_t dist = i - v;
        if (dist == 0) op |= OP_ZERO;
        else if (dist <= OP_WINDOW) op |= dist << (8 * k);
        else op |= k ? OP_FAR2 : OP_FAR1;
    }
    if ((int32_t)rd > 63) {
        if (rd - 64u >= d.W0) atomicOr(d.flags, EF_OOB);
        if (rd - 64u != i) odd = true;
        op |= fp ? OP_SELF | (37u << OP_CONST) : OP_SELF | OP_ALLOC;
    } else if ((int32_t)rd < 0) {
        odd = true;
    } else {
        op |= rd << OP_CONST;
    }
    return op;
}

// The used words, regalloc's view of them, and the walks' ops (one pass: the
// word's fields are at hand).  Streaming: 17 B read, 21 B written per word.
__global__ __launch_bounds__(256) void k_opt_final(Dev d) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    // the function of the wave's first word, then each lane steps to its own
    const uint64_t i0 = blockIdx.x * (uint64_t)blockDim.x + (threadIdx.x & ~63u);
    if (i0 >= d.W0) return;
    uint32_t f = prog_of(d.fstarts, d.F, (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)i0));
    if (i >= d.W0) return;
    while (f + 1 < d.F && d.fstarts[f + 1] <= (uint32_t)i) ++f;
    const uint32_t rd = d.w0_rd[i], rs1 = d.w0_rs1[i], rs2 = d.w0_rs2[i], ins = d.w0_instr[i];
    d.usedi[i] = (!((int32_t)rd > 63) || d.used[i]) ? 1 : 0;
    d.w0_f4[i] = make_uint4(rd, rs1, rs2, ins);  // regalloc's view of the word
    bool odd = false;
    const uint32_t s = d.fstarts[f];
    // (a word outside every function is walked by none)
    const bool in = (uint32_t)i - s < d.fsizes[f];
    const uint32_t op = in ? ra_op(d, f, (uint32_t)i, s, rd, rs1, rs2, ins, odd) : 0u;
    d.ops[i] = op;
    if (odd) { atomicOr(d.flags, EF_XCONFLICT); d.cflag[prog_of(d.pf, d.P, f)] = 1; }
}

// ================================================================= regalloc
struct RaStep {
    uint32_t ord, rs1, rs2, r1r, r2r, rdr;
    bool sw1, sw2, swd;
    uint64_t newlife;
};

// One allocation step of one function (rv_generator_avx.cpp:1062-1397), given
// the word's fields, the operands' gathered registers (raw1/raw2: 0 when not
// virtual) and their swapped states.
DEV RaStep ra_eval_raw(uint32_t ins, uint32_t ord, uint32_t rs1, uint32_t rs2, uint32_t raw1, uint32_t raw2,
                       bool s1, bool s2, uint64_t life) {
    RaStep r;
    r.rs1 = rs1; r.rs2 = rs2; r.ord = ord;
    const bool v1 = (int32_t)rs1 > 63, v2 = (int32_t)rs2 > 63;
    r.r1r = v1 ? raw1 : 0u;
    r.r2r = v2 ? raw2 : 0u;
    if (v1 && s1) r.r1r = (ins == 0xC0007053u || (ins & 0x7Fu) == 0x53u) ? 37u : 5u;
    if (v2 && s2) r.r2r = ((ins & 0x7Fu) == 0x53u) ? 38u : 6u;
    const uint64_t clr = ((1ull << r.r1r) | (1ull << r.r2r)) & ~1ull;
    const uint64_t cl = life & ~clr;
    uint32_t rdr = ord;
    if ((int32_t)ord > 63) {
        const bool rdf = ins == 0xD0007053u || (ins & 0x7Fu) == 0x53u;
        rdr = ffz_gcc(cl | (rdf ? 0xFFFFFFFFull : 0xFFFFFFFF00000000ull));
        if (rdr == 64) rdr = rdf ? 37u : 5u;
    }
    r.rdr = rdr;
    r.sw1 = r.r1r != 0 && ((life >> r.r1r) & 1ull);
    r.sw2 = r.r2r != 0 && ((life >> r.r2r) & 1ull);
    r.swd = rdr != 0 && ((cl >> rdr) & 1ull);
    r.newlife = cl | (1ull << rdr);
    return r;
}

// Whether v is a virtual register inside the words (one past them is flagged).
DEV bool virt_ok(const Dev &d, uint32_t v) {
    if ((int32_t)v <= 63) return false;
    if (v - 64u >= d.W0) { atomicOr(d.flags, EF_OOB); return false; }
    return true;
}

DEV RaStep ra_eval(const Dev &d, uint32_t off, uint64_t life, bool s1, bool s2) {
    const uint4 w = d.w0_f4[off];
    const uint32_t raw1 = virt_ok(d, w.y) ? (d.sym[w.y - 64u] & 0xFFu) : 0u;
    const uint32_t raw2 = virt_ok(d, w.z) ? (d.sym[w.z - 64u] & 0xFFu) : 0u;
    return ra_eval_raw(w.w, w.x, w.y, w.z, raw1, raw2, s1, s2, life);
}

DEV bool sym_swapped(const Dev &d, uint32_t v) { return (d.sym[v] & 0x100u) != 0; }

DEV void sym_mark(const Dev &d, uint32_t v) { reinterpret_cast<uint8_t *>(d.sym)[2u * v + 1u] = 1; }

// register_state updates of one step (rv_generator_avx.cpp:1356-1397): each
// named virtual register takes its register and, as the lane-0 lockstep
// commits, a cleared swapped flag.  The swapped flags of functions outside
// lane 0 are never set, so writing the whole entry is the same as writing the
// register alone there.
DEV void ra_commit_syms(const Dev &d, const RaStep &r) {
    if (((int32_t)r.ord > 63 && r.ord - 64u >= d.W0) || ((int32_t)r.rs1 > 63 && r.rs1 - 64u >= d.W0) ||
        ((int32_t)r.rs2 > 63 && r.rs2 - 64u >= d.W0)) { atomicOr(d.flags, EF_OOB); return; }
    if ((int32_t)r.ord > 63) d.sym[r.ord - 64u] = (uint16_t)r.rdr;
    if ((int32_t)r.rs1 > 63) d.sym[r.rs1 - 64u] = (uint16_t)r.r1r;
    if ((int32_t)r.rs2 > 63) d.sym[r.rs2 - 64u] = (uint16_t)r.r2r;
}

// Functions outside lane 0 of their group: their swapped flags are never set
// (only lane-0 registers are ever looked up), so each walks alone.  What the
// lane-0 functions need of them is which registers each group looks up at each
// step.  permw lists these functions by size, largest first, so that the 64
// walks of a workgroup take about the same number of steps.
//
// Workgroups spread their per-step lookup records over up to WALK_COPIES
// copies of the (step, register) tables (copy = workgroup mod copies), which
// k_walk_merge folds: one table shared by every workgroup serializes its
// atomics on the same few addresses.  Programs of at most RA0_WAVE_GROUPS
// groups have (step, group) tables of 64-bit register masks instead, in up to
// MASK_COPIES copies.
constexpr uint32_t WALK_COPIES = 16;
constexpr uint32_t MASK_COPIES = 2;
constexpr uint32_t RA0_WAVE_GROUPS = 64;
// Walk and lockstep may run at the same time: for each program whose lockstep
// does, each walk workgroup holding functions of it publishes the program's
// table rows in chunks of WALK_PUB rows, adding 1 to done[cbase + chunk]
// (release, agent scope) once it has posted every row of the chunk it takes
// part in (the lowest lane of the program in the workgroup publishes).  The
// lockstep reads a row after the counter reaches need[cbase + chunk], the
// number of walk workgroups holding a function of the program that still runs
// at the chunk's first row.  Walk workgroups never wait, so when both kernels are resident
// the lockstep's wait always ends.  Where dispatches are serialized (a profiler
// collecting counters), the walk cannot start before the lockstep ends: a wait
// that sees no progress for RA0_WAIT_TICKS of the 100 MHz wall clock gives up
// for the rest of the kernel (EF_WAIT), and the host redoes the allocation with
// the two kernels one after the other.
constexpr uint32_t WALK_PUB = 32;
constexpr uint32_t RA0_MAXCOPIES = 8;  // table copies the lockstep folds itself
constexpr uint64_t RA0_WAIT_TICKS = 25000000ull;  // 0.25 s

// One program's allocation: functions from fbase (nf of them) in groups of 8
// (L groups), maxsize = its longest function; its slices of the lane-0 group
// order (perm + poff) and of the lookup tables (+ gbase: (step, register)
// tables, or (step, group) masks when L is at most RA0_WAVE_GROUPS).  The
// tables hold `rows` steps: every step while a lane-0 function is running, then
// (when some other function runs longer) one last row that gathers all later
// steps.  Past its lane-0 functions the snapshot no longer changes and no owner
// reads, so a later lookup only marks, whatever its step.
// cbase: its first row chunk in the walk's publish counters (RA0_NOPUB when its
// lockstep does not run at the same time as the walk).  prg: its index.
struct Ra0Prog { uint32_t fbase, L, maxsize, poff; uint64_t gbase; uint32_t nf, rows, cbase, prg; };
constexpr uint32_t RA0_NOPUB = 0xFFFFFFFFu;

// OR of v over the 8 lanes of each group of a wave, every lane active (DPP:
// swap neighbours, swap pairs, then mirror each half row of 8).
DEV uint32_t sm_or8(uint32_t v) {
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false);  // row_half_mirror
    return v;
}
DEV uint64_t sm_or8_64(uint64_t v) { return (uint64_t)sm_or8((uint32_t)v) | ((uint64_t)sm_or8((uint32_t)(v >> 32)) << 32); }

// Ends a rarely taken branch that loads: without a wait of its own the compiler
// waits where the branch joins, on every step, and since loads and stores share
// the counter that wait is for every store and atomic before it too.
DEV void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)

// One step of a walk (rv_generator_avx.cpp:1062-1397) from the word's op, the
// registers its operands are read in and the function's lifetime mask: the
// registers freed (m; never x0), the one written (rdr, dm), the live registers
// looked up, the new lifetime.
struct OpStep { uint32_t rdr; uint64_t m, dm, look, life; };
DEV OpStep op_eval(uint32_t op, uint32_t r1, uint32_t r2, uint64_t life) {
    OpStep s;
    s.m = ((1ull << r1) | (1ull << r2)) & ~1ull;
    const uint64_t cl = life & ~s.m;
    const uint32_t fr = ~(uint32_t)cl;  // free integer registers (ffz_gcc); none: t0
    const uint32_t al = fr ? (uint32_t)__builtin_ctz(fr) : 5u;
    s.rdr = (op & OP_ALLOC) ? al : (op >> OP_CONST) & 63u;
    s.dm = 1ull << s.rdr;
    s.look = ((s.m & life) | (s.dm & cl)) & ~1ull;
    s.life = cl | s.dm;
    return s;
}

// The ops of four consecutive words (any 4-byte alignment).
struct __attribute__((packed, aligned(4))) Op4 { uint32_t o[4]; };
// Four consecutive states of a function's registers (any 2-byte alignment).
struct __attribute__((packed, aligned(2))) Sym4 { uint64_t v; };
struct __attribute__((packed, aligned(2))) Sym8 { uint32_t w[4]; };

// A function's ops in registers, 16 steps at a time: the load of the next 16 is
// waited for once in 16 steps (its wait also waits for every store before it),
// and `cur` moves down by four every four steps, so that it is indexed by
// constants alone.
struct OpBlock {
    Op4 cur[4], nxt[4];
    DEV void load(const uint32_t *ops, uint32_t i, uint32_t size) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) nxt[k] = *reinterpret_cast<const Op4 *>(ops + min(i + 4u * k, size));
    }
    DEV void step4(const uint32_t *ops, uint32_t i, uint32_t size) {  // before steps i .. i + 3 (i % 4 == 0)
        if (i % 16u == 0) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) cur[k] = nxt[k];
            load(ops, i + 16u, size);
        } else {
            cur[0] = cur[1]; cur[1] = cur[2]; cur[2] = cur[3];
        }
    }
};

// The same a step at a time: N loads of four ops ahead.
template <int N>
struct OpQueue {
    Op4 cur[N], nxt[N];
    DEV void load(const uint32_t *ops, uint32_t i, uint32_t size) {
#pragma unroll
        for (int k = 0; k < N; ++k) nxt[k] = *reinterpret_cast<const Op4 *>(ops + min(i + 4u * k, size));
    }
    DEV uint32_t next(const uint32_t *ops, uint32_t i, uint32_t size) {  // step i's op, from i % (4 * N) == 0 on
        if (i % (4u * N) == 0) {
#pragma unroll
            for (int k = 0; k < N; ++k) cur[k] = nxt[k];
            load(ops, i + 4u * N, size);
        } else if (N > 1 && i % 4u == 0) {
#pragma unroll
            for (int k = 0; k + 1 < N; ++k) cur[k] = cur[k + 1];
        }
        const uint32_t op = cur[0].o[0];
        cur[0].o[0] = cur[0].o[1]; cur[0].o[1] = cur[0].o[2]; cur[0].o[2] = cur[0].o[3];
        return op;
    }
};


DEV uint32_t rdlane(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }
extern "C" __device__ int ptl_writelane(int x, int l, int v) __asm("llvm.amdgcn.writelane.i32");
DEV uint32_t wrlane(uint32_t v, uint32_t l, uint32_t x) { return (uint32_t)ptl_writelane((int)x, (int)l, (int)v); }
DEV uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// A walk of one function on a whole wave: the step is scalar code (a scalar
// instruction takes about half a vector one's time in a dependent chain, has
// 64-bit masks and cheap branches), and what it needs of the last words is a lane
// of a vector register: `cur` has the ops of the block of 64 steps, `ringv` the
// states of the last 64 words (word mod 64), written and read by lane.  States
// go to HBM, and lookups to the tables, once a block, from all lanes.  Operands
// 64 words back and more are in the LDS ring `old`.
// Latency bound: 0.14 us a step against 0.30 as a lane (a function of 4115 words,
// 1.24 -> 0.58 ms).
constexpr uint32_t WALK_OLD = 16384;  // words of the LDS ring
DEV void walk_one(const Dev &d, uint8_t *old, unsigned long long *mtab, const Ra0Prog &pg, uint32_t f, uint32_t grp,
                  uint32_t lane, uint32_t *done) {
    const uint32_t start = uniform(d.fstarts[f]), size = uniform(d.fsizes[f]);
    const uint32_t L = pg.L, last = pg.rows - 1u;
    unsigned long long *tab = mtab + pg.gbase + grp;
    uint32_t ringv = 0, lo = 0, hi = 0;
    uint64_t life = 0x1Full;
    auto load = [&](uint32_t i) { return d.ops[start + min(i + lane, size)]; };
    uint32_t nxt = load(0);
    for (uint32_t b = 0; b < size; b += 64) {
        uint32_t cur = nxt;
        asm volatile("" : "+v"(cur) : : "memory");  // waited for before the next load is issued
        nxt = load(b + 64u);
        const uint32_t n = min(64u, size - b);
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t op = rdlane(cur, k);
            const uint32_t d1 = op & 0xFFu, d2 = (op >> 8) & 0xFFu;
            uint32_t r1 = d1 ? rdlane(ringv, (k - d1) & 63u) : 0u, r2 = d2 ? rdlane(ringv, (k - d2) & 63u) : 0u;
            if (__builtin_expect((op & (0xC0C0u | OP_FAR1 | OP_FAR2)) != 0, 0)) {
                const uint32_t i = b + k;
                const uint4 w = d.w0_f4[start + i];
                wait_loads();
                const uint32_t p1 = (op & OP_FAR1) ? uniform(w.y) - 64u - start : i - d1;
                const uint32_t p2 = (op & OP_FAR2) ? uniform(w.z) - 64u - start : i - d2;
                // (a word 64 or more back is in a block that has ended)
                auto state = [&](uint32_t p) {
                    uint32_t v = i - p < WALK_OLD - 64u ? old[p % WALK_OLD] : d.sym[start + p];
                    wait_loads();
                    return uniform(v) & 0x3Fu;
                };
                if ((op & OP_FAR1) || d1 > 63u) r1 = state(p1);
                if ((op & OP_FAR2) || d2 > 63u) r2 = state(p2);
            }
            const OpStep s = op_eval(op, r1, r2, life);
            life = s.life;
            ringv = wrlane(ringv, k, (op & (OP_SELF | OP_ZERO)) == OP_SELF ? s.rdr : 0u);
            lo = wrlane(lo, k, (uint32_t)s.look);
            hi = wrlane(hi, k, (uint32_t)(s.look >> 32));
        }
        if (lane < n) {
            const uint32_t i = b + lane;
            d.sym[start + i] = (uint16_t)ringv;
            old[i % WALK_OLD] = (uint8_t)ringv;
            const unsigned long long look = (unsigned long long)lo | ((unsigned long long)hi << 32);
            if (look) atomicOr(tab + (uint64_t)min(i, last) * L, look);
        }
        if (done && pg.cbase != RA0_NOPUB) {
            // the chunks of rows this block leaves (see k_ra_walk)
            const uint32_t nch = last / WALK_PUB + 1u, e = b + 64u;
            const uint32_t npub = min(nch, (size + WALK_PUB - 1u) / WALK_PUB);
            const uint32_t from = min(b / WALK_PUB, nch - 1u), to = e >= size ? npub : min(e / WALK_PUB, nch - 1u);
            if (from < to) {
                __threadfence();
                if (lane < to - from)
                    __hip_atomic_fetch_add(&done[pg.cbase + from + lane], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// One function per lane.  The states of a function's last OP_ROWS words are in
// an LDS ring of bytes, row = word mod OP_ROWS (a state here is just the
// register the word's rd was given; it never changes); operands further back
// are read from HBM.  Bound by the step's chain of instructions (latency; one
// wave per SIMD): steps run four at a time, on ops loaded 16 steps ahead and with
// one 8-byte store of states.  A 62-function program's
// 4115 steps: 4.7 -> 1.2 ms against words compared and states looked up in a
// tagged cache at each step.
__global__ __launch_bounds__(64) void k_ra_walk(Dev d, uint32_t *gmin_all, uint32_t *gmax_all, uint64_t stride,
                                                uint32_t copies, unsigned long long *mask_all, uint64_t mstride,
                                                uint32_t mcopies, const Ra0Prog *progs, const uint32_t *permw,
                                                uint32_t nw, uint32_t nreg, uint32_t solo, uint32_t *done) {
    __shared__ uint32_t smin[4][64], smax[4][64];
    __shared__ uint8_t ring[OP_ROWS * 64];
    static_assert(sizeof(ring) >= WALK_OLD, "walk_one's LDS ring");
    const uint32_t lane = threadIdx.x;
    // 64 functions to a workgroup: those of programs with (step, register) tables
    // (the first nreg, a workgroup's all of one program, padded), and the last
    // ones; `solo` between them have one each
    const uint32_t nb0 = (nreg + 63u) / 64u;
    uint32_t t = blockIdx.x * 64u + lane, tend = nreg;
    if (blockIdx.x >= nb0 + solo) { t = nreg + solo + (blockIdx.x - nb0 - solo) * 64u + lane; tend = nw; }
    else if (blockIdx.x >= nb0) {
        const uint32_t f = permw[nreg + blockIdx.x - nb0];
        const uint32_t prg = prog_of(d.pf, d.P, f);
        if (d.cflag[prg]) return;  // k_ra_serial's
        walk_one(d, ring, mask_all + (blockIdx.x % mcopies) * mstride, progs[prg], f, (f - d.pf[prg]) >> 3, lane, done);
        return;
    }
    const uint32_t f = t < tend ? permw[t] : d.F;
    const bool act = f < d.F;
    // group = function index within its program / 8; lookup table of the program
    const uint32_t prg = act ? prog_of(d.pf, d.P, f) : 0xFFFFFFFFu;
    const uint32_t grp = act ? (f - d.pf[prg]) >> 3 : 0u;
    const bool skip = act && d.cflag[prg] != 0;  // k_ra_serial's
    const uint32_t start = act ? d.fstarts[f] : 0u;
    const uint32_t size = act && !skip ? d.fsizes[f] : 0u;
    const uint32_t L = act ? progs[prg].L : 0u;
    const bool reg = blockIdx.x < nb0;  // (step, register) tables
    uint32_t *gmin = gmin_all + (blockIdx.x % copies) * stride;
    uint32_t *gmax = gmax_all + (blockIdx.x % copies) * stride;
    unsigned long long *mtab = mask_all + (blockIdx.x % mcopies) * mstride;
    const uint64_t mbase = act ? progs[prg].gbase : 0u;  // own program's table and its last row
    const uint32_t mlast = act ? progs[prg].rows - 1u : 0u;
    const uint64_t tb = (uint64_t)uniform((uint32_t)mbase) | ((uint64_t)uniform((uint32_t)(mbase >> 32)) << 32);
    const uint32_t tlast = uniform(mlast);  // (a workgroup's first lane has a function)
    // the lowest lane of each program in the workgroup publishes that program's
    // rows; pw = the size of the program's longest function here
    uint32_t pw = 0;
    bool lead = false;
    if (done) {
        uint64_t rem = __ballot(act);
        while (rem) {
            const uint32_t l = (uint32_t)__builtin_ctzll(rem);
            const uint32_t p = (uint32_t)__shfl((int)prg, (int)l, 64);
            const bool mine = act && prg == p;
            const uint64_t same = __ballot(mine);
            uint32_t m = mine ? size : 0u;
            for (int s = 32; s > 0; s >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, s, 64));
            if (mine) { pw = m; lead = lane == l; }
            rem &= ~same;
        }
    }
    const uint32_t cbase = act ? progs[prg].cbase : RA0_NOPUB;
    const bool publishes = done && lead && cbase != RA0_NOPUB && pw != 0;
    const uint32_t nch = mlast / WALK_PUB + 1u;
    const uint32_t npub = publishes ? min(nch, (pw + WALK_PUB - 1u) / WALK_PUB) : 0u;  // chunks it takes part in
    uint32_t pubd = 0;
    for (uint32_t q = 0; q < 4; ++q) { smin[q][lane] = 0xFFFFFFFFu; smax[q][lane] = 0; }
    uint32_t wmax = size;
    for (int s = 32; s > 0; s >>= 1) { uint32_t o = __shfl_xor(wmax, s, 64); wmax = wmax > o ? wmax : o; }
    uint64_t life = 0x1Full;
    const uint32_t *ops = d.ops + start;
    OpBlock ob;
    ob.load(ops, 0, size);
    __syncthreads();
    for (uint32_t i0 = 0; i0 < wmax; i0 += 4) {
        ob.step4(ops, i0, size);
        uint32_t st[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t i = i0 + q;
            const bool run = (int32_t)i < (int32_t)size;
            const uint32_t op = run ? ob.cur[0].o[q] : 0u;
            const uint32_t d1 = op & 0xFFu, d2 = (op >> 8) & 0xFFu;
            uint32_t r1 = ring[((i - d1) & (OP_ROWS - 1u)) * 64u + lane];
            uint32_t r2 = ring[((i - d2) & (OP_ROWS - 1u)) * 64u + lane];
            r1 = d1 ? r1 : 0u; r2 = d2 ? r2 : 0u;
            if (__ballot((op & (OP_FAR1 | OP_FAR2)) != 0)) {
                if (op & (OP_FAR1 | OP_FAR2)) {
                    const uint4 w = d.w0_f4[start + i];
                    if (op & OP_FAR1) r1 = d.sym[w.y - 64u] & 0xFFu;
                    if (op & OP_FAR2) r2 = d.sym[w.z - 64u] & 0xFFu;
                    wait_loads();
                }
            }
            const OpStep s = op_eval(op, r1, r2, life);
            life = s.life;
            st[q] = (op & OP_SELF) && !(op & OP_ZERO) ? s.rdr : 0u;
            ring[(i & (OP_ROWS - 1u)) * 64u + lane] = (uint8_t)st[q];
            if (!reg) {
                if (run && s.look) atomicOr(&mtab[mbase + (uint64_t)min(i, mlast) * L + grp], (unsigned long long)s.look);
            } else {
                uint64_t lk = run ? s.look : 0ull;
                while (lk) {
                    const uint32_t r = (uint32_t)__builtin_ctzll(lk);
                    lk &= lk - 1;
                    atomicMin(&smin[q][r], grp); atomicMax(&smax[q][r], grp + 1u);
                }
            }
        }
        if (reg) {  // the four steps' lookups, folded over the workgroup
            lds_barrier();
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t mn = smin[q][lane], mx = smax[q][lane];
                if (mx) {
                    const uint64_t e = tb + (uint64_t)min(i0 + q, tlast) * 64u + lane;
                    atomicMin(&gmin[e], mn);
                    atomicMax(&gmax[e], mx);
                    smin[q][lane] = 0xFFFFFFFFu; smax[q][lane] = 0;
                }
            }
            lds_barrier();
        }
        // (sym starts cleared: only words past the last whole four need care)
        if ((int32_t)(i0 + 3u) < (int32_t)size) {
            reinterpret_cast<Sym4 *>(d.sym + start + i0)->v =
                (uint64_t)(st[0] | (st[1] << 16)) | ((uint64_t)(st[2] | (st[3] << 16)) << 32);
        } else {
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if ((int32_t)(i0 + q) < (int32_t)size) d.sym[start + i0 + q] = (uint16_t)st[q];
        }
        if (done) {
            // chunks of the program's rows that its functions here are past
            // (steps past its last row all post to that row): published after
            // every lane's posts are visible; at most one chunk per four steps
            const uint32_t e = i0 + 4u;
            const uint32_t past = e >= pw ? npub : min(e / WALK_PUB, nch - 1u);
            const bool pub = publishes && past > pubd;
            if (__ballot(pub)) {
                __threadfence();
                __syncthreads();
                if (pub) {
                    __hip_atomic_fetch_add(&done[cbase + pubd], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ++pubd;
                }
            }
        }
    }
}

// gmin/gmax[e] = min/max over the copies (copy c at c * stride); mask[e] = OR
// over its copies.
__global__ void k_walk_merge(uint32_t *gmin, uint32_t *gmax, uint64_t stride, uint32_t copies,
                             unsigned long long *mask, uint64_t mstride, uint32_t mcopies) {
    const uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (copies > 1 && e < stride) {
        uint32_t mn = gmin[e], mx = gmax[e];
        for (uint32_t c = 1; c < copies; ++c) {
            mn = min(mn, gmin[c * stride + e]);
            mx = max(mx, gmax[c * stride + e]);
        }
        gmin[e] = mn; gmax[e] = mx;
    }
    if (mcopies > 1 && e < mstride) {
        unsigned long long m = mask[e];
        for (uint32_t c = 1; c < mcopies; ++c) m |= mask[c * mstride + e];
        mask[e] = m;
    }
}

// Waits (every lane of the wave) until the walk has published row chunk c;
// `ok` turns false, for good, when a wait sees no progress for RA0_WAIT_TICKS.
DEV void ra0_wait(const Dev &d, const uint32_t *done, const uint32_t *need, uint32_t c, bool &ok) {
    if (!ok) return;
    const uint32_t want = need[c];
    const uint64_t t0 = wall_clock64();
    // (the polls are relaxed: an acquire invalidates the compute unit's caches,
    // which the waves beside use; one at the end orders the rows' loads)
    while (__hip_atomic_load(&done[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want) {
        if (wall_clock64() - t0 > RA0_WAIT_TICKS) { ok = false; atomicOr(d.flags, EF_WAIT); return; }
        __builtin_amdgcn_s_sleep(8);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// The same for the wave's 64 chunks from c on: waits until c is published and
// returns the first chunk not known to be (a lockstep behind the walk then polls
// once in 64 chunks).
DEV uint32_t ra0_wait_run(const Dev &d, const uint32_t *done, const uint32_t *need, uint32_t c, uint32_t n, bool &ok) {
    if (!ok) return n;
    const uint32_t x = min(c + (threadIdx.x & 63u), n - 1u);
    const uint32_t want = need[x];
    const uint64_t t0 = wall_clock64();
    uint64_t got;
    while (got = __ballot(__hip_atomic_load(&done[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want), (got & 1u) == 0) {
        if (wall_clock64() - t0 > RA0_WAIT_TICKS) { ok = false; atomicOr(d.flags, EF_WAIT); return n; }
        __builtin_amdgcn_s_sleep(8);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return c + (got == ~0ull ? 64u : (uint32_t)__builtin_ctzll(~got));
}

// ---------------------------------------------- lane-0 functions in one wave
// Region 0 of the reference's register_state holds the last lane-0 write per
// physical register; every lookup of any function at step i reads its
// step-start snapshot and marks the virtual register found there as swapped.
// A lane steps one function; the snapshot is kept apart by owner: `own` has
// the entries that hold one of this function's virtual registers, hold[r] the
// word that defines it, `mk` the owned entries whose register is marked
// already.  A register can only be held by the entry of the register it was
// defined in, its home, so a state is
//     register | swapped << 8 | home << 9
// and the entry an operand is held by is found from its state alone.  States of
// the last OP_ROWS words are in an LDS ring; HBM (sym) has all of them, written
// through.
struct RaL0 { uint32_t start, size; uint64_t life, own, mk; };

template <int CTRL, int RMASK = 0xF>
DEV uint32_t dpp_or(uint32_t v) {
    return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RMASK, 0xF, RMASK == 0xF);
}
// Inclusive OR over the lanes up to this one, in the wave's first row of 16
// lanes (ROWS 1) or the whole wave; every lane active.
template <int ROWS>
DEV uint32_t scan_or(uint32_t v) {
    v = dpp_or<0x111>(v); v = dpp_or<0x112>(v); v = dpp_or<0x114>(v); v = dpp_or<0x118>(v);  // row_shr 1, 2, 4, 8
    if (ROWS > 1) { v = dpp_or<0x142, 0xA>(v); v = dpp_or<0x143, 0xC>(v); }                  // row_bcast 15, 31
    return v;
}
// The lane below's value (0 in lane 0).
template <int ROWS>
DEV uint32_t from_below(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ROWS > 1 ? 0x138 : 0x111, 0xF, 0xF, true);  // wave_shr / row_shr 1
}
// OR over the lanes above this one; `all` the OR over every lane.
template <int ROWS>
DEV uint32_t suffix_or(uint32_t v, uint32_t lane, uint32_t &all) {
    v = dpp_or<0x101>(v); v = dpp_or<0x102>(v); v = dpp_or<0x104>(v); v = dpp_or<0x108>(v);  // row_shl 1, 2, 4, 8
    uint32_t x = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x101, 0xF, 0xF, true);
    const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
    if (ROWS == 1) { all = t0; return x; }
    const uint32_t t1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16), t2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32),
                   t3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    x |= lane < 48u ? t3 : 0u;
    x |= lane < 32u ? t2 : 0u;
    x |= lane < 16u ? t1 : 0u;
    all = t0 | t1 | t2 | t3;
    return x;
}

// Lookups of the step by the walked functions, as a lane-0 step takes them: per
// lane a mask of the registers its group's other functions look up (W), or per
// register the least and greatest group + 1 (mn, mx) with the mask of those
// looked up at all (any).
struct RaLooks { uint64_t W; const uint32_t *mn, *mx; uint64_t any; };

// Register states of a lane's last words: an LDS ring of OP_ROWS rows, row = word
// mod OP_ROWS, and one row more that takes the writes of lanes whose function has
// ended (RC columns).  Rows leave it four at a time, before the steps of a block
// of four from b overwrite them, so that HBM gets one 8-byte store per four steps
// and no store for a change within the ring: words from ring_low(b) on are in
// the ring, older ones in HBM.
DEV uint32_t ring_low(uint32_t b, uint32_t size) {  // (the last block's for a function that has ended)
    const uint32_t e = min(b, (size - 1u) & ~3u);
    return e > OP_ROWS - 4u ? e - (OP_ROWS - 4u) : 0u;
}
template <int RC>
DEV void ra_evict(const Dev &d, const RaL0 &f, const uint16_t *ring, uint32_t rc, uint32_t b) {
    if (b >= OP_ROWS && (int32_t)b < (int32_t)f.size) {
        uint32_t e[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) e[q] = ring[((b + q) & (OP_ROWS - 1u)) * RC + rc];
        reinterpret_cast<Sym4 *>(d.sym + f.start + (b - OP_ROWS))->v =
            (uint64_t)(e[0] | (e[1] << 16)) | ((uint64_t)(e[2] | (e[3] << 16)) << 32);
    }
}
// The states still in the ring, after the last step.
template <int RC>
DEV void ra_flush(const Dev &d, const RaL0 &f, const uint16_t *ring, uint32_t rc) {
    if (f.size == 0) return;
    for (uint32_t p = ring_low(f.size, f.size); p < f.size; ++p)
        d.sym[f.start + p] = ring[(p & (OP_ROWS - 1u)) * RC + rc];
}

// One step i (of the block of four from b) of this lane's function on its word's
// op (0 where it has ended).  The wave's lanes walk the lane-0 functions of one
// program, the highest group in lane 0 (j: the lane's group), in the first row of
// 16 lanes (MODE 1) or all four (4, 5), the walk's lookups given by lane (1, 4) or
// by register (5).
// A lookup marks the virtual register its entry holds, except one the word names
// (its reset lands after a mark by its own or a lower group).  A lookup by a lower
// group is seen by the owner's operand read of the same
// step (a flip), settled by re-evaluation until the flips are stable: a group's
// depend on the groups below it alone, so this reaches the in-order result.  A
// lookup by a higher group lands after the owner's own reset, and the last group
// to write or free a register decides its entry.
// A wave runs alone on its SIMD, so a branch costs what ten instructions do
// whether it is taken or not: everything but the rare cases (a state read from
// HBM, a second mark, a flip) is straight-line, its writes going to a spare row or
// entry where there is nothing to write, and the rare cases are out of line (in
// line, jumped over: 0.55 us a step of 8 groups against 0.53).
// hold has an entry per register and one spare.
template <int MODE, int RC>
DEV void ra_l0_step(const Dev &d, RaL0 &f, uint16_t *ring, uint32_t *hold, uint32_t rc, uint32_t lane, uint32_t j,
                    uint32_t b, uint32_t i, uint32_t op, const RaLooks &lk) {
    constexpr int ROWS = MODE > 1 ? 4 : 1;
    constexpr int LAST = ROWS == 1 ? 15 : 63;
    const uint32_t d1 = op & 0xFFu, d2 = (op >> 8) & 0xFFu;
    const uint32_t ws = (int32_t)i < (int32_t)f.size ? i & (OP_ROWS - 1u) : OP_ROWS;  // this word's row
    uint32_t p1 = i - d1, p2 = i - d2;
    uint32_t w1 = d1 ? p1 & (OP_ROWS - 1u) : ws, w2 = d2 ? p2 & (OP_ROWS - 1u) : ws;
    uint32_t e1 = ring[w1 * RC + rc], e2 = ring[w2 * RC + rc];
    e1 = d1 ? e1 : 0u; e2 = d2 ? e2 : 0u;
    const uint32_t rl = ring_low(b, f.size);
    const bool far = __ballot((op & (OP_FAR1 | OP_FAR2)) != 0) != 0;
    if (__builtin_expect(far, 0)) {
        if (op & (OP_FAR1 | OP_FAR2)) {
            const uint4 w = d.w0_f4[f.start + i];
            if (op & OP_FAR1) {
                p1 = w.y - 64u - f.start;
                if (p1 >= rl) { w1 = p1 & (OP_ROWS - 1u); e1 = ring[w1 * RC + rc]; } else e1 = d.sym[f.start + p1];
            }
            if (op & OP_FAR2) {
                p2 = w.z - 64u - f.start;
                if (p2 >= rl) { w2 = p2 & (OP_ROWS - 1u); e2 = ring[w2 * RC + rc]; } else e2 = d.sym[f.start + p2];
            }
            wait_loads();
        }
    }
    // whether the entry of an operand's home holds it (no operand: home x0, which
    // is never held)
    const uint32_t h1 = e1 >> 9, h2 = e2 >> 9;
    const uint32_t q1 = hold[h1], q2 = hold[h2];
    uint32_t mn1 = 0, mn2 = 0, mx1 = 0, mx2 = 0;
    if (MODE == 5) { mn1 = lk.mn[h1]; mn2 = lk.mn[h2]; mx1 = lk.mx[h1]; mx2 = lk.mx[h2]; }
    const uint32_t sr1 = (op & OP_FP) ? 37u : 5u, sr2 = (op & OP_FP) ? 38u : 6u;
    bool s1 = (e1 & 0x100u) != 0, s2 = (e2 & 0x100u) != 0;
    uint32_t r1 = s1 ? sr1 : e1 & 0x3Fu, r2 = s2 ? sr2 : e2 & 0x3Fu;
    OpStep s = op_eval(op, r1, r2, f.life);
    const uint64_t nb1 = q1 == p1 ? f.own & (1ull << h1) : 0ull, nb2 = q2 == p2 ? f.own & (1ull << h2) : 0ull;
    const uint64_t nb = nb1 | nb2;
    const bool self = (op & OP_SELF) != 0;
    uint32_t tl = (uint32_t)s.look | (uint32_t)lk.W, th = (uint32_t)(s.look >> 32) | (uint32_t)(lk.W >> 32);
    // looked up by a lower group (the lanes above); the walk's by register
    const uint64_t wl = MODE == 5 ? (mn1 < j ? nb1 : 0ull) | (mn2 < j ? nb2 : 0ull) : 0ull;
    uint32_t x;
    uint64_t low = wl | (uint64_t)suffix_or<ROWS>(tl, lane, x) | ((uint64_t)suffix_or<ROWS>(th, lane, x) << 32);
    bool n1 = (nb1 & low) != 0, n2 = (nb2 & low) != 0;
    const bool z1 = s1, z2 = s2;  // swapped already
    if (__builtin_expect(__ballot((n1 && !z1) || (n2 && !z2)) != 0, 0)) {
        bool ch;
        do {
            const bool f1 = n1, f2 = n2;
            s1 = z1 || f1; s2 = z2 || f2;
            r1 = s1 ? sr1 : e1 & 0x3Fu; r2 = s2 ? sr2 : e2 & 0x3Fu;
            s = op_eval(op, r1, r2, f.life);
            tl = (uint32_t)s.look | (uint32_t)lk.W; th = (uint32_t)(s.look >> 32) | (uint32_t)(lk.W >> 32);
            low = wl | (uint64_t)suffix_or<ROWS>(tl, lane, x) | ((uint64_t)suffix_or<ROWS>(th, lane, x) << 32);
            n1 = (nb1 & low) != 0; n2 = (nb2 & low) != 0;
            ch = (n1 != f1 && !z1) || (n2 != f2 && !z2);
        } while (__ballot(ch));
    }
    const uint32_t il = scan_or<ROWS>(tl), ih = scan_or<ROWS>(th);
    uint64_t high = (uint64_t)from_below<ROWS>(il) | ((uint64_t)from_below<ROWS>(ih) << 32);
    if (MODE == 5) high |= (mx1 > j + 1u ? nb1 : 0ull) | (mx2 > j + 1u ? nb2 : 0ull);
    uint64_t T = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)il, LAST) |
        ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)ih, LAST) << 32);
    if (MODE == 5) T |= lk.any;
    // new marks: owned entries looked up whose mark does not stand yet
    f.mk &= ~nb;
    const uint64_t nm = f.own & ~f.mk & ((T & ~nb) | (high & nb));
    f.mk |= nm;
    const uint32_t mr = (uint32_t)__builtin_ctzll(nm | (1ull << 63));
    const uint32_t mp = hold[mr];
    // the registers written or freed: by any lane, by a higher group
    const uint64_t touch = s.m | ((op & (OP_SELF | (63u << OP_CONST))) ? s.dm : 0ull);
    const uint32_t wl2 = scan_or<ROWS>((uint32_t)touch), wh2 = scan_or<ROWS>((uint32_t)(touch >> 32));
    const uint64_t above = (uint64_t)from_below<ROWS>(wl2) | ((uint64_t)from_below<ROWS>(wh2) << 32);
    const uint64_t lost = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)wl2, LAST) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)wh2, LAST) << 32);
    const uint64_t won = self ? s.dm & ~above : 0ull;
    // the step's commit: swapped operands take the register they were read
    // through, and their flags are cleared (an operand not swapped keeps its
    // entry; without one, this word's row takes the write and its own after it)
    const uint32_t st1 = s1 ? r1 | (h1 << 9) : e1, st2 = s2 ? r2 | (h2 << 9) : e2;
    ring[w1 * RC + rc] = (uint16_t)st1;
    ring[w2 * RC + rc] = (uint16_t)st2;
    if (__builtin_expect(far, 0)) {
        if ((op & OP_FAR1) && s1 && p1 < rl) d.sym[f.start + p1] = (uint16_t)st1;
        if ((op & OP_FAR2) && s2 && p2 < rl) d.sym[f.start + p2] = (uint16_t)st2;
    }
    // the mark of the first marked entry; the flag byte of its state
    uint8_t *rb = reinterpret_cast<uint8_t *>(ring);
    const bool inr = nm != 0 && mp >= rl;
    rb[2u * ((inr ? mp & (OP_ROWS - 1u) : OP_ROWS) * RC + rc) + 1u] = (uint8_t)(1u | (mr << 1));
    if (__builtin_expect(__ballot((nm & (nm - 1)) != 0 || (nm != 0 && !inr)) != 0, 0)) {
        for (uint64_t m = nm; m; m &= m - 1) {
            const uint32_t r = (uint32_t)__builtin_ctzll(m), p = hold[r];
            const uint8_t fl = (uint8_t)(1u | (r << 1));
            if (p >= rl) rb[2u * ((p & (OP_ROWS - 1u)) * RC + rc) + 1u] = fl;
            else reinterpret_cast<uint8_t *>(d.sym + f.start)[2u * p + 1u] = fl;
        }
    }
    ring[ws * RC + rc] = (uint16_t)(self ? ((op & OP_ZERO) ? 0u : s.rdr) | (s.rdr << 9) : 0u);
    hold[won ? s.rdr : 64u] = i;
    f.life = s.life;
    f.own = (f.own & ~lost) | won;
    f.mk &= ~lost;
}

// The lane-0 function of a program of one group, on a whole wave as walk_one
// (`own`, `mk` and the state as in ra_l0_step): every entry of region 0 is this
// function's, so a step needs of the others only their lookups, a mask a step
// (`wlo`, `whi`: those of the block's steps, by lane).  hold is a vector register,
// lane = entry, and ringv the states of this block's words and the last one's: those
// before are in HBM and an LDS ring, and a change to one goes to both.
// Latency bound, ~7 cycles for each of a step's ~90 scalar instructions; the rare
// cases (an operand ONE_BLOCK or more back, a marked operand, a mark of an old
// word or a second one) are out of line.  1.5 -> 0.24 us a step (0.59 as a lane of
// eight programs' wave; 0.32 with every mark a loop and the walk's progress
// polled each block): a stress program of 91k steps, 32 -> 26.6 ms.
constexpr uint32_t ONE_OLD = 4096;    // words of the LDS ring
constexpr uint32_t ONE_BLOCK = 32;    // steps of a block: a chunk of the walk's rows
constexpr uint32_t ONE_SELF = 23, ONE_WRITES = 28;  // bits of an op here: OP_SELF, and one set a block
static_assert(OP_SELF == 1u << ONE_SELF, "");
// first bit that is 1 (0), ~0 if there is none
DEV uint32_t ff1(uint64_t x) { uint32_t r; asm("s_ff1_i32_b64 %0, %1" : "=s"(r) : "s"(x)); return r; }
DEV uint32_t ff0(uint32_t x) { uint32_t r; asm("s_ff0_i32_b32 %0, %1" : "=s"(r) : "s"(x)); return r; }
// The state of such a function and its steps, B at a time.  old: an LDS ring of OLD
// words, STRIDE entries apart.  MULTI: the one function left of a program of more
// groups (k_ra_lane0_wave): the other groups' walked functions still look registers
// up, those of a lower group in time for the step's own reads (a flip, ra_l0_step),
// and entries that ended functions hold (oth, defined at word holdv of the function
// that starts at obase) are still marked.
struct SoloLooks { uint64_t W, low, high; };  // of every group; of those below and above the function's
template <uint32_t B, uint32_t OLD, uint32_t STRIDE, bool MULTI>
struct Solo {
    const Dev &d;
    uint32_t start, lane;
    uint16_t *old;
    uint32_t ringv, holdv, obase;
    uint64_t life, own, mk, oth;
    DEV uint16_t &at(uint32_t p) { return old[(p % OLD) * STRIDE]; }
    DEV uint8_t *flag(uint32_t p) { return reinterpret_cast<uint8_t *>(&at(p)) + 1; }
    // the states of the words [lo, hi), hi - lo <= 64, leave the ring
    DEV void flush(uint32_t lo, uint32_t hi) {
        const uint32_t w = lo + ((lane - lo) & 63u);
        if (w < hi) {
            d.sym[start + w] = (uint16_t)ringv;
            at(w) = (uint16_t)ringv;
        }
    }
    // the first word the ring holds in the block from b
    static DEV uint32_t kept_at(uint32_t b) { return b > 64u - B ? b - (64u - B) : 0u; }
    // before the block from b; first: the first block's
    DEV void begin(uint32_t b, uint32_t first) {
        if (b >= 64u && b >= first + B) flush(b - 64u, b - 64u + B);
        if (((lane - b) & 63u) < B) ringv = 0;
    }
    // steps b .. b + n - 1 on the ops `cur` (by lane); looks(k): the walk's lookups of step b + k
    template <class Looks>
    DEV void steps(uint32_t b, uint32_t n, uint32_t cur, Looks looks) {
        // the ring holds the words from kept on; the lanes of this block's are 0
        // until they are written, which is also the state of no operand
        const uint32_t kept = kept_at(b);
        const uint64_t oldown = __ballot(holdv < kept);  // entries whose word may have left the ring
        // state of a word from its register, as a factor; whether it ends its entry's holding
        const uint32_t fac = (cur & OP_SELF) ? ((cur & OP_ZERO) ? 0x200u : 0x201u) : 0u;
        cur |= (cur & (OP_SELF | (63u << OP_CONST))) ? 1u << ONE_WRITES : 0u;
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t i = b + k;
            const uint32_t op = rdlane(cur, k);
            const SoloLooks lk = looks(k);
            uint32_t p1 = i - (op & 0xFFu), p2 = i - ((op >> 8) & 0xFFu);
            uint32_t e1 = rdlane(ringv, p1 & 63u), e2 = rdlane(ringv, p2 & 63u);
            // a word's state after a read through register r that finds it marked
            auto flipped = [&](uint32_t e, uint32_t r) { return (e & ~0x1FFu) | r | ((op & OP_FP) ? 32u : 0u); };
            auto put = [&](uint32_t p, uint32_t v) {  // of a word that may have left the ring
                if (p >= kept) { ringv = wrlane(ringv, p & 63u, v); return; }
                if (i - p < OLD) at(p) = (uint16_t)v;
                d.sym[start + p] = (uint16_t)v;
            };
            if (__builtin_expect((op & (0xE0E0u | OP_FAR1 | OP_FAR2)) != 0, 0)) {
                if (op & (OP_FAR1 | OP_FAR2)) {
                    const uint4 w = d.w0_f4[start + i];
                    wait_loads();
                    if (op & OP_FAR1) p1 = uniform(w.y) - 64u - start;
                    if (op & OP_FAR2) p2 = uniform(w.z) - 64u - start;
                }
                auto look = [&](uint32_t p, uint32_t e) {
                    if (p >= kept) return p == i ? 0u : rdlane(ringv, p & 63u);
                    uint32_t v;
                    if (i - p < OLD - 64u) v = at(p);
                    else { v = d.sym[start + p]; wait_loads(); }
                    return uniform(v);
                };
                e1 = look(p1, e1);
                e2 = look(p2, e2);
            }
            if (__builtin_expect(((e1 | e2) & 0x100u) != 0, 0)) {  // marked operands: flipped back
                // (both read before either is written: they may be the same word)
                if (e1 & 0x100u) { e1 = flipped(e1, 5u); put(p1, e1); }
                if (e2 & 0x100u) { e2 = flipped(e2, 6u); put(p2, e2); }
            }
            const uint32_t h1 = e1 >> 9, h2 = e2 >> 9;
            const uint64_t nb1 = rdlane(holdv, h1) == p1 ? 1ull << h1 : 0ull, nb2 = rdlane(holdv, h2) == p2 ? 1ull << h2 : 0ull;
            const uint64_t nb = own & (nb1 | nb2);
            if (MULTI && __builtin_expect((nb & lk.low) != 0, 0)) {
                if (nb1 & own & lk.low) { e1 = flipped(e1, 5u); put(p1, e1); }
                if (nb2 & own & lk.low) { e2 = flipped(e2, 6u); put(p2, e2); }
            }
            // the step's lookups, as op_eval
            const uint64_t m = ((1ull << (e1 & 63u)) | (1ull << (e2 & 63u))) & ~1ull, cl = life & ~m;
            const uint32_t fr = ff0((uint32_t)cl), al = fr != ~0u ? fr : 5u;
            const uint32_t rdr = (op & OP_ALLOC) ? al : (op >> OP_CONST) & 63u;
            const uint64_t dm = 1ull << rdr;
            const uint64_t T = (((m & life) | (dm & cl)) & ~1ull) | lk.W;
            mk &= ~nb;
            uint64_t nm = MULTI ? own & ~mk & ((T & ~nb) | (lk.high & nb)) : own & ~(mk | nb) & T;
            mk |= nm;
            // new marks: mostly none or one, of a word in the ring
            const uint64_t more = (nm & (nm - 1)) | (nm & oldown);
            const uint32_t q = rdlane(holdv, ff1(nm) & 63u) & 63u, fl = nm ? 0x100u : 0u;
            ringv = wrlane(ringv, q, rdlane(ringv, q) | (more ? 0u : fl));
            if (__builtin_expect(more != 0, 0)) {
                for (; nm; nm &= nm - 1) {
                    const uint32_t r = (uint32_t)__builtin_ctzll(nm), p = rdlane(holdv, r);
                    if (p >= kept) { ringv = wrlane(ringv, p & 63u, rdlane(ringv, p & 63u) | 0x100u); continue; }
                    if (i - p < OLD) *flag(p) = (uint8_t)(1u | (r << 1));
                    reinterpret_cast<uint8_t *>(d.sym + start + p)[1] = (uint8_t)(1u | (r << 1));
                }
            }
            const uint64_t lost = m | ((uint64_t)((op >> ONE_WRITES) & 1u) << rdr);
            if (MULTI) {
                if (__builtin_expect((oth & T) != 0, 0)) mark_others(T);
                oth &= ~lost;
            }
            ringv = wrlane(ringv, i & 63u, rdr * rdlane(fac, k));
            holdv = wrlane(holdv, rdr, i);  // (of an entry not won: not owned, never read)
            own = (own & ~lost) | ((uint64_t)((op >> ONE_SELF) & 1u) << rdr);
            mk &= ~lost;
            life = cl | dm;
        }
    }
    DEV void mark_others(uint64_t T) {
        if (((oth & T) >> lane) & 1u) reinterpret_cast<uint8_t *>(d.sym + obase + holdv)[1] = (uint8_t)(1u | (lane << 1));
        oth &= ~T;
    }
    // the row that gathers the steps past the last, after the last flush
    DEV void finish(uint64_t W) {
        const uint64_t nm = own & ~mk & W;
        if ((nm >> lane) & 1u) reinterpret_cast<uint8_t *>(d.sym + start + holdv)[1] = (uint8_t)(1u | (lane << 1));
        if (MULTI) mark_others(W);
    }
};

__global__ __launch_bounds__(64) void k_ra_lane0_one(Dev d, const Ra0Prog *progs, const unsigned long long *mask_all,
                                                     uint64_t mstride, uint32_t mcopies, const uint32_t *done,
                                                     const uint32_t *need) {
    __shared__ uint16_t old[ONE_OLD];
    const uint32_t lane = threadIdx.x;
    const Ra0Prog pg = progs[blockIdx.x];
    if (d.cflag[pg.prg]) return;  // k_ra_serial's
    if (pg.L > 1u) { if (lane == 0) atomicOr(d.flags, EF_OOB); return; }
    const uint32_t start = uniform(d.fstarts[pg.fbase]), size = uniform(d.fsizes[pg.fbase]), rows = pg.rows;
    const uint32_t *pdone = done && pg.cbase != RA0_NOPUB ? done + pg.cbase : nullptr;
    const uint32_t *pneed = pdone ? need + pg.cbase : nullptr;
    const unsigned long long *tab = mask_all + pg.gbase;
    const uint64_t m1 = mcopies > 1 ? mstride : 0u;
    bool wok = true;
    // ops and lookups of the steps i + lane, lane < ONE_BLOCK (rows past the last: none)
    struct Block { uint32_t op; unsigned long long a, b; };
    uint32_t ready = 0;  // chunks known to be published
    auto load = [&](uint32_t i) {
        if (pdone && i < rows && i / WALK_PUB >= ready)
            ready = uniform(ra0_wait_run(d, pdone, pneed, i / WALK_PUB, (rows - 1u) / WALK_PUB + 1u, wok));
        const uint32_t x = i + lane, e = min(x, rows - 1u);
        Block r{0, 0, 0};
        if (lane < ONE_BLOCK) {
            r.op = d.ops[start + min(x, size)];
            if (x < rows) { r.a = tab[e]; r.b = tab[m1 + e]; }
        }
        return r;
    };
    Solo<ONE_BLOCK, ONE_OLD, 1, false> f{d, start, lane, old, 0u, 0u, 0u, 0x1Full, 0ull, 0ull, 0ull};
    Block nx = load(0);
    for (uint32_t b = 0; b < size; b += ONE_BLOCK) {
        uint32_t cur = nx.op, wlo = (uint32_t)(nx.a | nx.b), whi = (uint32_t)((nx.a | nx.b) >> 32);
        asm volatile("" : "+v"(cur), "+v"(wlo), "+v"(whi) : : "memory");  // waited for before the next loads are issued
        nx = load(b + ONE_BLOCK);
        f.begin(b, 0u);
        f.steps(b, uniform(min(ONE_BLOCK, size - b)), cur, [&](uint32_t k) {
            return SoloLooks{(uint64_t)rdlane(wlo, k) | ((uint64_t)rdlane(whi, k) << 32), 0ull, 0ull};
        });
    }
    if (size) f.flush(f.kept_at((size - 1u) / ONE_BLOCK * ONE_BLOCK), size);
    if (rows > size) {
        if (pdone) ra0_wait(d, pdone, pneed, (rows - 1u) / WALK_PUB, wok);
        const unsigned long long W = tab[rows - 1u] | tab[m1 + rows - 1u];
        f.finish((uint64_t)uniform((uint32_t)W) | ((uint64_t)uniform((uint32_t)(W >> 32)) << 32));
    }
}

// The lane-0 functions of a program of 2 to 16 (ROWS 1) or 64 (4) groups, in
// step lockstep on one wave: what the groups exchange in a step goes
// through DPP scans of 64-bit register masks, so a step has no barrier.  A
// second wave fetches the ops and the walk's lookups (one mask per group and
// step) into LDS, RA0_FETCH steps ahead: the stepping wave then waits for no
// load, and so for none of its own stores either (they share a counter).
// Bound by the chain of a step's instructions (latency): 5.4 -> 0.53 us a step
// for 8 groups, against a workgroup exchanging lookups through LDS atomics and
// barriers with its states in HBM; 0.8 us with the loads in the stepping wave.
// From the block on in which one function is left, its steps are a one-group
// program's (Solo; a step as above has three LDS reads in a chain, and leaving out
// its scans alone gained nothing): 62 functions, a quarter of 3740 steps, 2.10 ->
// 1.94 ms; 60 programs 6.5 -> 6.25 ms summed.
constexpr uint32_t RA0_FETCH = 16;
template <int ROWS>
__global__ __launch_bounds__(128) void k_ra_lane0_wave(Dev d, const Ra0Prog *progs, const unsigned long long *mask_all,
                                                       uint64_t mstride, uint32_t mcopies, const uint32_t *done,
                                                       const uint32_t *need) {
    constexpr int NL = ROWS == 1 ? 16 : 64;
    __shared__ uint16_t ring[(OP_ROWS + 1) * NL];
    __shared__ uint32_t hold[65];
    __shared__ uint32_t fop[2][RA0_FETCH][NL];
    __shared__ unsigned long long fw[2][RA0_FETCH][NL];
    const uint32_t lane = threadIdx.x & 63u, col = lane % NL;
    const bool fetch = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) != 0;
    const Ra0Prog pg = progs[blockIdx.x];
    if (d.cflag[pg.prg]) return;  // k_ra_serial's
    if (pg.L > (uint32_t)NL) { if (threadIdx.x == 0) atomicOr(d.flags, EF_OOB); return; }
    const bool act = lane < pg.L;
    const uint32_t j = act ? pg.L - 1u - lane : 0u;  // the lane's group
    RaL0 f{act ? d.fstarts[pg.fbase + 8u * j] : 0u, act ? d.fsizes[pg.fbase + 8u * j] : 0u, 0x1Full, 0, 0};
    const uint32_t rows = pg.rows;
    // the longest function's lane, and the first block of steps it is alone in
    uint32_t top = f.size;
    for (uint32_t o = 32; o > 0; o >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, (int)o, 64));
    const uint32_t al = uniform((uint32_t)__builtin_ctzll(__ballot(f.size == top)));
    uint32_t second = lane == al ? 0u : f.size;
    for (uint32_t o = 32; o > 0; o >>= 1) second = max(second, (uint32_t)__shfl_xor((int)second, (int)o, 64));
    const uint32_t alone = uniform((second + RA0_FETCH - 1u) / RA0_FETCH * RA0_FETCH);
    if (fetch) {
        const uint32_t *pdone = done && pg.cbase != RA0_NOPUB ? done + pg.cbase : nullptr;
        const uint32_t *pneed = pdone ? need + pg.cbase : nullptr;
        const unsigned long long *mtab = mask_all + pg.gbase + j;
        const uint64_t m1 = mcopies > 1 ? mstride : 0u;
        bool wok = true;  // the walk's rows still arrive
        for (uint32_t i = 0;; i += RA0_FETCH) {  // steps i .. i + RA0_FETCH - 1, zeros past the last row
            if (i < rows) {
                const uint32_t b = (i / RA0_FETCH) & 1u;
                if (pdone && i % WALK_PUB == 0) ra0_wait(d, pdone, pneed, i / WALK_PUB, wok);
                Op4 o[RA0_FETCH / 4];
                unsigned long long w0[RA0_FETCH], w1[RA0_FETCH];
#pragma unroll
                for (uint32_t k = 0; k < RA0_FETCH / 4; ++k)
                    o[k] = *reinterpret_cast<const Op4 *>(d.ops + f.start + min(i + 4u * k, f.size));
#pragma unroll
                for (uint32_t k = 0; k < RA0_FETCH; ++k) {
                    const uint64_t e = (uint64_t)min(i + k, rows - 1u) * pg.L;
                    w0[k] = mtab[e];
                    w1[k] = mtab[m1 + e];
                }
                if (lane < (uint32_t)NL) {
#pragma unroll
                    for (uint32_t k = 0; k < RA0_FETCH; ++k) {
                        fop[b][k][col] = (int32_t)(i + k) < (int32_t)f.size ? o[k / 4].o[k % 4] : 0u;
                        if (i < alone) fw[b][k][col] = act && i + k < rows ? w0[k] | w1[k] : 0ull;
                    }
                }
                if (i >= alone) {  // the masks of RaLooks for one function
#pragma unroll
                    for (uint32_t k = 0; k < RA0_FETCH; ++k) {
                        const uint64_t w = act && i + k < rows ? w0[k] | w1[k] : 0ull;
                        const uint64_t wo = lane > al ? w : 0ull, wh = lane < al ? w : 0ull;
                        constexpr uint32_t LAST = NL - 1;
                        const uint32_t a = scan_or<ROWS>((uint32_t)wo), c = scan_or<ROWS>((uint32_t)(wo >> 32));
                        const uint32_t g = scan_or<ROWS>((uint32_t)wh), h = scan_or<ROWS>((uint32_t)(wh >> 32));
                        const uint64_t low = (uint64_t)rdlane(a, LAST) | ((uint64_t)rdlane(c, LAST) << 32);
                        const uint64_t high = (uint64_t)rdlane(g, LAST) | ((uint64_t)rdlane(h, LAST) << 32);
                        const uint64_t own = (uint64_t)rdlane((uint32_t)w, al) | ((uint64_t)rdlane((uint32_t)(w >> 32), al) << 32);
                        if (lane < 3u) fw[b][k][lane] = lane == 0 ? low : lane == 1 ? high : low | high | own;
                    }
                }
            }
            lds_barrier();
            if (i >= rows) break;
        }
        return;
    }
    lds_barrier();  // the first steps are in
    uint32_t i0 = 0;
    for (; i0 < min(alone, rows); i0 += RA0_FETCH) {
        const uint32_t b = (i0 / RA0_FETCH) & 1u;
        uint32_t op = fop[b][0][col];
        unsigned long long W = fw[b][0][col];
        for (uint32_t k = 0; k < RA0_FETCH; k += 4) {
            ra_evict<NL>(d, f, ring, col, i0 + k);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                // the next step's op and lookups, read a step ahead
                const uint32_t kn = (k + q + 1u) % RA0_FETCH;
                const uint32_t opn = fop[b][kn][col];
                const unsigned long long Wn = fw[b][kn][col];
                ra_l0_step<ROWS, NL>(d, f, ring, hold, col, lane, j, i0 + k, i0 + k + q,
                                     lane < (uint32_t)NL ? op : 0u,
                                     RaLooks{lane < (uint32_t)NL ? W : 0ull, nullptr, nullptr, 0});
                op = opn; W = Wn;
            }
        }
        lds_barrier();  // the next steps are in
    }
    if (i0 >= rows) {
        if (lane < (uint32_t)NL) ra_flush<NL>(d, f, ring, col);
        return;
    }
    // One function left, the one of lane al: stepped as a one-group program's.  The
    // states of the others go to HBM, and those of its last words: the LDS ring
    // keeps these, the last of them go to the register ring.
    const uint32_t start = rdlane(f.start, al), size = rdlane(f.size, al);
    if (lane < (uint32_t)NL && (lane != al || size <= i0)) ra_flush<NL>(d, f, ring, col);
    if (size > i0)
        for (uint32_t p = (i0 > OP_ROWS ? i0 - OP_ROWS : 0u) + lane; p < i0; p += 64u)
            d.sym[start + p] = ring[(p & (OP_ROWS - 1u)) * NL + al];
    auto of = [&](uint64_t v, uint32_t l) { return (uint64_t)rdlane((uint32_t)v, l) | ((uint64_t)rdlane((uint32_t)(v >> 32), l) << 32); };
    Solo<RA0_FETCH, OP_ROWS, NL, true> g{d, start, lane, ring + al, 0u, hold[lane], 0u, of(f.life, al), of(f.own, al), of(f.mk, al), 0ull};
    for (uint32_t l = 0; l < pg.L; ++l) {
        const uint64_t o = l == al ? 0ull : of(f.own & ~f.mk, l);
        g.oth |= o;
        if ((o >> lane) & 1u) g.obase = rdlane(f.start, l);
    }
    {
        const uint32_t lo = i0 > 64u - RA0_FETCH ? i0 - (64u - RA0_FETCH) : 0u, w = lo + ((lane - lo) & 63u);
        if (w < i0) g.ringv = ring[(w & (OP_ROWS - 1u)) * NL + al];
    }
    wait_loads();  // (the others' states are written before a mark of one of them)
    const uint32_t first = i0;
    for (; i0 < rows; i0 += RA0_FETCH) {
        const uint32_t b = (i0 / RA0_FETCH) & 1u, kl = lane % RA0_FETCH;
        const uint32_t cur = fop[b][kl][al];
        const uint64_t lo = fw[b][kl][0], hi = fw[b][kl][1], W = fw[b][kl][2];
        if (i0 < size) {
            g.begin(i0, first);
            g.steps(i0, uniform(min(RA0_FETCH, size - i0)), cur, [&](uint32_t k) { return SoloLooks{of(W, k), of(lo, k), of(hi, k)}; });
            if (size - i0 <= RA0_FETCH) g.flush(g.kept_at(i0), size);  // the last block
        }
        if (rows > size && size / RA0_FETCH == i0 / RA0_FETCH) g.finish(of(W, size % RA0_FETCH));
        lds_barrier();
    }
}

// ============================================================ small programs
// Programs of at most 64 functions (at most 8 groups of 8) whose words fit
// the LDS budget are allocated by one wave: lane = function (its index in the
// program, so lanes 8g .. 8g+7 are group g), each lane keeping the states of
// its function's virtual registers in LDS, one byte per word (register |
// touched << 6 | swapped << 7), and its lifetime in registers.  A step is the
// reference's step (rv_generator_avx.cpp:1041-1418 at one thread) for every
// function of the program at once:
//   * a function's state reads see its own group's body's view: the only
//     effect of the lower groups' bodies in the same step is a mark on a
//     region-0 entry (only lane-0 functions write region 0, and every lookup
//     reads it), which an owner sees as a swapped operand (a flip) when it
//     reads that register.  Owners that read an entry they own are settled in
//     group order, each from the final lookups of the groups below it, so one
//     pass reaches the in-order result;
//   * a lookup of register r marks the virtual that region 0 held at r at the
//     start of the step.  The owner's commit resets the swapped flag of the
//     registers it names, so a mark stands if a higher group made it, or if
//     the owner does not name that register in this step;
//   * region 0 of the next step: each lane-0 function's rd write, then its rs1
//     and rs2 frees, groups in order (the last one wins).
// Several programs can share the wave (program k on lanes seg[k] .. seg[k] +
// nf - 1, seg[k] a multiple of 8).  Lanes exchange values with DPP inside a
// group's 8 lanes and with readlane across groups; region 0 of each program
// is an LDS table read by lane = register, double-buffered by step parity.
// (Programs naming registers outside their own function are reallocated by
// k_ra_serial, whatever this kernel makes of them.)
constexpr uint32_t SM_CHUNK = 32;        // steps per staged chunk of words
constexpr uint32_t SM_PROGS = 8;         // programs per wave at most
constexpr uint32_t SM_STATE_OFF = 40960; // LDS bytes before the register states
constexpr uint32_t SM_STATE_MAX = 40960;   // LDS bytes of register states per wave at most (80 KB of
                                           // LDS in all: two waves per compute unit)
constexpr uint32_t SM_STATE_SMALL = 40960;
constexpr uint32_t SM_MIN_FUNCS = 9;       // programs of one group keep k_ra_lane0_one

struct SmWave { uint32_t np, state_bytes, prog[SM_PROGS], seg[SM_PROGS]; };

DEV uint32_t sm_rl(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }
DEV uint64_t sm_rl64(uint64_t v, uint32_t l) { return (uint64_t)sm_rl((uint32_t)v, l) | ((uint64_t)sm_rl((uint32_t)(v >> 32), l) << 32); }

DEV uint64_t sm_look(const RaStep &r) {
    uint64_t m = 0;
    if (r.swd) m |= 1ull << r.rdr;
    if (r.sw1) m |= 1ull << r.r1r;
    if (r.sw2) m |= 1ull << r.r2r;
    return m;
}

__global__ __launch_bounds__(64) void k_ra_small(Dev d, const SmWave *waves) {
    extern __shared__ __align__(16) uint8_t sm_lds[];
    uint4 (*words)[64] = reinterpret_cast<uint4 (*)[64]>(sm_lds);                        // [SM_CHUNK][64]
    int32_t (*Sv)[SM_PROGS][64] = reinterpret_cast<int32_t (*)[SM_PROGS][64]>(sm_lds + 32768);  // [2]
    int8_t (*So)[SM_PROGS][64] = reinterpret_cast<int8_t (*)[SM_PROGS][64]>(sm_lds + 36864);    // [2]
    uint32_t *slot_base = reinterpret_cast<uint32_t *>(sm_lds + 37888);  // per group slot: lane-0 function's
    uint32_t *slot_start = slot_base + 8;                                // state base and first word
    uint32_t *slot_size = slot_base + 16;
    uint32_t *prog_slots = slot_base + 24;  // per program: first group slot | end slot << 8
    uint8_t *st = sm_lds + SM_STATE_OFF;
    __shared__ uint32_t fstart[64], fsize[64];
    const uint32_t lane = threadIdx.x;
    const SmWave wv = waves[blockIdx.x];
    // this lane's program, function and group slot
    uint32_t pk = 0;
    for (uint32_t k = 1; k < wv.np; ++k) if (wv.seg[k] <= lane) pk = k;
    const uint32_t prg = wv.prog[pk], seg = wv.seg[pk];
    const uint32_t fb = d.pf[prg], nf = d.pf[prg + 1] - fb;
    const uint32_t li = lane - seg;
    const bool has = li < nf;
    const uint32_t f = fb + li;
    const uint32_t start = has ? d.fstarts[f] : 0u;
    const uint32_t size = has ? d.fsizes[f] : 0u;
    const uint32_t slot = lane >> 3, k8 = lane & 7u;
    // state bytes: exclusive scan of the sizes rounded up to 4
    const uint32_t sz4 = (size + 3u) & ~3u;
    uint32_t incl = sz4;
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)incl, o, 64);
        if (lane >= o) incl += u;
    }
    const uint32_t base = incl - sz4;
    uint8_t *my = st + base;
    for (uint32_t x = 0; x < sz4; x += 4) *reinterpret_cast<uint32_t *>(my + x) = 0u;
    fstart[lane] = start; fsize[lane] = size;
    if (k8 == 0) { slot_base[slot] = base; slot_start[slot] = start; slot_size[slot] = size; }
    if (lane == seg) prog_slots[pk] = (seg >> 3) | (((seg + nf + 7u) >> 3) << 8);
    for (uint32_t p = 0; p < wv.np; ++p) { Sv[0][p][lane] = -1; So[0][p][lane] = -1; }
    const uint32_t np = wv.np;
    uint32_t wmax = size;
    for (int s = 32; s > 0; s >>= 1) { const uint32_t o = (uint32_t)__shfl_xor((int)wmax, s, 64); wmax = max(wmax, o); }
    uint64_t life = 0x1Full;
    uint64_t own = 0;  // lane-0 functions: the region-0 entries this group owns
    bool bad = false;  // a word names a register past the program's words: this lane stops (EF_OOB)
    __syncthreads();
    // state of virtual register v as read by this function: (register, swapped);
    // v is within the words (checked when its chunk was staged)
    auto rd_state = [&](uint32_t v, uint32_t &reg, bool &sw) {
        reg = 0; sw = false;
        if (!((int32_t)v > 63)) return;
        const uint32_t x = v - 64u - start;
        if (x < size) { const uint32_t b = my[x]; reg = b & 0x3Fu; sw = (b >> 7) != 0; }
        else { const uint32_t g = d.sym[v - 64u]; reg = g & 0xFFu; sw = (g >> 8) != 0; }
    };
    auto wr_state = [&](uint32_t v, uint32_t reg) {
        const uint32_t x = v - 64u - start;
        if (x < size) my[x] = (uint8_t)(reg | 0x40u);
        else d.sym[v - 64u] = (uint16_t)reg;
    };
    for (uint32_t i = 0; i < wmax; ++i) {
        if (i % SM_CHUNK == 0) {
            // thread t stages word i + t % 32 of functions t / 32, t / 32 + 2, ...
            const uint32_t kk = lane % SM_CHUNK, g0 = lane / SM_CHUNK;
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                uint4 tmp[16];
#pragma unroll
                for (uint32_t r = 0; r < 16; ++r) {
                    const uint32_t g = g0 + 2u * (16u * h + r);
                    tmp[r] = i + kk < fsize[g] ? d.w0_f4[fstart[g] + i + kk] : make_uint4(0, 0, 0, 0);
                }
#pragma unroll
                for (uint32_t r = 0; r < 16; ++r) words[kk][g0 + 2u * (16u * h + r)] = tmp[r];
            }
            __syncthreads();
            // this function's words of the chunk: registers past the words
            for (uint32_t k = 0; k < SM_CHUNK && i + k < size; ++k) {
                const uint4 wk = words[k][lane];
                if (((int32_t)wk.x > 63 && wk.x - 64u >= d.W0) || ((int32_t)wk.y > 63 && wk.y - 64u >= d.W0) ||
                    ((int32_t)wk.z > 63 && wk.z - 64u >= d.W0)) {
                    atomicOr(d.flags, EF_OOB);
                    bad = true;
                }
            }
        }
        const uint32_t c = i & 1u, nx = c ^ 1u;
        const bool act = (int32_t)i < (int32_t)size && !bad;
        const uint4 w = act ? words[i % SM_CHUNK][lane] : make_uint4(0, 0, 0, 0);
        uint32_t raw1, raw2;
        bool s1, s2;
        rd_state(w.y, raw1, s1);
        rd_state(w.z, raw2, s2);
        RaStep r = ra_eval_raw(w.w, w.x, w.y, w.z, raw1, raw2, s1, s2, life);
        uint64_t look = act ? sm_look(r) : 0ull;
        uint64_t gl = sm_or8_64(look);
        // owners reading an entry they own: settled in group order
        uint64_t or1 = 0, or2 = 0;
        if (k8 == 0 && act && own) {
            uint64_t m = own;
            while (m) {
                const uint32_t reg = (uint32_t)__builtin_ctzll(m);
                m &= m - 1;
                const int32_t v = Sv[c][pk][reg];
                if ((int32_t)w.y > 63 && v == (int32_t)w.y) or1 |= 1ull << reg;
                if ((int32_t)w.z > 63 && v == (int32_t)w.z) or2 |= 1ull << reg;
            }
        }
        uint64_t cand = __ballot(k8 == 0 && act && (or1 | or2) != 0);
        while (cand) {
            const uint32_t L0 = (uint32_t)__builtin_ctzll(cand);
            cand &= cand - 1;
            const uint32_t s = L0 >> 3, first = sm_rl(seg, L0) >> 3;
            uint64_t lower = 0;
            for (uint32_t t = first; t < s; ++t) lower |= sm_rl64(gl, 8u * t);
            const bool f1 = lane == L0 && (or1 & lower) != 0, f2 = lane == L0 && (or2 & lower) != 0;
            if (__ballot(f1 || f2)) {
                if (f1 || f2) { r = ra_eval_raw(w.w, w.x, w.y, w.z, raw1, raw2, s1 || f1, s2 || f2, life); look = sm_look(r); }
                gl = sm_or8_64(look);
            }
        }
        // commit: rd, then rs1, then rs2 (a later one wins); the lifetime
        if (act) {
            if ((int32_t)r.ord > 63) wr_state(r.ord, r.rdr);
            if ((int32_t)r.rs1 > 63) wr_state(r.rs1, r.r1r);
            if ((int32_t)r.rs2 > 63) wr_state(r.rs2, r.r2r);
            life = r.newlife;
        }
        // per program: marks on region 0's virtuals (entry `lane`), then region 0
        // of the next step.  Entry `lane` needs bit `lane` of the lookups of the
        // groups below its owner, of its owner's group and of the groups above it.
        for (uint32_t p = 0; p < np; ++p) {
            const uint32_t ps = prog_slots[p];
            const uint32_t s0 = ps & 0xFFu, s1e = ps >> 8;
            const int32_t v = Sv[c][p][lane];
            const int32_t o = So[c][p][lane];
            int32_t nv = v, no = o;
            bool lowb = false, ownb = false, highb = false, named = false;
            for (uint32_t t = s0; t < s1e; ++t) {
                const uint32_t L0 = 8u * t;
                const bool bt = ((sm_rl64(gl, L0) >> lane) & 1ull) != 0;
                lowb |= (int32_t)t < o && bt;
                highb |= (int32_t)t > o && bt;
                const bool at = sm_rl((uint32_t)act, L0) != 0;
                const uint32_t ot = sm_rl(w.x, L0), o1 = sm_rl(w.y, L0), o2 = sm_rl(w.z, L0);
                if ((int32_t)t == o) {
                    ownb = bt;
                    named = at && ((uint32_t)v == ot || (uint32_t)v == o1 || (uint32_t)v == o2);
                }
                // group t's lane-0 function acts on region 0: rd write, rs1 and rs2 frees
                if (at) {
                    const uint32_t rdt = sm_rl(r.rdr, L0), r1t = sm_rl(r.r1r, L0), r2t = sm_rl(r.r2r, L0);
                    if (ot && rdt == lane) { nv = (int32_t)ot; no = (int32_t)t; }
                    if (r1t != rdt && r1t == lane) { nv = -1; no = -1; }
                    if (r2t != rdt && r2t == lane) { nv = -1; no = -1; }
                }
            }
            if (o >= 0 && v >= 64 && (highb || (!named && (lowb || ownb)))) {
                const uint32_t x = (uint32_t)v - 64u - slot_start[o];
                if (x < slot_size[o]) st[slot_base[o] + x] |= 0x80u;
                else { atomicOr(d.flags, EF_XCONFLICT); d.cflag[waves[blockIdx.x].prog[p]] = 1; }
            }
            Sv[nx][p][lane] = nv;
            So[nx][p][lane] = (int8_t)no;
            for (uint32_t t = s0; t < s1e; ++t) {
                const uint64_t m = __ballot(no == (int32_t)t);
                if (lane == 8u * t) own = m;
            }
        }
    }
    __syncthreads();
    // final states to HBM (the bytes a function wrote or a mark set), the wave
    // storing each function's range with consecutive lanes
    for (uint32_t l = 0; l < 64; ++l) {
        const uint32_t bl = sm_rl(base, l), sl = sm_rl(start, l), zl = sm_rl(size, l);
        for (uint32_t x = lane; x < zl; x += 64u) {
            const uint32_t b = st[bl + x];
            if (b & 0xC0u) d.sym[sl + x] = (uint16_t)((b & 0x3Fu) | ((b >> 7) << 8));
        }
    }
}

// Lane-0 functions in step lockstep, one workgroup.  Region 0 of the
// reference's register_state holds the last lane-0 write per physical register;
// every lookup of any function at step i reads its step-start snapshot S and
// marks the virtual register found there as swapped.  A lookup by a lower group
// at step i is seen by the owner's operand read at step i; one by a higher group
// lands after the owner's own reset.  Intra-step effects between lane-0
// functions are settled by re-evaluation until stable (lower groups settle
// first, so this converges to the reference's in-order result).
constexpr int RA0_THREADS = 1024;

struct Ra0Rec { uint32_t ord, rs1, rs2; uint32_t regs; /* r1r | r2r<<8 | rdr<<16 */ };

DEV void ra0_flips(const int32_t *So, const uint32_t *fbits, uint32_t j, bool &f1, bool &f2) {
    f1 = false; f2 = false;
#pragma unroll 8
    for (int r = 0; r < 64; ++r)
        if (So[r] == (int32_t)j) { f1 |= (fbits[r] & 1u) != 0; f2 |= (fbits[r] & 2u) != 0; }
}

DEV RaStep ra0_eval(const Dev &d, uint32_t off, uint64_t life, bool f1, bool f2) {
    const uint32_t rs1 = d.w0_f4[off].y, rs2 = d.w0_f4[off].z;
    bool s1 = ((int32_t)rs1 > 63 && rs1 - 64u < d.W0 && sym_swapped(d, rs1 - 64u)) || f1;
    bool s2 = ((int32_t)rs2 > 63 && rs2 - 64u < d.W0 && sym_swapped(d, rs2 - 64u)) || f2;
    return ra_eval(d, off, life, s1, s2);
}


__global__ __launch_bounds__(RA0_THREADS) void k_ra_lane0_generic(Dev d, const Ra0Prog *progs, const uint32_t *gmin_all,
                                                         const uint32_t *gmax_all, uint64_t *life0, Ra0Rec *rec) {
    __shared__ int32_t Rv[64], Ro[64], Sv[64], So[64];
    __shared__ uint32_t Lmin[64], Lmax[64], fbits[64], wkey[64];
    __shared__ int changed;
    const uint32_t tid = threadIdx.x;
    const Ra0Prog pg = progs[blockIdx.x];
    const uint32_t L = pg.L, maxsize = pg.rows, fbase = pg.fbase;
    const uint32_t *gmin = gmin_all + pg.gbase, *gmax = gmax_all + pg.gbase;
    life0 += pg.poff; rec += pg.poff;
    if (tid < 64) { Rv[tid] = -1; Ro[tid] = -1; }
    for (uint32_t j = tid; j < L; j += RA0_THREADS) life0[j] = 0x1Full;
    __syncthreads();
    for (uint32_t i = 0; i < maxsize; ++i) {
        if (tid < 64) { Sv[tid] = Rv[tid]; So[tid] = Ro[tid]; fbits[tid] = 0; wkey[tid] = 0; }
        __syncthreads();
        for (uint32_t round = 0;; ++round) {
            if (tid < 64) { Lmin[tid] = gmin[(uint64_t)i * 64u + tid]; Lmax[tid] = gmax[(uint64_t)i * 64u + tid]; }
            if (tid == 0) changed = 0;
            __syncthreads();
            for (uint32_t j = tid; j < L; j += RA0_THREADS) {
                const uint32_t f = fbase + 8u * j;
                if (!((int32_t)i < (int32_t)d.fsizes[f])) continue;
                bool f1, f2;
                ra0_flips(So, fbits, j, f1, f2);
                RaStep r = ra0_eval(d, d.fstarts[f] + i, life0[j], f1, f2);
                if (r.swd) { atomicMin(&Lmin[r.rdr], j); atomicMax(&Lmax[r.rdr], j + 1u); }
                if (r.sw1) { atomicMin(&Lmin[r.r1r], j); atomicMax(&Lmax[r.r1r], j + 1u); }
                if (r.sw2) { atomicMin(&Lmin[r.r2r], j); atomicMax(&Lmax[r.r2r], j + 1u); }
            }
            __syncthreads();
            if (tid < 64) {
                uint32_t nb = 0;
                if (Sv[tid] >= 64 && So[tid] >= 0) {
                    const uint32_t o = (uint32_t)So[tid];
                    const uint32_t f = fbase + 8u * o;
                    if ((int32_t)i < (int32_t)d.fsizes[f] && Lmin[tid] < o) {
                        const uint32_t off = d.fstarts[f] + i;
                        if (d.w0_f4[off].y == (uint32_t)Sv[tid]) nb |= 1u;
                        if (d.w0_f4[off].z == (uint32_t)Sv[tid]) nb |= 2u;
                    }
                }
                if (nb != fbits[tid]) changed = 1;
                Lmin[tid] = nb;  // staged; fbits is updated after the barrier
            }
            __syncthreads();
            int again = changed;
            if (again && round > L + 1) { again = 0; if (tid == 0) atomicOr(d.flags, EF_OOB); }
            if (tid < 64 && again) fbits[tid] = Lmin[tid];
            __syncthreads();
            if (!again) break;
        }
        // commit: lifetime, records, region-0 write keys (group order: last writer wins)
        for (uint32_t j = tid; j < L; j += RA0_THREADS) {
            const uint32_t f = fbase + 8u * j;
            if (!((int32_t)i < (int32_t)d.fsizes[f])) continue;
            bool f1, f2;
            ra0_flips(So, fbits, j, f1, f2);
            RaStep r = ra0_eval(d, d.fstarts[f] + i, life0[j], f1, f2);
            life0[j] = r.newlife;
            rec[j] = Ra0Rec{r.ord, r.rs1, r.rs2, r.r1r | (r.r2r << 8) | (r.rdr << 16)};
            if (r.ord) atomicMax(&wkey[r.rdr], ((j + 1u) << 2) | 1u);
            if (r.r1r != r.rdr) atomicMax(&wkey[r.r1r], ((j + 1u) << 2) | 2u);
            if (r.r2r != r.rdr) atomicMax(&wkey[r.r2r], ((j + 1u) << 2) | 3u);
        }
        __syncthreads();
        for (uint32_t j = tid; j < L; j += RA0_THREADS) {
            const uint32_t f = fbase + 8u * j;
            if (!((int32_t)i < (int32_t)d.fsizes[f])) continue;
            const Ra0Rec q = rec[j];
            RaStep r;
            r.ord = q.ord; r.rs1 = q.rs1; r.rs2 = q.rs2;
            r.r1r = q.regs & 0xFFu; r.r2r = (q.regs >> 8) & 0xFFu; r.rdr = (q.regs >> 16) & 0xFFu;
            if (r.ord && wkey[r.rdr] == (((j + 1u) << 2) | 1u)) { Rv[r.rdr] = (int32_t)r.ord; Ro[r.rdr] = (int32_t)j; }
            if (r.r1r != r.rdr && wkey[r.r1r] == (((j + 1u) << 2) | 2u)) { Rv[r.r1r] = -1; Ro[r.r1r] = -1; }
            if (r.r2r != r.rdr && wkey[r.r2r] == (((j + 1u) << 2) | 3u)) { Rv[r.r2r] = -1; Ro[r.r2r] = -1; }
            ra_commit_syms(d, r);
        }
        __syncthreads();
        // marks on the snapshot's virtual registers
        if (tid < 64 && Sv[tid] >= 64 && Lmax[tid] != 0) {
            const uint32_t v = (uint32_t)Sv[tid];
            bool mark = true;
            if (So[tid] >= 0) {
                const uint32_t o = (uint32_t)So[tid];
                const uint32_t f = fbase + 8u * o;
                if ((int32_t)i < (int32_t)d.fsizes[f]) {
                    const Ra0Rec q = rec[o];
                    bool reset = (q.ord == v) || (q.rs1 == v) || (q.rs2 == v);
                    if (reset) mark = Lmax[tid] > o + 1u;
                }
            }
            if (mark) {
                if (v - 64u < d.W0) sym_mark(d, v - 64u);
                else atomicOr(d.flags, EF_OOB);
            }
        }
        __syncthreads();
    }
}


// Register-resident lockstep: each thread owns PER lane-0 functions (slots
// t = tid + q*blockDim; slot t runs group perm[t], the groups ordered by
// function size, largest first, so that the functions still running at a step
// fill the first waves and finished waves skip each phase) and keeps their
// state in registers: the fields of step i+1 and the packed operand state of
// step i.  The fields of step i sit in LDS (cur_*), where the snapshot checks
// read them too.  A function's virtual registers are read and written only by
// its own thread (marks by other groups reach the owner through LDS), so the
// barriers of a step order LDS alone.  Each step ends with the loads for the
// next: the operands' symbol states (waited for), the walk's row two steps
// ahead (by the loading waves) and the fields two steps ahead (waited for a
// step later).  Per-step LDS tables are double-buffered by step parity so that
// no barrier is needed between the end of a step and the start of the next.
//
// Snapshot owners: only a group owning an entry of the region-0 snapshot (a
// virtual register it wrote there) can see a swap made earlier in the same
// step, so only owners take part in the in-order settle; every other group's
// step result is final after its first evaluation.  Each function keeps the
// set of snapshot registers it may own (`own`, a superset refreshed against
// the snapshot every step), so owners find their flips and marks by register
// without any table.
//
// Of an instruction word, register allocation looks only at whether its major
// opcode is OP-FP (0x53): the other word tests of ra_eval_raw (0xC0007053,
// 0xD0007053) are OP-FP words themselves, so the lockstep keeps that bit alone.
struct Ra0Fn {
    uint32_t j, start, size;              // group, first word, word count
    uint64_t life;
    uint64_t own;                         // snapshot registers this function may own
    uint32_t ord, rs1, rs2;               // step i (reloaded from LDS in every phase)
    uint4 nw;                             // step i+1: rd, rs1, rs2, instruction (zeros past the end)
    uint32_t rr;                          // step i's result: r1r | r2r << 8 | rdr << 16
    uint32_t pk;                          // step i: raw1 | raw2 << 8 | s1 << 16 | s2 << 17 | flips << 18 |
                                          // won << 20 | OP-FP << 31 (won: 0x40 | the snapshot entry its
                                          // step i-1 commit won, 0 for none)
};

DEV RaStep ra0_step(const Ra0Fn &f) {
    const uint32_t fl = (f.pk >> 18) & 3u;
    return ra_eval_raw((f.pk >> 31) ? 0x53u : 0u, f.ord, f.rs1, f.rs2, f.pk & 0xFFu, (f.pk >> 8) & 0xFFu,
                       ((f.pk >> 16) & 1u) || (fl & 1u), ((f.pk >> 17) & 1u) || (fl & 2u), f.life);
}

// Word `step` of the function (zeros past its end).
DEV uint4 ra0_word(const Dev &d, const Ra0Fn &f, uint32_t step) {
    return (int32_t)step < (int32_t)f.size ? d.w0_f4[f.start + step] : make_uint4(0, 0, 0, 0);
}

DEV uint32_t ra0_fpbit(uint32_t ins) { return (ins & 0x7Fu) == 0x53u ? 1u : 0u; }

// sym entries of a word's operands (0 for physical operands).
DEV void ra0_gather(const Dev &d, uint32_t rs1, uint32_t rs2, uint32_t &g1, uint32_t &g2) {
    g1 = virt_ok(d, rs1) ? d.sym[rs1 - 64u] : 0u;
    g2 = virt_ok(d, rs2) ? d.sym[rs2 - 64u] : 0u;
}

// (bit 31 of g1, the OP-FP bit where the caller sets it, is kept)
DEV uint32_t ra0_pack(uint32_t g1, uint32_t g2) {
    return (g1 & 0x800000FFu) | ((g2 & 0xFFu) << 8) | (((g1 >> 8) & 1u) << 16) | (((g2 >> 8) & 1u) << 17);
}

// The commit of ra_commit_syms, storing only entries whose value changes:
// old1/old2 are the operands' entries before the commit; a destination entry is
// always stored unless an operand names the same entry (the later store wins).
DEV void ra0_commit(const Dev &d, const RaStep &r, uint32_t old1, uint32_t old2) {
    const bool vo = (int32_t)r.ord > 63, v1 = (int32_t)r.rs1 > 63, v2 = (int32_t)r.rs2 > 63;
    if ((vo && r.ord - 64u >= d.W0) || (v1 && r.rs1 - 64u >= d.W0) || (v2 && r.rs2 - 64u >= d.W0)) {
        atomicOr(d.flags, EF_OOB);
        return;
    }
    if (vo && !(v1 && r.rs1 == r.ord) && !(v2 && r.rs2 == r.ord)) d.sym[r.ord - 64u] = (uint16_t)r.rdr;
    if (v1 && !(v2 && r.rs2 == r.rs1) && r.r1r != old1) d.sym[r.rs1 - 64u] = (uint16_t)r.r1r;
    if (v2 && r.r2r != old2) d.sym[r.rs2 - 64u] = (uint16_t)r.r2r;
}

// The flip bits of the snapshot entries of `own` that group j owns, each
// entry's owner, register and flip bits read together.
DEV uint32_t ra0_owned_flips(uint64_t own, const int32_t *Sv, const int32_t *So, const uint32_t *flip, uint32_t j) {
    uint32_t f = 0;
    while (own) {
        const uint32_t r = (uint32_t)__builtin_ctzll(own);
        own &= own - 1;
        const int32_t so = So[r], sv = Sv[r];
        const uint32_t fl = flip[r];
        f |= fl & (0u - (uint32_t)((so == (int32_t)j) & (sv >= 64)));
    }
    return f;
}

constexpr uint32_t RA0_LDS_FNS = 8192;  // lane-0 functions whose current fields fit in LDS

// A function's fields of step i, from LDS.
DEV void ra0_cur(Ra0Fn &f, const uint32_t *crd, const uint32_t *crs1, const uint32_t *crs2, uint32_t j) {
    f.ord = crd[j]; f.rs1 = crs1[j]; f.rs2 = crs2[j];
}

DEV void ra0_lookups(uint32_t *mn, uint32_t *mx, const RaStep &r, uint32_t j) {
    if (r.swd) { atomicMin(&mn[r.rdr], j); atomicMax(&mx[r.rdr], j + 1u); }
    if (r.sw1) { atomicMin(&mn[r.r1r], j); atomicMax(&mx[r.r1r], j + 1u); }
    if (r.sw2) { atomicMin(&mn[r.r2r], j); atomicMax(&mx[r.r2r], j + 1u); }
}

DEV void ra0_keys(uint32_t *wkey, const RaStep &r, uint32_t j) {
    if (r.ord) atomicMax(&wkey[r.rdr], ((j + 1u) << 2) | 1u);
    if (r.r1r != r.rdr) atomicMax(&wkey[r.r1r], ((j + 1u) << 2) | 2u);
    if (r.r2r != r.rdr) atomicMax(&wkey[r.r2r], ((j + 1u) << 2) | 3u);
}

// Lookups of table row r by the walked functions (entry `tid`): min and max
// over the table's `copies` copies, `stride` apart.  Every load is issued
// before the first is used.
DEV void ra0_row(const uint32_t *gmin, const uint32_t *gmax, uint64_t stride, uint32_t copies, uint32_t r,
                 uint32_t tid, uint32_t &mn, uint32_t &mx) {
    const uint64_t e = (uint64_t)r * 64u + tid;
    uint32_t a[RA0_MAXCOPIES], b[RA0_MAXCOPIES];
#pragma unroll
    for (uint32_t c = 0; c < RA0_MAXCOPIES; ++c) {
        const uint64_t o = (c < copies ? c : 0u) * stride + e;
        a[c] = gmin[o]; b[c] = gmax[o];
    }
    mn = a[0]; mx = b[0];
#pragma unroll
    for (uint32_t c = 1; c < RA0_MAXCOPIES; ++c) { mn = min(mn, a[c]); mx = max(mx, b[c]); }
}

// Folds row r of the walk's tables into the lockstep's lookup row of its step
// (mn / mx, cleared beforehand; min / max over the copies by LDS atomics):
// copy k is loaded by wave nwv-1-(k mod nwv), the last waves holding the
// shortest functions (idle through most steps), so that no wave with work
// waits for rows coming from HBM.  A loading wave waits for the row's chunk to
// be published (`first`: for the chunk of a first row).
DEV void ra0_stage(const Dev &d, const uint32_t *gmin, const uint32_t *gmax, uint64_t stride, uint32_t copies,
                   uint32_t r, const uint32_t *pdone, const uint32_t *pneed, bool first, bool &ok,
                   uint32_t *mn, uint32_t *mx, uint32_t wid, uint32_t nwv, uint32_t lane) {
    const uint32_t k0 = nwv - 1u - wid;
    if (k0 >= copies) return;
    if (pdone && (first || r % WALK_PUB == 0)) ra0_wait(d, pdone, pneed, r / WALK_PUB, ok);
    for (uint32_t k = k0; k < copies; k += nwv) {
        const uint64_t o = (uint64_t)k * stride + (uint64_t)r * 64u + lane;
        atomicMin(&mn[lane], gmin[o]);
        atomicMax(&mx[lane], gmax[o]);
    }
}

template <int PER, uint32_t NL>
__global__ __launch_bounds__(1024) void k_ra_lane0(Dev d, const Ra0Prog *progs, const uint32_t *gmin_all,
                                                   const uint32_t *gmax_all, const uint32_t *perm_all,
                                                   const uint32_t *done, const uint32_t *need, uint32_t copies,
                                                   uint64_t stride) {
    __shared__ uint32_t cur_rd[NL], cur_rs1[NL], cur_rs2[NL];
    __shared__ int32_t Sv[2][64], So[2][64];                  // region-0 snapshot of step i / i+1
    // lookups by all groups but the owners, and by the walk: the walk's row of
    // a step is folded in two steps ahead, into the table cleared after its last
    // read
    __shared__ uint32_t Lmin[2][64], Lmax[2][64];
    __shared__ uint32_t Omin[2][64], Omax[2][64];             // lookups by the (possible) owners
    __shared__ uint32_t wkey[2][64];
    __shared__ uint32_t flip[64];                             // flip bits per snapshot entry
    __shared__ uint32_t fmk[2];                               // snapshot entries with flip bits
    __shared__ uint32_t mk[2][2];                             // snapshot entries marked at step i
    __shared__ uint32_t keyed[2][2];                          // snapshot entries rewritten in the commit of step i
    __shared__ int changed;
    const uint32_t tid = threadIdx.x, nth = blockDim.x;
    const uint32_t wid = tid >> 6, nwv = nth >> 6, lane = tid & 63u;
    // with one table copy per loading wave, a loading wave holds its copy's
    // row of step i+2 in registers, loaded a step before it is staged
    const uint32_t k0 = nwv - 1u - wid;
    const bool reg_rows = nwv >= copies;
    uint32_t rmn = 0xFFFFFFFFu, rmx = 0;
    // this workgroup's program: groups of 8 functions from fbase, L of them
    const Ra0Prog pg = progs[blockIdx.x];
    if (d.cflag[pg.prg]) return;  // k_ra_serial's
    const uint32_t L = pg.L, maxsize = pg.rows, fbase = pg.fbase;  // steps: the table's rows
    const uint32_t *perm = perm_all + pg.poff;
    const uint32_t *gmin = gmin_all + pg.gbase, *gmax = gmax_all + pg.gbase;
    const uint32_t cb = nth > 64 ? 64u : 0u;  // first thread of the table-clearing threads
    // this program's publish counters (none: the walk has finished)
    const uint32_t *pdone = done && pg.cbase != RA0_NOPUB ? done + pg.cbase : nullptr;
    const uint32_t *pneed = pdone ? need + pg.cbase : nullptr;
    Ra0Fn fn[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const uint32_t t = tid + q * nth;
        Ra0Fn &f = fn[q];
        f.j = 0; f.start = 0; f.size = 0; f.life = 0x1Full; f.own = 0; f.rr = 0;
        if (t < L) {
            f.j = perm[t];
            if (f.j < L) { f.start = d.fstarts[fbase + 8u * f.j]; f.size = d.fsizes[fbase + 8u * f.j]; }
            else { atomicOr(d.flags, EF_OOB); f.j = 0; }
        }
        const uint4 w0 = ra0_word(d, f, 0);
        f.ord = w0.x; f.rs1 = w0.y; f.rs2 = w0.z;
        f.nw = ra0_word(d, f, 1);
        uint32_t g1 = 0, g2 = 0;
        if ((int32_t)f.size > 0) ra0_gather(d, f.rs1, f.rs2, g1, g2);
        f.pk = ra0_pack(g1, g2) | (ra0_fpbit(w0.w) << 31);
        if (t < L) {
            const bool act = (int32_t)f.size > 0;
            cur_rd[f.j] = act ? f.ord : 0u; cur_rs1[f.j] = act ? f.rs1 : 0u; cur_rs2[f.j] = act ? f.rs2 : 0u;
        }
    }
    bool wok = true;  // the walk's rows still arrive (waves that wait for them)
    if (tid < 64) {
        Sv[0][tid] = -1; So[0][tid] = -1; wkey[0][tid] = 0;
        if (tid < 2) keyed[1][tid] = 0;
        uint32_t m0 = 0xFFFFFFFFu, x0 = 0u;
        if (maxsize) {
            if (pdone) ra0_wait(d, pdone, pneed, 0, wok);
            ra0_row(gmin, gmax, stride, copies, 0, tid, m0, x0);
        }
        Lmin[0][tid] = m0; Lmax[0][tid] = x0;
        Lmin[1][tid] = 0xFFFFFFFFu; Lmax[1][tid] = 0u;
        Omin[0][tid] = Omin[1][tid] = 0xFFFFFFFFu; Omax[0][tid] = Omax[1][tid] = 0;
    }
    __syncthreads();
    if (maxsize > 1) ra0_stage(d, gmin, gmax, stride, copies, 1, pdone, pneed, true, wok, Lmin[1], Lmax[1], wid, nwv, lane);
    if (reg_rows && k0 < copies && maxsize > 2) {
        if (pdone && 2u % WALK_PUB == 0) ra0_wait(d, pdone, pneed, 2u / WALK_PUB, wok);
        const uint64_t o = (uint64_t)k0 * stride + 2u * 64u + lane;
        rmn = gmin[o]; rmx = gmax[o];
    }
    __syncthreads();
    uint32_t fb = 0;   // wave 0: flip bits of snapshot register tid
    uint32_t om = 0xFFFFFFFFu, ox = 0;  // wave 0: owners' lookups of register tid at step i
    for (uint32_t i = 0; i < maxsize; ++i) {
        const uint32_t c = i & 1u, n = c ^ 1u;
        // P1: every group evaluates with no flips; a group that cannot own a
        // snapshot entry finalizes its step, a possible owner keeps its
        // lookups apart
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            Ra0Fn &f = fn[q];
            const uint32_t j = f.j;
            if ((int32_t)i < (int32_t)f.size) {
                ra0_cur(f, cur_rd, cur_rs1, cur_rs2, j);
                const RaStep r = ra0_step(f);
                if (f.own) {
                    ra0_lookups(Omin[c], Omax[c], r, j);
                    f.rr = r.r1r | (r.r2r << 8) | (r.rdr << 16);  // final unless a settle round re-evaluates
                } else {
                    ra0_lookups(Lmin[c], Lmax[c], r, j);
                    f.rr = r.r1r | (r.r2r << 8) | (r.rdr << 16);
                    f.life = r.newlife;
                    ra0_keys(wkey[c], r, j);
                }
            }
        }
        lds_barrier();
        // P2: an owner of a snapshot entry reading it as an operand sees the
        // swap when a lower group looked the register up in this step
        if (tid < 64) {
            om = Omin[c][tid]; ox = Omax[c][tid];
            Omin[c][tid] = 0xFFFFFFFFu; Omax[c][tid] = 0;  // cleared for the settle rounds and step i+2
            uint32_t nb = 0;
            const int32_t o = So[c][tid], v = Sv[c][tid];
            const uint32_t lm = Lmin[c][tid];  // read with the entry, not behind its test
            if ((v >= 64) & (o >= 0) & (min(lm, om) < (uint32_t)o)) {
                if (cur_rs1[o] == (uint32_t)v) nb |= 1u;
                if (cur_rs2[o] == (uint32_t)v) nb |= 2u;
            }
            flip[tid] = nb;
            fb = nb;
            const uint64_t any = __ballot(nb != 0);
            if (tid == 0) { changed = any != 0; fmk[0] = (uint32_t)any; fmk[1] = (uint32_t)(any >> 32); }
        }
        if (tid >= cb)
            for (uint32_t k = tid - cb; k < 64; k += nth - cb) wkey[n][k] = 0;
        lds_barrier();
        // (the flipped entries read with the flag, for the first round)
        const uint64_t fm0 = ((uint64_t)fmk[1] << 32) | fmk[0];
        if (changed) {
            // settle intra-step flips among the owners: re-evaluate until the
            // flip bits are stable (lower groups settle first, so this reaches
            // the in-order result); O[c] was cleared when wave 0 last read it
            for (uint32_t round = 0;; ++round) {
                // only entries with flip bits can give an owner flips
                const uint64_t fm = round == 0 ? fm0 : ((uint64_t)fmk[1] << 32) | fmk[0];
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    const uint32_t j = fn[q].j;
                    if (fn[q].own && (int32_t)i < (int32_t)fn[q].size) {
                        fn[q].pk = (fn[q].pk & ~(3u << 18)) |
                                   (ra0_owned_flips(fn[q].own & fm, Sv[c], So[c], flip, j) << 18);
                        ra0_cur(fn[q], cur_rd, cur_rs1, cur_rs2, j);
                        const RaStep r = ra0_step(fn[q]);
                        ra0_lookups(Omin[c], Omax[c], r, j);
                        fn[q].rr = r.r1r | (r.r2r << 8) | (r.rdr << 16);
                    }
                }
                lds_barrier();
                if (tid < 64) {
                    om = Omin[c][tid]; ox = Omax[c][tid];
                    Omin[c][tid] = 0xFFFFFFFFu; Omax[c][tid] = 0;
                    uint32_t nb = 0;
                    const int32_t o = So[c][tid], v = Sv[c][tid];
                    const uint32_t lm = Lmin[c][tid];
                    if ((v >= 64) & (o >= 0) & (min(lm, om) < (uint32_t)o)) {
                        if (cur_rs1[o] == (uint32_t)v) nb |= 1u;
                        if (cur_rs2[o] == (uint32_t)v) nb |= 2u;
                    }
                    flip[tid] = nb;
                    const uint64_t diff = __ballot(nb != fb), any = __ballot(nb != 0);
                    fb = nb;
                    if (tid == 0) { changed = diff != 0; fmk[0] = (uint32_t)any; fmk[1] = (uint32_t)(any >> 32); }
                }
                lds_barrier();
                if (!changed) break;
                if (round > L + 1) { if (tid == 0) atomicOr(d.flags, EF_OOB); break; }
            }
        }
        // P3: possible owners finalize, from the registers of their last
        // evaluation (P1's, or the last settle round's: the same inputs, so the
        // same result) and the lifetime update of ra_eval_raw; marks on the
        // snapshot's virtual registers; the snapshot of step i+1 starts as a copy
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const uint32_t j = fn[q].j;
            if (fn[q].own && (int32_t)i < (int32_t)fn[q].size) {
                const uint32_t rr = fn[q].rr;
                RaStep r;
                r.ord = cur_rd[j];
                r.r1r = rr & 0xFFu; r.r2r = (rr >> 8) & 0xFFu; r.rdr = (rr >> 16) & 0xFFu;
                const uint64_t clr = ((1ull << r.r1r) | (1ull << r.r2r)) & ~1ull;
                fn[q].life = (fn[q].life & ~clr) | (1ull << r.rdr);
                ra0_keys(wkey[c], r, j);
            }
        }
        if (tid < 64) {
            const int32_t v = Sv[c][tid], o = So[c][tid];
            Sv[n][tid] = v; So[n][tid] = o;
            const uint32_t mx = max(Lmax[c][tid], ox);
            Lmin[c][tid] = 0xFFFFFFFFu; Lmax[c][tid] = 0u;  // last read: cleared for the walk's row of step i+2
            bool mark = false;
            if (v >= 64 && o >= 0 && mx != 0) {
                mark = true;
                const uint32_t uv = (uint32_t)v;
                const uint32_t a = cur_rd[o], b = cur_rs1[o], e = cur_rs2[o];  // read together
                if ((a == uv) | (b == uv) | (e == uv)) mark = mx > (uint32_t)o + 1u;
            }
            const uint64_t m = __ballot(mark);
            if (tid == 0) { mk[c][0] = (uint32_t)m; mk[c][1] = (uint32_t)(m >> 32); }
        }
        lds_barrier();
        // P4: snapshot of step i+1, commit of the symbol state, marks; then the
        // fields of step i+1 into LDS and one batch of loads for the next step.
        // The fields of step i+1, loaded a step ago, are in: one wait for every
        // vector load (vmcnt 0) here leaves none outstanding across the
        // branches below, so the gathers issue back to back.
        __builtin_amdgcn_s_waitcnt(0x0F70);
        const uint64_t marked = ((uint64_t)mk[c][1] << 32) | mk[c][0];
        // entries whose region-0 state the commit of step i-1 rewrote; every
        // other entry a group owned at the start of step i-1 it still owns
        const uint64_t kprev = ((uint64_t)keyed[n][1] << 32) | keyed[n][0];
        if (tid < 64) {
            const uint64_t kb = __ballot(wkey[c][tid] != 0);
            if (tid == 0) { keyed[c][0] = (uint32_t)kb; keyed[c][1] = (uint32_t)(kb >> 32); }
        }
        uint32_t wb[PER];  // the entry each function's commit wins: 0x40 | register, 0 for none
        // the operand states of step i+1 (sym entries), loaded right after each
        // function's commit (the commit's stores come first in program order);
        // a mark of one of them that follows, and the OP-FP bit, are added at
        // packing (pm: bit 0 / 1 operand marked, bit 2 OP-FP)
        uint32_t g1[PER], g2[PER], pm[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const uint32_t t = tid + q * nth;
            Ra0Fn &f = fn[q];
            const uint32_t j = f.j;
            wb[q] = 0; g1[q] = 0; g2[q] = 0; pm[q] = 0;
            if (t >= L) continue;
            uint64_t won = 0;
            if ((int32_t)i < (int32_t)f.size) {
                ra0_cur(f, cur_rd, cur_rs1, cur_rs2, j);
                const uint32_t rr = f.rr;
                RaStep r;
                r.ord = f.ord; r.rs1 = f.rs1; r.rs2 = f.rs2;
                r.r1r = rr & 0xFFu; r.r2r = (rr >> 8) & 0xFFu; r.rdr = (rr >> 16) & 0xFFu;
                // the three keys read together (registers are below 64), then compared
                const uint32_t kd = wkey[c][r.rdr & 63u], k1 = wkey[c][r.r1r & 63u], k2 = wkey[c][r.r2r & 63u];
                const bool wd = (r.ord != 0u) & (kd == (((j + 1u) << 2) | 1u));
                const bool w1 = (r.r1r != r.rdr) & (k1 == (((j + 1u) << 2) | 2u));
                const bool w2 = (r.r2r != r.rdr) & (k2 == (((j + 1u) << 2) | 3u));
                if (wd) {
                    Sv[n][r.rdr] = (int32_t)r.ord; So[n][r.rdr] = (int32_t)j;
                    if ((int32_t)r.ord >= 64) { won = 1ull << r.rdr; wb[q] = 0x40u | r.rdr; }
                }
                if (w1) { Sv[n][r.r1r] = -1; So[n][r.r1r] = -1; }
                if (w2) { Sv[n][r.r2r] = -1; So[n][r.r2r] = -1; }
                ra0_commit(d, r, (f.pk & 0xFFu) | (((f.pk >> 16) & 1u) << 8), ((f.pk >> 8) & 0xFFu) | (((f.pk >> 17) & 1u) << 8));
                const bool nx = (int32_t)(i + 1) < (int32_t)f.size;
                cur_rd[j] = nx ? f.nw.x : 0u; cur_rs1[j] = nx ? f.nw.y : 0u; cur_rs2[j] = nx ? f.nw.z : 0u;
            }
            if ((int32_t)(i + 1) < (int32_t)f.size) {
                ra0_gather(d, f.nw.y, f.nw.z, g1[q], g2[q]);
                pm[q] = ra0_fpbit(f.nw.w) << 2;  // (not ORed into g1 here: that would wait for the load)
            }
            if (f.own) {
                // the entries it owns now: those it owned that the commit of step
                // i-1 left alone, and the one it won in that commit (a won entry
                // is keyed, and a keyed entry is won by one group alone)
                const uint32_t pw = (f.pk >> 20) & 0x7Fu;
                const uint64_t wprev = (pw & 0x40u) ? 1ull << (pw & 63u) : 0ull;
                const uint64_t o = (f.own & ~kprev) | (f.own & kprev & wprev);
                uint64_t m = o & marked;
                while (m) {
                    const uint32_t reg = (uint32_t)__builtin_ctzll(m);
                    m &= m - 1;
                    const uint32_t v = (uint32_t)Sv[c][reg];
                    if (v - 64u < d.W0) sym_mark(d, v - 64u);
                    else atomicOr(d.flags, EF_OOB);
                    pm[q] |= (v == f.nw.y ? 1u : 0u) | (v == f.nw.z ? 2u : 0u);
                }
                f.own = o;
            }
            f.own |= won;
        }
        if (reg_rows) {
            if (k0 < copies && i + 2 < maxsize) { atomicMin(&Lmin[c][lane], rmn); atomicMax(&Lmax[c][lane], rmx); }
        } else if (i + 2 < maxsize) {
            ra0_stage(d, gmin, gmax, stride, copies, i + 2, pdone, pneed, false, wok, Lmin[c], Lmax[c], wid, nwv, lane);
        }
        // (packed for every slot, finished ones too: no gather stays pending
        // on any path into the next step)
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            fn[q].pk = ra0_pack(g1[q] | ((pm[q] & 1u) << 8) | ((pm[q] >> 2) << 31), g2[q] | ((pm[q] & 2u) << 7)) |
                       (wb[q] << 20);
            asm volatile("" : "+v"(fn[q].pk) : : "memory");  // packed here, before the loads below
        }
        // the walk's row of step i+3, staged at the end of step i+1, and the
        // fields of step i+2, first read at the end of step i+1: issued after
        // every load this step waits for (loads complete in order), so that
        // their latency overlaps step i+1
        if (reg_rows && k0 < copies && i + 3 < maxsize) {
            if (pdone && (i + 3) % WALK_PUB == 0) ra0_wait(d, pdone, pneed, (i + 3) / WALK_PUB, wok);
            const uint64_t o = (uint64_t)k0 * stride + (uint64_t)(i + 3) * 64u + lane;
            rmn = gmin[o]; rmx = gmax[o];
        }
#pragma unroll
        for (int q = 0; q < PER; ++q)
            if ((int32_t)(i + 1) < (int32_t)fn[q].size) fn[q].nw = ra0_word(d, fn[q], i + 2);
    }
}

// The lane-0 functions of a program of more than RA0_WAVE_GROUPS groups, in step
// lockstep on one workgroup.  Lanes hold functions in group order, the highest
// first, 64 to a wave slot (slot k on wave k mod the computing waves, PER slots
// a wave at most), so what a step exchanges between groups is an OR over the
// lanes below or above within a slot (DPP) and one pair of 64-bit masks per slot
// through LDS: the registers looked up and the ones written or freed.
//
// A step takes one barrier.  Flips (ra_l0_step) are settled within the slot
// before it, against the walk's lookups and the slot's own; a lane whose operand
// none of them looks up says so (chk), and only where a lower slot turns out to
// look it up do the slots settle together, at a barrier a round: the walk has
// seven functions to each of these, so mostly it has looked the register up.
//
// Every RA0_PACK steps the functions still running (or still holding a snapshot
// entry) are packed into as few slots as they fit, through memory, and waves
// left without one end; the LDS ring of states gets as many rows as the slots
// leave room for, reloaded from HBM.  One slot left steps as k_ra_lane0_wave
// does.  The last wave only fetches the walk's table rows (the fold of their
// copies), four to eight steps ahead of use.
//
// Bound by the chain of a step's instructions, LDS reads and the barrier
// (latency), and with more than a slot per SIMD by instruction issue on the one
// compute unit: 157 groups, 5267 steps: 19.0 -> 5.1 ms; 2500 groups, 5658 steps:
// 24.1 -> 14.2 ms, against lookups exchanged by LDS atomics with the states in
// HBM; 5.7 and 21.5 ms with a barrier more on nearly every step to settle flips.
//
// States in the ring are bytes: register | swapped << 6 | 0x80 when the register
// is not the home (which matters only while the home's entry holds it, and is
// then found among the few entries the lane owns).
constexpr uint32_t RA0_PACK = 64;
constexpr uint32_t RA0_WROWS = 16;         // walk rows in LDS
constexpr uint32_t RA0_RING_MAX = 147456;  // bytes of ring at most (160 KB of LDS per compute unit)
struct Ra0Tot { unsigned long long look, touch; };  // look bit 0 (x0 is never looked up): changed in this round
struct Ra0Move { uint32_t j, start, size, pad; uint64_t life, own, mk; };

DEV uint64_t lane64(uint32_t lo, uint32_t hi, uint32_t l) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)lo, (int)l) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, (int)l) << 32);
}

// A function of k_ra_lane0_wg; pr: the entry it won in the step before (0: none),
// not in hold yet.
template <int N> struct WgFn { uint32_t j, start, size, pr; uint64_t life, own, mk; OpQueue<N> ops; };
// Its step between the barriers: the op; packed, the operands' state bytes (8
// bits each), homes (6 bits each, at 16 and 22), flips taken (28, 29) and whether
// the homes' entries hold them (30, 31); the words defining them.
struct WgMid { uint32_t op, x, p1, p2; };

DEV void wg_regs(const WgMid &m, uint32_t fl, uint32_t &r1, uint32_t &r2) {
    const bool s1 = ((m.x >> 6) & 1u) || (fl & 1u), s2 = ((m.x >> 14) & 1u) || (fl & 2u);
    r1 = s1 ? ((m.op & OP_FP) ? 37u : 5u) : m.x & 0x3Fu;
    r2 = s2 ? ((m.op & OP_FP) ? 38u : 6u) : (m.x >> 8) & 0x3Fu;
}
DEV uint64_t wg_touch(uint32_t op, const OpStep &s) {
    return s.m | ((op & (OP_SELF | (63u << OP_CONST))) ? s.dm : 0ull);
}

template <int PER>
__global__ __launch_bounds__(1024) void k_ra_lane0_wg(Dev d, const Ra0Prog *progs, const uint32_t *gmin_all,
                                                      const uint32_t *gmax_all, const uint32_t *done,
                                                      const uint32_t *need, uint32_t copies, uint64_t stride,
                                                      Ra0Move *move_all, uint32_t ring_bytes) {
    extern __shared__ __align__(16) uint8_t wg_ring[];
    __shared__ Ra0Tot tot[2][64], settle[2][64];
    __shared__ uint32_t chk[2][64];  // by register: step << 6 | slot of a holder that no lookup flips yet
    __shared__ uint32_t Wmn[RA0_WROWS][64], Wmx[RA0_WROWS][64];
    __shared__ unsigned long long Wany[RA0_WROWS];
    __shared__ uint32_t hold[65], cnt[64];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t CW = (blockDim.x >> 6) - 1u;  // computing waves
    const bool helper = wave == CW;
    const Ra0Prog pg = progs[blockIdx.x];
    if (d.cflag[pg.prg]) return;  // k_ra_serial's
    const uint32_t steps = pg.rows;
    uint32_t NW = (pg.L + 63u) / 64u;
    if (NW > 64u || NW > CW * PER) { if (threadIdx.x == 0) atomicOr(d.flags, EF_OOB); return; }
    if (!helper && wave >= NW) return;  // (ended waves count as arrived at every barrier)
    const uint32_t *gmin = gmin_all + pg.gbase, *gmax = gmax_all + pg.gbase;
    const uint32_t *pdone = done && pg.cbase != RA0_NOPUB ? done + pg.cbase : nullptr;
    const uint32_t *pneed = pdone ? need + pg.cbase : nullptr;
    if (threadIdx.x < 128u) (&chk[0][0])[threadIdx.x] = 0xFFFFFFFFu;  // (two slots at least: those waves are there)
    // the totals of every slot, one per lane
    auto totals = [&](const Ra0Tot *t) {
        Ra0Tot r{0, 0};
        if (lane < NW) r = t[lane];
        return r;
    };
    // whether a holder that no lookup flips within its slot is looked up by a
    // lower slot (a higher slot number): then the slots settle together
    auto unsettled = [&](const Ra0Tot &t, uint32_t i) {
        const uint32_t key = chk[i & 1u][lane];
        bool any = false;
        for (uint64_t z = __ballot((key >> 6) == (i & 0x3FFFFFFu)); z; z &= z - 1) {
            const int r = __builtin_ctzll(z);
            const uint32_t es = (uint32_t)__builtin_amdgcn_readlane((int)key, r) & 63u;
            any = any || (__ballot((t.look >> r) & 1ull) >> es >> 1) != 0;
        }
        return any;
    };
    // packing at step i: the functions kept, inclusive over the slots
    auto pack_count = [&](uint32_t &before) {
        before = lane < NW ? cnt[lane] : 0u;
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)before, o, 64);
            if (lane >= o) before += u;
        }
        return (uint32_t)__builtin_amdgcn_readlane((int)before, 63);
    };
    if (helper) {
        // four rows at a time, their loads issued four steps before they are
        // folded and eight before the first is used; the barriers are the
        // computing waves'
        bool wok = true;  // the walk's rows still arrive
        uint32_t a[4][RA0_MAXCOPIES], b[4][RA0_MAXCOPIES];
        auto load4 = [&](uint32_t r) {
            if (pdone && r < steps && r % WALK_PUB == 0) ra0_wait(d, pdone, pneed, r / WALK_PUB, wok);
#pragma unroll
            for (uint32_t y = 0; y < 4; ++y) {
                const uint64_t e = (uint64_t)min(r + y, steps - 1u) * 64u + lane;
#pragma unroll
                for (uint32_t k = 0; k < RA0_MAXCOPIES; ++k) {
                    const uint64_t o = (k < copies ? k : 0u) * stride + e;
                    a[y][k] = gmin[o]; b[y][k] = gmax[o];
                }
            }
        };
        auto put4 = [&](uint32_t r) {
#pragma unroll
            for (uint32_t y = 0; y < 4; ++y) {
                uint32_t mn = a[y][0], mx = b[y][0];
#pragma unroll
                for (uint32_t k = 1; k < RA0_MAXCOPIES; ++k) { mn = min(mn, a[y][k]); mx = max(mx, b[y][k]); }
                const uint32_t w = (r + y) % RA0_WROWS;
                Wmn[w][lane] = mn; Wmx[w][lane] = mx;
                const uint64_t any = __ballot(mx != 0);
                if (lane == 0) Wany[w] = any;
            }
        };
        load4(0); put4(0); load4(4);
        __syncthreads();
        uint32_t i = 0;
        for (; i < steps; ++i) {
            if (i % RA0_PACK == 0 && i) {
                __syncthreads();
                __syncthreads();
                uint32_t before;
                const uint32_t nn = max(1u, (pack_count(before) + 63u) / 64u);
                if (nn < NW) {
                    __syncthreads();
                    NW = nn;
                    __syncthreads();
                    if (NW == 1u) break;
                }
            }
            lds_barrier();
            // rows i + 4 .. i + 7, over rows no wave reads any more
            if (i % 4u == 0) { put4(i + 4u); load4(i + 8u); }
            if (unsettled(totals(tot[i & 1u]), i)) {
                uint32_t r = 0;
                do { lds_barrier(); } while (__ballot(totals(settle[r++ & 1u]).look & 1ull));
            }
        }
        for (; i < steps; i += 4) {  // one slot left: a barrier per four steps
            lds_barrier();
            put4(i + 4u);
            load4(i + 8u);
        }
        return;
    }
    Ra0Move *mv = move_all + pg.poff;
    // the ring: `rows` rows of `slots` bytes and a spare one, word i in row ri
    uint32_t slots, rows, ri;
    auto ring_shape = [&](uint32_t i) {
        slots = NW * 64u;
        rows = min(OP_ROWS, ring_bytes / slots - 1u);
        ri = i % rows;
    };
    auto row_of = [&](uint32_t dist) { return ri >= dist ? ri - dist : ri + rows - dist; };  // dist <= rows
    ring_shape(0);
    // whether entry h of this lane holds word p (h: an operand's home), or for a
    // state that left its home (odd) which entry does
    auto home_of = [&](uint32_t e, uint32_t p, uint64_t own, uint32_t pr, uint32_t i) {
        uint32_t h = 0;
        if (e & 0x80u)
            for (uint64_t m = own; m; m &= m - 1) {
                const uint32_t r = (uint32_t)__builtin_ctzll(m);
                if ((r == pr ? i - 1u : hold[r]) == p) h = r;
            }
        return (e & 0x80u) ? h : e & 0x3Fu;
    };
    // the first part of a function's step: its operands' states (ring column k)
    auto operands = [&](uint32_t op, uint32_t i, uint32_t k, uint32_t start, uint64_t own, uint32_t pr, WgMid &m) {
        m.op = op;
        const uint32_t d1 = op & 0xFFu, d2 = (op >> 8) & 0xFFu;
        m.p1 = i - d1; m.p2 = i - d2;
        uint32_t e1 = wg_ring[row_of(min(d1, rows)) * slots + k], e2 = wg_ring[row_of(min(d2, rows)) * slots + k];
        e1 = d1 ? e1 : 0u; e2 = d2 ? e2 : 0u;
        // operands older than the ring: from HBM
        const bool o1 = (op & OP_FAR1) || d1 >= rows, o2 = (op & OP_FAR2) || d2 >= rows;
        if (__builtin_expect(__ballot(o1 || o2) != 0, 0)) {
            if (o1 || o2) {
                if (op & (OP_FAR1 | OP_FAR2)) {
                    const uint4 w = d.w0_f4[start + i];
                    if (op & OP_FAR1) m.p1 = w.y - 64u - start;
                    if (op & OP_FAR2) m.p2 = w.z - 64u - start;
                }
                const uint32_t g1 = d.sym[start + (o1 ? m.p1 : 0u)], g2 = d.sym[start + (o2 ? m.p2 : 0u)];
                wait_loads();
                if (o1) e1 = (g1 & 0x3Fu) | (((g1 >> 8) & 1u) << 6) | ((g1 & 0x3Fu) != g1 >> 9 ? 0x80u : 0u);
                if (o2) e2 = (g2 & 0x3Fu) | (((g2 >> 8) & 1u) << 6) | ((g2 & 0x3Fu) != g2 >> 9 ? 0x80u : 0u);
            }
        }
        uint32_t h1 = e1 & 0x3Fu, h2 = e2 & 0x3Fu;
        if (__builtin_expect(__ballot(((e1 | e2) & 0x80u) != 0) != 0, 0)) {
            h1 = home_of(e1, m.p1, own, pr, i);
            h2 = home_of(e2, m.p2, own, pr, i);
        }
        m.x = e1 | (e2 << 8) | (h1 << 16) | (h2 << 22);
    };
    // the second: commit and marks (new marks nm), and the word's own state
    auto commit = [&](const WgMid &m, const OpStep &s, uint32_t r1, uint32_t r2, uint32_t i, uint32_t k, uint32_t start,
                      bool run, uint64_t nm) {
        const uint32_t fl = (m.x >> 28) & 3u, h1 = (m.x >> 16) & 0x3Fu, h2 = (m.x >> 22) & 0x3Fu;
        const bool s1 = ((m.x >> 6) & 1u) || (fl & 1u), s2 = ((m.x >> 14) & 1u) || (fl & 2u);
        if (__ballot(s1 || s2)) {
            if (s1) {
                if (i - m.p1 < rows) wg_ring[row_of(i - m.p1) * slots + k] = (uint8_t)(r1 | 0x80u);
                d.sym[start + m.p1] = (uint16_t)(r1 | (h1 << 9));
            }
            if (s2) {
                if (i - m.p2 < rows) wg_ring[row_of(i - m.p2) * slots + k] = (uint8_t)(r2 | 0x80u);
                d.sym[start + m.p2] = (uint16_t)(r2 | (h2 << 9));
            }
        }
        while (nm) {
            const uint32_t r = (uint32_t)__builtin_ctzll(nm);
            nm &= nm - 1;
            const uint32_t p = hold[r];
            if (i - p < rows) wg_ring[row_of(i - p) * slots + k] |= 0x40u;
            reinterpret_cast<uint8_t *>(d.sym + start)[2u * p + 1u] = (uint8_t)(1u | (r << 1));
        }
        const bool self = (m.op & OP_SELF) != 0;
        if (run) {
            const uint32_t reg = self && !(m.op & OP_ZERO) ? s.rdr : 0u;
            wg_ring[ri * slots + k] = (uint8_t)(reg | (self && reg != s.rdr ? 0x80u : 0u));
            if (self) d.sym[start + i] = (uint16_t)(reg | (s.rdr << 9));
        }
    };
    // the states of a function's words [lo, last) from HBM, 32 a round: one round's
    // loads are in flight together (2500 groups, 26 packings: 14.40 -> 14.27 ms
    // against a load and its wait every four words)
    auto reload = [&](uint32_t start, uint32_t lo, uint32_t last, auto put) {
        for (uint32_t p = lo & ~7u; __ballot(p < last); p += 32) {
            Sym8 v[4];
#pragma unroll
            for (uint32_t x = 0; x < 4; ++x)
                v[x] = *reinterpret_cast<const Sym8 *>(d.sym + start + min(p + 8u * x, last ? (last - 1u) & ~7u : 0u));
#pragma unroll
            for (uint32_t x = 0; x < 4; ++x)
#pragma unroll
                for (uint32_t y = 0; y < 8; ++y)
                    if (p + 8u * x + y < last) put(p + 8u * x + y, (v[x].w[y / 2u] >> (16u * (y & 1u))) & 0xFFFFu);
        }
    };
    // packs the slots of fn[] (slot wave + q * CW in fn[q]) at step i; true when
    // this wave goes on
    auto pack = [&](auto &fn, uint32_t i) {
        constexpr int N = (int)(sizeof(fn) / sizeof(fn[0]));
        __syncthreads();  // every store of the steps before is done
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const uint32_t ws = wave + q * CW;
            if (ws >= NW) continue;
            if (fn[q].pr) { hold[fn[q].pr] = i - 1u; fn[q].pr = 0; }
            const uint64_t m = __ballot((int32_t)i < (int32_t)fn[q].size || fn[q].own != 0);
            if (lane == 0) cnt[ws] = (uint32_t)__popcll(m);
        }
        __syncthreads();
        uint32_t before;
        const uint32_t all = pack_count(before);
        const uint32_t nn = max(1u, (all + 63u) / 64u);
        if (nn >= NW) return true;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const uint32_t ws = wave + q * CW;
            if (ws >= NW) continue;
            const auto &f = fn[q];
            const bool keep = (int32_t)i < (int32_t)f.size || f.own != 0;
            const uint64_t m = __ballot(keep);
            const uint32_t b = ws ? (uint32_t)__builtin_amdgcn_readlane((int)before, (int)ws - 1) : 0u;
            if (keep) mv[b + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] =
                Ra0Move{f.j, f.start, f.size, 0u, f.life, f.own, f.mk};
        }
        __syncthreads();
        NW = nn;
        if (wave >= NW) return false;
        ring_shape(i);
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const uint32_t ws = wave + q * CW;
            if (ws >= NW) continue;
            auto &f = fn[q];
            const uint32_t k = ws * 64u + lane;
            const Ra0Move r = k < all ? mv[k] : Ra0Move{0, 0, 0, 0, 0x1Full, 0, 0};
            f.j = r.j; f.start = r.start; f.size = r.size; f.life = r.life; f.own = r.own; f.mk = r.mk;
            f.ops.load(d.ops + f.start, i, f.size);
            if (NW == 1u) {  // the ring as ra_l0_step has it, of functions that have ended too
                uint16_t *ring = reinterpret_cast<uint16_t *>(wg_ring);
                const uint32_t last = min(i, f.size);
                reload(f.start, last > OP_ROWS ? last - OP_ROWS : 0u, last,
                       [&](uint32_t p, uint32_t e) { ring[(p & (OP_ROWS - 1u)) * 64u + lane] = (uint16_t)e; });
            } else {
                const bool run = (int32_t)i < (int32_t)f.size;
                reload(f.start, i > rows ? i - rows : 0u, run ? i : 0u, [&](uint32_t p, uint32_t e) {
                    const uint32_t reg = e & 0x3Fu;
                    if (i - p <= rows)
                        wg_ring[(p % rows) * slots + k] =
                            (uint8_t)(reg | (((e >> 8) & 1u) << 6) | (reg != (e >> 9) ? 0x80u : 0u));
                });
            }
        }
        __syncthreads();
        return true;
    };
    auto next_row = [&]() { ri = ri + 1u == rows ? 0u : ri + 1u; };
    uint32_t i = 0;
    WgFn<4> f1[1];
    if (PER > 1) {
        // more slots than waves: each wave steps its slots one after the other,
        // keeping of each between the barriers only a WgMid
        WgFn<1> fn[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            WgFn<1> &f = fn[q];
            const uint32_t k = (wave + q * CW) * 64u + lane;
            const bool act = k < pg.L;
            f.j = act ? pg.L - 1u - k : 0u; f.pr = 0; f.life = 0x1Full; f.own = 0; f.mk = 0;
            f.start = act ? d.fstarts[pg.fbase + 8u * f.j] : 0u;
            f.size = act ? d.fsizes[pg.fbase + 8u * f.j] : 0u;
            f.ops.load(d.ops + f.start, 0, f.size);
        }
        __syncthreads();
        for (; i < steps && NW > CW; ++i) {
            if (i % RA0_PACK == 0 && i) {
                if (!pack(fn, i)) return;
                if (NW <= CW) break;
            }
            WgMid md[PER];
            bool has_nb[PER];
            // settles slot q's flips against `below` (what lower slots look up)
            // and returns its totals
            auto settle_slot = [&](int q, uint64_t below) {
                const WgFn<1> &f = fn[q];
                WgMid &m = md[q];
                uint32_t fl = (m.x >> 28) & 3u, r1, r2, x;
                OpStep s;
                if (has_nb[q]) {
                    const uint32_t h1 = (m.x >> 16) & 0x3Fu, h2 = (m.x >> 22) & 0x3Fu;
                    const bool b1 = (m.x >> 30) & 1u, b2 = (m.x >> 31) & 1u;
                    const uint32_t *wmn = Wmn[i % RA0_WROWS];
                    const bool w1 = b1 && (wmn[h1] < f.j || ((below >> h1) & 1u)), w2 = b2 && (wmn[h2] < f.j || ((below >> h2) & 1u));
                    bool ch;
                    do {
                        wg_regs(m, fl, r1, r2);
                        s = op_eval(m.op, r1, r2, f.life);
                        const uint64_t low = (uint64_t)suffix_or<4>((uint32_t)s.look, lane, x) |
                                             ((uint64_t)suffix_or<4>((uint32_t)(s.look >> 32), lane, x) << 32);
                        const uint32_t nf = (w1 || (b1 && ((low >> h1) & 1u)) ? 1u : 0u) |
                                            (w2 || (b2 && ((low >> h2) & 1u)) ? 2u : 0u);
                        ch = nf != fl;
                        fl = nf;
                    } while (__ballot(ch));
                    m.x = (m.x & ~(3u << 28)) | (fl << 28);
                }
                wg_regs(m, fl, r1, r2);
                s = op_eval(m.op, r1, r2, f.life);
                const uint64_t tc = wg_touch(m.op, s);
                const uint32_t a = scan_or<4>((uint32_t)s.look), b = scan_or<4>((uint32_t)(s.look >> 32));
                const uint32_t e = scan_or<4>((uint32_t)tc), g = scan_or<4>((uint32_t)(tc >> 32));
                return Ra0Tot{lane64(a, b, 63), lane64(e, g, 63)};
            };
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const uint32_t ws = wave + q * CW;
                has_nb[q] = false;
                if (ws >= NW) continue;
                WgFn<1> &f = fn[q];
                const uint32_t op = f.ops.next(d.ops + f.start, i, f.size);
                operands((int32_t)i < (int32_t)f.size ? op : 0u, i, ws * 64u + lane, f.start, f.own, f.pr, md[q]);
                if (__ballot(f.own != 0)) {
                    const uint32_t h1 = (md[q].x >> 16) & 0x3Fu, h2 = (md[q].x >> 22) & 0x3Fu;
                    const uint32_t q1 = h1 == f.pr ? i - 1u : hold[h1], q2 = h2 == f.pr ? i - 1u : hold[h2];
                    const bool b1 = q1 == md[q].p1 && ((f.own >> h1) & 1u), b2 = q2 == md[q].p2 && ((f.own >> h2) & 1u);
                    has_nb[q] = __ballot(b1 || b2) != 0;
                    md[q].x |= (b1 ? 1u << 30 : 0u) | (b2 ? 1u << 31 : 0u);
                }
                const Ra0Tot r = settle_slot(q, 0ull);
                if (has_nb[q]) {
                    const uint32_t x = md[q].x, key = ((i & 0x3FFFFFFu) << 6) | ws;
                    if (((x >> 30) & 1u) && !((x >> 28) & 1u) && !((x >> 6) & 1u)) chk[i & 1u][(x >> 16) & 0x3Fu] = key;
                    if (((x >> 31) & 1u) && !((x >> 29) & 1u) && !((x >> 14) & 1u)) chk[i & 1u][(x >> 22) & 0x3Fu] = key;
                }
                if (lane == 0) tot[i & 1u][ws] = r;
            }
            lds_barrier();
#pragma unroll
            for (int q = 0; q < PER; ++q)
                if (fn[q].pr) { hold[fn[q].pr] = i - 1u; fn[q].pr = 0; }
            Ra0Tot t = totals(tot[i & 1u]);
            if (unsettled(t, i)) {
                for (uint32_t r = 0;; ++r) {
                    uint32_t x;
                    const uint32_t bl = suffix_or<4>((uint32_t)t.look, lane, x), bh = suffix_or<4>((uint32_t)(t.look >> 32), lane, x);
#pragma unroll
                    for (int q = 0; q < PER; ++q) {
                        const uint32_t ws = wave + q * CW;
                        if (ws >= NW) continue;
                        Ra0Tot n{lane64((uint32_t)t.look, (uint32_t)(t.look >> 32), ws) & ~1ull,
                                 lane64((uint32_t)t.touch, (uint32_t)(t.touch >> 32), ws)};
                        if (has_nb[q]) {
                            const Ra0Tot o = n;
                            n = settle_slot(q, lane64(bl, bh, ws));
                            if (n.look != o.look || n.touch != o.touch) n.look |= 1ull;
                        }
                        if (lane == 0) settle[r & 1u][ws] = n;
                    }
                    lds_barrier();
                    t = totals(settle[r & 1u]);
                    if (!__ballot(t.look & 1ull)) break;
                }
            }
            // every slot's totals are final: of all, of the slots above each
            const uint32_t la = scan_or<4>((uint32_t)t.look), lb = scan_or<4>((uint32_t)(t.look >> 32));
            const uint32_t ta = scan_or<4>((uint32_t)t.touch), tb = scan_or<4>((uint32_t)(t.touch >> 32));
            const uint64_t T = (lane64(la, lb, 63) | Wany[i % RA0_WROWS]) & ~1ull, lost = lane64(ta, tb, 63);
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const uint32_t ws = wave + q * CW;
                if (ws >= NW) continue;
                WgFn<1> &f = fn[q];
                const WgMid &m = md[q];
                uint32_t r1, r2;
                wg_regs(m, (m.x >> 28) & 3u, r1, r2);
                const OpStep s = op_eval(m.op, r1, r2, f.life);
                const uint64_t tc = wg_touch(m.op, s);
                uint64_t won = (m.op & OP_SELF) ? s.dm & ~(ws ? lane64(ta, tb, ws - 1u) : 0ull) : 0ull;
                if (__ballot(won != 0))
                    won &= ~((uint64_t)from_below<4>(scan_or<4>((uint32_t)tc)) |
                             ((uint64_t)from_below<4>(scan_or<4>((uint32_t)(tc >> 32))) << 32));
                uint64_t nm = 0;
                if (__ballot(f.own != 0)) {
                    uint64_t mset = f.own & T;
                    if (has_nb[q]) {
                        const uint32_t h1 = (m.x >> 16) & 0x3Fu, h2 = (m.x >> 22) & 0x3Fu;
                        uint64_t high = (uint64_t)from_below<4>(scan_or<4>((uint32_t)s.look)) |
                                        ((uint64_t)from_below<4>(scan_or<4>((uint32_t)(s.look >> 32))) << 32);
                        if (ws) high |= lane64(la, lb, ws - 1u);
                        const uint64_t nb1 = (m.x >> 30) & 1u ? 1ull << h1 : 0ull, nb2 = (m.x >> 31) & 1u ? 1ull << h2 : 0ull;
                        if (Wmx[i % RA0_WROWS][h1] > f.j + 1u) high |= nb1;
                        if (Wmx[i % RA0_WROWS][h2] > f.j + 1u) high |= nb2;
                        const uint64_t nb = nb1 | nb2;
                        mset = f.own & ((T & ~nb) | (high & nb));
                        f.mk &= ~nb;
                    }
                    nm = mset & ~f.mk;
                    f.mk |= mset;
                }
                commit(m, s, r1, r2, i, ws * 64u + lane, f.start, (int32_t)i < (int32_t)f.size, nm);
                f.life = s.life;
                f.own = (f.own & ~lost) | won;
                f.mk &= ~lost;
                f.pr = won ? s.rdr : 0u;
            }
            next_row();
        }
        if (i >= steps) return;
        f1[0].j = fn[0].j; f1[0].start = fn[0].start; f1[0].size = fn[0].size; f1[0].life = fn[0].life;
        f1[0].own = fn[0].own; f1[0].mk = fn[0].mk;
    } else {
        const uint32_t k = wave * 64u + lane;
        const bool act = k < pg.L;
        f1[0].j = act ? pg.L - 1u - k : 0u; f1[0].life = 0x1Full; f1[0].own = 0; f1[0].mk = 0;
        f1[0].start = act ? d.fstarts[pg.fbase + 8u * f1[0].j] : 0u;
        f1[0].size = act ? d.fsizes[pg.fbase + 8u * f1[0].j] : 0u;
        __syncthreads();
    }
    f1[0].pr = 0;
    f1[0].ops.load(d.ops + f1[0].start, i, f1[0].size);
    bool packed = true;  // (the pack at this step is done)
    // a slot a wave: the step's results stay in registers over the barrier
    for (; NW > 1u && i < steps; ++i) {
        if (i % RA0_PACK == 0 && i && !packed) {
            if (!pack(f1, i)) return;
            if (NW == 1u) break;
        }
        packed = false;
        WgFn<4> &f = f1[0];
        const uint32_t k = wave * 64u + lane;
        const uint32_t op = f.ops.next(d.ops + f.start, i, f.size);
        const bool run = (int32_t)i < (int32_t)f.size;
        WgMid m;
        operands(run ? op : 0u, i, k, f.start, f.own, f.pr, m);
        const uint32_t h1 = (m.x >> 16) & 0x3Fu, h2 = (m.x >> 22) & 0x3Fu;
        // (an entry won in the step before is not in hold yet)
        const uint32_t q1 = h1 == f.pr ? i - 1u : hold[h1], q2 = h2 == f.pr ? i - 1u : hold[h2];
        const uint32_t mn1 = Wmn[i % RA0_WROWS][h1], mn2 = Wmn[i % RA0_WROWS][h2];
        const uint32_t mx1 = Wmx[i % RA0_WROWS][h1], mx2 = Wmx[i % RA0_WROWS][h2];
        const bool z1 = (m.x >> 6) & 1u, z2 = (m.x >> 14) & 1u;  // swapped already
        uint32_t fl = 0, r1, r2, x;
        wg_regs(m, 0u, r1, r2);
        OpStep s = op_eval(m.op, r1, r2, f.life);
        const uint64_t nb1 = q1 == m.p1 ? f.own & (1ull << h1) : 0ull, nb2 = q2 == m.p2 ? f.own & (1ull << h2) : 0ull;
        const uint64_t nb = nb1 | nb2;
        const uint64_t wl = (mn1 < f.j ? nb1 : 0ull) | (mn2 < f.j ? nb2 : 0ull);
        // flips against the slot's own lookups, the walk's and `below`
        auto settle_slot = [&](uint64_t below) {
            uint64_t low = below | (uint64_t)suffix_or<4>((uint32_t)s.look, lane, x) |
                           ((uint64_t)suffix_or<4>((uint32_t)(s.look >> 32), lane, x) << 32);
            uint32_t nf = ((nb1 & low) && !z1 ? 1u : 0u) | ((nb2 & low) && !z2 ? 2u : 0u);
            while (__ballot(nf != fl)) {
                fl = nf;
                wg_regs(m, fl, r1, r2);
                s = op_eval(m.op, r1, r2, f.life);
                low = below | (uint64_t)suffix_or<4>((uint32_t)s.look, lane, x) |
                      ((uint64_t)suffix_or<4>((uint32_t)(s.look >> 32), lane, x) << 32);
                nf = ((nb1 & low) && !z1 ? 1u : 0u) | ((nb2 & low) && !z2 ? 2u : 0u);
            }
        };
        settle_slot(wl);
        uint64_t tc = wg_touch(m.op, s);
        uint32_t la = scan_or<4>((uint32_t)s.look), lb = scan_or<4>((uint32_t)(s.look >> 32));
        uint32_t ta = scan_or<4>((uint32_t)tc), tb = scan_or<4>((uint32_t)(tc >> 32));
        if (lane == 63u) tot[i & 1u][wave] = Ra0Tot{(uint64_t)la | ((uint64_t)lb << 32), (uint64_t)ta | ((uint64_t)tb << 32)};
        const bool c1 = nb1 != 0 && !(fl & 1u) && !z1, c2 = nb2 != 0 && !(fl & 2u) && !z2;
        if (c1 || c2) {
            const uint32_t key = ((i & 0x3FFFFFFu) << 6) | wave;
            if (c1) chk[i & 1u][h1] = key;
            if (c2) chk[i & 1u][h2] = key;
        }
        lds_barrier();
        hold[f.pr ? f.pr : 64u] = i - 1u;
        Ra0Tot t = totals(tot[i & 1u]);
        if (unsettled(t, i)) {
            for (uint32_t r = 0;; ++r) {
                const uint64_t below = lane64(suffix_or<4>((uint32_t)t.look, lane, x), suffix_or<4>((uint32_t)(t.look >> 32), lane, x), wave);
                const uint64_t ol = lane64(la, lb, 63), ot = lane64(ta, tb, 63);
                settle_slot(wl | below);
                tc = wg_touch(m.op, s);
                la = scan_or<4>((uint32_t)s.look); lb = scan_or<4>((uint32_t)(s.look >> 32));
                ta = scan_or<4>((uint32_t)tc); tb = scan_or<4>((uint32_t)(tc >> 32));
                const uint64_t nl = lane64(la, lb, 63), nt = lane64(ta, tb, 63);
                if (lane == 0) settle[r & 1u][wave] = Ra0Tot{nl | (nl != ol || nt != ot ? 1ull : 0ull), nt};
                lds_barrier();
                t = totals(settle[r & 1u]);
                if (!__ballot(t.look & 1ull)) break;
            }
        }
        // every slot's totals are final: of all, of the slots above (at most 16
        // slots: one row of lanes)
        const uint32_t sa = scan_or<1>((uint32_t)t.look), sb = scan_or<1>((uint32_t)(t.look >> 32));
        const uint32_t ua = scan_or<1>((uint32_t)t.touch), ub = scan_or<1>((uint32_t)(t.touch >> 32));
        const uint64_t T = (lane64(sa, sb, 15) | Wany[i % RA0_WROWS]) & ~1ull, lost = lane64(ua, ub, 15);
        const uint32_t wp = wave ? wave - 1u : 31u;  // (lanes past the first row hold nothing)
        uint64_t high = (uint64_t)from_below<4>(la) | ((uint64_t)from_below<4>(lb) << 32) | lane64(sa, sb, wp);
        high |= (mx1 > f.j + 1u ? nb1 : 0ull) | (mx2 > f.j + 1u ? nb2 : 0ull);
        const uint64_t above = (uint64_t)from_below<4>(ta) | ((uint64_t)from_below<4>(tb) << 32) | lane64(ua, ub, wp);
        const uint64_t won = (m.op & OP_SELF) ? s.dm & ~above : 0ull;
        f.mk &= ~nb;
        const uint64_t nm = f.own & ~f.mk & ((T & ~nb) | (high & nb));
        f.mk |= nm;
        m.x |= fl << 28;
        commit(m, s, r1, r2, i, k, f.start, run, nm);
        f.life = s.life;
        f.own = (f.own & ~lost) | won;
        f.mk &= ~lost;
        f.pr = won ? s.rdr : 0u;
        next_row();
    }
    if (i >= steps) return;
    // one slot left: its steps need no exchange with other waves
    RaL0 f{f1[0].start, f1[0].size, f1[0].life, f1[0].own, f1[0].mk};
    uint16_t *ring = reinterpret_cast<uint16_t *>(wg_ring);
    const uint32_t *ops = d.ops + f.start;
    OpBlock ob;
    ob.load(ops, i, f.size);  // (i is a multiple of RA0_PACK)
    for (; i < steps; i += 4) {
        lds_barrier();  // the walk's rows of the four steps are in
        ob.step4(ops, i, f.size);
        ra_evict<64>(d, f, ring, lane, i);
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t r = (i + q) % RA0_WROWS;
            const uint32_t op = (int32_t)(i + q) < (int32_t)f.size ? ob.cur[0].o[q] : 0u;
            ra_l0_step<5, 64>(d, f, ring, hold, lane, lane, f1[0].j, i, i + q, op,
                                 RaLooks{0ull, Wmn[r], Wmx[r], i + q < steps ? Wany[r] : 0ull});
        }
    }
    ra_flush<64>(d, f, ring, lane);
}

// Exact fallback for programs in which a function names a register that another
// one defines (ra_op): the reference's allocation walk as written
// (rv_generator_avx.cpp:1041-1418 at one thread), one wave: steps in order,
// groups of 8 functions in order within a step, the 8 functions of a group on
// lanes 0-7.  Each group body reads its operands' states before any of its
// writes; its writes follow the reference's order (marks, lifetimes,
// register_state, then the symbol entries of rd, rs1, rs2, lane by lane).
// register_state keeps 8 regions of 64 (region = lane); lookups read region 0
// of the step's snapshot.
__global__ __launch_bounds__(64) void k_ra_serial(Dev d, const Ra0Prog *progs, const uint32_t *plist,
                                                  uint64_t *life_all) {
    __shared__ int32_t reg[8][64];
    __shared__ int32_t snap[64];
    const uint32_t lane = threadIdx.x;
    const uint32_t prg = plist[blockIdx.x];
    const Ra0Prog pg = progs[prg];
    const uint32_t maxsize = pg.maxsize, fbase = pg.fbase, nf = pg.nf;
    uint64_t *life = life_all + fbase;
    for (uint32_t k = lane; k < 8 * 64; k += 64) reg[k / 64][k % 64] = -1;
    for (uint32_t f = lane; f < nf; f += 64) life[f] = 0x1Full;
    for (uint32_t e = d.pw[prg] + lane; e < d.pw[prg + 1]; e += 64) d.sym[e] = 0;  // the program's states restart
    __syncthreads();
    const uint32_t G = (nf + 7u) / 8u;
    for (uint32_t i = 0; i < maxsize; ++i) {
        snap[lane] = reg[0][lane];
        __syncthreads();
        for (uint32_t g = 0; g < G; ++g) {
            const uint32_t f = 8u * g + lane;  // within the program
            const bool nc = lane < 8 && f < nf && (int32_t)i < (int32_t)d.fsizes[fbase + f];
            uint4 w = make_uint4(0, 0, 0, 0);
            uint64_t lt = 0;
            if (nc) { w = d.w0_f4[d.fstarts[fbase + f] + i]; lt = life[f]; }
            const uint32_t raw1 = nc && virt_ok(d, w.y) ? d.sym[w.y - 64u] : 0u;
            const uint32_t raw2 = nc && virt_ok(d, w.z) ? d.sym[w.z - 64u] : 0u;
            const RaStep r = ra_eval_raw(w.w, w.x, w.y, w.z, raw1 & 0xFFu, raw2 & 0xFFu, (raw1 >> 8) != 0,
                                         (raw2 >> 8) != 0, lt);
            __syncthreads();  // every lane has read before any lane writes
            if (nc && r.swd) { const int32_t x = snap[r.rdr] - 64; if (x >= 0) sym_mark(d, (uint32_t)x); }
            if (nc && r.sw1) { const int32_t x = snap[r.r1r] - 64; if (x >= 0) sym_mark(d, (uint32_t)x); }
            if (nc && r.sw2) { const int32_t x = snap[r.r2r] - 64; if (x >= 0) sym_mark(d, (uint32_t)x); }
            if (nc) {
                life[f] = r.newlife;
                if (r.ord) reg[lane][r.rdr] = (int32_t)r.ord;
                if (r.r1r != r.rdr) reg[lane][r.r1r] = -1;
                if (r.r2r != r.rdr) reg[lane][r.r2r] = -1;
            }
            const bool oob = nc && (((int32_t)r.ord > 63 && r.ord - 64u >= d.W0) ||
                                    ((int32_t)r.rs1 > 63 && r.rs1 - 64u >= d.W0) ||
                                    ((int32_t)r.rs2 > 63 && r.rs2 - 64u >= d.W0));
            if (oob) atomicOr(d.flags, EF_OOB);
            const bool ok = nc && !oob;
            for (uint32_t k = 0; k < 8; ++k) { if (ok && lane == k && (int32_t)r.ord > 63) d.sym[r.ord - 64u] = (uint16_t)r.rdr; __syncthreads(); }
            for (uint32_t k = 0; k < 8; ++k) { if (ok && lane == k && (int32_t)r.rs1 > 63) d.sym[r.rs1 - 64u] = (uint16_t)r.r1r; __syncthreads(); }
            for (uint32_t k = 0; k < 8; ++k) { if (ok && lane == k && (int32_t)r.rs2 > 63) d.sym[r.rs2 - 64u] = (uint16_t)r.r2r; __syncthreads(); }
        }
    }
}

// Instruction counts after allocation (:1473-1495): used words plus one load
// per swapped operand and one store for a swapped destination.
struct RaCountOp {
    Dev d;
    DEV uint32_t sw(uint32_t r) const { return ((int32_t)r > 63 && r - 64u < d.W0 && sym_swapped(d, r - 64u)) ? 1u : 0u; }
    DEV uint32_t value(uint64_t i) const {
        if (!d.usedi[i]) return 0;
        const uint4 w = d.w0_f4[i];  // rd, rs1, rs2, instruction
        return 1u + sw(w.y) + sw(w.z) + sw(w.x);
    }
    DEV void emit(uint64_t i, uint32_t excl, uint32_t) const { d.ra_off[i] = excl; }
};

// spill_offsets (:1450-1469): each function's words copy the flag at its start.
DEV uint32_t spill_of(const Dev &d, uint32_t v) {
    uint32_t lo = 0, hi = d.F;  // last start <= v
    while (hi - lo > 1) { uint32_t m = (lo + hi) / 2; if (d.fstarts[m] <= v) lo = m; else hi = m; }
    return sym_swapped(d, d.fstarts[lo]) ? 1u : 0u;
}

// Emit (:1552-1697).
__global__ __launch_bounds__(256) void k_ra_emit(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    // the function of the wave's first word, looked up once for the wave: a
    // word's operands are mostly registers of its own function, and the
    // wave's words mostly of one function (spill_of of any other register)
    const uint64_t i0 = blockIdx.x * (uint64_t)blockDim.x + (threadIdx.x & ~63u);
    uint32_t fi = 0, fs = 0, fe = 0;
    if (i0 < d.W0 && d.F) {
        uint32_t lo = 0, hi = d.F;  // last start <= i0
        while (hi - lo > 1) { const uint32_t m = (lo + hi) / 2; if (d.fstarts[m] <= (uint32_t)i0) lo = m; else hi = m; }
        fi = lo;
        fs = d.fstarts[lo];
        fe = lo + 1 < d.F ? d.fstarts[lo + 1] : 0xFFFFFFFFu;
    }
    const uint32_t fsp = fe > fs && sym_swapped(d, fs) ? 1u : 0u;
    // the function of this lane's own word, stepping on from the wave's (a
    // wave's words span few functions), for a lane past the wave's function
    uint32_t ls = fs, le = fe, lsp = fsp;
    if (i < d.W0 && d.F && (uint32_t)i >= fe) {
        uint32_t li = fi + 1;
        while (li + 1 < d.F && d.fstarts[li + 1] <= (uint32_t)i) ++li;
        ls = d.fstarts[li];
        le = li + 1 < d.F ? d.fstarts[li + 1] : 0xFFFFFFFFu;
        lsp = sym_swapped(d, ls) ? 1u : 0u;
    }
    auto spill = [&](uint32_t v) -> uint32_t {
        return v >= ls && v < le ? lsp : v >= fs && v < fe ? fsp : spill_of(d, v);
    };
    // slots no word's range covers: the pad at W1 and, when the last word is
    // unused, the reference's last slot W1 - 1 (W1 = last offset + 1)
    auto zero = [&](uint32_t o) {
        d.w1_instr[o] = 0; d.w1_rd[o] = 0; d.w1_rs1[o] = 0; d.w1_rs2[o] = 0; d.w1_jt[o] = 0;
    };
    if (i == 0) zero(d.W1);
    if (i + 1 == d.W0 && !d.usedi[i] && d.ra_off[i] < d.W1) zero(d.ra_off[i]);
    if (i >= d.W0 || !d.usedi[i]) return;
    const int32_t base = (int32_t)d.ra_off[i];
    const uint4 wf = d.w0_f4[i];  // rd, rs1, rs2, instruction
    const uint32_t ins = wf.w;
    const uint32_t r1 = wf.y, r2 = wf.z, rdv = wf.x;
    int32_t l1 = -1, l2 = -1, rdo = -1;
    uint32_t a1 = r1, a2 = r2, ad = rdv, st1 = 0, st2 = 0, std_ = 0;
    if (((int32_t)r1 > 63 && r1 - 64u >= d.W0) || ((int32_t)r2 > 63 && r2 - 64u >= d.W0) ||
        ((int32_t)rdv > 63 && rdv - 64u >= d.W0)) { atomicOr(d.flags, EF_OOB); return; }
    if ((int32_t)r1 > 63) {
        const uint32_t e = d.sym[r1 - 64u];
        const bool sw = (e & 0x100u) != 0;
        l1 = sw ? base : -1;
        st1 = spill(r1 - 64u);
        a1 = sw ? (((ins == 0xC0007053u) || (ins & 0x7Fu) == 0x53u) ? 37u : 5u) : (e & 0xFFu);
    }
    if ((int32_t)r2 > 63) {
        const uint32_t e = d.sym[r2 - 64u];
        const bool sw = (e & 0x100u) != 0;
        l2 = sw ? base : -1;  // the reference tests its own, still -1, offset (D6)
        st2 = spill(r2 - 64u);
        a2 = sw ? (((ins & 0x7Fu) == 0x53u) ? 38u : 6u) : (e & 0xFFu);
    }
    const int32_t mo = base + (l1 > 0 ? 1 : 0) + (l2 > 0 ? 1 : 0);
    if ((int32_t)rdv > 63) {
        const uint32_t e = d.sym[rdv - 64u];
        const bool sw = (e & 0x100u) != 0;
        rdo = sw ? mo + 1 : -1;
        std_ = spill(rdv - 64u);
        ad = e & 0xFFu;
    }
    // The word's slots are [base, base + n) (its count in RaCountOp); the
    // reference's stores land in them as below, later ones over earlier ones,
    // and a slot none of them reaches stays zero.  Each slot of the range is
    // written once, all five fields, so the arrays need no clearing.
    const uint32_t n = 1u + (l1 >= 0 ? 1u : 0u) + (l2 >= 0 ? 1u : 0u) + (rdo >= 0 ? 1u : 0u);
    const uint32_t end = (uint32_t)base + n;
    if ((rdo >= 0 && (uint32_t)rdo >= end) || (uint32_t)mo >= end || end > d.W1) { atomicOr(d.flags, EF_OOB); return; }
    uint32_t wi[4] = {0, 0, 0, 0}, wd[4] = {0, 0, 0, 0}, w1[4] = {0, 0, 0, 0}, w2[4] = {0, 0, 0, 0}, wj[4] = {0, 0, 0, 0};
    auto at = [&](int32_t slot) -> uint32_t { return (uint32_t)(slot - base); };  // < n for every slot stored
    if (l1 >= 0) { wi[at(l1)] = (((st1 - 1u) * 4u) << 20) | 0x2003u; wd[at(l1)] = 5; }
    if (l2 >= 0) { wi[at(l2)] = (((st2 - 1u) * 4u) << 20) | 0x2003u; wd[at(l2)] = 6; }
    {
        const uint32_t k = at(mo);
        wi[k] = ins; wd[k] = ad; w1[k] = a1; w2[k] = a2;
        wj[k] = d.ra_off[d.w0_jt[i] < d.W0 ? d.w0_jt[i] : 0];
        if (d.w0_jt[i] >= d.W0) atomicOr(d.flags, EF_OOB);
    }
    if (rdo >= 0) {
        const uint32_t k = at(rdo);
        uint32_t imm = (std_ - 1u) * (uint32_t)-4;
        wi[k] = 0x2023u | ((imm & 0x1Fu) << 7) | ((imm & 0xFEu) << 19);
        wd[k] = 0; w1[k] = ad; w2[k] = 0; wj[k] = 0;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (k < n) {
            const uint32_t o = (uint32_t)base + k;
            d.w1_instr[o] = wi[k]; d.w1_rd[o] = wd[k]; d.w1_rs1[o] = w1[k]; d.w1_rs2[o] = w2[k]; d.w1_jt[o] = wj[k];
        }
}

// fix_func_tab (:1816-1837) against an offset array; pend[p] is the end of
// program p's range of that array (a function ending there takes the last
// offset + 1, as the reference does at the end of its array).
__global__ void k_fixtab(Dev d, const uint32_t *off, const uint32_t *pend) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= d.F) return;
    const uint32_t len = pend[prog_of(d.pf, d.P, k)];
    uint32_t s = d.fstarts[k], e = s + d.fsizes[k];
    uint32_t so = off[s];
    uint32_t eo = (int32_t)e >= (int32_t)len ? off[len - 1] + 1u : off[e];
    d.fstarts[k] = so; d.fends[k] = eo; d.fsizes[k] = eo - so;
}

// Per-program bounds after regalloc (the reference's W1 = last offset + 1,
// :1542) and after fix_jumps (last offset + size of the last word, :1891):
// b1[p] = start of program p's allocated words, e1[p] = its W1 end; b2/e2 the
// same for the final words.
__global__ void k_prog_w1(Dev d, uint32_t *b1, uint32_t *e1) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= d.P) return;
    b1[p] = d.ra_off[d.pw[p]];
    e1[p] = d.ra_off[d.pw[p + 1] - 1] + 1u;
}

// Frame words (:1714-1811): lui s0, 0 / addi s0, s0, 8 after the prologue
// stores and before the epilogue; no callee-saved preservation (never written).
__global__ void k_ra_frame(Dev d) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= d.F) return;
    const uint32_t upper = 0x437u, lower = (8u << 20) | 0x40413u;
    uint32_t s = d.fstarts[k], e = s + d.fsizes[k];
    uint32_t pos[4] = {s + 2, s + 3, e - 6, e - 5};
    for (int q = 0; q < 4; ++q) {
        uint32_t x = pos[q];
        if (x >= d.W1) { atomicOr(d.flags, EF_OOB); continue; }
        d.w1_instr[x] = (q & 1) ? lower : upper;
        d.w1_rd[x] = 0; d.w1_rs1[x] = 0; d.w1_rs2[x] = 0; d.w1_jt[x] = 0;
    }
}

// ================================================================ fix_jumps
DEV uint32_t fj_size(uint32_t w) {
    bool jmp = ((w & 0x7Fu) == 0x67u) && w != 0x8067u;
    return jmp ? 2u : (w != 0 ? 1u : 0u);
}

__global__ void k_prog_w2(Dev d, const uint32_t *b1, const uint32_t *e1, uint32_t *b2, uint32_t *e2) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= d.P) return;
    b2[p] = d.fj_off[b1[p]];
    e2[p] = d.fj_off[e1[p] - 1] + fj_size(d.w1_instr[e1[p] - 1]);
}

struct FjSizeOp {
    Dev d;
    DEV uint32_t value(uint64_t i) const { return fj_size(d.w1_instr[i]); }
    DEV void emit(uint64_t i, uint32_t excl, uint32_t) const { d.fj_off[i] = excl; }
};

// Move + jump/branch encoding + postprocess in one pass (:1895-1993, :1995-2011).
__global__ __launch_bounds__(256) void k_fj_move(Dev d) {
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= d.W1) return;
    const uint32_t w = d.w1_instr[i];
    if (w == 0) return;
    const uint32_t k = d.fj_off[i];
    const bool jmp = ((w & 0x7Fu) == 0x67u) && w != 0x8067u;
    const bool br = (w & 0x7Fu) == 0x63u;
    const uint32_t pp = ((d.w1_rd[i] & 31u) << 7) | ((d.w1_rs1[i] & 31u) << 15) | ((d.w1_rs2[i] & 31u) << 20);
    if (jmp || br) {
        const uint32_t jt1 = d.w1_jt[i];
        if (jt1 >= d.W1) atomicOr(d.flags, EF_OOB);
        const uint32_t tgt = 4u * d.fj_off[jt1 < d.W1 ? jt1 : 0];
        const uint32_t delta = tgt - k * 4u;
        if (jmp) {
            const uint32_t upper = (delta & 0xFFFFF000u) >> 12, lower = delta & 0xFFFu, sign = (delta >> 11) & 1u;
            d.words[k] = ((upper + sign) << 12) | 0x97u;
            d.words[k + 1] = w | (lower << 20) | (1u << 15);
            return;
        }
        const uint32_t sign = (delta >> 12) & 1u, b11 = (delta >> 11) & 1u;
        const uint32_t b105 = (delta >> 5) & 0x1Fu, b14 = (delta >> 1) & 0xFu;
        d.words[k] = w | (sign << 31) | (b11 << 7) | (b105 << 25) | (b14 << 8) | pp;
        return;
    }
    d.words[k] = w | pp;
}

// ============================================================== text output
// rv_generator::to_asm (src/codegen/rv_generator.cpp:114-120): one line per
// word, rvdisasm::instruction(word) (src/disassembler.cpp:453-462) and '\n':
// the mnemonic (instr_name, :83-222), a space, the operands (format_args,
// :224-407, no colour, address 0).  The reference's switches continue with the
// next case in source order wherever an inner switch finds no match; asm_name
// walks its cases as such a chain, so a branch with funct3 2 is named "lw" and
// a SYSTEM word other than ecall/ebreak "flw", exactly as the reference prints
// them.  Lines are at most 48 bytes.  Each word is formatted by one thread: a
// scan of the line lengths gives every line's offset, and the rescan writes
// each thread's 16 consecutive lines (4-byte stores inside its own byte range,
// byte stores at its two ends).
enum : uint8_t {
    M_LUI, M_AUIPC, M_JAL, M_JALR, M_BEQ, M_BNE, M_BLT, M_BGE, M_BLTU, M_BGEU, M_LB, M_LH, M_LW, M_LBU, M_LHU,
    M_SB, M_SH, M_SW, M_ADDI, M_SLLI, M_SLTI, M_SLTIU, M_XORI, M_SRLI, M_SRAI, M_ORI, M_ANDI, M_ADD, M_MUL,
    M_SUB, M_SLL, M_MULH, M_SLT, M_MULHSU, M_SLTU, M_MULHU, M_XOR, M_DIV, M_SRL, M_DIVU, M_SRA, M_OR, M_REM,
    M_AND, M_REMU, M_FENCE, M_ECALL, M_EBREAK, M_FLW, M_FSW, M_FMADD, M_FMSUB, M_FNMSUB, M_FNMADD, M_FADD,
    M_FSUB, M_FMUL, M_FDIV, M_FSQRT, M_FSGNJ, M_FSGNJN, M_FSGNJX, M_FMIN, M_FMAX, M_FCVT_W_S, M_FCVT_WU_S,
    M_FMV_X_W, M_FCLASS, M_FLE, M_FLT, M_FEQ, M_FCVT_S_W, M_FCVT_S_WU, M_FMV_W_X, M_UNKNOWN, M_ZERO, M_COUNT
};
// names and registers in 16- and 8-byte slots, read as 8-byte words
__constant__ __align__(16) char c_asm_name[M_COUNT][16] = {
    "lui", "auipc", "jal", "jalr", "beq", "bne", "blt", "bge", "bltu", "bgeu", "lb", "lh", "lw", "lbu", "lhu",
    "sb", "sh", "sw", "addi", "slli", "slti", "sltiu", "xori", "srli", "srai", "ori", "andi", "add", "mul",
    "sub", "sll", "mulh", "slt", "mulhsu", "sltu", "mulhu", "xor", "div", "srl", "divu", "sra", "or", "rem",
    "and", "remu", "fence", "ecall", "ebreak", "flw", "fsw", "fmadd.s", "fmsub.s", "fnmsub.s", "fnmadd.s",
    "fadd.s", "fsub.s", "fmul.s", "fdiv.s", "fsqrt.s", "fsgnj.s", "fsgnjn.s", "fsgnjx.s", "fmin.s", "fmax.s",
    "fcvt.w.s", "fcvt.wu.s", "fmv.x.w", "fclass.s", "fle.s", "flt.s", "feq.s", "fcvt.s.w", "fcvt.s.wu",
    "fmv.w.x", "unknown", "(zero)"};
// ABI register names (:15-50)
__constant__ __align__(8) char c_asm_x[32][8] = {"zero", "ra", "sp", "gp", "tp", "t0", "t1", "t2", "s0", "s1", "a0",
                                    "a1", "a2", "a3", "a4", "a5", "a6", "a7", "s2", "s3", "s4", "s5",
                                    "s6", "s7", "s8", "s9", "s10", "s11", "t3", "t4", "t5", "t6"};
__constant__ __align__(8) char c_asm_f[32][8] = {"ft0", "ft1", "ft2", "ft3", "ft4", "ft5", "ft6", "ft7", "fs0", "fs1", "fa0",
                                    "fa1", "fa2", "fa3", "fa4", "fa5", "fa6", "fa7", "fs2", "fs3", "fs4", "fs5",
                                    "fs6", "fs7", "fs8", "fs9", "fs10", "fs11", "ft8", "ft9", "ft10", "ft11"};

// instr_name: the case chain entered at the word's opcode.
DEV uint32_t asm_name(uint32_t w) {
    const uint32_t op = w & 0x7Fu, f3 = (w >> 12) & 7u, f7 = (w >> 25) & 0x7Fu, r2 = (w >> 20) & 0x1Fu;
    // cases in source order: 0 lui, 1 auipc, 2 jal, 3 jalr, 4 BRANCH, 5 LOAD,
    // 6 STORE, 7 OP-IMM, 8 OP, 9 fence, 10 SYSTEM, 11 flw, 12 fsw, 13-16 the
    // fused multiply-adds, 17 OP-FP
    int k;
    switch (op) {
        case 0x37: k = 0; break;  case 0x17: k = 1; break;  case 0x6F: k = 2; break;  case 0x67: k = 3; break;
        case 0x63: k = 4; break;  case 0x03: k = 5; break;  case 0x23: k = 6; break;  case 0x13: k = 7; break;
        case 0x33: k = 8; break;  case 0x0F: k = 9; break;  case 0x73: k = 10; break; case 0x07: k = 11; break;
        case 0x27: k = 12; break; case 0x43: k = 13; break; case 0x47: k = 14; break; case 0x4B: k = 15; break;
        case 0x4F: k = 16; break; case 0x53: k = 17; break;
        default: return w ? M_UNKNOWN : M_ZERO;
    }
    for (; k < 18; ++k) {
        switch (k) {
            case 0: return M_LUI;
            case 1: return M_AUIPC;
            case 2: return M_JAL;
            case 3: return M_JALR;
            case 4: { constexpr uint8_t t[8] = {M_BEQ, M_BNE, 0xFF, 0xFF, M_BLT, M_BGE, M_BLTU, M_BGEU};
                      if (t[f3] != 0xFF) return t[f3]; break; }
            case 5: { constexpr uint8_t t[8] = {M_LB, M_LH, M_LW, 0xFF, M_LBU, M_LHU, 0xFF, 0xFF};
                      if (t[f3] != 0xFF) return t[f3]; break; }
            case 6: if (f3 < 3) return M_SB + f3; break;
            case 7: { constexpr uint8_t t[8] = {M_ADDI, M_SLLI, M_SLTI, M_SLTIU, M_XORI, 0xFF, M_ORI, M_ANDI};
                      if (f3 == 5) return f7 == 0 ? M_SRLI : f7 == 0x20 ? M_SRAI : M_ORI;  // else into funct3 6
                      return t[f3]; }
            case 8: {
                // funct3 cases from the word's own on, each matching funct7 0, 1
                // (and 0x20 for add/sub, srl/sra), else the next funct3 case
                constexpr uint8_t base[8] = {M_ADD, M_SLL, M_SLT, M_SLTU, M_XOR, M_SRL, M_OR, M_AND};
                constexpr uint8_t mext[8] = {M_MUL, M_MULH, M_MULHSU, M_MULHU, M_DIV, M_DIVU, M_REM, M_REMU};
                for (uint32_t g = f3; g < 8; ++g) {
                    if (f7 == 0) return base[g];
                    if (f7 == 1) return mext[g];
                    if (f7 == 0x20 && g == 0) return M_SUB;
                    if (f7 == 0x20 && g == 5) return M_SRA;
                }
                break;
            }
            case 9: return M_FENCE;
            case 10: if (f7 == 0) return M_ECALL; if (f7 == 1) return M_EBREAK; break;
            case 11: return M_FLW;
            case 12: return M_FSW;
            case 13: return M_FMADD;
            case 14: return M_FMSUB;
            case 15: return M_FNMSUB;
            case 16: return M_FNMADD;
            case 17: {
                // funct7 cases in source order, entered at the word's own
                constexpr uint8_t sev[12] = {0x00, 0x04, 0x08, 0x0C, 0x2C, 0x10, 0x14, 0x60, 0x70, 0x50, 0x68, 0x78};
                uint32_t t = 0;
                while (t < 12 && sev[t] != f7) ++t;
                for (; t < 12; ++t) {
                    switch (t) {
                        case 0: return M_FADD;
                        case 1: return M_FSUB;
                        case 2: return M_FMUL;
                        case 3: return M_FDIV;
                        case 4: return M_FSQRT;
                        case 5: if (f3 < 3) return M_FSGNJ + f3; break;
                        case 6: if (f3 < 2) return M_FMIN + f3; break;
                        case 7: if (r2 < 2) return M_FCVT_W_S + r2; break;
                        case 8: if (f3 < 2) return M_FMV_X_W + f3; break;
                        case 9: if (f3 < 3) return M_FLE + f3; break;
                        case 10: if (r2 < 2) return M_FCVT_S_W + r2; break;
                        default: return M_FMV_W_X;
                    }
                }
                break;
            }
        }
    }
    return w ? M_UNKNOWN : M_ZERO;
}

// the bytes of v up to the first zero; true when all eight were emitted
template <class S> DEV bool asm_8(S &s, uint64_t v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const char c = (char)(v >> (8 * i));
        if (!c) return false;
        s.put(c);
    }
    return true;
}
template <class S> DEV void asm_str16(S &s, const char *p) {  // a 16-byte slot
    const uint64_t *q = reinterpret_cast<const uint64_t *>(p);
    const uint64_t lo = q[0], hi = q[1];
    if (asm_8(s, lo)) asm_8(s, hi);
}
template <class S> DEV void asm_str8(S &s, const char *p) { asm_8(s, *reinterpret_cast<const uint64_t *>(p)); }
template <class S> DEV void asm_dec(S &s, int32_t x) {
    uint32_t u = (uint32_t)x;
    if (x < 0) { s.put('-'); u = 0u - u; }
    uint64_t dig = 0;  // decimal digits, 4 bits each, least significant first
    int nd = 0;
    do { dig |= (uint64_t)(u % 10u) << (4 * nd); u /= 10u; ++nd; } while (u);
    for (int k = nd - 1; k >= 0; --k) s.put((char)('0' + ((dig >> (4 * k)) & 15u)));
}
// std::hex << std::showbase: "0x" and the digits, a bare "0" for zero
template <class S> DEV void asm_hex(S &s, uint64_t v) {
    if (!v) { s.put('0'); return; }
    s.put('0'); s.put('x');
    for (int k = (67 - __clzll((long long)v)) / 4 - 1; k >= 0; --k) {
        const uint32_t d = (uint32_t)(v >> (4 * k)) & 15u;
        s.put((char)(d < 10 ? '0' + d : 'a' + d - 10));
    }
}

struct AsmCount {
    uint32_t n = 0;
    DEV void put(char) { ++n; }
};

// rvdisasm::disassemble (src/disassembler.cpp:411-451), one line per word for
// rv_generator::print(os, true) (src/codegen/rv_generator.cpp:100-103): before
// a word at a function start a label line (cd + hd + 18 spaces, "func<k>:",
// k in hex after word 0);
// then the word index (decimal, right-aligned in cd columns), three spaces, the
// byte address (hex, zero-padded to hd digits), ": ", the four bytes (hex, high
// byte first), three spaces, the mnemonic left-aligned in 9 columns, a space
// and format_args with colour and the word's address (branch targets are
// absolute).  Colours are the reference's ANSI escapes.
struct AsmList {
    uint64_t first;          // word index of the first word formatted
    const uint32_t *fstarts; // function starts (word indices), sorted, distinct
    uint32_t nf, cd, hd;     // functions; decimal digits of the word count; hex digits of the addresses
};
#define ASM_WHITE "\033[37m"
#define ASM_INSTR "\033[38;5;186m"
#define ASM_REG "\033[38;5;117m"
#define ASM_IMM "\033[38;5;114m"
#define ASM_EXTRA "\033[38;5;114m"
template <class S> DEV void asm_cstr(S &s, const char *p) { while (*p) s.put(*p++); }
// width-padded numbers of the listing's prefix
template <class S> DEV void asm_udec_w(S &s, uint64_t u, uint32_t width, char fill) {
    char b[20];
    int nd = 0;
    do { b[nd++] = (char)('0' + u % 10u); u /= 10u; } while (u);
    for (int k = nd; k < (int)width; ++k) s.put(fill);
    while (nd) s.put(b[--nd]);
}
template <class S> DEV void asm_uhex_w(S &s, uint64_t u, uint32_t width) {
    char b[16];
    int nd = 0;
    do { const uint32_t d = (uint32_t)(u & 15u); b[nd++] = (char)(d < 10 ? '0' + d : 'a' + d - 10); u >>= 4; } while (u);
    for (int k = nd; k < (int)width; ++k) s.put('0');
    while (nd) s.put(b[--nd]);
}

template <bool LIST, class S> DEV void asm_line(S &s, uint32_t w, const AsmList &L, uint64_t idx) {
    const uint32_t op = w & 0x7Fu, f3 = (w >> 12) & 7u, f7 = (w >> 25) & 0x7Fu;
    const uint32_t rd = (w >> 7) & 31u, rs1 = (w >> 15) & 31u, rs2 = (w >> 20) & 31u, rs3 = (w >> 27) & 31u;
    const uint32_t nm = asm_name(w);
    if (LIST) {
        // label: the index of this start among the distinct starts
        uint32_t lo = 0, hi = L.nf;
        while (lo < hi) { const uint32_t m = (lo + hi) >> 1; if (L.fstarts[m] < idx) lo = m + 1; else hi = m; }
        if (lo < L.nf && L.fstarts[lo] == idx) {
            for (uint32_t k = 0; k < L.cd + 3u + L.hd + 2u + 12u + 1u; ++k) s.put(' ');
            // the stream is still in hex from the previous word's line (format_args
            // restores the flags it found), so only a label before word 0 is decimal
            asm_cstr(s, "func");
            if (idx == 0) asm_udec_w(s, lo, 0, ' '); else asm_uhex_w(s, lo, 0);
            s.put(':'); s.put('\n');
        }
        asm_cstr(s, ASM_EXTRA); asm_udec_w(s, idx, L.cd, ' '); asm_cstr(s, ASM_WHITE);
        s.put(' '); s.put(' '); s.put(' ');
        asm_uhex_w(s, 4 * idx, L.hd); s.put(':'); s.put(' ');
        for (int b = 3; b >= 0; --b) {
            s.put(' '); asm_cstr(s, ASM_EXTRA); asm_uhex_w(s, (w >> (8 * b)) & 0xFFu, 2); asm_cstr(s, ASM_WHITE);
        }
        s.put(' '); s.put(' '); s.put(' ');
        asm_cstr(s, ASM_INSTR);
        AsmCount nc;
        asm_str16(nc, c_asm_name[nm]);
        asm_str16(s, c_asm_name[nm]);
        for (uint32_t k = nc.n; k < 9; ++k) s.put(' ');
        asm_cstr(s, ASM_WHITE);
    } else {
        asm_str16(s, c_asm_name[nm]);
    }
    s.put(' ');
    auto X = [&](uint32_t r) { if (LIST) asm_cstr(s, ASM_REG); asm_str8(s, c_asm_x[r]); if (LIST) asm_cstr(s, ASM_WHITE); };
    auto F = [&](uint32_t r) { if (LIST) asm_cstr(s, ASM_REG); asm_str8(s, c_asm_f[r]); if (LIST) asm_cstr(s, ASM_WHITE); };
    auto I0 = [&]() { if (LIST) asm_cstr(s, ASM_IMM); };
    auto I1 = [&]() { if (LIST) asm_cstr(s, ASM_WHITE); };
    auto sep = [&]() { s.put(','); s.put(' '); };
    switch (op) {
        case 0x33:  // R
            X(rd); sep(); X(rs1); sep(); X(rs2);
            break;
        case 0x53:  // R, OP-FP: register files by funct7 (:250-281)
            if (f7 == 0x78 || f7 == 0x68) { F(rd); sep(); X(rs1); }
            else if (f7 == 0x60 || (f7 == 0x70 && f3 == 0)) { X(rd); sep(); F(rs1); }
            else { F(rd); sep(); F(rs1); sep(); F(rs2); }
            break;
        case 0x67: case 0x03: case 0x13: case 0x0F: case 0x73: case 0x07: {  // I
            const int32_t imm = (int32_t)w >> 20;
            if (op == 0x07 || op == 0x03 || op == 0x67) {
                if (op == 0x07) F(rd); else X(rd);
                sep(); I0(); asm_dec(s, imm); I1(); s.put('('); X(rs1); s.put(')');
            } else {
                X(rd); sep(); X(rs1); sep(); I0(); asm_dec(s, imm); I1();
            }
            break;
        }
        case 0x23: case 0x27: {  // S; an fsw names its register by the rs1 field (:357-361)
            const int32_t imm = ((int32_t)(w & 0xFE000000u) >> 20) | (int32_t)((w >> 7) & 0x1Fu);
            if (op == 0x27) F(rs1); else X(rs2);
            sep(); I0(); asm_dec(s, imm); I1(); s.put('('); X(rs1); s.put(')');
            break;
        }
        case 0x63: {  // B: bits 4:1, 9:5 (not 10) and 11, the sign over bits 31:11 (:366-372)
            uint32_t imm = ((w >> 7) & 0x1Eu) | ((w >> 20) & 0x3E0u) | (((w >> 7) & 1u) << 11);
            if (w >> 31) imm |= 0xFFFFF800u;
            const uint64_t addr = LIST ? 4 * idx : 0;
            X(rs1); sep(); X(rs2); sep(); I0(); asm_hex(s, addr + (uint64_t)(int64_t)(int32_t)imm); I1();
            break;
        }
        case 0x37: case 0x17:  // U
            X(rd); sep(); I0(); asm_dec(s, (int32_t)(w & 0xFFFFF000u)); I1();
            break;
        case 0x6F: {  // J: bits 10:1, 11, 19:12, the sign over bits 31:19 (:384-392)
            uint32_t imm = ((w >> 20) & 0x7FEu) | (((w >> 20) & 1u) << 11) | (w & 0xFF000u);
            if (w >> 31) imm |= 0xFFF80000u;
            X(rd); sep(); I0(); asm_dec(s, (int32_t)imm); I1();
            break;
        }
        case 0x43: case 0x47: case 0x4B: case 0x4F:  // R4 (integer names, :395-403)
            X(rd); sep(); X(rs1); sep(); X(rs2); sep(); X(rs3);
            break;
        default:
            break;
    }
    s.put('\n');
}

// Writes bytes from pos on; a 4-byte word lying inside [lo, hi) (the thread's
// own lines) goes out as one store, the bytes of a word shared with a
// neighbour's lines one by one.
struct AsmWrite {
    uint8_t *out;
    uint64_t pos, lo, hi;
    uint32_t acc = 0;
    DEV void put(char ch) {
        const uint64_t wb = pos & ~3ull;
        if (wb >= lo && wb + 4 <= hi) {
            acc |= (uint32_t)(uint8_t)ch << (8u * (uint32_t)(pos & 3u));
            if ((pos & 3u) == 3u) { *reinterpret_cast<uint32_t *>(out + wb) = acc; acc = 0; }
        } else {
            out[pos] = (uint8_t)ch;
        }
        ++pos;
    }
};

// line lengths: formatted once with a counting sink (the tile sums), kept per
// word for the rescan (one byte for to_asm lines, two for listing lines)
template <bool LIST>
struct AsmLenOp {
    using Len = typename std::conditional<LIST, uint16_t, uint8_t>::type;
    const uint32_t *w;
    Len *len;
    AsmList L;
    DEV uint32_t value(uint64_t i) const {
        AsmCount c;
        asm_line<LIST>(c, w[i], L, L.first + i);
        len[i] = (Len)c.n;
        return c.n;
    }
    DEV void emit(uint64_t, uint32_t, uint32_t) const {}
};
template <class Len>
struct AsmLenRead {
    const Len *len;
    DEV uint32_t value(uint64_t i) const { return len[i]; }
};

template <bool LIST>
__global__ __launch_bounds__(SCAN_BLOCK) void k_asm_write(const uint32_t *w, const typename AsmLenOp<LIST>::Len *lens,
                                                          uint64_t n, const uint32_t *tile_pre, uint8_t *out, AsmList L) {
    __shared__ uint32_t s_w[SCAN_BLOCK / 64];
    __shared__ uint32_t s_v[SCAN_TILE + SCAN_TILE / 16];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    const uint32_t run = scan_tile(AsmLenRead<typename AsmLenOp<LIST>::Len>{lens}, n, tile_pre, s_w, s_v, v);
    uint32_t len = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) len += v[k];
    AsmWrite s{out, run, run, (uint64_t)run + len};
    for (int k = 0; k < SCAN_ITEMS; ++k)
        if (base + k < n) asm_line<LIST>(s, w[base + k], L, L.first + base + k);
}

// ================================================================ host side
#include "ptl_host.inc"
