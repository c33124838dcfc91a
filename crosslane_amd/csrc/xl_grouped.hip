// CDNA4 (gfx950) grouped routed-expert path: T tokens, each with its own k
// picks, reading every touched expert's weights once per task of its (token,
// pick) pairs. The result is that of T independent layer calls
// (WarmRedirect::warm_compute_many per token, engine/strata/warm/runtime.hpp:13,
// then the fixed-order join of runtime.cpp:183-188): per (row, pair) the same
// exact integer block partials and the same fp16(d) * d_x fma over blocks in
// block order as the row kernels.
//
//   bucket_kernel    one workgroup: pairs bucketed by expert id into tasks of
//                    at most 16 or 64 pairs of one expert
//   q8k_rows_kernel  Q8_K (q8k_core.hpp:30-38) of token rows (x) and pair rows
//                    (h), written in the operand order of the MFMA kernels
//   grouped_kernel   gate/up + SwiGLU of every task, then down of every task
//   gcombine_kernel  fixed-order combine per token, + shared
//
// MFMA: v_mfma_i32_16x16x32_i8 with M = pairs, N = weight rows, K = the 32
// weights of one sub-block. Lane l supplies A[l % 16][8 (l / 16) .. + 7] (8
// quants of pair l % 16), B[8 (l / 16) .. + 7][l % 16] (grid entry l / 16 of
// row l % 16: 8 weights) and receives D[4 (l / 16) + r][l % 16], r = 0..3. The
// lane that decodes a row's entry therefore also holds that row's outputs and
// applies the row's sub-block scale (2s + 1) to them as integers: the block
// partials are exact. Any K order works as long as A and B agree, which the
// chunk-major activation layouts below guarantee.
//
// IQ1_M needs neither: its sub-scale (2s + 1 <= 15) times its grid value (-1, 0, 1)
// is an int8 (the LDS table holds byte selectors, v_perm picks the scale, its
// negative or zero by them), so that a block's eight MFMAs accumulate into one
// result, and any lane may hold any of the block's entries (lane group e4 keeps
// values 64 e4 .. + 63: the activations have an order of their own). The delta term, (2s + 1) * (+-1) times
// the sum of an entry's 8 quants, is a product over the block's 32 entries: two
// more MFMAs on those sums (11 bits, split 16 hi + lo by the quantizer).
//
// Work: a wave takes one tile at a time, two streams of 16 rows that share the
// activations (gate and up rows, or 32 down rows; 16 where tiles are few), from its
// workgroup's current bundle; a wave that finds the bundle empty fetches the next one from the
// device's queue of the type. Waves never wait for each other inside a type (a
// workgroup barrier per item left every wave waiting for the item's chain of
// dependent loads: task, matrix, scales, weights). A layer of several types has
// one queue per type; a workgroup starts with the type its place in the grid falls
// on (by estimated cost) and goes on with the others' remainders, each after
// filling its LDS tables for that type.
//
// Weights stream from HBM through registers: each wave loads its rows' next block
// while it computes the current one (one dword per row that touched the line four
// blocks ahead made calls up to 22 % slower: 13 tokens, 384 experts; the other waves
// cover the latency). The texture data path costs one cycle per cache access, and a
// quad of lanes makes one access only when it reads 64 contiguous bytes: so each lane
// loads just the 16 B of its row's block that it decodes (the entries then move
// between lane groups by permlane swaps), activations are laid out so that a quad's
// four slots are adjacent, and the small per-block scales are staged once per tile in
// the wave's own LDS. An IQ1_M lane needs 8, 4 and 8 bytes of three planes per block:
// loaded directly, those kept the texture unit busy for the whole kernel (1,415 us for
// gate/up of 512 tokens at 4096 x 3072, 384 experts), so four blocks of the 16 rows
// come as whole 16-byte pieces and go through the wave's LDS.
//
// Bound by the decode work per weight byte: at 512 tokens (4096 x 3072, 384 experts,
// 6 picks, IQ2) VALU issue takes 79 % of the gate/up launch's SIMD cycles (765 us) and
// 71 % of the down launch's (531), LDS 36 % of its cycles in both; at 2,048 tokens, by
// 64 pairs, 82 and 84 %. Whole calls at 512 tokens: IQ2 1,307 to 1,350 us, IQ1_M 1,149,
// mixed types 1,335 (10,999 and 12,992 as 512 layer calls).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "xl_dev.hpp"
#include "xl_format.hpp"
#include "xl_internal.hpp"

namespace xl::dev {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kTile = 16;   // pairs per tile (the MFMA M dimension)
// GroupArgs::pos: slot of a pair, and whether its x / h go there in the IQ1_M order.
constexpr int kSlotX1 = 1 << 30, kSlotH1 = 1 << 29, kSlotMask = kSlotH1 - 1;
// Tasks hold up to 64 pairs, in kernels of 8 waves (2 per SIMD: their registers), from
// kMultiPairs pairs per expert on (several types: kMultiPairsMix) if that leaves more
// than kMultiTiles tiles per workgroup, or half of them and four times the pairs. 4096
// x 3072, 384 experts, IQ2: 12 per expert 1,582 us, 32 per expert 2,341 us (3,075 by
// 16-pair tasks); 11 per expert 1,587 against 1,548, 8 per expert 1,528 against 1,449.
// With few tiles the pairs of a task are a chain that idle waves could have shared: 256
// tokens of one pick over 8 experts (6 tiles) 104.6 us against 94.5, 1024 x 512, 64
// tokens of 8 over 8 experts (1 tile) 45.0 against 40.1, but 512 tokens there (8 tiles)
// 69.7 against 103.1, and 5120 x 2304, 512 tokens of one over 8 (5 tiles, 64 per expert)
// 129.2 against 158.1. Several types: 12 per expert 357 against 347 us, 24 454 and 502.
// IQ1_M decodes faster and gains earlier: 128 tokens of 2 over 8 experts (6 tiles) 84.1
// against 96.9, 5120 x 2304, 32 of 6 over 8 (5 tiles) 76.0 against 81.0.
constexpr int kMultiPairs = 12, kMultiPairsMix = 16, kMultiTiles = 6, kMultiTilesIQ1 = 4;
// Relative cost of a tile by type (XXS, XS, IQ1_M), for the first share of a mixed
// layer's workgroups (the queues even out what it misses).
__device__ constexpr int kTileCost[3] = {10, 11, 8};
// Expanded codebook tables (layer_tables() in xl_api.cpp): 128 sign entries of
// 16 B (byte mask, then the mask's low bits), the IQ2_XXS grid (256 x 8 B), the
// IQ2_XS grid (512 x 8 B).
constexpr int kTabSgn = 0, kTabXXS = 2048, kTabXS = 4096;

// LDS tables of one type (128 KB). IQ2: grid entries as 16 B (g, -g) in C copies
// per entry (lane copy = lane % C, so the 16 lanes of one ds_read_b128 pass never
// share a bank), then sign masks as 8 B in 32 copies (the 32 lanes of one
// ds_read_b64 pass never share a bank) indexed by a whole byte whose top bit is not
// a sign bit. IQ1_M (16 KB): the grid as 8 B of v_perm selectors (0: 1, 1: -1, 0x0C: 0).
constexpr int kL_GRID = 0, kL_SGN = 65536, kL_TAB = 131072, kL_TAB1 = 16384;
constexpr int kTabIQ1 = 8192;   // IQ1 grid in the expanded tables
// Then each wave's staging: its tile's 16 pairs' activation scales [block][tile
// position] (f32), then its two streams' fp16 row scales [row][block].
constexpr int kGrpNb = kMaxRowK / 256;
constexpr int kL_WAVE = 64 * kGrpNb + 2 * 16 * kGrpNb * 2;
// IQ1_M waves: the activation scales, then per stream four blocks of 16 rows:
// [block][row] 32 B of indices, then 16 B of nibbles, then 8 B of scale words.
// (block strides a quarter more than the 512, 256 and 128 bytes: the pieces of one
// store then fall into different banks)
constexpr int kR1q = 576, kR1h = 320, kR1s = 192, kR1ho = 4 * kR1q, kR1so = kR1ho + 4 * kR1h;
constexpr int kRaw1 = kR1so + 4 * kR1s, kL_WAVE1 = 64 * kGrpNb + 2 * kRaw1;
constexpr int grp_lds_bytes(int mask, int nw) {
    const int iq2 = mask & 3 ? kL_TAB + nw * kL_WAVE : 0, iq1 = mask & 4 ? kL_TAB1 + nw * kL_WAVE1 : 0;
    return iq2 > iq1 ? iq2 : iq1;
}
static_assert(grp_lds_bytes(7, 12) + 64 <= 160 * 1024, "LDS budget");
constexpr int kCopiesXXS = 16;   // 256 entries x 256 B: the entry byte lands in address byte 1
constexpr int kCopiesXS = 8;     // 512 entries x 128 B: the 9-bit entry lands at address bit 7

// Values every lane of the wave holds alike, moved to scalar registers (buffer
// descriptors built from them stay scalar: no waterfall loops).
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const uint8_t* uni(const uint8_t* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v)), hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return reinterpret_cast<const uint8_t*>((uint64_t(hi) << 32) | lo);
}
__device__ __forceinline__ int4 task_at(const int4* tasks, int i) {
    const int4 t = tasks[i];
    return make_int4(uni(t.x), uni(t.y), uni(t.z), 0);
}
__device__ __forceinline__ MatRef mat_at(const ExpertDesc* d, int e, int role) {
    const MatRef m = d[e].m[role];
    MatRef u;
    u.base = uni(m.base);
    u.off1 = (uint64_t(uint32_t(uni(int(m.off1 >> 32)))) << 32) | uint32_t(uni(int(uint32_t(m.off1))));
    u.off2 = (uint64_t(uint32_t(uni(int(m.off2 >> 32)))) << 32) | uint32_t(uni(int(uint32_t(m.off2))));
    u.type = uni(m.type);
    u.nb = uni(m.nb);
    return u;
}

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t x, uint32_t y) { return (m & x) | (~m & y); }
__device__ __forceinline__ long pack64(uint32_t lo, uint32_t hi) {
    return static_cast<long>((uint64_t(hi) << 32) | lo);
}
__device__ __forceinline__ v4i mfma(long a, long b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int mad24(int a, int b, int c) {   // v_mad_i32_i24
    // the opaque result keeps the add from merging into a v_add3 (mul + add3 per
    // pair of terms instead of one mad each)
    int r = __mul24(a, b) + c;
    asm volatile("" : "+v"(r));
    return r;
}
// Bytewise negation of grid bytes (all in 1..127, so no byte borrows).
__device__ __forceinline__ uint64_t neg_grid(uint64_t g) { return ~g + 0x0101010101010101ull; }

// Sign tables: 256 rows (row r = sign entry r & 127) x 32 copies x 8 B.
__device__ __forceinline__ void fill_signs(uint8_t* lds, const uint64_t* tab, int t, int nt) {
    for (int i = t; i < 256 * 32; i += nt)
        *reinterpret_cast<uint64_t*>(lds + kL_SGN + 8 * i) = tab[kTabSgn / 8 + 2 * ((i >> 5) & 127)];
}
// Grid tables: E entries x C copies x 16 B (g, -g).
template <int E, int C>
__device__ __forceinline__ void fill_grid(uint8_t* lds, const uint64_t* grid, int t, int nt) {
    for (int i = t; i < E * C; i += nt) {
        const uint64_t g = grid[i / C], n = neg_grid(g);
        *reinterpret_cast<uint4*>(lds + kL_GRID + 16 * i) =
            make_uint4(uint32_t(g), uint32_t(g >> 32), uint32_t(n), uint32_t(n >> 32));
    }
}

// The tables of block type ty.
template <int NT>
__device__ __forceinline__ void fill_tables(uint8_t* lds, int ty, const uint64_t* tab, int t) {
    if (ty == kIQ2_XXS) {
        fill_grid<256, kCopiesXXS>(lds, tab + kTabXXS / 8, t, NT);
        fill_signs(lds, tab, t, NT);
    } else if (ty == kIQ2_XS) {
        fill_grid<512, kCopiesXS>(lds, tab + kTabXS / 8, t, NT);
        fill_signs(lds, tab, t, NT);
    } else {
        constexpr uint64_t kOnes = 0x0101010101010101ull;
        for (int i = t; i < 2048; i += NT) {
            const uint64_t g = tab[kTabIQ1 / 8 + i], n = (g >> 1) & kOnes;   // bytes 0xff
            *reinterpret_cast<uint64_t*>(lds + 8 * i) = (kOnes ^ (g & kOnes)) * 0x0Cu + n;
        }
    }
}

// ---------------------------------------------------------------------------
// Buckets: counts per expert in LDS, one scan of tiles and tasks, then each valid
// pair takes a slot of its expert's tiles (tile i: slots 16 i .. + 15). A task is
// up to a.cap pairs of one expert, in consecutive tiles. The tasks are listed
// twice, by the expert's gate type and by its down type (kIQ2_XXS, kIQ2_XS,
// kIQ1_M in turn), each list's type counts beside it. The slot order inside an
// expert varies run to run; no result depends on it (every output of a pair is
// computed from that pair's operands only, in a fixed order).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int type_index(int t) { return t == kIQ2_XXS ? 0 : t == kIQ2_XS ? 1 : 2; }
// One count per type in 21 bits each (tasks of a call are below 2^17).
__device__ __forceinline__ uint64_t type_count(int ti, int n) { return uint64_t(uint32_t(n)) << (21 * ti); }
__device__ __forceinline__ int type_part(uint64_t v, int ti) { return int((v >> (21 * ti)) & 0x1fffff); }
// Inclusive scan over the workgroup's 1024 threads; sh: 17 words (the total last).
__device__ __forceinline__ uint64_t scan1024(uint64_t v, uint64_t* sh, int t) {
    const int lane = t & 63, wv = t >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    __syncthreads();   // an earlier scan's words are read
    if (lane == 63) sh[wv] = v;
    __syncthreads();
    uint64_t before = 0;
    for (int i = 0; i < wv; ++i) before += sh[i];
    v += before;
    if (t == 1023) sh[16] = v;
    __syncthreads();
    return v;
}
__global__ __launch_bounds__(1024) void bucket_kernel(GroupArgs a) {
    __shared__ int cnt[kGroupMaxExperts];
    __shared__ int cur[kGroupMaxExperts];
    __shared__ uint64_t sh[17];
    const int t = threadIdx.x, P = a.T * a.k, E = a.n_experts;
    // this thread's first expert's types, loaded under the counting
    const int ef = min(E - 1, t * ((E + 1023) / 1024));
    const int g_first = a.descs[ef].m[0].type, d_first = a.descs[ef].m[2].type;
    for (int e = t; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int p = t; p < P; p += 1024) {
        const int e = a.ids[p];
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
        else atomicOr(a.err, kDevErrExpertId);
    }
    __syncthreads();
    const auto gate_type = [&](int e) { return type_index(e == ef ? g_first : a.descs[e].m[0].type); };
    const auto down_type = [&](int e) { return type_index(e == ef ? d_first : a.descs[e].m[2].type); };
    const int per = (E + 1023) / 1024, e0 = min(E, t * per), e1 = min(E, e0 + per);
    uint64_t tiles = 0, gu = 0, dn = 0;
    for (int e = e0; e < e1; ++e) {
        const int c = cnt[e], n = (c + a.cap - 1) / a.cap;
        tiles += uint64_t((c + kTile - 1) / kTile) | (uint64_t(n) << 32);
        gu += type_count(gate_type(e), n);
        dn += type_count(down_type(e), n);
    }
    const uint64_t tt = scan1024(tiles, sh, t) - tiles;   // tiles, tasks << 32
    int tile = int(uint32_t(tt));
    uint64_t g_at, g_all, d_at, d_all;
    if (a.gu_first && a.dn_first) {   // one type each: their lists are the tasks in turn
        const int gt = type_index(g_first), dt = type_index(d_first);
        g_at = type_count(gt, int(tt >> 32));
        d_at = type_count(dt, int(tt >> 32));
        g_all = type_count(gt, int(sh[16] >> 32));
        d_all = type_count(dt, int(sh[16] >> 32));
    } else {
        g_at = scan1024(gu, sh, t) - gu;
        g_all = sh[16];
        d_at = scan1024(dn, sh, t) - dn;
        d_all = sh[16];
    }
    // the types' lists one after the other
    const uint64_t g0 = type_count(1, type_part(g_all, 0)) + type_count(2, type_part(g_all, 0) + type_part(g_all, 1));
    const uint64_t d0 = type_count(1, type_part(d_all, 0)) + type_count(2, type_part(d_all, 0) + type_part(d_all, 1));
    g_at += g0;
    d_at += d0;
    for (int e = e0; e < e1; ++e) {
        const int c = cnt[e];
        const int gt = gate_type(e), dt = down_type(e);
        // the expert's first slot; its pairs fill its tiles' slots in turn. Bits 30
        // and 29: x and h in the IQ1_M order
        cur[e] = (kTile * tile) | (gt == 2 ? kSlotX1 : 0) | (dt == 2 ? kSlotH1 : 0);
        for (int i = 0; i * a.cap < c; ++i) {
            const int4 task = make_int4(e, kTile * tile, min(a.cap, c - a.cap * i), 0);
            a.tasks[type_part(g_at, gt)] = task;
            a.dtasks[type_part(d_at, dt)] = task;
            g_at += type_count(gt, 1);
            d_at += type_count(dt, 1);
            tile += (task.z + kTile - 1) / kTile;
        }
    }
    if (t < 3) {
        a.queue->gu_tasks[t] = type_part(g_all, t);
        a.queue->dn_tasks[t] = type_part(d_all, t);
        a.queue->gu_next[t] = a.gu_first;
        a.queue->dn_next[t] = a.dn_first;
    }
    __syncthreads();
    for (int p = t; p < P; p += 1024) {
        const int e = a.ids[p];
        int slot = -1;
        if (e >= 0 && e < E) {
            slot = atomicAdd(&cur[e], 1);   // consecutive per expert: its tiles' slots have no gaps before the last
            a.order[slot & kSlotMask] = p;
        }
        a.pos[p] = slot;
    }
}

// ---------------------------------------------------------------------------
// Q8_K of 256-value blocks of rows, one wave per block, written to the slots of
// the row's pairs (ROWS_X: a token row goes to its k pairs' slots; ROWS_H: a
// pair row to its slot; bad ids have none) in the operand order of the MFMA
// kernels. A tile's slots form one region of nb * 4 KiB, in which, per block b, the
// 16-B piece i of chunk e of slot s sits at ((4 b + i) * 4 + e) * 256 + 16 s, so that
// four lanes of consecutive slots read 64 contiguous bytes. IQ2 order: piece i of
// chunk e is the 8 quants of entry e of sub-blocks 2i and 2i + 1. IQ1_M order: chunk e
// is values 64 e .. + 63, piece i 16 of them; and in a region of their own, nb KiB per
// tile (which only banks with IQ1_M have), the sums S of each 8 values as S = 16 hi +
// lo: slot s's 16 bytes at (4 b + e) * 256 + 16 s hold lo, then hi, of chunk e's entries 0, 2,
// 4, 6, 1, 3, 5, 7. The block scale goes to the tile's [block][slot] floats.
// ---------------------------------------------------------------------------
// The j-th pair of a tile (slot 16 i + j) sits at tile position 4 (j % 4) + j / 4
// (M index of the MFMAs; the map is its own inverse): the lane holding M rows
// 4 e + r, r = 0..3, gets pairs 4 r + e, so a tile of n pairs has results only
// in the lanes' first ceil(n / 4) output registers.
__device__ __forceinline__ int tile_pos(int j) { return ((j & 3) << 2) | (j >> 2); }
__device__ __forceinline__ size_t tile_off(int tile, int nb) { return size_t(tile) * size_t(nb) * 4096; }
__device__ __forceinline__ size_t sum_off(int tile, int nb) { return size_t(tile) * size_t(nb) * 1024; }
enum { ROWS_X = 0, ROWS_H = 1 };
// trace (null outside the parity trace): the row's blocks also as 292-byte Q8_K
// blocks, row-major (a token's for ROWS_X, a pair's for ROWS_H).
// IQ1: some slots may be in the IQ1_M order.
template <int MODE, bool IQ1, bool TR>
__global__ __launch_bounds__(256) void q8k_rows_kernel(const float* __restrict__ src, int rows, int nb,
                                                       int8_t* __restrict__ q, int8_t* __restrict__ sums,
                                                       float* __restrict__ d, const int32_t* __restrict__ pos, int k,
                                                       int* __restrict__ err, uint8_t* __restrict__ trace) {
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= rows * nb) return;   // wave-uniform
    const int row = b / nb, blk = b - row * nb;
    if (MODE == ROWS_H && pos[row] < 0) return;
    const int lane = threadIdx.x & 63;
    const float4 v4 = reinterpret_cast<const float4*>(src + size_t(b) * 256)[lane];
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    const Q8Lane r = q8k_lane(v, lane);
    if (!r.finite && lane == 0) atomicOr(err, kDevErrNonFinite);
    // values 4 lane .. + 3 in the IQ2 order: sub-block c, entry e
    const int c = lane >> 3, e = (lane >> 1) & 3;
    const int o2 = ((4 * blk + (c >> 1)) * 4 + e) * 256 + 8 * (c & 1) + 4 * (lane & 1);
    // in the IQ1_M order: chunk lane / 16, piece (lane / 4) % 4; its entry's sum
    const int o1 = ((4 * blk + ((lane >> 2) & 3)) * 4 + (lane >> 4)) * 256 + 4 * (lane & 3);
    int sum = __builtin_amdgcn_sdot4(int(r.packed), 0x01010101, 0, false);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, false);   // lane ^ 1: the entry's 8 values
    const int j = (lane >> 1) & 7, lo = ((sum + 8) & 15) - 8, hi = (sum - lo) >> 4;
    const int os = (4 * blk + (lane >> 4)) * 256 + (j >> 1) + 4 * (j & 1);
    const int np = MODE == ROWS_X ? k : 1;
    for (int i = 0; i < np; ++i) {
        const int slot = pos[MODE == ROWS_X ? row * k + i : row];
        if (slot < 0) continue;
        const int s = slot & kSlotMask, tp = tile_pos(s & 15);
        int8_t* t = q + tile_off(s >> 4, nb) + 16 * tp;
        if (IQ1 && (slot & (MODE == ROWS_X ? kSlotX1 : kSlotH1))) {
            *reinterpret_cast<uint32_t*>(t + o1) = r.packed;
            if (!(lane & 1)) {
                int8_t* ts = sums + sum_off(s >> 4, nb) + 16 * tp + os;
                ts[0] = int8_t(lo);
                ts[8] = int8_t(hi);
            }
        } else {
            *reinterpret_cast<uint32_t*>(t + o2) = r.packed;
        }
        if (lane == 0) d[(size_t(s >> 4) * nb + blk) * 16 + tp] = r.d;
    }
    if constexpr (TR) {
        if (trace) trace_q8_block(trace + size_t(b) * 292, r.d, r.packed, lane);
    }
}

// Buffer loads: the base in a scalar descriptor, the per-lane byte offset in
// voffset, a uniform plane offset in soffset.
typedef uint32_t v4u32 __attribute__((ext_vector_type(4)));
typedef uint32_t v2u32 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00020000);
}
__device__ __forceinline__ uint4 ld128(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t so = 0) {
    const v4u32 q = __builtin_amdgcn_raw_buffer_load_b128(r, v, so, 0);
    return make_uint4(q.x, q.y, q.z, q.w);
}
__device__ __forceinline__ uint2 ld64(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t so = 0) {
    const v2u32 q = __builtin_amdgcn_raw_buffer_load_b64(r, v, so, 0);
    return make_uint2(q.x, q.y);
}
__device__ __forceinline__ uint32_t ld32(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t so = 0) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, v, so, 0);
}
__device__ __forceinline__ uint16_t ld16(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t so = 0) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, v, so, 0);
}

// Exchanges across the four 16-lane groups (e4 = lane / 16) of a wave.
__device__ __forceinline__ void swap32(uint32_t& x, uint32_t& y) {   // lanes 32.. of x <-> lanes ..31 of y
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
__device__ __forceinline__ void swap16(uint32_t& x, uint32_t& y) {   // odd groups of x <-> even groups of y
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
// v[j] of group g -> v[g] of group j, lane by lane within the groups.
__device__ __forceinline__ void xpose4(uint32_t (&v)[4]) {
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}
// Every group's byte x (placed at byte e4 by the caller) in every group.
__device__ __forceinline__ uint32_t gather4(uint32_t x) {
    uint32_t y = x;
    swap32(x, y);
    x |= y;
    y = x;
    swap16(x, y);
    return x | y;
}

// IQ2_XXS block of the MFMA lane (col, e4) from 16-B parts: lane (col, g) loaded
// bytes 16 g .. + 15 of row col's block (sub-blocks 2g and 2g + 1: grid bytes,
// then aux bytes = 7 sign bits | scale bit k in byte k). Afterwards u[j] holds
// {grid, aux} bytes of entry e4 of sub-blocks 2j (bytes 0, 1) and 2j + 1 (bytes
// 2, 3), and byte j of ls[c & 1] holds sub-block c = 2j + (c & 1)'s factor
// 2 s + 1 (s its 4-bit scale).
struct XxsLane {
    uint32_t u[4], ls[2];
};
__device__ __forceinline__ XxsLane xxs_lane(const uint4& w, int e4) {
    const uint32_t p01 = perm(w.y, w.x, 0x05010400u), p01b = perm(w.y, w.x, 0x07030602u);
    const uint32_t p23 = perm(w.w, w.z, 0x05010400u), p23b = perm(w.w, w.z, 0x07030602u);
    XxsLane r;
    r.u[0] = perm(p23, p01, 0x05040100u);    // entry 0 of both sub-blocks
    r.u[1] = perm(p23, p01, 0x07060302u);
    r.u[2] = perm(p23b, p01b, 0x05040100u);
    r.u[3] = perm(p23b, p01b, 0x07060302u);
    xpose4(r.u);
    const uint32_t sa = __builtin_amdgcn_udot4((w.y >> 7) & 0x01010101u, 0x08040201u, 0u, false);
    const uint32_t sb = __builtin_amdgcn_udot4((w.w >> 7) & 0x01010101u, 0x08040201u, 0u, false);
    const uint32_t s = gather4((sa | (sb << 4)) << (8 * e4));   // sub-block c's scale at bits 4c .. 4c + 3
    r.ls[0] = ((s << 1) & 0x1E1E1E1Eu) | 0x01010101u;
    r.ls[1] = ((s >> 3) & 0x1E1E1E1Eu) | 0x01010101u;
    return r;
}
// IQ2_XS block of the MFMA lane (col, e4) from 16-B parts, as xxs_lane: u[j]
// holds the 16-bit code (9-bit grid index at bits 7..15, sign bits 0..6) of
// entry e4 of sub-block 2j (low half) and 2j + 1 (high half).
__device__ __forceinline__ void xs_lane(const uint4& w, uint32_t (&u)[4]) {
    u[0] = perm(w.z, w.x, 0x05040100u);
    u[1] = perm(w.z, w.x, 0x07060302u);
    u[2] = perm(w.w, w.y, 0x05040100u);
    u[3] = perm(w.w, w.y, 0x07060302u);
    xpose4(u);
}

// One stream (16 rows) of a tile: where its blocks are. Lane (col, e4) holds row
// row0 + col; at = that row's first block.
struct Stream {
    __amdgpu_buffer_rsrc_t r;
    uint32_t at;          // row * nb
    uint32_t o1, o2;      // plane offsets
};
// A lane's raw words of one block of one stream: IQ2_XXS q = 16-B part e4 of the
// row's block; IQ2_XS also s = the block's 8 scale bytes; IQ1_M (from LDS) q.xy = the
// 8 low index bytes of values 64 e4 .. + 63, q.z their 8 nibbles, s = the scale words.
struct Raw {
    uint4 q;
    uint2 s;
};
template <int TY>
__device__ __forceinline__ void load_raw(Raw& o, const Stream& st, int blk, int e4) {
    const uint32_t b = st.at + uint32_t(blk);
    o.q = ld128(st.r, 64u * b + 16u * e4);
    if constexpr (TY == kIQ2_XS) o.s = ld64(st.r, 8u * b, st.o1);
}
// Four IQ1_M blocks (blk0 .. + 3, past the row's end the last one) of a stream's 16
// rows, as pieces: row0nb = the stream's first row * nb.
struct Raw1 {
    uint4 q[2], h;
    uint2 s;
};
__device__ __forceinline__ void load_raw1(Raw1& o, const Stream& st, uint32_t row0nb, int blk0, int nb, int lane) {
    const int bq = min(blk0 + ((lane >> 1) & 3), nb - 1), bh = min(blk0 + (lane & 3), nb - 1);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        o.q[i] = ld128(st.r, 32u * (row0nb + uint32_t((8 * i + (lane >> 3)) * nb + bq)) + 16u * (lane & 1));
    const uint32_t b = row0nb + uint32_t((lane >> 2) * nb + bh);
    o.h = ld128(st.r, 16u * b, st.o1);
    o.s = ld64(st.r, 8u * b, st.o2);
}
__device__ __forceinline__ void store_raw1(uint8_t* p, const Raw1& o, int lane) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
        *reinterpret_cast<uint4*>(p + kR1q * ((lane >> 1) & 3) + 32 * (8 * i + (lane >> 3)) + 16 * (lane & 1)) = o.q[i];
    *reinterpret_cast<uint4*>(p + kR1ho + kR1h * (lane & 3) + 16 * (lane >> 2)) = o.h;
    *reinterpret_cast<uint2*>(p + kR1so + kR1s * (lane & 3) + 8 * (lane >> 2)) = o.s;
}
__device__ __forceinline__ void read_raw1(Raw& o, const uint8_t* p, int i, int col, int e4) {   // block i of the four
    const uint2 q = *reinterpret_cast<const uint2*>(p + kR1q * i + 32 * col + 8 * e4);
    o.q.x = q.x;
    o.q.y = q.y;
    o.q.z = *reinterpret_cast<const uint32_t*>(p + kR1ho + kR1h * i + 16 * col + 4 * e4);
    o.s = *reinterpret_cast<const uint2*>(p + kR1so + kR1s * i + 8 * col);
}

// Decoded block of one stream: the MFMA operands of its eight steps and what
// scales their results. IQ2: step c is sub-block c (32 weights), B its signed
// grid bytes; XXS: byte c >> 1 of s[c & 1] its factor 2 s + 1; XS: byte c & 3 of
// s[c >> 2] the factor ls2 of entries 2, 3 and of s[2 + (c >> 2)], signed, ls1 - ls2.
// IQ1_M: step j is entry j of the lane's 64 values, B scaled; D the factors
// (2 s + 1) * delta of those entries, in the order of the activations' sums.
struct Dec {
    long B[8];
    uint32_t s[4];
    long D;
    float d;   // IQ1_M: the block's fp16 scale
};
template <int TY>
__device__ __forceinline__ void decode(Dec& o, const Raw& w, const uint8_t* lds, int lane, int e4) {
    if constexpr (TY == kIQ2_XXS) {
        const uint32_t lo_g = uint32_t(lane & (kCopiesXXS - 1)) << 4;        // kL_GRID = 0
        const uint32_t lo_s = (uint32_t(lane & 31) << 3) | (1u << 16);       // kL_SGN = 1 << 16
        const XxsLane X = xxs_lane(w.q, e4);
        o.s[0] = X.ls[0];
        o.s[1] = X.ls[1];
#pragma unroll
        for (int c = 0; c < 8; ++c) {   // grid byte -> address byte 1, then the aux byte
            const uint32_t u = X.u[c >> 1], h = uint32_t(c & 1) * 2u;
            const uint4 g = *reinterpret_cast<const uint4*>(lds + perm(u, lo_g, 0x0C020000u | ((4u + h) << 8)));
            const uint2 m = *reinterpret_cast<const uint2*>(lds + perm(u, lo_s, 0x0C020000u | ((5u + h) << 8)));
            o.B[c] = pack64(bfi(m.x, g.z, g.x), bfi(m.y, g.w, g.y));
        }
    } else if constexpr (TY == kIQ2_XS) {
        const uint32_t lo_x = uint32_t(lane & (kCopiesXS - 1)) << 4;
        const uint32_t lo_s = (uint32_t(lane & 31) << 3) | (1u << 16);
        // Scale byte c holds nibbles lo (entries 0, 1) and hi (entries 2, 3): ls2 =
        // 2 hi + 1 and ls1 - ls2 = 2 (lo - hi); 128 + 2 lo - 2 hi never borrows.
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t v = h ? w.s.y : w.s.x;
            const uint32_t hi2 = (v >> 3) & 0x1E1E1E1Eu, lo2 = (v << 1) & 0x1E1E1E1Eu;
            o.s[h] = hi2 | 0x01010101u;
            o.s[2 + h] = ((lo2 | 0x80808080u) - hi2) ^ 0x80808080u;
        }
        uint32_t u[4];
        xs_lane(w.q, u);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint32_t v = u[c >> 1], code = (c & 1) ? v >> 16 : v;
            const uint4 g = *reinterpret_cast<const uint4*>(lds + ((code & 0xff80u) | lo_x));
            const uint2 m = *reinterpret_cast<const uint2*>(lds + perm(v, lo_s, (c & 1) ? 0x0C020600u : 0x0C020400u));
            o.B[c] = pack64(bfi(m.x, g.z, g.x), bfi(m.y, g.w, g.y));
        }
    } else {
        // the lane's scale word: s of entries 2k, 2k + 1 at bits 3k; f = those four 2s + 1 as bytes
        const uint32_t sw = ((e4 & 2) ? w.s.y : w.s.x) >> (16 * (e4 & 1));
        const uint32_t f = ((sw << 1) & 0xEu) | ((sw << 6) & 0xE00u) | ((sw << 11) & 0xE0000u) | ((sw << 16) & 0xE000000u) | 0x01010101u;
        const uint32_t nf = ~f + 0x01010101u;   // -(2s + 1) bytewise (f >= 1: no carry)
        const uint32_t h = w.q.z;   // byte k: nibbles of entries 2k (low) and 2k + 1
        const uint32_t te = h & 0x07070707u, to = (h >> 4) & 0x07070707u;   // index bits 8..10
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t q = j < 4 ? w.q.x : w.q.y, t = (j & 1) ? to : te;
            const uint32_t row = perm(t, q, 0x0C0C0000u | uint32_t(j & 3) | ((4u + uint32_t(j >> 1)) << 8));
            const uint2 g = *reinterpret_cast<const uint2*>(lds + (row << 3));
            const uint32_t sc = perm(nf, f, 0x0C0C0000u | uint32_t(j >> 1) | ((4u + uint32_t(j >> 1)) << 8));   // 2s + 1, -(2s + 1)
            o.B[j] = pack64(perm(0u, sc, g.x), perm(0u, sc, g.y));
        }
        const uint32_t ne = (h >> 3) & 0x01010101u, no = (h >> 7) & 0x01010101u;   // delta -1
        const uint32_t me = (ne << 8) - ne, mo = (no << 8) - no;
        o.D = pack64(bfi(me, nf, f), bfi(mo, nf, f));
        const uint32_t d16 = ((w.s.x >> 12) & 15u) | ((w.s.x >> 24) & 0xf0u) | ((w.s.y >> 4) & 0xf00u) | ((w.s.y >> 16) & 0xf000u);
        o.d = h2f(d16);
    }
}
// A block's activations of one tile, a lane's chunk: the four pieces, and IQ1_M's sums.
template <int TY>
struct Act {
    uint4 a[TY == kIQ1_M ? 5 : 4];
};
template <int TY>
__device__ __forceinline__ long act8(const Act<TY>& x, int c) {
    const uint32_t* av = reinterpret_cast<const uint32_t*>(x.a) + 2 * c;
    return pack64(av[0], av[1]);
}
// Block integers of one IQ1_M stream, bi[r], r < RR: 8 * main + delta, exact.
template <int RR>
__device__ __forceinline__ void products1(const Dec& w, const Act<kIQ1_M>& x, int (&bi)[4]) {
    const v4i L = mfma(act8<kIQ1_M>(x, 8), w.D, v4i{0, 0, 0, 0}), Hs = mfma(act8<kIQ1_M>(x, 9), w.D, v4i{0, 0, 0, 0});
    v4i M = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) M = mfma(act8<kIQ1_M>(x, j), w.B[j], M);
#pragma unroll
    for (int r = 0; r < RR; ++r) bi[r] = 8 * M[r] + (16 * Hs[r] + L[r]);
}
// Block integers of the NS IQ2 streams, bi[s][r], r < RR: exact.
template <int TY, int RR, int NS>
__device__ __forceinline__ void products(const Dec (&w)[NS], const Act<TY>& x, uint32_t mk, int (&bi)[NS][4]) {
    // each step's MFMA is issued before the previous step's multiply-adds read theirs
    v4i C[8 * NS], C1[TY == kIQ2_XS ? 8 * NS : 1];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) bi[s][r] = 0;
#pragma unroll
    for (int i = 0; i <= 8 * NS; ++i) {
        if (i < 8 * NS) {
            const long A = act8<TY>(x, i / NS);
            C[i] = mfma(A, w[i % NS].B[i / NS], v4i{0, 0, 0, 0});
            // entries 2, 3 masked out (lanes e4 >= 2 hold them on both sides)
            if constexpr (TY == kIQ2_XS)
                C1[i] = mfma(pack64(uint32_t(uint64_t(A)) & mk, uint32_t(uint64_t(A) >> 32) & mk), w[i % NS].B[i / NS], v4i{0, 0, 0, 0});
        }
        if (i > 0) {
            const int s = (i - 1) % NS, c = (i - 1) / NS;
            if constexpr (TY == kIQ2_XS) {   // ls1 C1 + ls2 (C - C1) as ls2 C + (ls1 - ls2) C1, exactly
                const int ls2 = int(__builtin_amdgcn_ubfe(w[s].s[c >> 2], 8 * (c & 3), 8));
                const int dls = __builtin_amdgcn_sbfe(int(w[s].s[2 + (c >> 2)]), 8 * (c & 3), 8);
#pragma unroll
                for (int r = 0; r < RR; ++r) bi[s][r] = mad24(ls2, C[i - 1][r], mad24(dls, C1[i - 1][r], bi[s][r]));
            } else {
                const int ls = int(__builtin_amdgcn_ubfe(w[s].s[c & 1], 8 * (c >> 1), 8));
#pragma unroll
                for (int r = 0; r < RR; ++r) bi[s][r] = mad24(ls, C[i - 1][r], bi[s][r]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Tiles. GU: rows 16 tl .. + 15 of gate and of up; down: 16 NS rows from 16 NS tl on.
// ---------------------------------------------------------------------------
// LDS written by one wave and read by its other lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// The float sum of a row, over its blocks in order: one fma chain, or (F8) a chain
// per eight blocks, the chains' results added up in order. Layers of other types
// than IQ2_XXS gate/up with IQ2_XS down take F8: with fewer than kGroupAnyTokens
// tokens they are layer calls, whose sums are trees, and one chain over 12 to 20
// blocks is further from 64 bits than those. Tokens without a moved quant of h,
// IQ1_M, from 64 bits: 4096 x 3072 one chain 1.44e-7, layer calls 1.32e-7, by eights
// 1.26e-7; 5120 x 2304 1.47e-7, 1.33e-7, 1.27e-7; mixed types 1.38e-7, 1.26e-7,
// 1.20e-7. By fours 1.24e-7, but the several-tile kernels then spill (IQ1_M, 2,048
// tokens of 64 experts: 2,053 us; by eights 1,427; one chain 1,418).
// Before block b > 0, and past the row's last block with b = 0:
template <bool F8, int N>
__device__ __forceinline__ void next_chain(float* acc, float* total, int b, int nb) {
    if (!F8 || (b & 7) || (b == 0 && nb <= 8)) return;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float v = b == 8 ? acc[i] : __fadd_rn(total[i], acc[i]);
        total[i] = v;
        acc[i] = b == 0 ? v : 0.0f;
    }
}
// TR: also write each pair's block integers (GroupArgs::tint).
template <bool GU, int TY, bool TR, bool DB, bool F8, int NS>
__device__ __forceinline__ void do_tile(const GroupArgs& a, const int4& tk, int tl, uint8_t* lds, uint8_t* wl, int lane) {
    const int col = lane & 15, e4 = lane >> 4, nb = (GU ? a.dim : a.ff) / 256;
    const uint32_t mk = e4 < 2 ? ~0u : 0u;   // lanes of entries 0, 1
    static_assert(!GU || NS == 2, "gate and up");
    Stream st[NS];
    const uint8_t* planes[NS];   // fp16 scales of the streams' rows
    uint32_t row0nb[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const MatRef m = mat_at(a.descs, tk.x, GU ? s : 2);
        const int row0 = GU ? 16 * tl : 16 * (NS * tl + s);
        row0nb[s] = uint32_t(row0 * nb);
        st[s] = Stream{rsrc(m.base), uint32_t((row0 + col) * nb), uint32_t(m.off1), uint32_t(m.off2)};
        planes[s] = m.base + (TY == kIQ2_XXS ? m.off1 : m.off2) + size_t(row0) * nb * 2;
    }
    // A operand: slot col of the tile (past its pairs: unused slot memory, whose
    // outputs are discarded), the lane's chunk e4
    const __amdgpu_buffer_rsrc_t rx = rsrc((GU ? a.xq : a.hq) + tile_off(tk.y >> 4, nb));
    const __amdgpu_buffer_rsrc_t rs = TY == kIQ1_M ? rsrc((GU ? a.xs : a.hs) + sum_off(tk.y >> 4, nb)) : rx;
    const uint32_t va = 256u * e4 + 16u * col;
    Act<TY> x0, x1;
    auto load_x = [&](Act<TY>& x, int blk) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x.a[i] = ld128(rx, va + 4096u * blk + 1024u * i);
        if constexpr (TY == kIQ1_M) x.a[4] = ld128(rs, va + 1024u * blk);
    };
    Raw w0[NS], w1[NS];   // IQ2
    auto load = [&](Raw (&w)[NS], Act<TY>& x, int blk) {
#pragma unroll
        for (int s = 0; s < NS; ++s) load_raw<TY>(w[s], st[s], blk, e4);
        load_x(x, blk);
    };
    Raw1 r1[NS];         // IQ1_M
    if constexpr (TY == kIQ1_M) {
#pragma unroll
        for (int s = 0; s < NS; ++s) load_raw1(r1[s], st[s], row0nb[s], 0, nb, lane);
        if (DB) load_x(x0, 0);
    } else {
        load(w0, x0, 0);
    }
    // the tile's pair scales and rows' scales into the wave's own LDS
    float* pd = reinterpret_cast<float*>(wl);
    uint16_t* rd = reinterpret_cast<uint16_t*>(wl + 64 * kGrpNb);
    const float4* pds = reinterpret_cast<const float4*>((GU ? a.xd : a.hd) + size_t(tk.y >> 4) * nb * 16);
    wave_sync();   // the previous tile's are read
    for (int i = lane; i < 4 * nb; i += 64) reinterpret_cast<float4*>(pd)[i] = pds[i];
    if constexpr (TY != kIQ1_M) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            for (int i = lane; i < 2 * nb; i += 64)   // 16 rows x nb halves, 16 B a piece
                reinterpret_cast<uint4*>(rd + 16 * kGrpNb * s)[i] = reinterpret_cast<const uint4*>(planes[s])[i];
    }
    int po[4];   // the pairs of the lane's four outputs (tile positions 4 e4 + r)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = 4 * r + e4;
        po[r] = j < tk.z ? a.order[tk.y + j] : -1;
    }
    wave_sync();
    // RR: output registers that can hold a pair (ceil(pairs / 4), rounded up to 2 or 4)
    auto run = [&]<int RR>() {
        float acc[NS][4] = {}, total[NS][4];
        int blk_c = 0;   // block the next compute() handles
        auto compute = [&](const Raw (&w)[NS], const Act<TY>& x) {
            const int b = blk_c++;
            Dec dec[NS];
            int bi[NS][4];
            if constexpr (TY == kIQ1_M) {
#pragma unroll
                for (int s = 0; s < NS; ++s) {   // one stream after the other: both at once spill
                    decode<TY>(dec[s], w[s], lds, lane, e4);
                    products1<RR>(dec[s], x, bi[s]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int s = 0; s < NS; ++s) decode<TY>(dec[s], w[s], lds, lane, e4);
                products<TY, RR, NS>(dec, x, mk, bi);
            }
            if constexpr (TR) {   // pair po[r]'s block integers of this lane's rows
                const size_t gu = size_t(a.ff) * (a.dim / 256), rec = 2 * gu + size_t(a.dim) * (a.ff / 256);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int r = 0; r < RR; ++r)
                        if (a.tint && po[r] >= 0)
                            a.tint[size_t(po[r]) * rec + (GU ? s * gu : 2 * gu) + st[s].at + size_t(b)] = bi[s][r];
            }
            const float4 xd4 = *reinterpret_cast<const float4*>(pd + 16 * b + 4 * e4);
            const float xd[4] = {xd4.x, xd4.y, xd4.z, xd4.w};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const float d = TY == kIQ1_M ? dec[s].d : h2f(rd[16 * kGrpNb * s + col * nb + b]);
#pragma unroll
                for (int r = 0; r < RR; ++r) acc[s][r] = fmaf(__fmul_rn(d, xd[r]), float(bi[s][r]), acc[s][r]);
            }
        };
        if constexpr (TY == kIQ1_M) {
            // four blocks at a time through the wave's LDS, the next four in registers
            // meanwhile
            uint8_t* raw = wl + 64 * kGrpNb;
            for (int b = 0; b < nb; b += 4) {
                if (b > 0) next_chain<F8, 4 * NS>(acc[0], total[0], b, nb);
                wave_sync();   // the previous four are read
#pragma unroll
                for (int s = 0; s < NS; ++s) store_raw1(raw + kRaw1 * s, r1[s], lane);
                wave_sync();
#pragma unroll
                for (int s = 0; s < NS; ++s) load_raw1(r1[s], st[s], row0nb[s], min(b + 4, nb - 1), nb, lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    Act<TY>& now = DB && (i & 1) ? x1 : x0;
                    Act<TY>& then = DB && !(i & 1) ? x1 : x0;
                    if (DB) load_x(then, min(b + i + 1, nb - 1));
                    if (b + i < nb) {
                        if (!DB) load_x(now, b + i);   // under the first stream's decode (a second set spills)
                        __builtin_amdgcn_sched_barrier(0);
                        Raw w[NS];
#pragma unroll
                        for (int s = 0; s < NS; ++s) read_raw1(w[s], raw + kRaw1 * s, i, col, e4);
                        compute(w, now);
                    }
                }
            }
        } else {
            // Two operand sets alternate over a 4-step unrolled loop (no register copies,
            // so no wait ever covers a load issued in the same step).
            for (int b = 0; b < nb; b += 4) {
                if (b > 0) next_chain<F8, 4 * NS>(acc[0], total[0], b, nb);
                load(w1, x1, min(b + 1, nb - 1));
                __builtin_amdgcn_sched_barrier(0);   // the loads stay ahead of the compute
                compute(w0, x0);
                load(w0, x0, min(b + 2, nb - 1));
                __builtin_amdgcn_sched_barrier(0);
                if (b + 1 < nb) compute(w1, x1);
                load(w1, x1, min(b + 3, nb - 1));
                __builtin_amdgcn_sched_barrier(0);
                if (b + 2 < nb) compute(w0, x0);
                load(w0, x0, min(b + 4, nb - 1));
                __builtin_amdgcn_sched_barrier(0);
                if (b + 3 < nb) compute(w1, x1);
            }
        }
        next_chain<F8, 4 * NS>(acc[0], total[0], 0, nb);
#pragma unroll
        for (int r = 0; r < RR; ++r)
            if (po[r] >= 0) {
                if constexpr (GU) {
                    a.h[size_t(po[r]) * a.ff + 16 * tl + col] =
                        silu_mul3(__fmul_rn(0.125f, acc[0][r]), __fmul_rn(0.125f, acc[1][r]), a.lim);
                } else {
                    float* y = a.y + size_t(po[r]) * a.dim + 16 * NS * tl + col;
#pragma unroll
                    for (int s = 0; s < NS; ++s) y[16 * s] = __fmul_rn(0.125f, acc[s][r]);
                }
            }
    };
    if (tk.z <= 8) run.template operator()<2>();
    else run.template operator()<4>();
}

// A tile of a task of 16 (NT - 1) + 1 .. 16 NT pairs: each block's two streams are
// decoded once for all NT tiles of pairs. As do_tile otherwise (the same float
// operations per pair); the pair scales come from memory (LDS has no room for NT
// sets beside the tables), one step ahead with the activations.
template <bool GU, int TY, int NT, bool F8>
__device__ __forceinline__ void do_tiles(const GroupArgs& a, const int4& tk, int tl, uint8_t* lds, uint8_t* wl, int lane) {
    const int col = lane & 15, e4 = lane >> 4, nb = (GU ? a.dim : a.ff) / 256;
    const uint32_t mk = e4 < 2 ? ~0u : 0u;
    Stream st[2];
    const uint8_t* planes[2];
    uint32_t row0nb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const MatRef m = mat_at(a.descs, tk.x, GU ? s : 2);
        const int row0 = GU ? 16 * tl : 32 * tl + 16 * s;
        row0nb[s] = uint32_t(row0 * nb);
        st[s] = Stream{rsrc(m.base), uint32_t((row0 + col) * nb), uint32_t(m.off1), uint32_t(m.off2)};
        planes[s] = m.base + (TY == kIQ2_XXS ? m.off1 : m.off2) + size_t(row0) * nb * 2;
    }
    const __amdgpu_buffer_rsrc_t rx = rsrc((GU ? a.xq : a.hq) + tile_off(tk.y >> 4, nb));
    const __amdgpu_buffer_rsrc_t rs = TY == kIQ1_M ? rsrc((GU ? a.xs : a.hs) + sum_off(tk.y >> 4, nb)) : rx;
    const __amdgpu_buffer_rsrc_t rp = rsrc((GU ? a.xd : a.hd) + size_t(tk.y >> 4) * nb * 16);
    const uint32_t va = 256u * e4 + 16u * col;
    struct Step {   // one block's activations and scales of one tile
        Act<TY> x;
        uint4 d;
    };
    Step p0, p1;
    auto load_p = [&](Step& p, int blk, int mt) {
        const uint32_t t = uint32_t(mt) * uint32_t(nb) * 4096u;
#pragma unroll
        for (int i = 0; i < 4; ++i) p.x.a[i] = ld128(rx, va + 4096u * blk + 1024u * i, t);
        if constexpr (TY == kIQ1_M) p.x.a[4] = ld128(rs, va + 1024u * blk, t / 4);
        p.d = ld128(rp, 64u * blk + 16u * e4, uint32_t(mt) * uint32_t(nb) * 64u);
    };
    Raw w0[2], w1[2];   // IQ2
    auto load_w = [&](Raw (&w)[2], int blk) {
#pragma unroll
        for (int s = 0; s < 2; ++s) load_raw<TY>(w[s], st[s], blk, e4);
    };
    Raw1 r1[2];         // IQ1_M
    if constexpr (TY == kIQ1_M) {
#pragma unroll
        for (int s = 0; s < 2; ++s) load_raw1(r1[s], st[s], row0nb[s], 0, nb, lane);
    } else {
        load_w(w0, 0);
    }
    load_p(p0, 0, 0);
    uint16_t* rd = reinterpret_cast<uint16_t*>(wl + 64 * kGrpNb);
    if constexpr (TY != kIQ1_M) {
        wave_sync();   // the previous tile's are read
#pragma unroll
        for (int s = 0; s < 2; ++s)
            for (int i = lane; i < 2 * nb; i += 64)
                reinterpret_cast<uint4*>(rd + 16 * kGrpNb * s)[i] = reinterpret_cast<const uint4*>(planes[s])[i];
        wave_sync();
    }
    float acc[NT][2][4] = {}, total[NT][2][4];
    // Block b from its raw words; `odd` (with NT odd, the block's parity) says which
    // set holds its first step.
    auto block = [&](const Raw (&w)[2], int b, auto odd) {
        Dec dec[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) decode<TY>(dec[s], w[s], lds, lane, e4);
        float d[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) d[s] = TY == kIQ1_M ? dec[s].d : h2f(rd[16 * kGrpNb * s + col * nb + b]);
#pragma unroll
        for (int mt = 0; mt < NT; ++mt) {
            Step& now = (mt + odd.value) & 1 ? p1 : p0;
            Step& then = (mt + odd.value) & 1 ? p0 : p1;
            load_p(then, mt + 1 < NT ? b : min(b + 1, nb - 1), mt + 1 < NT ? mt + 1 : 0);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay ahead of the compute
            int bi[2][4];
            if constexpr (TY == kIQ1_M) {
#pragma unroll
                for (int s = 0; s < 2; ++s) products1<4>(dec[s], now.x, bi[s]);
            } else {
                products<TY, 4, 2>(dec, now.x, mk, bi);
            }
            const float xd[4] = {__uint_as_float(now.d.x), __uint_as_float(now.d.y), __uint_as_float(now.d.z), __uint_as_float(now.d.w)};
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[mt][s][r] = fmaf(__fmul_rn(d[s], xd[r]), float(bi[s][r]), acc[mt][s][r]);
        }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, NT & 1> second{};   // odd NT: the second block of a pair starts in p1
    if constexpr (TY == kIQ1_M) {
        uint8_t* raw = wl + 64 * kGrpNb;
        for (int b = 0; b < nb; b += 4) {
            if (b > 0) next_chain<F8, 8 * NT>(acc[0][0], total[0][0], b, nb);
            wave_sync();   // the previous four are read
#pragma unroll
            for (int s = 0; s < 2; ++s) store_raw1(raw + kRaw1 * s, r1[s], lane);
            wave_sync();
#pragma unroll
            for (int s = 0; s < 2; ++s) load_raw1(r1[s], st[s], row0nb[s], min(b + 4, nb - 1), nb, lane);
            for (int i = 0; i < 4; i += 2) {
                if (b + i >= nb) break;
                Raw w[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) read_raw1(w[s], raw + kRaw1 * s, i, col, e4);
                block(w, b + i, even);
                if (b + i + 1 >= nb) break;
#pragma unroll
                for (int s = 0; s < 2; ++s) read_raw1(w[s], raw + kRaw1 * s, i + 1, col, e4);
                block(w, b + i + 1, second);
            }
        }
    } else {
        for (int b = 0; b < nb; b += 2) {
            if (b > 0) next_chain<F8, 8 * NT>(acc[0][0], total[0][0], b, nb);
            load_w(w1, min(b + 1, nb - 1));
            block(w0, b, even);
            load_w(w0, min(b + 2, nb - 1));
            if (b + 1 < nb) block(w1, b + 1, second);
        }
    }
    next_chain<F8, 8 * NT>(acc[0][0], total[0][0], 0, nb);
#pragma unroll
    for (int mt = 0; mt < NT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 16 * mt + 4 * r + e4;   // the pair of tile position 4 e4 + r
            if (j < tk.z) {
                const size_t p = size_t(a.order[tk.y + j]);
                if constexpr (GU) {
                    a.h[p * a.ff + 16 * tl + col] =
                        silu_mul3(__fmul_rn(0.125f, acc[mt][0][r]), __fmul_rn(0.125f, acc[mt][1][r]), a.lim);
                } else {
                    float* y = a.y + p * a.dim + 32 * tl + col;
                    y[0] = __fmul_rn(0.125f, acc[mt][0][r]);
                    y[16] = __fmul_rn(0.125f, acc[mt][1][r]);
                }
            }
        }
}

// MASK: block types among the launch's matrices (bits 1 IQ2_XXS, 2 IQ2_XS, 4 IQ1_M).
// MT: tasks may hold up to 16 MT pairs. NS: streams per tile (down of 16 or 32 rows).
// F8: the order of the float sums (do_tile).
template <bool GU, int MASK, int NW, int MT, bool TR, bool F8, int NS = 2>
__global__ __launch_bounds__(NW * 64, 1) void grouped_kernel(GroupArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[grp_lds_bytes(MASK, NW)];
    __shared__ uint32_t s_bundle;   // current bundle << 8 | its next tile
    __shared__ int s_open;
    const int t = threadIdx.x, lane = t & 63, wv = uni(t >> 6);
    const int tiles = GU ? a.ff / 16 : a.dim / (16 * NS);   // per task
    int n[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) n[i] = uni(GU ? a.queue->gu_tasks[i] : a.queue->dn_tasks[i]);
    int* next = GU ? a.queue->gu_next : a.queue->dn_next;
    // the type this workgroup starts with: its place in the tasks weighted by their cost
    int first = 0;
    if constexpr (MASK == 7) {
        const int c0 = kTileCost[0] * n[0], c1 = c0 + kTileCost[1] * n[1], all = c1 + kTileCost[2] * n[2];
        const int64_t at = int64_t(all) * (2 * blockIdx.x + 1);
        first = at < int64_t(c0) * 2 * gridDim.x ? 0 : at < int64_t(c1) * 2 * gridDim.x ? 1 : 2;
    }
    for (int i = 0; i < (MASK == 7 ? 3 : 1); ++i) {
        const int ti = MASK == 7 ? (first + i) % 3 : MASK == 1 ? 0 : MASK == 2 ? 1 : 2;
        const int base = ti == 0 ? 0 : ti == 1 ? n[0] : n[0] + n[1];   // the type's tasks in the list
        const int total = n[ti] * tiles;
        // tiles per bundle: a workgroup's waves on one task's activations, or fewer
        // where that would leave the last round of bundles short
        // (few tiles of one type: an even share each, no queue)
        const bool even = MASK != 7 && total <= 2 * NW * int(gridDim.x);
        const int start = even ? int(int64_t(total) * blockIdx.x / gridDim.x) : 0;
        const int bs = even ? int(int64_t(total) * (blockIdx.x + 1) / gridDim.x) - start
                            : total >= 16 * NW * int(gridDim.x) ? NW : 4;
        uint8_t* wl = ti == 2 ? lds + kL_TAB1 + wv * kL_WAVE1 : lds + kL_TAB + wv * kL_WAVE;
        if (MASK == 7 || i == 0) {
            __syncthreads();   // every wave is done with the previous type's tables
            if (t == 0) {
                s_open = total > 0 && (i == 0 || __hip_atomic_load(next + ti, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * bs < total);
                // one type: the first bundle is the workgroup's own; several: none yet
                s_bundle = even ? 0u : MASK != 7 ? uint32_t(blockIdx.x) << 8 : uint32_t(bs);
            }
            __syncthreads();
        }
        if (!s_open) continue;   // nothing left of this type (workgroup-uniform)
        if (MASK != 7 && bs == 0) break;   // workgroup-uniform
        fill_tables<NW * 64>(lds, ti == 0 ? kIQ2_XXS : ti == 1 ? kIQ2_XS : kIQ1_M, a.tables, t);
        __syncthreads();
        for (;;) {
            uint32_t got = 0;
            for (;;) {   // this wave's next tile
                if (lane == 0) got = atomicAdd(&s_bundle, 1u);
                got = uint32_t(uni(int(got)));
                const uint32_t at = got & 255u;
                if (at < uint32_t(bs) || even) break;
                if (at == uint32_t(bs)) {   // empty: this wave fetches the next bundle and takes its first tile
                    int b = 0;
                    if (lane == 0) b = atomicAdd(next + ti, 1);
                    b = min(uni(b), (total + bs - 1) / bs);   // past the last: an empty bundle that ends every wave
                    got = uint32_t(b) << 8;
                    if (lane == 0) __hip_atomic_store(&s_bundle, got | 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    break;
                }
                // Past bs: another wave is fetching one (it waits for nothing but the queue's
                // atomic). At bs itself nobody is: a wave that missed a whole bundle
                // between two looks must draw again, or, with every other wave gone
                // after the last bundle, it would wait for good.
                while ((__hip_atomic_load(&s_bundle, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & 255u) > uint32_t(bs))
                    __builtin_amdgcn_s_sleep(1);
            }
            if (even && got >= uint32_t(bs)) break;
            const int tile = even ? start + int(got) : int(got >> 8) * bs + int(got & 255u);
            if (tile >= total) break;
            const int task = tile / tiles, tl = tile - task * tiles;
            const int4 tk = task_at((GU ? a.tasks : a.dtasks) + base, task);
            const auto tile_of = [&]<int TY>() {
                if constexpr (MT == 1) {
                    do_tile<GU, TY, TR, NW <= 8, F8, NS>(a, tk, tl, lds, wl, lane);
                } else {
                    if (tk.z <= 16) do_tiles<GU, TY, 1, F8>(a, tk, tl, lds, wl, lane);
                    else if (tk.z <= 32) do_tiles<GU, TY, 2, F8>(a, tk, tl, lds, wl, lane);
                    else if (tk.z <= 48) do_tiles<GU, TY, 3, F8>(a, tk, tl, lds, wl, lane);
                    else do_tiles<GU, TY, 4, F8>(a, tk, tl, lds, wl, lane);
                }
            };
            if (MASK == 1 || (MASK == 7 && ti == 0)) tile_of.template operator()<kIQ2_XXS>();
            else if (MASK == 2 || (MASK == 7 && ti == 1)) tile_of.template operator()<kIQ2_XS>();
            else tile_of.template operator()<kIQ1_M>();
        }
    }
}

// ---------------------------------------------------------------------------
// Fixed-order combine per token (runtime.cpp:183-188): ascending expert id,
// out = fma(w, y, out) from +0, then + shared. A bad id contributes nothing.
// Wave 0 ranks the token's picks once (ascending id, equal ids in pick order:
// the stable order of an insertion sort) into LDS; every thread then issues
// its column's loads of all the token's rows before the fma chain.
// ---------------------------------------------------------------------------
// V values per thread (V = 4: 16-byte loads and stores; out and shared 16-byte
// aligned), each combined exactly as with V = 1.
template <int V>
__global__ __launch_bounds__(256) void gcombine_kernel(GroupArgs a) {
    __shared__ int s_row[16];     // pair row of rank r
    __shared__ float s_w[16];
    __shared__ int s_n;
    const int tok = blockIdx.y, t = threadIdx.x, k = a.k;
    if (t < 64) {
        const int id = t < k ? a.ids[size_t(tok) * k + t] : -1;
        const bool ok = t < k && id >= 0 && id < a.n_experts;
        int rank = 0;
        for (int j = 0; j < k; ++j) {
            const int idj = __shfl(id, j);
            const bool okj = idj >= 0 && idj < a.n_experts;
            rank += int(okj && (idj < id || (idj == id && j < t)));
        }
        if (ok) {
            s_row[rank] = tok * k + t;
            s_w[rank] = a.w[size_t(tok) * k + t];
        }
        const int n = __popcll(__ballot(ok));
        if (t == 0) s_n = n;
    }
    __syncthreads();
    const int c = (blockIdx.x * 256 + t) * V;
    if (c >= a.dim) return;   // dim is a multiple of 256
    const int n = s_n;
    using VT = std::conditional_t<V == 4, float4, float>;
    auto lanes = [](VT& x) -> float* { return reinterpret_cast<float*>(&x); };
    VT v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = r < n ? *reinterpret_cast<const VT*>(a.y + size_t(s_row[r]) * a.dim + c) : VT{};
    VT acc{};
#pragma unroll
    for (int r = 0; r < 16; ++r)
        if (r < n)
#pragma unroll
            for (int e = 0; e < V; ++e) lanes(acc)[e] = fmaf(s_w[r], lanes(v[r])[e], lanes(acc)[e]);
    if (a.shared) {
        VT sh = *reinterpret_cast<const VT*>(a.shared + size_t(tok) * a.dim + c);
#pragma unroll
        for (int e = 0; e < V; ++e) lanes(acc)[e] = __fadd_rn(lanes(acc)[e], lanes(sh)[e]);
    }
    *reinterpret_cast<VT*>(a.out + size_t(tok) * a.dim + c) = acc;
}

// How a call's tasks and kernels are cut, from what the host knows: T draws of k of
// the E experts touch E (1 - (1 - k / E)^T) of them. No result depends on it.
struct GroupPlan {
    bool multi;      // tasks of up to 64 pairs
    bool gu8, dn8;   // gate/up, down: the kernels of 8 waves instead of 12
    bool dn_half;    // down tiles of 16 rows instead of 32, 12 waves
};
GroupPlan group_plan(const GroupArgs& a, int gu_types, int dn_types, bool trace, int cus) {
    GroupPlan p{};
    if (trace) return p;   // one kernel each
    const double E = a.n_experts, pairs = double(a.T) * a.k;
    const double touched = E * (1.0 - std::pow(1.0 - std::min(1.0, a.k / E), a.T));
    const double gu_tiles = a.ff / 16, dn_tiles = a.dim / 32;   // per task
    const auto per_wg = [&](double tasks, double tiles) { return tasks * tiles / cus; };
    const auto mixed = [](int types) { return types != 1 && types != 2 && types != 4; };
    const int least = mixed(gu_types) || mixed(dn_types) ? kMultiPairsMix : kMultiPairs;
    const double wide = per_wg(std::max(touched, pairs / 64), std::max(gu_tiles, dn_tiles));
    const bool iq2 = gu_types == 1 && dn_types == 2;
    p.multi = pairs >= least * E && (wide > (iq2 || least == kMultiPairsMix ? kMultiTiles : kMultiTilesIQ1) ||
                                     (wide >= kMultiTiles / 2 && pairs >= 4 * least * E));
    p.gu8 = p.dn8 = p.multi;
    if (p.multi) return p;
    if (!iq2) {   // where 12 waves would share at most 8 tiles
        p.gu8 = p.dn8 = per_wg(std::min(pairs, E), std::max(gu_tiles, dn_tiles)) <= 8;
        return p;
    }
    // IQ2_XXS / IQ2_XS, tiles per workgroup, each way timed over five shapes, 8 to 384
    // experts and 1 to 512 tokens. Gate/up: 8 waves to 8 tiles (0.90 to 1.00 of 12 waves'
    // call); from there 12 to 24, past which the tiles come from a queue, one bundle at a
    // time: 1.01 to 1.05 the other way; past 24 rows of four blocks are faster on 8 waves
    // (0.97), and long rows to 36 tiles (0.95 to 0.99), the rest on 12 (1.00 to 1.04).
    // Down: tiles of 16 rows to 12 tiles (0.87 to 1.00; past them 1.02 to 1.2), with rows of
    // two blocks to 6, where 8 waves follow to 16 and past 24 (0.92 to 1.0).
    const double tasks = std::max(touched, pairs / 16), gu = per_wg(tasks, gu_tiles), dn = per_wg(tasks, dn_tiles);
    p.gu8 = gu <= 8 || (gu > 24 && (a.dim <= 1024 || (a.dim > 2048 && gu <= 36)));
    p.dn_half = dn <= (a.ff <= 512 ? 6 : 12);
    p.dn8 = !p.dn_half && a.ff <= 512 && (dn <= 16 || dn > 24);
    return p;
}

}  // namespace

hipError_t launch_grouped(GroupArgs args, int gu_types, int dn_types, int cus, hipStream_t s) {
    // Waves per workgroup: 3 per SIMD; layers of several types 2: at 3 their kernels spill
    // 39 to 60 registers (512 tokens, 4096 x 3072, 384 experts: 1,512 us against 1,335), at
    // 2 up to 16, and 44 to 90 with 64-pair tasks, which still win (kMultiPairsMix).
    constexpr int NW = 12, NWM = 8;
    if (args.T < 1 || args.k < 1 || args.k > 16 || args.n_experts > kGroupMaxExperts || args.dim % 256 || args.ff % 256 ||
        args.dim > kGrpNb * 256 || args.ff > 4096)   // (longer hidden rows would fit: not measured)
        return hipErrorNotSupported;
    const bool trace = args.tq8x || args.tq8h || args.th || args.tint, iq2 = gu_types == 1 && dn_types == 2;
    if (trace && !iq2) return hipErrorNotSupported;
    if (((gu_types & 4) && !args.xs) || ((dn_types & 4) && !args.hs)) return hipErrorInvalidValue;
    const GroupPlan plan = group_plan(args, gu_types, dn_types, trace, cus);
    args.cap = plan.multi ? 64 : 16;
    const int P = args.T * args.k, nbx = args.dim / 256, nbh = args.ff / 256;
    const auto grouped = [&](auto kernel, int nw = 12) { hipLaunchKernelGGL(kernel, dim3(cus), dim3(nw * 64), 0, s, args); };
    const auto rows = [&](auto kernel, const float* src, int n, int nb, int8_t* q, int8_t* sums, float* d, uint8_t* tr) {
        hipLaunchKernelGGL(kernel, dim3((n * nb + 3) / 4), dim3(256), 0, s, src, n, nb, q, sums, d, args.pos, args.k, args.err, tr);
    };
    // sums by eights (next_chain), where a row has more than eight blocks: without, it is
    // one chain all the same, and several-type kernels spill less (1024 x 512, 256 tokens
    // of 6 over 64 experts 97.9 to 93.1 us)
    const bool gu_f8 = !iq2 && nbx > 8, dn_f8 = !iq2 && nbh > 8;
    const auto sums = [&](bool f8, auto chain, auto eights, int nw) { grouped(f8 ? eights : chain, nw); };
    // the queues start past the workgroups' own first bundles (launches of one type)
    args.gu_first = gu_types == 1 || gu_types == 4 ? cus : 0;
    args.dn_first = dn_types == 2 || dn_types == 4 ? cus : 0;
    hipLaunchKernelGGL(bucket_kernel, dim3(1), dim3(1024), 0, s, args);
    if (trace) {   // the parity trace (separate instances)
        rows((q8k_rows_kernel<ROWS_X, false, true>), args.x, args.T, nbx, args.xq, args.xs, args.xd, args.tq8x);
        grouped(grouped_kernel<true, 1, NW, 1, true, false>);
        rows((q8k_rows_kernel<ROWS_H, false, true>), args.h, P, nbh, args.hq, args.hs, args.hd, args.tq8h);
        grouped(grouped_kernel<false, 2, NW, 1, true, false>);
    } else {
        rows(gu_types & 4 ? q8k_rows_kernel<ROWS_X, true, false> : q8k_rows_kernel<ROWS_X, false, false>, args.x, args.T, nbx,
             args.xq, args.xs, args.xd, nullptr);
        if (gu_types == 1) {
            if (plan.gu8) sums(gu_f8, grouped_kernel<true, 1, 8, 4, false, false>, grouped_kernel<true, 1, 8, 4, false, true>, 8);
            else sums(gu_f8, grouped_kernel<true, 1, NW, 1, false, false>, grouped_kernel<true, 1, NW, 1, false, true>, NW);
        } else if (gu_types == 4) {
            if (plan.gu8) sums(gu_f8, grouped_kernel<true, 4, 8, 4, false, false>, grouped_kernel<true, 4, 8, 4, false, true>, 8);
            else sums(gu_f8, grouped_kernel<true, 4, NW, 1, false, false>, grouped_kernel<true, 4, NW, 1, false, true>, NW);
        } else {
            if (plan.multi) sums(gu_f8, grouped_kernel<true, 7, NWM, 4, false, false>, grouped_kernel<true, 7, NWM, 4, false, true>, NWM);
            else sums(gu_f8, grouped_kernel<true, 7, NWM, 1, false, false>, grouped_kernel<true, 7, NWM, 1, false, true>, NWM);
        }
        rows(dn_types & 4 ? q8k_rows_kernel<ROWS_H, true, false> : q8k_rows_kernel<ROWS_H, false, false>, args.h, P, nbh,
             args.hq, args.hs, args.hd, nullptr);
        if (plan.dn_half) {   // IQ2 layers only
            grouped(grouped_kernel<false, 2, NW, 1, false, false, 1>);
        } else if (dn_types == 2) {
            if (plan.dn8) sums(dn_f8, grouped_kernel<false, 2, 8, 4, false, false>, grouped_kernel<false, 2, 8, 4, false, true>, 8);
            else sums(dn_f8, grouped_kernel<false, 2, NW, 1, false, false>, grouped_kernel<false, 2, NW, 1, false, true>, NW);
        } else if (dn_types == 4) {
            if (plan.dn8) sums(dn_f8, grouped_kernel<false, 4, 8, 4, false, false>, grouped_kernel<false, 4, 8, 4, false, true>, 8);
            else sums(dn_f8, grouped_kernel<false, 4, NW, 1, false, false>, grouped_kernel<false, 4, NW, 1, false, true>, NW);
        } else {
            if (plan.multi) sums(dn_f8, grouped_kernel<false, 7, NWM, 4, false, false>, grouped_kernel<false, 7, NWM, 4, false, true>, NWM);
            else sums(dn_f8, grouped_kernel<false, 7, NWM, 1, false, false>, grouped_kernel<false, 7, NWM, 1, false, true>, NWM);
        }
    }
    const bool al16 = (reinterpret_cast<uintptr_t>(args.out) | reinterpret_cast<uintptr_t>(args.shared)) % 16 == 0;
    if (al16) hipLaunchKernelGGL(gcombine_kernel<4>, dim3((args.dim / 4 + 255) / 256, args.T), dim3(256), 0, s, args);
    else hipLaunchKernelGGL(gcombine_kernel<1>, dim3((args.dim + 255) / 256, args.T), dim3(256), 0, s, args);
    return hipGetLastError();
}

}  // namespace xl::dev
