// CDNA4 (gfx950) shared-expert FFN of several tokens over the dense formats
// (Q8_0, Q4_K, Q5_K, Q6_K) in the per32 arithmetic (hip_backend.cpp:664-666;
// the row arithmetic of sycl/moe/core.hpp:56-84), bit-identical to the row
// kernels of xl_per32.hip run token by token:
//
//   quant32t_kernel  per-32 quantization of the token rows, written in the
//                    operand order of the MFMA kernels
//   ffn_gu_kernel    gate and up of 32 rows x 16 or 32 tokens, SwiGLU, and the
//                    per-32 quantization of those 32 h values (one sub-block of
//                    every token of the tile), so that h never leaves the chip
//   ffn_dn_kernel    down of 32 rows x 16 or 32 tokens
//
// MFMA: v_mfma_i32_16x16x32_i8 with M = 16 rows, N = 16 tokens, K = the 32
// values of one sub-block, whose integer dot is what the row arithmetic scales.
// Lane l supplies the 8 weights 8 (l / 16) .. + 7 of row l % 16 and the same 8
// quants of token l % 16, and receives rows 4 (l / 16) + r, r = 0..3, of token
// l % 16. The sums of the activations that the min term of Q4_K / Q5_K takes
// come from the same unit (ones as weights).
//
// Order of the sums: a row of the row kernels is 32 lanes, lane l taking
// sub-blocks l, l + 32, ... as one fma chain, then a 16-8-4-2-1 butterfly. A tile
// has eight waves: wave (c, p) takes the sub-blocks i of parity p of the 256-value
// blocks b = c (mod 4), each the next link of lane 8 (b % 4) + i's chain, so that
// it holds four chains per output. The butterfly's first two steps add the
// waves' chains through LDS (c and c ^ 2, then c and c ^ 1), the next two a wave's
// own four, the last the two parities.
//
// What bounds it: VALU issue, and the copies to LDS, whose latency is not hidden
// (stage_step). The float part is five VALU instructions per output and sub-block for
// Q4_K / Q5_K and Q6_K (three for Q8_0) against a quarter of an MFMA: at 512 tokens of
// 4096 x 3072 77 of the 160 us that all VALU instructions take to issue; the rest is
// decode, scales and the sums' exchange. There, Q5_K gate/up and Q6_K down: 205 us, 189
// TFLOP/s (traced 127 us gate/up, VALU issue 84 % of its SIMD cycles, 95 us down, 65 %; the
// row kernels, which decode every weight once per token: 2,913 us); 16 tokens: 32 us
// (120). The 32-token instances spill (Q8_0 13, Q4_K 2, Q5_K 9, Q6_K 41 registers of
// gate/up; Q5_K 2, Q6_K 18 of down).
#include <hip/hip_runtime.h>

#include "xl_dev.hpp"
#include "xl_format.hpp"
#include "xl_internal.hpp"

namespace xl::dev {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kRowsT = 32;   // rows per workgroup: one sub-block of h

__device__ __forceinline__ long pack64(uint32_t lo, uint32_t hi) { return long((uint64_t(hi) << 32) | lo); }
__device__ __forceinline__ v4i mfma(long a, long b) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4i{0, 0, 0, 0}, 0, 0, 0);
}
__device__ __forceinline__ uint32_t ld16u(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
// LDS written by one wave and read by its other lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Activations of the tokens 16 tile .. (nt of them, 16 but in the last tile):
// quants from byte 16 tile * K on, where the 8 values 8 e .. + 7 of sub-block i
// of block b of the tile's token t sit at ((4 b + s / 2) * 4 + e) * 16 nt + 16 t
// + 8 (s % 2), s = act_slot(i) (four lanes of consecutive tokens read 64
// contiguous bytes, and a lane's 16 bytes are two sub-blocks of one parity);
// scales from float 16 tile * K / 32 on, that sub-block's at (b nt + t) * 8 + s.
__host__ __device__ constexpr int act_slot(int i) { return (i >> 1) | ((i & 1) << 2); }
struct ActTile {
    const int8_t* q;
    const float* d;
    int nt, t;   // tokens of the tile, the lane's token (clamped to a valid one)
};
__device__ __forceinline__ ActTile act_tile(const int8_t* q, const float* d, int T, int K, int tile, int lane) {
    ActTile a;
    const int tl = min(tile, (T - 1) / 16);   // a tile past the end reads the last one and stores nothing
    a.nt = min(16, T - 16 * tl);
    a.t = min(lane & 15, a.nt - 1);
    a.q = q + size_t(tl) * 16 * K;
    a.d = d + size_t(tl) * 16 * (K / 32);
    return a;
}

__host__ __device__ constexpr int row_block_bytes(int ty) { return ty == kQ8_0 ? 8 * 34 : dense_block_bytes(ty); }

// The weights go through LDS, 32 rows of four 256-value blocks at a time (one per
// c), copied there directly as whole 16-byte pieces (a lane's 8-byte slices straight
// from memory cost the texture unit one access per lane, and bounded the kernel). The
// copies of step s + 1 go out before the products of step s, but not ahead of its first
// LDS read: the compiler cannot tell the halves of the stage apart and waits there for
// every copy in flight, so that each step shows a copy's latency. Row stride: an odd number of pieces, so that the 16
// rows' slices fall into different banks. A Q6_K block starts at any even byte:
// its pieces start at the 16-byte boundary before it and 14 hold it (n and k are
// multiples of 256, so that the last block's pieces end with the matrix).
template <int TY>
constexpr int kPieces = TY == kQ8_0 ? 17 : TY == kQ6_K ? 15 : TY == kQ5_K ? 11 : 9;
template <int TY>
constexpr int kStride = 16 * kPieces<TY>;
template <int TY>
constexpr int kStepBytes = 4 * 32 * kStride<TY>;   // a multiple of 1 KiB

// Copies step s (blocks 4 s .. + 3, past the row's end the last one) of the 32
// rows at W to LDS; wave w of eight.
template <int TY>
__device__ __forceinline__ void stage_step(uint8_t* st, const uint8_t* W, size_t row_bytes, int nb, int s, int w, int lane) {
    constexpr int P = kPieces<TY>;
    for (int g = w; g * 1024 < kStepBytes<TY>; g += 8) {
        const int c = 64 * g + lane, blk = c / (32 * P), rp = c - blk * (32 * P), row = rp / P;
        int p = rp - row * P;
        size_t at = size_t(row) * row_bytes + size_t(min(4 * s + blk, nb - 1)) * row_block_bytes(TY);
        if constexpr (TY == kQ6_K) {
            at &= ~size_t(15);
            p = min(p, 13);   // the 15th piece pads the stride
        }
        __builtin_amdgcn_global_load_lds((const void*)(W + at + 16 * p),
                                         (__attribute__((address_space(3))) void*)(st + 1024 * g), 16, 0, 0);
    }
}
// 8 bytes at a 2-byte-aligned LDS address from the aligned words that cover them.
__device__ __forceinline__ uint2 lds8_a2(const uint8_t* p, uint32_t sh) {   // sh: p's offset from p - sh, a multiple of 4
    const uint32_t* w = reinterpret_cast<const uint32_t*>(p - sh);
    const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
    return make_uint2(__builtin_amdgcn_alignbyte(w1, w0, sh), __builtin_amdgcn_alignbyte(w2, w1, sh));
}
// The lane's view of its row of a staged block: the bytes that hold values 8 e .. + 7.
template <int TY>
struct RowBlk {
    const uint8_t* p;   // the block's first byte in LDS
    uint32_t sh;        // Q6_K: 2 where p is not 4-byte aligned
    uint32_t h[4];      // Q5_K: fifth bits; Q6_K: high bits of both halves
};
template <int TY>
__device__ __forceinline__ RowBlk<TY> row_blk(const uint8_t* st, int m, uint32_t off, int e) {
    RowBlk<TY> r;
    r.p = st + m * kStride<TY> + off;
    r.sh = off & 2u;
    if constexpr (TY == kQ5_K) {
        const uint2 h = *reinterpret_cast<const uint2*>(r.p + 16 + 8 * e);
        r.h[0] = h.x; r.h[1] = h.y;
    } else if constexpr (TY == kQ6_K) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint2 h = lds8_a2(r.p + 128 + 32 * i + 8 * e, r.sh);
            r.h[2 * i] = h.x; r.h[2 * i + 1] = h.y;
        }
    }
    return r;
}
// The lane's 8 weights of sub-block 2 i + par as int8.
template <int TY>
__device__ __forceinline__ long weights8(const RowBlk<TY>& r, int i, int e, int par) {
    uint32_t w[2];
    const int ib = 2 * i + par;   // par is wave-uniform: its shifts are scalar
    if constexpr (TY == kQ8_0) {
        const uint2 v = lds8_a2(r.p + 34 * ib + 2 + 8 * e, 2u - 2u * uint32_t(par));
        w[0] = v.x; w[1] = v.y;
    } else if constexpr (TY == kQ6_K) {   // half ib / 4, quarter ib % 4: lows of 32-byte run 2 half + (quarter & 1)
        const int qt = ib & 3;
        const uint2 v = lds8_a2(r.p + 32 * (2 * (i >> 1) + par) + 8 * e, r.sh);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t lo = ((j ? v.y : v.x) >> (4 * (qt >> 1))) & 0x0f0f0f0fu;
            const uint32_t hi = (r.h[2 * (i >> 1) + j] >> (2 * qt)) & 0x03030303u;
            // q - 32 bytewise: q ^ 0x20 has the value's low six bits, whose sign bit 5 fills bits 6 and 7
            const uint32_t x = (lo | (hi << 4)) ^ 0x20202020u;
            const uint32_t s = x & 0x20202020u;
            w[j] = x | (s << 1) | (s << 2);
        }
    } else {
        const uint2 v = *reinterpret_cast<const uint2*>(r.p + (TY == kQ5_K ? 48 : 16) + 32 * i + 8 * e);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            w[j] = ((j ? v.y : v.x) >> (4 * par)) & 0x0f0f0f0fu;
            if constexpr (TY == kQ5_K) w[j] |= ((r.h[j] >> ib) & 0x01010101u) << 4;
        }
    }
    return pack64(w[0], w[1]);
}
// Scales of a wave's four sub-blocks of one block of 16 rows in LDS: plane 0 / 1
// [sub-block][row] (K-quants: d * scale and dmin * min, exact products of an fp16
// and a 6-bit integer; Q6_K: the two half scales as integers; Q8_0: d), then
// Q6_K's d [row]. Lane (m, e) writes sub-block 2 e + par of row m.
struct ScaleLds {
    float p[2][4][16];
    float d[16];
};
template <int TY>
__device__ __forceinline__ void stage_scales(ScaleLds& S, const RowBlk<TY>& r, int m, int e, int par) {
    if constexpr (TY == kQ8_0) {
        S.p[0][e][m] = h2f(ld16u(r.p + 34 * (2 * e + par)));
    } else if constexpr (TY == kQ6_K) {
        const uint32_t s = ld16u(r.p + 192 + 4 * e + 2 * par);
        S.p[0][e][m] = __int_as_float(__builtin_amdgcn_sbfe(int(s), 0, 8));
        S.p[1][e][m] = __int_as_float(__builtin_amdgcn_sbfe(int(s), 8, 8));
        if (e == 0) S.d[m] = h2f(ld16u(r.p + 208));
    } else {
        // 6-bit scale and min of sub-blocks 0..3 and 4..7 (core.hpp:30-39), one byte each
        const uint4 hd = *reinterpret_cast<const uint4*>(r.p);
        const uint32_t a = hd.y, b = hd.z, c = hd.w;
        const uint32_t lo = e < 2 ? ~0u : 0u;   // masks, not branches
        const uint32_t sc = (a & 0x3f3f3f3fu & lo) | (((c & 0x0f0f0f0fu) | ((a >> 2) & 0x30303030u)) & ~lo);
        const uint32_t mn = (b & 0x3f3f3f3fu & lo) | ((((c >> 4) & 0x0f0f0f0fu) | ((b >> 2) & 0x30303030u)) & ~lo);
        const int sh = 16 * (e & 1) + 8 * par;
        S.p[0][e][m] = __fmul_rn(h2f(hd.x & 0xffffu), float((sc >> sh) & 255u));
        S.p[1][e][m] = __fmul_rn(h2f(hd.x >> 16), float((mn >> sh) & 255u));
    }
}

// The 32 x 16 NT tile of rows (W: the first one's bytes) times tokens, by eight
// waves (w): out[rt][tt][r] is row 16 rt + 4 (lane / 16) + r of token lane % 16 of
// tile tt, in wave 0 only. nb: 256-value blocks per row. lds: tile_lds_bytes.
template <int TY, int NT>
__device__ __forceinline__ void tile_rows(const uint8_t* W, int nb, const ActTile (&act)[NT], ScaleLds (&sl)[2], uint8_t* lds,
                                          int w, int lane, float (&out)[2][NT][4]) {
    const int m = lane & 15, e = lane >> 4, c = w & 3, par = w >> 2;
    const size_t row_bytes = size_t(nb) * row_block_bytes(TY);
    const long ones_a = e < 2 ? 0x0101010101010101l : 0l, ones_b = e < 2 ? 0l : 0x0101010101010101l;
    const long half_a = e < 2 ? -1l : 0l;
    float acc[4][2][NT][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][rt][tt][r] = 0.0f;
    stage_step<TY>(lds, W, row_bytes, nb, 0, w, lane);
    const int steps = (nb + 3) / 4;
    for (int s = 0; s < steps; ++s) {
        const int b = 4 * s + c;
        // This wave's copies of step s arrive before the barrier that hands them over,
        // stated here: nothing in the language ties a copy to LDS to a barrier. Ahead of
        // the activations' loads, which then are in flight across the barrier (512 tokens
        // of 4096 x 3072, Q5_K / Q6_K 204.8 us, Q8_0 140.9; behind them 207.6 and 147.3).
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        u32x4_t aq[NT][2];
        float4 xd[NT];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
            const int bc = min(b, nb - 1);
#pragma unroll
            for (int i = 0; i < 2; ++i)
                aq[tt][i] = *reinterpret_cast<const u32x4_t*>(act[tt].q + size_t((4 * bc + 2 * par + i) * 4 + e) * 16 * act[tt].nt +
                                                              16 * act[tt].t);
            xd[tt] = *reinterpret_cast<const float4*>(act[tt].d + size_t(bc * act[tt].nt + act[tt].t) * 8 + 4 * par);
        }
        __syncthreads();   // step s is in LDS, and every wave is done with step s - 1
        if (s + 1 < steps) stage_step<TY>(lds + ((s + 1) & 1) * kStepBytes<TY>, W, row_bytes, nb, s + 1, w, lane);
        if (b >= nb) continue;   // wave-uniform; the step's barriers are the loop's
        const uint8_t* st = lds + (s & 1) * kStepBytes<TY> + c * 32 * kStride<TY>;
        RowBlk<TY> raw[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const uint32_t off = TY == kQ6_K ? uint32_t(size_t(16 * rt + m) * row_bytes + size_t(b) * 210) & 15u : 0u;
            raw[rt] = row_blk<TY>(st + 16 * rt * kStride<TY>, m, off, e);
            stage_scales<TY>(sl[rt], raw[rt], m, e, par);
        }
        wave_sync();
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // sub-block 2 i + par
            if (NT > 1) __builtin_amdgcn_sched_barrier(0);   // no later sub-block's operands in registers
            long bq[NT];
            float sa[NT], sb[NT], xi[NT];
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
                xi[tt] = i == 0 ? xd[tt].x : i == 1 ? xd[tt].y : i == 2 ? xd[tt].z : xd[tt].w;
                const u32x4_t v = aq[tt][i >> 1];
                bq[tt] = (i & 1) ? pack64(v.z, v.w) : pack64(v.x, v.y);
                if constexpr (TY == kQ4_K || TY == kQ5_K) {
                    sa[tt] = float(mfma(ones_a, bq[tt])[0]);
                    sb[tt] = float(mfma(ones_b, bq[tt])[0]);
                }
            }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const long w = weights8<TY>(raw[rt], i, e, par);
                const float4 p0 = *reinterpret_cast<const float4*>(&sl[rt].p[0][i][4 * e]);
                const float s0[4] = {p0.x, p0.y, p0.z, p0.w};
                float s1[4], d6[4];
                if constexpr (TY != kQ8_0) {
                    const float4 p1 = *reinterpret_cast<const float4*>(&sl[rt].p[1][i][4 * e]);
                    s1[0] = p1.x; s1[1] = p1.y; s1[2] = p1.z; s1[3] = p1.w;
                }
                if constexpr (TY == kQ6_K) {
                    const float4 p2 = *reinterpret_cast<const float4*>(&sl[rt].d[4 * e]);
                    d6[0] = p2.x; d6[1] = p2.y; d6[2] = p2.z; d6[3] = p2.w;
                }
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) {
                    float (&ac)[4] = acc[i][rt][tt];
                    if constexpr (TY == kQ6_K) {
                        const v4i ca = mfma(w & half_a, bq[tt]), cb = mfma(w & ~half_a, bq[tt]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int isum = __mul24(__float_as_int(s0[r]), ca[r]) + __mul24(__float_as_int(s1[r]), cb[r]);
                            ac[r] = fmaf(xi[tt], __fmul_rn(d6[r], float(isum)), ac[r]);
                        }
                    } else {
                        const v4i c = mfma(w, bq[tt]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if constexpr (TY == kQ8_0) {
                                ac[r] = fmaf(__fmul_rn(s0[r], xi[tt]), float(c[r]), ac[r]);
                            } else {
                                // core.hpp:62-65 with the block's d * scale as one factor (both products exact)
                                const float corr = fmaf(s1[r], sa[tt], __fmul_rn(s1[r], sb[tt]));
                                ac[r] = fmaf(xi[tt], fmaf(s0[r], float(c[r]), -corr), ac[r]);
                            }
                        }
                    }
                }
            }
        }
    }
    // the butterfly: lanes l and l ^ 16 are waves c and c ^ 2, l and l ^ 8 waves c and
    // c ^ 1, l and l ^ 4 and l and l ^ 2 a wave's chains, l and l ^ 1 the parities
    const auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) f(acc[i][rt][tt][r], ((i * 2 + rt) * NT + tt) * 4 + r);
    };
    float* red = reinterpret_cast<float*>(lds) + lane;
    const int slots = 32 * NT * 64;                     // floats of one wave's chains
    float* mine = red + (2 * par + (c & 1)) * slots;
    __syncthreads();   // every wave is done with the staged steps
    if (c >= 2) each([&](float& v, int at) { mine[64 * at] = v; });
    __syncthreads();
    if (c < 2) each([&](float& v, int at) { v = __fadd_rn(v, mine[64 * at]); });
    if (c == 1) each([&](float& v, int at) { mine[64 * at] = v; });   // its own slots, which only it read
    __syncthreads();
    if (c == 0) {
        each([&](float& v, int at) { v = __fadd_rn(v, mine[slots + 64 * at]); });
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto a = [&](int i) { return acc[i][rt][tt][r]; };   // sub-block 2 i + par
                    out[rt][tt][r] = __fadd_rn(__fadd_rn(a(0), a(2)), __fadd_rn(a(1), a(3)));
                }
        if (par == 1)
#pragma unroll
            for (int j = 0; j < 8 * NT; ++j) red[64 * j] = out[j / (4 * NT)][(j / 4) % NT][j % 4];   // wave (0, 0)'s slots, read
    }
    __syncthreads();
    if (w == 0)
#pragma unroll
        for (int j = 0; j < 8 * NT; ++j) {
            float& v = out[j / (4 * NT)][(j / 4) % NT][j % 4];
            v = __fadd_rn(__fadd_rn(v, red[64 * j]), 0.0f);
        }
    __syncthreads();   // the sums are read: the next tile stages over them
}
// LDS of one tile: two staged steps, over them the sums' exchange.
template <int TY, int NT>
constexpr int tile_lds_bytes = 2 * kStepBytes<TY> > 4 * 32 * NT * 64 * 4 ? 2 * kStepBytes<TY> : 4 * 32 * NT * 64 * 4;

// Per-32 quantization of T rows of K values (quant32_kernel's arithmetic), one
// wave per 256-value block, into the layout of ActTile.
__global__ __launch_bounds__(256) void quant32t_kernel(const float* __restrict__ x, int T, int K, int8_t* __restrict__ q,
                                                       float* __restrict__ d, int* __restrict__ err, int wide) {
    const int nb = K / 256, w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= T * nb) return;   // wave-uniform
    const int tok = w / nb, b = w - tok * nb;
    const float* p = x + size_t(w) * 256 + 4 * lane;
    float v[4];
    if (wide) {
        const float4 f = *reinterpret_cast<const float4*>(p);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = p[j];
    }
    float am = fabsf(v[0]);   // no start value: a block of NaNs keeps NaN, as in quant32_kernel
    bool finite = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        am = fmaxf(am, fabsf(v[j]));
        finite = finite && (fabsf(v[j]) <= 3.402823466e38f);
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
    if (__any(!finite) && lane == 0) atomicOr(err, kDevErrNonFinite);
    const float sc = __fdiv_rn(am, 127.0f);
    uint32_t packed = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        packed |= uint32_t(uint8_t(int8_t(am > 0.0f ? __float2int_rn(__fdiv_rn(v[j], sc)) : 0))) << (8 * j);
    const int i = act_slot(lane >> 3), e = (lane >> 1) & 3, tile = tok >> 4, t = tok & 15, nt = min(16, T - 16 * tile);
    *reinterpret_cast<uint32_t*>(q + size_t(tile) * 16 * K + size_t((4 * b + (i >> 1)) * 4 + e) * 16 * nt + 16 * t +
                                 8 * (i & 1) + 4 * (lane & 1)) = packed;
    if ((lane & 7) == 0) d[size_t(tile) * 16 * (K / 32) + size_t(b * nt + t) * 8 + i] = sc;
}

// Workgroup (x, y): rows 32 x .. + 31 of gate and up, tokens 16 NT y .. of T.
// SPLIT: waves 8..15 take up while waves 0..7 take gate (few tokens: half the
// serial work per wave); else eight waves take one after the other (many tokens:
// two workgroups per CU, one's sums under the other's products).
template <int TY, int NT, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 1024 : 512, 4) void ffn_gu_kernel(const uint8_t* __restrict__ G,
                                                                       const uint8_t* __restrict__ U, int T, int K, int ff,
                                                                       const int8_t* __restrict__ q,
                                                                       const float* __restrict__ d, float lim,
                                                                       int8_t* __restrict__ hq, float* __restrict__ hd) {
    constexpr int R = SPLIT ? 2 : 1;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[R][tile_lds_bytes<TY, NT>];
    __shared__ __attribute__((aligned(16))) ScaleLds sl[8 * R][2];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wv & 7, role = wv >> 3;
    const int row0 = blockIdx.x * kRowsT, nb = K / 256;
    const size_t at = size_t(row0) * size_t(nb) * row_block_bytes(TY);
    ActTile act[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) act[tt] = act_tile(q, d, T, K, blockIdx.y * NT + tt, lane);
    float g[2][NT][4], u[2][NT][4];
    if constexpr (SPLIT) {
        tile_rows<TY, NT>((role ? U : G) + at, nb, act, sl[wv], lds[role], w, lane, g);
        float* x = reinterpret_cast<float*>(lds[1]) + lane;   // up's rows to gate's wave
        if (wv == 8)
#pragma unroll
            for (int j = 0; j < 8 * NT; ++j) x[64 * j] = g[j / (4 * NT)][(j / 4) % NT][j % 4];
        __syncthreads();
        if (wv == 0)
#pragma unroll
            for (int j = 0; j < 8 * NT; ++j) u[j / (4 * NT)][(j / 4) % NT][j % 4] = x[64 * j];
    } else {
        // gate's rows wait in LDS where two workgroups' worth of it is left (in
        // registers they spill the next tile's operands)
        constexpr bool KEEP = sizeof(lds) + sizeof(sl) + 8 * NT * 256 <= 80 * 1024;
        __shared__ float keep[KEEP ? 8 * NT * 64 : 1];
        tile_rows<TY, NT>(G + at, nb, act, sl[wv], lds[0], w, lane, g);
        if (KEEP && wv == 0)
#pragma unroll
            for (int j = 0; j < 8 * NT; ++j) keep[64 * j + lane] = g[j / (4 * NT)][(j / 4) % NT][j % 4];
        tile_rows<TY, NT>(U + at, nb, act, sl[wv], lds[0], w, lane, u);
        if (KEEP && wv == 0)
#pragma unroll
            for (int j = 0; j < 8 * NT; ++j) g[j / (4 * NT)][(j / 4) % NT][j % 4] = keep[64 * j + lane];
    }
    if (wv != 0) return;
    const int m = lane & 15, e = lane >> 4, i = act_slot((row0 >> 5) & 7), b = row0 >> 8;   // h's sub-block of block b
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
        const int tile = blockIdx.y * NT + tt, tok = 16 * tile + m;
        float am = 0.0f;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                g[rt][tt][r] = silu_mul3(g[rt][tt][r], u[rt][tt][r], lim);
                // the first value starts the maximum: a block of NaNs keeps NaN, as in swiglu_quant32_kernel
                am = rt + r == 0 ? fabsf(g[rt][tt][r]) : fmaxf(am, fabsf(g[rt][tt][r]));
            }
        am = fmaxf(am, __shfl_xor(am, 16));
        am = fmaxf(am, __shfl_xor(am, 32));
        const float sc = __fdiv_rn(am, 127.0f);
        if (tok >= T) continue;
        const int nt = min(16, T - 16 * tile);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {   // rows 16 rt + 4 e .. + 3: eighth 2 rt + e / 2, half e % 2
            uint32_t packed = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                packed |= uint32_t(uint8_t(int8_t(am > 0.0f ? __float2int_rn(__fdiv_rn(g[rt][tt][r], sc)) : 0))) << (8 * r);
            *reinterpret_cast<uint32_t*>(hq + size_t(tile) * 16 * ff +
                                         size_t((4 * b + (i >> 1)) * 4 + 2 * rt + (e >> 1)) * 16 * nt + 16 * m +
                                         8 * (i & 1) + 4 * (e & 1)) = packed;
        }
        if (e == 0) hd[size_t(tile) * 16 * (ff / 32) + size_t(b * nt + m) * 8 + i] = sc;
    }
}
template <int TY, int NT>
__global__ __launch_bounds__(512, 4) void ffn_dn_kernel(const uint8_t* __restrict__ D, int T, int K, int n, const int8_t* __restrict__ q,
                                                     const float* __restrict__ d, float* __restrict__ out, int wide) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[tile_lds_bytes<TY, NT>];
    __shared__ __attribute__((aligned(16))) ScaleLds sl[8][2];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row0 = blockIdx.x * kRowsT;
    ActTile act[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) act[tt] = act_tile(q, d, T, K, blockIdx.y * NT + tt, lane);
    float y[2][NT][4];
    tile_rows<TY, NT>(D + size_t(row0) * size_t(K / 256) * row_block_bytes(TY), K / 256, act, sl[w], lds, w, lane, y);
    if (w != 0) return;
    const int m = lane & 15, e = lane >> 4;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
        const int tok = 16 * (blockIdx.y * NT + tt) + m;
        if (tok >= T) continue;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            float* o = out + size_t(tok) * n + row0 + 16 * rt + 4 * e;
            if (wide) {
                *reinterpret_cast<float4*>(o) = make_float4(y[rt][tt][0], y[rt][tt][1], y[rt][tt][2], y[rt][tt][3]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = y[rt][tt][r];
            }
        }
    }
}

// Few tokens of a small FFN, where the row kernels' many short rows fill the chip
// better than a few tiles whose blocks come one after the other. Timed both ways at 2 to
// 12 tokens over dim 256 .. 5120, ff 256 .. 6144 and four type sets: 3 tokens, ff up to
// 512 (rows of 2,048 on 1,024; Q8_0, cheaper to decode: 256) 0.99 to 1.10 of the row kernels' time (4096 x 256
// 26.0 against 24.8 us, 512 x 256 18.9 against 17.1), ff of 2048 0.80 to 0.99; 4 tokens of
// up to 2^18 weights a matrix 1.01 to 1.11; to 8 of 256 x 256 1.02 to 1.06. Two tokens are
// faster by rows almost everywhere (kFfnTokensMin), 5120 x 512 from three on by tiles.
bool rows_faster(int T, int dim, int ff, bool q8) {
    if (T == 3) return ff <= (q8 ? 256 : dim >= 2048 ? 1024 : 512) && dim < 5120;
    if (T == 4) return q8 ? ff <= 256 && dim <= 512 : ff <= 512 && dim * ff <= 1 << 18;
    return T <= 8 && !q8 && dim * ff <= 1 << 16;
}

}  // namespace

hipError_t launch_ffn_tokens(const MatRef& gate, const MatRef& up, const MatRef& down, int T, int dim, int ff,
                             const float* x, float* out, int8_t* xq, float* xd, int8_t* hq, float* hd, float lim,
                             int* err, int cus, hipStream_t s) {
    if (T < kFfnTokensMin || !dense_type(gate.type) || up.type != gate.type || !dense_type(down.type) || dim % 256 ||
        ff % 256 || rows_faster(T, dim, ff, gate.type == kQ8_0))
        return hipErrorNotSupported;
    const int nb = dim / 256, t16 = (T + 15) / 16, t32 = (T + 31) / 32, out16 = reinterpret_cast<uintptr_t>(out) % 16 == 0;
    hipLaunchKernelGGL(quant32t_kernel, dim3((T * nb + 3) / 4), dim3(256), 0, s, x, T, dim, xq, xd, err,
                       int(reinterpret_cast<uintptr_t>(x) % 16 == 0));
    // 16 tokens and both matrices at once per workgroup while the grid is at most
    // one (gate/up) or two (down) workgroups per CU: 32 tokens 36.6 us, against 59.1
    // by 32-token tiles; past that the 32-token tiles, which decode half as often
    // (64 tokens: 57.0 us).
    const auto gu = [&](auto few, auto many) {
        if (ff / kRowsT * t16 <= cus)
            hipLaunchKernelGGL(few, dim3(ff / kRowsT, t16), dim3(1024), 0, s, gate.base, up.base, T, dim, ff, xq, xd, lim,
                               hq, hd);
        else
            hipLaunchKernelGGL(many, dim3(ff / kRowsT, t32), dim3(512), 0, s, gate.base, up.base, T, dim, ff, xq, xd, lim,
                               hq, hd);
    };
    const auto dn = [&](auto few, auto many) {
        const bool one = dim / kRowsT * t16 <= 2 * cus;
        hipLaunchKernelGGL(one ? few : many, dim3(dim / kRowsT, one ? t16 : t32), dim3(512), 0, s, down.base, T, ff, dim, hq,
                           hd, out, out16);
    };
    switch (gate.type) {
    case kQ8_0: gu(ffn_gu_kernel<kQ8_0, 1, true>, ffn_gu_kernel<kQ8_0, 2, false>); break;
    case kQ4_K: gu(ffn_gu_kernel<kQ4_K, 1, true>, ffn_gu_kernel<kQ4_K, 2, false>); break;
    case kQ5_K: gu(ffn_gu_kernel<kQ5_K, 1, true>, ffn_gu_kernel<kQ5_K, 2, false>); break;
    default: gu(ffn_gu_kernel<kQ6_K, 1, true>, ffn_gu_kernel<kQ6_K, 2, false>); break;
    }
    switch (down.type) {
    case kQ8_0: dn(ffn_dn_kernel<kQ8_0, 1>, ffn_dn_kernel<kQ8_0, 2>); break;
    case kQ4_K: dn(ffn_dn_kernel<kQ4_K, 1>, ffn_dn_kernel<kQ4_K, 2>); break;
    case kQ5_K: dn(ffn_dn_kernel<kQ5_K, 1>, ffn_dn_kernel<kQ5_K, 2>); break;
    default: dn(ffn_dn_kernel<kQ6_K, 1>, ffn_dn_kernel<kQ6_K, 2>); break;
    }
    return hipGetLastError();
}

}  // namespace xl::dev
