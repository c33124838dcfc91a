// CDNA4 (gfx950) row kernels of the per32 layer over bank matrices: the rows of
// every pick with the bits of mv32_kernel (xl_per32.hip; the arithmetic of the
// reference's engine/strata/warm/hip_experts.hip:17-39), 16 waves per CU.
//
// What bounded mv32_kernel here: codebook lookups. Lanes look up random rows of
// one 2- to 16-KB copy, so the 16 lanes that LDS serves at a time meet in the
// same banks, and every row reads its activations again (4x its own bytes).
// Here each lookup is one v_perm_b32 or v_and_or_b32 address into copies
// interleaved over the banks (IQ2_XXS grid and signs x32, IQ2_XS grid x16, no
// conflicts; layers of several types x16 / x8; IQ1_M value rows, one lookup per
// 8 weights, x1), x is quantized in the launch and stays in registers, the
// hidden rows are staged in LDS, and a wave loads its next two rows before it
// decodes two.
//
// Lane l of a half wave takes sub-blocks l, l + 32, ... of its row, as there;
// the integer dots are exact however they are formed, and the float chain and
// the butterfly keep their order.
//
// Per layer call, weights from HBM, mv32_kernel -> here: 4096 x 3072 IQ2, 6 picks
// 45.9 -> 33.5 us, one pick 20.7 -> 19.3, IQ1_M 63.9 -> 30.8, mixed 59.2 -> 33.8;
// 5120 x 2304 IQ2 51.5 -> 33.7; 1024 x 512 IQ2 29.5 -> 15.7 (every shape, type and
// pick count measured is faster, so the rule takes whatever fits). Rows of at
// most 5,120 values are all that a layer has; 16 waves need <= 128 registers.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "xl_dev.hpp"
#include "xl_format.hpp"
#include "xl_internal.hpp"
#include "xl_iq2.hpp"

namespace xl::dev {
namespace {

constexpr int kWaves = 16, kThreads = 64 * kWaves;
constexpr int kMaxIt = 5;          // sub-blocks per lane: rows of up to 5,120 values
constexpr int kActBytes = 27648;   // quants and scales in LDS (8 picks x 3,072 values)
constexpr int kYsFloats = 640;     // a workgroup's rows of every pick
constexpr int kMaxPicks = 16;
constexpr int kMix = 7;            // more than one block type

// LDS tables by the launch's types: [0, 64K) then [64K, 128K).
//   IQ2_XXS  grid x32 | signs x32        IQ2_XS  grid x16 | signs x32
//   IQ1_M    value rows x1 (32 KB)       mixed   rows of 16 grid then 16 sign copies | IQ2_XS grid x8, value rows
template <int MASK>
constexpr int tab_bytes() { return MASK == 4 ? 32768 : 131072; }

struct Raw {
    uint32_t w0, w1, d, s;   // IQ2: codes, fp16 d, IQ2_XS scale byte. IQ1_M: qs, qh, the block's scale words
};

struct Args {
    const ExpertDesc* descs;
    const int32_t* ids;
    int picks, n_experts, role0, n, k;
    const float* x;           // gate/up: the token's vector
    const int8_t* q;          // down: hidden quants, pick-major
    const float* d;
    float *y0, *y1;
    const uint64_t* tab;
    int* err;
    Mv32Comb cb;
    int rp;                   // down: row pairs per workgroup
};

// lane ^ 16, 8, 4, 2, 1 in this order, for each 32-lane half; each step's
// operands are those of the xor butterfly once its earlier steps have made the
// row periodic, so every lane holds the butterfly's result.
__device__ __forceinline__ float butterfly32(float v) {
    const uint32_t u = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
    v = __fadd_rn(v, dppf<0x128>(v));   // row_ror:8
    v = __fadd_rn(v, dppf<0x124>(v));   // row_ror:4
    v = __fadd_rn(v, dppf<0x122>(v));   // row_ror:2
    return __fadd_rn(v, dppf<0x121>(v));
}

template <int T>
__device__ __forceinline__ void load_raw(Raw& r, const MatRef& m, uint32_t rowblk, int kb) {
    const uint32_t blk = rowblk + uint32_t(kb >> 3);
    if constexpr (T == kIQ1_M) {
        r.w0 = *reinterpret_cast<const uint32_t*>(m.base + (size_t(rowblk) * 32 + 4 * kb));
        r.w1 = *reinterpret_cast<const uint16_t*>(m.base + m.off1 + (size_t(rowblk) * 16 + 2 * kb));
        const uint2 s = *reinterpret_cast<const uint2*>(m.base + m.off2 + size_t(blk) * 8);
        r.d = s.x;
        r.s = s.y;
    } else {
        const uint2 w = *reinterpret_cast<const uint2*>(m.base + (size_t(rowblk) * 64 + 8 * kb));
        r.w0 = w.x;
        r.w1 = w.y;
        if constexpr (T == kIQ2_XXS) {
            r.d = *reinterpret_cast<const uint16_t*>(m.base + m.off1 + size_t(blk) * 2);
        } else {
            r.s = m.base[m.off1 + (size_t(rowblk) * 8 + kb)];
            r.d = *reinterpret_cast<const uint16_t*>(m.base + m.off2 + size_t(blk) * 2);
        }
    }
}

// One sub-block: the integer sum_h s_h * dot_h and the block's d * 0.125.
template <int T, int MASK>
__device__ __forceinline__ float sub_dot(const Raw& r, int kb, const uint32_t* a, const uint8_t* lds, uint32_t lo_g,
                                         uint32_t lo_s) {
    int isum;
    uint32_t d16;
    if constexpr (T == kIQ2_XXS) {
        int acc = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint2 m = *reinterpret_cast<const uint2*>(lds + perm(r.w1, lo_s, sel_b(g)));
            const uint2 v = *reinterpret_cast<const uint2*>(lds + perm(r.w0, lo_g, sel_b(g)));
            acc = g == 0 ? sdot4_0(signed_grid(v.x, m.x), a[0]) : sdot4(signed_grid(v.x, m.x), a[2 * g], acc);
            acc = sdot4(signed_grid(v.y, m.y), a[2 * g + 1], acc);
        }
        isum = __mul24(acc, xxs_sc(r.w1));
        d16 = r.d;
    } else if constexpr (T == kIQ2_XS) {
        int part[2];
        const uint32_t copy = lo_g & 255u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t w = g < 2 ? r.w0 : r.w1;
            const uint2 m = *reinterpret_cast<const uint2*>(lds + perm(w, lo_s, sel_b(2 * (g & 1))));
            const uint32_t c = (g & 1) ? w >> 16 : w;   // sign7 | grid9 << 7: 128-B rows need no shift
            const uint32_t at = MASK == kMix ? 65536u + (((c >> 1) & 0x7fc0u) | (copy & 0x38u)) : ((c & 0xff80u) | (copy & 0x78u));
            const uint2 v = *reinterpret_cast<const uint2*>(lds + at);
            int& acc = part[g >> 1];
            acc = (g & 1) ? sdot4(signed_grid(v.x, m.x), a[2 * g], acc) : sdot4_0(signed_grid(v.x, m.x), a[2 * g]);
            acc = sdot4(signed_grid(v.y, m.y), a[2 * g + 1], acc);
        }
        isum = __mul24(part[0], int(2u * (r.s & 15u) + 1u)) + __mul24(part[1], int(2u * (r.s >> 4) + 1u));
        d16 = r.d;
    } else {
        int part[2];
        constexpr uint32_t base = MASK == kMix ? 98304u : 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t row = ((r.w0 >> (8 * g)) & 255u) | (((r.w1 >> (4 * g)) & 15u) << 8);
            const uint2 v = *reinterpret_cast<const uint2*>(lds + base + 8u * row);
            int& acc = part[g >> 1];
            acc = (g & 1) ? sdot4(v.x, a[2 * g], acc) : sdot4_0(v.x, a[2 * g]);
            acc = sdot4(v.y, a[2 * g + 1], acc);
        }
        const int ib = kb & 7;
        const uint32_t w = ((ib & 4) ? r.s : r.d) >> (16 * ((ib >> 1) & 1) + 6 * (ib & 1));
        isum = __mul24(part[0], int(2u * (w & 7u) + 1u)) + __mul24(part[1], int(2u * ((w >> 3) & 7u) + 1u));
        d16 = ((r.d >> 12) & 0xfu) | ((r.d >> 24) & 0xf0u) | ((r.s >> 4) & 0xf00u) | ((r.s >> 16) & 0xf000u);
    }
    return __fmul_rn(__fmul_rn(h2f(d16), 0.125f), float(isum));
}

// copies 16-byte pairs of table row v: chunk c of the rows' copies
__device__ __forceinline__ void put2(uint8_t* lds, int c, uint64_t v) {
    reinterpret_cast<ulonglong2*>(lds)[c] = make_ulonglong2(v, v);
}

// GU: the gate and up rows of every pick (x quantized here); the waves of the
// grid take row pairs wave-major, so every CU gets the same number to within one
// per wave. Else the down rows: workgroup b owns row pairs [b * rp, ...) of every
// pick, so that it can join them in the combine's order.
template <int IT, int MASK, bool GU>
__global__ __launch_bounds__(kThreads) void rows32_kernel(Args A) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[tab_bytes<MASK>()];
    __shared__ __attribute__((aligned(16))) uint8_t act[GU ? IT * 1024 * 9 / 8 : kActBytes];
    __shared__ float ys[GU ? 1 : kYsFloats];
    __shared__ MatRef s_mat[2 * kMaxPicks];
    __shared__ int s_ok[kMaxPicks], s_order[kMaxPicks];
    const int tid = int(threadIdx.x), lane = tid & 63, l = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nk = A.k / 32, na = GU ? 1 : A.picks;
    float* actd = reinterpret_cast<float*>(act + na * A.k);

    if (tid < A.picks) {
        const int id = A.ids[tid];
        const bool ok = id >= 0 && id < A.n_experts;
        if (!ok && blockIdx.x == 0) atomicOr(A.err, kDevErrExpertId);
        s_ok[tid] = ok;
        s_mat[2 * tid] = A.descs[ok ? id : 0].m[A.role0];   // an invalid pick's rows are read from expert 0 and dropped
        if (GU) s_mat[2 * tid + 1] = A.descs[ok ? id : 0].m[A.role0 + 1];
        int rank = 0;   // combine_one's order: ascending expert id, equal ids in pick order
        for (int j = 0; j < A.picks; ++j) rank += A.ids[j] < id || (A.ids[j] == id && j < tid);
        s_order[rank] = tid;
    }
    // tables
    if constexpr (MASK == 1 || MASK == 2) {
        for (int c = tid; c < 4096; c += kThreads) {
            put2(lds, c, MASK == 1 ? A.tab[256 + (c >> 4)] : A.tab[512 + (c >> 3)]);
            put2(lds + 65536, c, A.tab[2 * ((c >> 4) & 127)]);
        }
    } else if constexpr (MASK == 4) {
        for (int c = tid; c < 2048; c += kThreads)
            reinterpret_cast<uint4*>(lds)[c] = reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(A.tab) + kTableIQ1X)[c];
    } else {
        for (int c = tid; c < 4096; c += kThreads) put2(lds, c, (c & 8) ? A.tab[2 * ((c >> 4) & 127)] : A.tab[256 + (c >> 4)]);
        for (int c = tid; c < 2048; c += kThreads) {
            put2(lds + 65536, c, A.tab[512 + (c >> 2)]);
            reinterpret_cast<uint4*>(lds + 98304)[c] =
                reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(A.tab) + kTableIQ1X)[c];
        }
    }
    // activations
    if constexpr (GU) {
        bool bad = false;
        for (int i = tid; i < A.k; i += kThreads) {   // quant32_kernel's arithmetic; k is a multiple of 256
            const float v = A.x[i];
            float am = fabsf(v);
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o, 32));
            bad = bad || !(fabsf(v) <= 3.402823466e38f);
            const float sc = __fdiv_rn(am, 127.0f);
            reinterpret_cast<int8_t*>(act)[i] = int8_t(am > 0.0f ? __float2int_rn(__fdiv_rn(v, sc)) : 0);
            if ((i & 31) == 0) actd[i >> 5] = sc;
        }
        if (bad && blockIdx.x == 0) atomicOr(A.err, kDevErrNonFinite);
    } else {
        for (int i = tid; i < na * A.k / 16; i += kThreads)
            reinterpret_cast<uint4*>(act)[i] = reinterpret_cast<const uint4*>(A.q)[i];
        for (int i = tid; i < na * nk; i += kThreads) actd[i] = A.d[i];
    }
    __syncthreads();

    const uint32_t lo_g = 8u * uint32_t(MASK == kMix ? lane & 15 : l);
    const uint32_t lo_s = MASK == kMix ? lo_g + 128u : lo_g | 0x10000u;
    const int hp = A.n / 2;   // n is a multiple of 256
    const int rp0 = GU ? 0 : int(blockIdx.x) * A.rp;
    const int rpb = GU ? hp : min(A.rp, hp - rp0);
    const int total = GU ? 2 * A.picks * hp : A.picks * rpb;
    const int step = GU ? kWaves * int(gridDim.x) : kWaves;
    const int first = GU ? wave * int(gridDim.x) + int(blockIdx.x) : wave;

    uint32_t a[IT][8];
    float xd[IT];
    const auto load_act32 = [&](int pick) {
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int kr = l + 32 * it, kb = kr < nk ? kr : 0;
            const uint4* p = reinterpret_cast<const uint4*>(act + pick * A.k + 32 * kb);
            const uint4 lo = p[0], hi = p[1];
            a[it][0] = lo.x; a[it][1] = lo.y; a[it][2] = lo.z; a[it][3] = lo.w;
            a[it][4] = hi.x; a[it][5] = hi.y; a[it][6] = hi.z; a[it][7] = hi.w;
            xd[it] = actd[pick * nk + kb];
        }
    };
    if constexpr (GU) load_act32(0);

    struct Unit {
        MatRef m;
        int pick, role, row;
        uint32_t rowblk;
    };
    const auto unit = [&](int u) {
        Unit U;
        const int slot = u / rpb, rp = u - slot * rpb;
        const int mi = GU ? slot : 2 * slot;   // (pick, role)
        U.pick = GU ? slot >> 1 : slot;
        U.role = GU ? slot & 1 : 0;
        const uint64_t b = reinterpret_cast<uint64_t>(s_mat[mi].base);
        const auto s64 = [](uint64_t v) {
            return uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))))) |
                   uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))))) << 32;
        };
        U.m.base = reinterpret_cast<const uint8_t*>(s64(b));
        U.m.off1 = s64(s_mat[mi].off1);
        U.m.off2 = s64(s_mat[mi].off2);
        U.m.type = __builtin_amdgcn_readfirstlane(s_mat[mi].type);
        U.m.nb = nk >> 3;
        U.row = 2 * (rp0 + rp) + half;
        U.rowblk = uint32_t(U.row) * uint32_t(U.m.nb);
        return U;
    };
    const auto fetch = [&]<int T>(const Unit& U, Raw* R) {
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int kr = l + 32 * it;
            load_raw<T>(R[it], U.m, U.rowblk, kr < nk ? kr : 0);
        }
    };
    const auto rows = [&]<int T>(const Raw* R) {
        float acc = 0.0f;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int kr = l + 32 * it;
            const float next = fmaf(xd[it], sub_dot<T, MASK>(R[it], kr, a[it], lds, lo_g, lo_s), acc);
            acc = kr < nk ? next : acc;
        }
        return acc;
    };
    const auto finish = [&](const Unit& U, float acc) {
        const float v = __fadd_rn(butterfly32(acc), 0.0f);
        if (l == 0 && s_ok[U.pick]) {
            (U.role ? A.y1 : A.y0)[size_t(U.pick) * A.n + U.row] = v;
            if constexpr (!GU) ys[U.pick * 2 * A.rp + U.row - 2 * rp0] = v;
        }
    };
    if constexpr (MASK == kMix) {   // a type per unit: its loads inside its branch, other waves in flight meanwhile
        for (int u = first; u < total; u += step) {
            const Unit U = unit(u);
            if constexpr (!GU) load_act32(U.pick);
            const auto one = [&]<int T>() {
                Raw R[IT];
                fetch.template operator()<T>(U, R);
                finish(U, rows.template operator()<T>(R));
            };
            if (U.m.type == kIQ2_XXS) one.template operator()<kIQ2_XXS>();
            else if (U.m.type == kIQ2_XS) one.template operator()<kIQ2_XS>();
            else one.template operator()<kIQ1_M>();
        }
    } else {
        constexpr int T = MASK == 1 ? int(kIQ2_XXS) : MASK == 2 ? int(kIQ2_XS) : int(kIQ1_M);
        if (first < total) {
            // two operand sets in turn, so that no copy of a register waits for the load in flight
            Raw R0[IT], R1[IT];
            Unit U0 = unit(first), U1 = U0;
            fetch.template operator()<T>(U0, R0);
            for (int u = first;;) {
                int v = u + step;
                U1 = unit(v < total ? v : u);
                fetch.template operator()<T>(U1, R1);
                if constexpr (!GU) load_act32(U0.pick);
                finish(U0, rows.template operator()<T>(R0));
                u = v;
                if (u >= total) break;
                v = u + step;
                U0 = unit(v < total ? v : u);
                fetch.template operator()<T>(U0, R0);
                if constexpr (!GU) load_act32(U1.pick);
                finish(U1, rows.template operator()<T>(R1));
                u = v;
                if (u >= total) break;
            }
        }
    }
    if constexpr (!GU) {
        if (!A.cb.out) return;
        __syncthreads();
        if (tid < 2 * rpb) {
            float c = 0.0f;   // fma(w, y, .) in the combine's order from +0, then + shared
            for (int i = 0; i < A.picks; ++i) {
                const int p = s_order[i];
                if (s_ok[p]) c = fmaf(A.cb.w[p], ys[p * 2 * A.rp + tid], c);
            }
            const int row = 2 * rp0 + tid;
            A.cb.out[row] = A.cb.shared ? __fadd_rn(c, A.cb.shared[row]) : c;
        }
    }
}

template <int IT, bool GU>
void go_mask(int mask, int grid, const Args& a, hipStream_t s) {
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, s, a); };
    if (mask == 1) go(rows32_kernel<IT, 1, GU>);
    else if (mask == 2) go(rows32_kernel<IT, 2, GU>);
    else if (mask == 4) go(rows32_kernel<IT, 4, GU>);
    else go(rows32_kernel<IT, kMix, GU>);
}
template <bool GU>
hipError_t launch(int mask, int grid, const Args& a, hipStream_t s) {
    switch ((a.k / 32 + 31) / 32) {
    case 1: go_mask<1, GU>(mask, grid, a, s); break;
    case 2: go_mask<2, GU>(mask, grid, a, s); break;
    case 3: go_mask<3, GU>(mask, grid, a, s); break;
    case 4: go_mask<4, GU>(mask, grid, a, s); break;
    default: go_mask<5, GU>(mask, grid, a, s); break;
    }
    return hipGetLastError();
}
bool shape_ok(int picks, int n, int k) {
    return picks >= 1 && picks <= kMaxPicks && n >= 256 && n % 256 == 0 && k >= 256 && k % 256 == 0 && k <= 1024 * kMaxIt;
}

}  // namespace

hipError_t launch_gate_up32(const ExpertDesc* descs, const int32_t* ids, int picks, int n_experts, int mask, int n,
                            int k, const float* x, float* g, float* u, const uint64_t* tables, int cus, int* err,
                            hipStream_t s) {
    if (!shape_ok(picks, n, k)) return hipErrorInvalidValue;
    Args a{};
    a.descs = descs; a.ids = ids; a.picks = picks; a.n_experts = n_experts; a.role0 = 0; a.n = n; a.k = k;
    a.x = x; a.y0 = g; a.y1 = u; a.tab = tables; a.err = err;
    const int waves = picks * n;   // row pairs of both roles
    return launch<true>(mask, std::min(cus, (waves + kWaves - 1) / kWaves), a, s);
}

// hipErrorNotSupported: the hidden rows of all picks or a workgroup's outputs do
// not fit beside the 128 KB of tables (more than 8 picks of 3,072 values; one
// limit for all instances, though IQ1_M's tables of 32 KB would leave room);
// mv32_kernel, which stages neither, takes those.
hipError_t launch_down32(const ExpertDesc* descs, const int32_t* ids, int picks, int n_experts, int mask, int n, int k,
                         const int8_t* q, const float* d, float* y, const Mv32Comb& cb, const uint64_t* tables, int cus,
                         int* err, hipStream_t s) {
    const int rp = (n / 2 + cus - 1) / cus;
    if (!shape_ok(picks, n, k) || picks * (k + k / 8) > kActBytes || 2 * rp * picks > kYsFloats || 2 * rp > kThreads)
        return hipErrorNotSupported;
    Args a{};
    a.descs = descs; a.ids = ids; a.picks = picks; a.n_experts = n_experts; a.role0 = 2; a.n = n; a.k = k;
    a.q = q; a.d = d; a.y0 = y; a.tab = tables; a.err = err; a.cb = cb; a.rp = rp;
    return launch<false>(mask, (n / 2 + rp - 1) / rp, a, s);
}

}  // namespace xl::dev
