// tc_prefill_common.hpp -- what the prefill GEMM kernels share: the launch
// arguments, stream-K work ranges, MFMA and LDS helpers, direct-to-LDS loads
// and the kernel that sums tiles split over many workgroups.
#pragma once

#include "tc_kernels.hpp"

namespace tc {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));

constexpr uint32_t PW = 8;  // waves per workgroup (two per SIMD)

struct PfArgs {
    const uint8_t *W;
    const int8_t *qs;   // block-major [nblk][M][256]
    const float *d8;    // Q4_K: [nblk][M]
    const int8_t *xs;   // Q4_K sum pieces [nblk][M][32 B]; Q8_0 d pieces [nblk][M][64 B]
    float *out;         // [M][N]
    float *ws;          // partial tiles [G][2][TT][PR]
    uint32_t *ctr;      // per tile: contributors arrived (zero before the launch, zero after it)
    uint32_t fused;     // split tiles summed by their last contributor (else by k_pf_fixup)
    uint32_t M, N, K;
    uint32_t row_bytes, nblk;
    uint32_t ntm, ntn, ntiles;  // token tiles, row blocks, tiles
    uint32_t G;                 // workgroups
    // Grouped (MoE) mode: token tile i covers rows [mt[3i], mt[3i+1]) of the
    // expert-sorted activations and uses expert mt[3i+2]'s matrix at W +
    // expert * wstride; the tile count is read from *ntm_dev (written on the
    // device by the router).
    const uint32_t *mt;
    const uint32_t *ntm_dev;
    uint64_t wstride;
    // Grouped mode with two matrices of one shape (MoE gate and up): the
    // tiles of W2 / out2 follow those of W / out in one launch.
    const uint8_t *W2;
    float *out2;
    uint32_t nb32;  // 32-blocks of a row (the last superblock of ragged Q8_0 rows has fewer than 8)
};

// A tile's token rows [m0, mend), weight matrix and output.
struct PfTile {
    uint32_t m0, mend, n0;
    const uint8_t *W;
    float *out;
};
template <bool GRP>
__device__ __forceinline__ PfTile pf_tile(const PfArgs &a, uint32_t tile, uint32_t TT, uint32_t PR) {
    PfTile t;
    if constexpr (GRP) {
        const uint32_t nt1 = *a.ntm_dev * a.ntn;  // tiles of one matrix
        const bool second = a.W2 != nullptr && tile >= nt1;
        if (second) tile -= nt1;
        const uint32_t tn = tile % a.ntn, tm = tile / a.ntn;
        t.n0 = tn * PR;
        // (wave-uniform: readfirstlane keeps them, and the load descriptors
        // built from them, in scalar registers)
        t.m0 = __builtin_amdgcn_readfirstlane(a.mt[3 * tm]);
        t.mend = __builtin_amdgcn_readfirstlane(a.mt[3 * tm + 1]);
        t.W = (second ? a.W2 : a.W) + uint64_t(__builtin_amdgcn_readfirstlane(a.mt[3 * tm + 2])) * a.wstride;
        t.out = second ? a.out2 : a.out;
    } else {
        const uint32_t tn = tile % a.ntn, tm = tile / a.ntn;
        t.n0 = tn * PR;
        t.m0 = tm * TT;
        t.mend = a.M;
        t.W = a.W;
        t.out = a.out;
    }
    return t;
}
template <bool GRP>
__device__ __forceinline__ uint32_t pf_ntiles(const PfArgs &a) {
    if constexpr (GRP)
        return *a.ntm_dev * a.ntn * (a.W2 != nullptr ? 2u : 1u);
    else
        return a.ntiles;
}

__device__ __forceinline__ v16i mfma(v4i a, v4i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v16f mfma_bf16(v4i a, v4i b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0,
                                                  0, 0);
}
__device__ __forceinline__ u4 lds4(const unsigned char *p) { return *reinterpret_cast<const u4 *>(p); }
__device__ __forceinline__ uint32_t lds1(const unsigned char *p) { return *reinterpret_cast<const uint32_t *>(p); }
__device__ __forceinline__ v4i as_v4i(u4 v) { return __builtin_bit_cast(v4i, v); }

// The lane's index recomputed where it is used (v_mbcnt on an opaque zero):
// a value the compiler cannot hoist, so that no register holds the lane
// across the kernel's loops (held, it was spilled, and the reload's wait also
// waited for the stage loads just issued).
__device__ __forceinline__ uint32_t lane_now() {
    uint32_t z = 0;
    asm volatile("" : "+s"(z));
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
}

// ---- loads into LDS ---------------------------------------------------------

// Direct-to-LDS buffer loads (no registers, no LDS stores): lane l's 16 (or
// 4) bytes land at lds_dst + 16 l (4 l). Inline, so that the compiler, which
// cannot tell which LDS bytes these write, does not wait for them before the
// wave's other LDS reads; the kernel waits (vmcnt) before its barrier. m0 (the
// LDS destination) is restored afterwards: the compiler may hold a value there.
__device__ __forceinline__ void lds_load16(uint32_t lds_dst, v4i rs, uint32_t voff) {
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "s"(__builtin_amdgcn_readfirstlane(lds_dst)), "v"(voff), "s"(rs), "s"(0u)
                 : "memory");
}
__device__ __forceinline__ void lds_load4(uint32_t lds_dst, v4i rs, uint32_t voff) {
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\tbuffer_load_dword %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "s"(__builtin_amdgcn_readfirstlane(lds_dst)), "v"(voff), "s"(rs), "s"(0u)
                 : "memory");
}

__device__ __forceinline__ v4i rs4(const void *p, uint32_t bytes) {
    const uint64_t base = reinterpret_cast<uint64_t>(p);
    return v4i{int(uint32_t(base)), int(uint32_t(base >> 32) & 0xFFFF), int(bytes), 0x00020000};
}
__device__ __forceinline__ uint32_t lds_addr(const unsigned char *p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void *)(p)));
}

// Wave instruction k of N (k = w, w + PW, ...) -- the loads of one stage are
// spread over the waves.
// Waves 0-3 issue all of a stage's loads: the second wave on each SIMD
// (w + 4) runs behind the first (the hardware favours the older wave), and
// measured 2-8% faster with no loads to issue (the first waves otherwise wait
// for it at the barrier).
constexpr uint32_t LW = 4;
template <uint32_t N, typename F>
__device__ __forceinline__ void each_inst(uint32_t w, F &&f) {
    if (w >= LW) return;
#pragma unroll
    for (uint32_t i = 0; i < (N + LW - 1) / LW; ++i) {
        const uint32_t k = w + LW * i;
        if (N % LW == 0 || k < N) f(k);
    }
}

__host__ __device__ inline uint32_t sk_begin(uint32_t units, uint32_t grid, uint32_t v) {
    return uint32_t(uint64_t(units) * v / grid);
}
// Range number of workgroup `bid`: the workgroups of one XCD take
// consecutive ranges (bid % 8 is the XCD under round-robin dispatch).
__device__ __forceinline__ uint32_t sk_logical(uint32_t bid, uint32_t G) {
    return (G & 7) ? bid : (bid & 7) * (G >> 3) + (bid >> 3);
}

// Tiles split over many workgroups (launches with more than kFusedMax
// contributors per tile): out = the partial segments summed in workgroup
// (range) order. A split tile is summed by kFixSlices(TT, PR)
// workgroups, each a slice of kFixNI float4 per thread; group j takes the
// tile holding range boundary j + 1 when that boundary splits it and is the
// first to do so. A thread issues the loads of up to kFixC contributors
// before adding them (in order, in fp64: Q4_K 3584x18944 at 8 tokens, 18 partials,
// 0.97e-7 -> 0.58e-7 from the 64-bit results, no slower), so that a CU has many
// partial lines in flight.
constexpr uint32_t kFixNI = 2;
// contributors whose loads are issued before they are added (Q4_K 5120x17408
// M = 128: 50.0 -> 48.3 us with 16 instead of 4; 8 in between)
constexpr uint32_t kFixC = 16;
__host__ __device__ constexpr uint32_t kFixSlices(uint32_t TT, uint32_t PR) { return TT * PR / 4 / (256 * kFixNI); }
template <uint32_t TT, uint32_t PR, bool GRP>
__global__ __launch_bounds__(256) void k_pf_fixup(PfArgs a) {
    constexpr uint32_t NS = kFixSlices(TT, PR);
    static_assert(NS * 256 * kFixNI * 4 == TT * PR, "a fixup slice is a whole number of 256-thread rounds");
    const uint32_t ntiles = pf_ntiles<GRP>(a);
    const uint32_t units = ntiles * a.nblk, G = a.G;
    const uint32_t slice = blockIdx.x % NS;
    const uint32_t wb = blockIdx.x / NS + 1, ubd = sk_begin(units, G, wb);
    const uint32_t tile = ubd / a.nblk;
    if (ubd % a.nblk == 0 || sk_begin(units, G, wb - 1) > tile * a.nblk) return;
    if (tile >= ntiles) return;
    const uint32_t t0 = tile * a.nblk, t1 = t0 + a.nblk;
    // contributors: the nonempty ranges from vf (the one holding t0) to vl
    // (the one holding t1 - 1); grouped launches size the grid for the
    // largest tile count, so some ranges may be empty there
    uint32_t vf = uint32_t(uint64_t(t0) * G / units);
    while (vf + 1 < G && sk_begin(units, G, vf + 1) <= t0) ++vf;
    while (vf > 0 && sk_begin(units, G, vf) > t0) --vf;
    uint32_t vl = vf;
    while (vl + 1 < G && sk_begin(units, G, vl + 1) < t1) ++vl;
    const uint32_t first_slot = sk_begin(units, G, vf) < t0 ? 1u : 0u;  // vf's second segment
    const PfTile tg_ = pf_tile<GRP>(a, tile, TT, PR);
    const uint32_t n0 = tg_.n0, m0 = tg_.m0;
    const uint32_t e0 = slice * (256 * kFixNI) + threadIdx.x;  // float4 index of item k: e0 + 256 k
    double s[kFixNI][4];
#pragma unroll
    for (uint32_t k = 0; k < kFixNI; ++k) s[k][0] = s[k][1] = s[k][2] = s[k][3] = 0.0;
    for (uint32_t v = vf; v <= vl; v += kFixC) {
        float4 p[kFixC][kFixNI];
        bool live[kFixC];
#pragma unroll
        for (uint32_t c = 0; c < kFixC; ++c) {
            const uint32_t vc = v + c;
            live[c] = vc <= vl && (!GRP || sk_begin(units, G, vc) != sk_begin(units, G, vc + 1));
            if (live[c]) {
                const float4 *src = reinterpret_cast<const float4 *>(
                    a.ws + (size_t(vc) * 2 + (vc == vf ? first_slot : 0u)) * (TT * PR));
#pragma unroll
                for (uint32_t k = 0; k < kFixNI; ++k) p[c][k] = src[e0 + 256 * k];
            }
        }
#pragma unroll
        for (uint32_t c = 0; c < kFixC; ++c) {
            if (live[c]) {
#pragma unroll
                for (uint32_t k = 0; k < kFixNI; ++k) {
                    s[k][0] += p[c][k].x;
                    s[k][1] += p[c][k].y;
                    s[k][2] += p[c][k].z;
                    s[k][3] += p[c][k].w;
                }
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kFixNI; ++k) {
        const uint32_t i = e0 + 256 * k;
        const uint32_t ml = (4 * i) / PR, nl = (4 * i) % PR;
        const uint32_t m = m0 + ml, n = n0 + nl;
        if (m >= tg_.mend) continue;
        float *o = tg_.out + size_t(m) * a.N + n;
        const float sv[4] = {float(s[k][0]), float(s[k][1]), float(s[k][2]), float(s[k][3])};
        if (n + 3 < a.N && (a.N & 3) == 0) {
            *reinterpret_cast<float4 *>(o) = make_float4(sv[0], sv[1], sv[2], sv[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < a.N) o[e] = sv[e];
        }
    }
}

// Whether some workgroup boundary of a launch cuts a tile.
inline bool pf_splits(uint32_t units, uint32_t G, uint32_t nblk) {
    for (uint32_t v = 1; v < G; ++v)
        if (sk_begin(units, G, v) % nblk != 0) return true;
    return false;
}

}  // namespace
}  // namespace tc
