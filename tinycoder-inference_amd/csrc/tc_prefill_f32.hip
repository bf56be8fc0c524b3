// tc_prefill_f32.hip -- prefill GEMM out[m][n] = W[n] . x[m] for the weight
// types whose products take fp32 activations as they are (IQ4_NL, Q5_0,
// IQ2_XS: their reference CPU paths do not quantize x), on the bf16 matrix
// cores (v_mfma_f32_32x32x16_bf16).
//
// x = h + m + l exactly, three bf16 pieces of 8 significant bits each (the
// sign and the 24 bits of an fp32; of |x| below 2^-103 what lies under the
// smallest normal number may be lost), split once per call by k_split_bf16; the
// integer weights (|q| <= 127) are exact in bf16, so every product q * piece
// is exact and only the sums round, in fp32 as in the decode kernel. Per
// 32-block (16 weights for IQ2_XS, whose scales are per 16) six (three) MFMAs
// form the sums of the m and l pieces and of the h pieces apart (the matrix
// core truncates what it adds to a larger sum: one chain over all pieces had
// 1.7e-7 of error where two have 1.1e-7); then acc += d * sum on the VALU.
//
// Sums are kept short so that rounding does not grow with K: block sums add
// up per superblock, up to kChain superblocks in the accumulator, which then
// goes into the workgroup's partial tile; partial tiles are summed in fp64.
//
// Decomposition. 8 waves of RB x TB blocks of 32 rows x 32 tokens; waves in
// TG token groups. A step is 64 columns: the three pieces of the tile's tokens
// (384 bytes each) go straight into LDS, double-buffered, with the raw weight
// blocks of 128 columns (IQ2_XS: 256). A wave instruction reads 1 KB of
// activations from LDS per 32 tokens x 16 columns, which feeds RB MFMAs of
// 32 cycles: at RB = 1 the eight waves would ask for all of the LDS
// bandwidth (128 bytes per cycle), so 128-token tiles take RB = 2.
// Work split, partial tiles and their sum as in tc_prefill.hip.
//
// Bound by MFMA and VALU issue together (per 32-block and wave at RB = TB = 2:
// 24 MFMAs of 32 cycles; ~96 conversion and 128 summing VALU instructions of 4).
// Against the decode kernel over groups of tokens (one token per launch at
// 18944 columns, whose fp32 x fills the LDS): IQ4_NL 3584x18944 M = 100 2025
// -> 89 us, 18944x3584 M = 512 8087 -> 278 us (751 TFLOP/s of bf16 work), M =
// 9 143 -> 38 us; Q5_0 and IQ2_XS M = 512 8114 -> 311 and 6383 -> 324 us.
// Error against 64-bit results (2-norm): IQ4_NL 1.1e-7 -> 0.8e-7 there, 0.94e-7
// at M = 1024; Q5_0 1.18e-7 -> 0.94e-7, IQ2_XS 1.35e-7 -> 1.06e-7.
#include <algorithm>

#include "tc_prefill_common.hpp"

namespace tc {
namespace {

// Per type: raw bytes of one weight stage in LDS per row (16-byte chunks,
// loaded CPR per row; strides whose 16-byte reads of 16 rows fall on distinct
// banks), its columns, and the bytes between stages in a row.
template <int TYPE>
struct FType;
template <>
struct FType<kIQ4_NL> {
    static constexpr uint32_t WB = 80, COLS = 128, STEP = 72, CHUNKS = 5, TAB = 0;
};
template <>
struct FType<kQ5_0> {
    static constexpr uint32_t WB = 112, COLS = 128, STEP = 88, CHUNKS = 6, TAB = 0;
};
// (74-byte units, 2-byte aligned: the window from the 4-byte-aligned start;
// the codebook as bf16, 8 magnitudes per entry, and the signs of a 7-bit index
// as xor masks)
template <>
struct FType<kIQ2_XS> {
    static constexpr uint32_t WB = 80, COLS = 256, STEP = 74, CHUNKS = 5, TAB = 512 * 16 + 128 * 16;
};

constexpr uint32_t kRows = 256;  // weight rows per workgroup tile
constexpr uint32_t kChain = 12;  // superblocks the accumulator holds

template <int TYPE, int TT>
struct FLds {
    using T = FType<TYPE>;
    static constexpr uint32_t PLANE = TT * 128;  // one piece of one step
    static constexpr uint32_t X = T::TAB;
    static constexpr uint32_t W = X + 2 * 3 * PLANE;
    static constexpr uint32_t total = W + 2 * kRows * T::WB;
};

__constant__ uint64_t c_f_iq2xs_grid[512] = {
#include "iq2xs_grid.inc"
};

// ---- the pieces of x --------------------------------------------------------

// x[m][k] as bf16 pieces: step ks (64 columns), piece p (high, middle, low),
// token m at ((3 ks + p) M + m) * 64 values. Truncations, so that each
// remainder is exact; an infinity or NaN is its own high piece.
__device__ __forceinline__ void split3(float x, uint32_t &h, uint32_t &m, uint32_t &l) {
    const uint32_t b = __builtin_bit_cast(uint32_t, x);
    const bool finite = (b & 0x7F800000u) != 0x7F800000u;
    const bool nan = !finite && (b & 0x007FFFFFu) != 0;
    h = (b >> 16) | (nan ? 0x40u : 0u);
    const float r = x - __builtin_bit_cast(float, b & 0xFFFF0000u);
    const uint32_t rb = finite ? __builtin_bit_cast(uint32_t, r) : 0u;
    m = rb >> 16;
    l = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, rb) - __builtin_bit_cast(float, rb & 0xFFFF0000u)) >> 16;
}
__global__ __launch_bounds__(256) void k_split_bf16(const float *__restrict__ x, unsigned char *__restrict__ xs,
                                                    uint32_t M, uint32_t K, uint32_t ngroups) {
    // one thread per 8 columns of a token; consecutive threads walk the
    // tokens' 64-column steps, so that a wave writes 1 KB runs of each piece
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ngroups) return;
    const uint32_t c = i & 7, mt = i >> 3, ks = mt / M, m = mt - ks * M;
    const float4 *src = reinterpret_cast<const float4 *>(x + size_t(m) * K + 64 * ks + 8 * c);
    const float4 a = src[0], b = src[1];
    const float e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    u4 o[3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split3(e[2 * k], h0, m0, l0);
        split3(e[2 * k + 1], h1, m1, l1);
        o[0][k] = h0 | (h1 << 16);
        o[1][k] = m0 | (m1 << 16);
        o[2][k] = l0 | (l1 << 16);
    }
#pragma unroll
    for (uint32_t p = 0; p < 3; ++p)
        *reinterpret_cast<u4 *>(xs + (size_t(3 * ks + p) * M + m) * 128 + 16 * c) = o[p];
}

// ---- weights to bf16 --------------------------------------------------------

// This lane's B operands of one 32-block of its row: columns 16 kh + 8 g ..
// + 7, and the scale(s).
struct FFrag {
    v4i bw[2];
    float d[2];  // (d[1]: IQ2_XS, the second 16 weights')
};

constexpr uint32_t bf16_of(float f) { return __builtin_bit_cast(uint32_t, f) >> 16; }
// Byte `hi` (0 or 1) of the bf16 of IQ4_NL's table entries 4i .. 4i + 3.
constexpr uint32_t nl_bytes(int i, int hi) {
    constexpr float kv[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
    uint32_t r = 0;
    for (int k = 0; k < 4; ++k) r |= ((bf16_of(kv[4 * i + k]) >> (8 * hi)) & 0xFFu) << (8 * k);
    return r;
}
// bf16 table values of four nibbles (bytes of nib): both bytes of each by a
// 16-entry byte lookup (entries 0-7 and 8-15 by the low 3 bits, then a pick by
// bit 3), interleaved.
__device__ __forceinline__ void nl_bf16(uint32_t nib, int &w01, int &w23) {
    constexpr uint32_t L0 = nl_bytes(0, 0), L1 = nl_bytes(1, 0), L2 = nl_bytes(2, 0), L3 = nl_bytes(3, 0);
    constexpr uint32_t H0 = nl_bytes(0, 1), H1 = nl_bytes(1, 1), H2 = nl_bytes(2, 1), H3 = nl_bytes(3, 1);
    const uint32_t low = nib & 0x07070707u, pick = ((nib >> 1) & 0x04040404u) | 0x03020100u;
    const uint32_t lo = __builtin_amdgcn_perm(__builtin_amdgcn_perm(L3, L2, low), __builtin_amdgcn_perm(L1, L0, low), pick);
    const uint32_t hi = __builtin_amdgcn_perm(__builtin_amdgcn_perm(H3, H2, low), __builtin_amdgcn_perm(H1, H0, low), pick);
    w01 = int(__builtin_amdgcn_perm(hi, lo, 0x05010400u));
    w23 = int(__builtin_amdgcn_perm(hi, lo, 0x07030602u));
}
// bf16 of q - 16 for the four bytes of q (0..31).
__device__ __forceinline__ void q5_bf16(uint32_t q, int &w01, int &w23) {
    float f[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = float((q >> (8 * k)) & 0xFFu) - 16.0f;
    w01 = int(__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f[1]), __builtin_bit_cast(uint32_t, f[0]), 0x07060302u));
    w23 = int(__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f[3]), __builtin_bit_cast(uint32_t, f[2]), 0x07060302u));
}

// 32-block 2q + bl (bl a compile-time index once unrolled, which alone decides
// the alignment) of the weight stage at `row`; sh: the unit's byte offset in
// its window (IQ2_XS).
template <int TYPE>
__device__ __forceinline__ void f_convert(const unsigned char *row, int q2, int bl, uint32_t g, uint32_t sh,
                                          const unsigned char *tab, FFrag &f) {
    if constexpr (TYPE == kIQ2_XS) {
        const int blk = q2 + bl;
        const uint16_t *u = reinterpret_cast<const uint16_t *>(row + sh);
        const float d = h2f(u[0]);
        const uint32_t scb = (uint32_t(u[33 + blk / 2]) >> (8 * (blk & 1))) & 0xFFu;
        f.d[0] = d * (0.5f + float(scb & 15u)) * 0.25f;
        f.d[1] = d * (0.5f + float(scb >> 4)) * 0.25f;
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
            const uint32_t q = u[1 + 4 * blk + 2 * kh + g];
            f.bw[kh] = as_v4i(lds4(tab + 16 * (q & 511u)) ^ lds4(tab + 512 * 16 + 16 * (q >> 9)));
        }
    } else {
        constexpr int BB = TYPE == kIQ4_NL ? 18 : 22, Q = TYPE == kIQ4_NL ? 2 : 6;
        row += BB * q2;
        f.d[0] = h2f(*reinterpret_cast<const uint16_t *>(row + BB * bl));
        // the 8 quant bytes of k-half g: from dword-aligned reads
        const int o = BB * bl + Q;
        const unsigned char *p = row + (o & ~3) + 8 * g;
        uint32_t q[2];
        if ((o & 3) == 0) {
            q[0] = lds1(p), q[1] = lds1(p + 4);
        } else {
            const uint32_t v0 = lds1(p), v1 = lds1(p + 4), v2 = lds1(p + 8);
            q[0] = __builtin_amdgcn_alignbyte(v1, v0, 2), q[1] = __builtin_amdgcn_alignbyte(v2, v1, 2);
        }
        if constexpr (TYPE == kIQ4_NL) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                int a, b;
                nl_bf16(q[i] & 0x0F0F0F0Fu, a, b);
                f.bw[0][2 * i] = a, f.bw[0][2 * i + 1] = b;
                nl_bf16((q[i] >> 4) & 0x0F0F0F0Fu, a, b);
                f.bw[1][2 * i] = a, f.bw[1][2 * i + 1] = b;
            }
        } else {
            const uint16_t *hp = reinterpret_cast<const uint16_t *>(row + BB * bl + 2);
            const uint32_t h0 = uint32_t(hp[0]) >> (8 * g), h1 = uint32_t(hp[1]) >> (8 * g);  // fifth bits: bytes g and 2 + g
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                auto bits = [&](uint32_t h) __attribute__((always_inline)) {
                    return (__umul24((h >> (4 * i)) & 15u, 0x00204081u) & 0x01010101u) << 4;
                };
                int a, b;
                q5_bf16((q[i] & 0x0F0F0F0Fu) | bits(h0), a, b);
                f.bw[0][2 * i] = a, f.bw[0][2 * i + 1] = b;
                q5_bf16(((q[i] >> 4) & 0x0F0F0F0Fu) | bits(h1), a, b);
                f.bw[1][2 * i] = a, f.bw[1][2 * i + 1] = b;
            }
        }
    }
}

// ---- stages -----------------------------------------------------------------

// The pieces of step ks for the tile's tokens: 16-byte chunk c of token t at
// slot c ^ ((t / 2) & 7) of its 128 bytes (the reads of 16 tokens fall on
// distinct banks).
template <int TYPE, int TT>
__device__ __forceinline__ void stage_x(const PfArgs &a, uint32_t m0, uint32_t ks, uint32_t dst, uint32_t w) {
    const uint32_t ln = lane_now();
    const v4i rx = rs4(a.xs, a.M * a.K * 6);
    each_inst<3 * TT / 8>(w, [&](uint32_t k) {
        const uint32_t p = k / (TT / 8), t = 8 * (k % (TT / 8)) + ln / 8;
        lds_load16(dst + 1024 * k, rx, ((3 * ks + p) * a.M + m0 + t) * 128 + 16 * ((ln & 7) ^ ((t >> 1) & 7)));
    });
}
// Weight stage gi (FType::COLS columns) of rows n0 .. n0 + 255.
template <int TYPE>
__device__ __forceinline__ void stage_w(const PfArgs &a, uint32_t n0, uint32_t gi, uint32_t dst, uint32_t w) {
    using T = FType<TYPE>;
    const uint32_t ln = lane_now();
    // (whole dwords: the range check zeroes one that is only partly in range)
    const v4i rw = rs4(a.W, (a.N * a.row_bytes + 3) & ~3u);
    constexpr uint32_t CPR = T::WB / 16;
    each_inst<kRows * CPR / 64>(w, [&](uint32_t k) {
        const uint32_t c = 64 * k + ln, r = c / CPR, p = c - CPR * r;
        lds_load16(dst + 1024 * k, rw, (((n0 + r) * a.row_bytes + gi * T::STEP) & ~3u) + 16 * min(p, T::CHUNKS - 1));
    });
}

template <int TYPE, int RB, int TB, int TG>
__global__ __launch_bounds__(64 * PW) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_prefill_f32(PfArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    using T = FType<TYPE>;
    constexpr uint32_t TT = 32 * TB * TG, PR = kRows;
    static_assert(32 * RB * PW / TG == PR, "256 rows per workgroup");
    using L = FLds<TYPE, TT>;
    constexpr int WSTEPS = T::COLS / 64;        // steps per weight stage
    constexpr uint32_t GPU = 256 / T::COLS;     // weight stages per superblock
    constexpr int NS = TYPE == kIQ2_XS ? 2 : 1;  // scales per 32-block
    const uint32_t tid = threadIdx.x;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t rg = w / TG, tg = w % TG;  // row group, token group
    auto xbuf = [&](uint32_t p) __attribute__((always_inline)) { return L::X + (p & 1) * 3 * L::PLANE; };
    auto wbuf = [&](uint32_t p) __attribute__((always_inline)) { return L::W + (p & 1) * kRows * T::WB; };
    const uint32_t lbase = lds_addr(lds);

    if constexpr (TYPE == kIQ2_XS) {
        uint32_t *t32 = reinterpret_cast<uint32_t *>(lds);
        for (uint32_t e = tid; e < 512 * 4; e += 64 * PW) {  // magnitudes 2i, 2i + 1 of an entry
            const uint32_t v = uint32_t(c_f_iq2xs_grid[e >> 2] >> (16 * (e & 3)));
            t32[e] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, float((v >> 8) & 0xFFu)),
                                           __builtin_bit_cast(uint32_t, float(v & 0xFFu)), 0x07060302u);
        }
        for (uint32_t e = tid; e < 128 * 4; e += 64 * PW) {  // the signs of 7 bits and their parity
            const uint32_t si = e >> 2, s8 = si | ((__builtin_popcount(si) & 1u) << 7), b = s8 >> (2 * (e & 3));
            t32[512 * 4 + e] = ((b & 1u) << 15) | ((b & 2u) << 30);
        }
        // first read after the first step's barrier
    }

    const uint32_t v = sk_logical(blockIdx.x, a.G);
    const uint32_t units = a.ntiles * a.nblk;
    const uint32_t ub = sk_begin(units, a.G, v), ue = sk_begin(units, a.G, v + 1);
    uint32_t px = 0, pw = 0;  // the buffers of the step and the weight stage being computed
    if (ub < ue) {
        const uint32_t tile = ub / a.nblk, b = ub - tile * a.nblk;
        const PfTile t0 = pf_tile<false>(a, tile, TT, PR);
        stage_x<TYPE, TT>(a, t0.m0, 4 * b, lbase + xbuf(px), w);
        stage_w<TYPE>(a, t0.n0, GPU * b, lbase + wbuf(pw), w);
    }
    for (uint32_t u = ub; u < ue;) {
        const uint32_t tile = u / a.nblk;
        const uint32_t b0 = u - tile * a.nblk, b1 = min(a.nblk, b0 + (ue - u));
        const bool whole = b0 == 0 && b1 == a.nblk;
        float *const part = a.ws + (size_t(v) * 2 + (u == ub ? 0 : 1)) * (TT * PR);
        u += b1 - b0;
        const uint32_t ln = lane_now(), j = ln & 31, g = ln >> 5;
        const PfTile tl = pf_tile<false>(a, tile, TT, PR);
        const uint32_t ntile = u / a.nblk;  // (u < ue: the next segment's tile, starting at superblock 0)

        // block sums of a superblock, and of the superblocks so far
        float sum[RB][TB][16], acc[RB][TB][16];
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][t][r] = sum[i][t][r] = 0.0f;

        // lane: rows 32 (RB rg + i) + j of the tile, tokens 32 (TB tg + t) + 8 q + 4 g + e
        // (the lane recomputed, so that no addresses are held across the loop)
        auto each_out = [&](auto &&f) __attribute__((always_inline)) {
            const uint32_t ln = lane_now(), j = ln & 31, g = ln >> 5;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int t = 0; t < TB; ++t)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            f(32 * (TB * tg + t) + 8 * q + 4 * g + e, 32 * (RB * rg + i) + j, acc[i][t][4 * q + e]);
        };
        uint32_t held = 0;      // superblocks in acc
        bool flushed = false;  // earlier ones are in part
        const uint32_t ge = GPU * b1;
        for (uint32_t gi = GPU * b0; gi < ge; ++gi) {
#pragma unroll 1
            for (int q = 0; q < WSTEPS; ++q) {
                __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this step's loads
                __syncthreads();
                // the next step's loads into the other buffers
                const uint32_t xn = lbase + xbuf(px + 1);
                if (q + 1 < WSTEPS) {
                    stage_x<TYPE, TT>(a, tl.m0, WSTEPS * gi + q + 1, xn, w);
                } else if (gi + 1 < ge) {
                    stage_x<TYPE, TT>(a, tl.m0, WSTEPS * (gi + 1), xn, w);
                    stage_w<TYPE>(a, tl.n0, gi + 1, lbase + wbuf(pw + 1), w);
                } else if (u < ue) {
                    const PfTile nt = pf_tile<false>(a, ntile, TT, PR);
                    stage_x<TYPE, TT>(a, nt.m0, 0, xn, w);
                    stage_w<TYPE>(a, nt.n0, 0, lbase + wbuf(pw + 1), w);
                }
                const unsigned char *xb = lds + xbuf(px) + (32 * TB * tg + j) * 128;
                const unsigned char *wb = lds + wbuf(pw) + (32 * RB * rg + j) * T::WB;
                const uint32_t sw = 16 * (g ^ ((j >> 1) & 7));
#pragma unroll
                for (int bl = 0; bl < 2; ++bl) {
                    __builtin_amdgcn_sched_barrier(0);
                    FFrag f[RB];
#pragma unroll
                    for (int i = 0; i < RB; ++i) {
                        const uint32_t sh = TYPE == kIQ2_XS ? ((tl.n0 + 32 * (RB * rg + i) + j) * a.row_bytes + gi * T::STEP) & 3u : 0u;
                        f_convert<TYPE>(wb + 32 * i * T::WB, 2 * q, bl, g, sh, lds, f[i]);
                    }
#pragma unroll
                    for (int t = 0; t < TB; ++t) {
                        __builtin_amdgcn_sched_barrier(0);
                        v4i x[3][2];
#pragma unroll
                        for (int p = 0; p < 3; ++p)
#pragma unroll
                            for (int kh = 0; kh < 2; ++kh)
                                x[p][kh] = as_v4i(lds4(xb + p * L::PLANE + 32 * 128 * t + (sw ^ (64 * bl + 32 * kh))));
#pragma unroll
                        for (int n = 0; n < NS; ++n) {  // the k-halves under scale n
                            v16f s[2][RB];  // of the lower pieces, of the high piece
#pragma unroll
                            for (int i = 0; i < RB; ++i) s[0][i] = s[1][i] = v16f{};
#pragma unroll
                            for (int p = 2; p >= 0; --p)
#pragma unroll
                                for (int kh = n; kh < (NS == 1 ? 2 : n + 1); ++kh)
#pragma unroll
                                    for (int i = 0; i < RB; ++i)
                                        s[p == 0][i] = mfma_bf16(x[p][kh], f[i].bw[kh], s[p == 0][i]);
#pragma unroll
                            for (int i = 0; i < RB; ++i)
#pragma unroll
                                for (int r = 0; r < 16; ++r)
                                    sum[i][t][r] = fmaf(f[i].d[n], s[1][i][r] + s[0][i][r], sum[i][t][r]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                px ^= 1;
            }
            pw ^= 1;
            if ((gi + 1) % GPU != 0) continue;
            if (held == kChain) {
                each_out([&](uint32_t ml, uint32_t rl, float &v) __attribute__((always_inline)) {
                    float &p = part[ml * PR + rl];
                    p = flushed ? p + v : v;
                    v = 0.0f;
                });
                held = 0;
                flushed = true;
            }
            ++held;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int t = 0; t < TB; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[i][t][r] += sum[i][t][r];
                        sum[i][t][r] = 0.0f;
                    }
        }

        each_out([&](uint32_t ml, uint32_t rl, float &v) __attribute__((always_inline)) {
            float &p = part[ml * PR + rl];
            if (flushed) v += p;
            const uint32_t m = tl.m0 + ml, n = tl.n0 + rl;
            if (!whole)
                p = v;
            else if (m < a.M && n < a.N)
                a.out[size_t(m) * a.N + n] = v;
        });
    }
}

// Tile geometry from M: 32, 64 or 128 tokens.
struct FGeom {
    uint32_t tt, ntm, ntn, ntiles, G;
};
FGeom f_geom(uint32_t M, uint32_t N, uint32_t K, int num_cu) {
    FGeom g;
    g.tt = M <= 32 ? 32 : M <= 64 ? 64 : 128;
    g.ntm = (M + g.tt - 1) / g.tt;
    g.ntn = (N + kRows - 1) / kRows;
    g.ntiles = g.ntm * g.ntn;
    const uint64_t units = uint64_t(g.ntiles) * (K / 256);
    g.G = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(uint64_t(num_cu), units)));
    return g;
}

template <int TYPE, int RB, int TB, int TG>
hipError_t f_launch(const PfArgs &a, hipStream_t st) {
    constexpr uint32_t TT = 32 * TB * TG;
    using L = FLds<TYPE, TT>;
    static_assert(L::total <= 160 * 1024, "LDS of one workgroup");
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_prefill_f32<TYPE, RB, TB, TG>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, L::total);
    if (attr != hipSuccess) return attr;
    k_prefill_f32<TYPE, RB, TB, TG><<<dim3{a.G, 1u, 1u}, 64 * PW, L::total, st>>>(a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !pf_splits(a.ntiles * a.nblk, a.G, a.nblk)) return e;
    k_pf_fixup<TT, kRows, false><<<dim3{(a.G - 1) * kFixSlices(TT, kRows), 1u, 1u}, 256, 0, st>>>(a);
    return hipGetLastError();
}
template <int TYPE>
hipError_t f_launch_tt(uint32_t tt, const PfArgs &a, hipStream_t st) {
    switch (tt) {
        case 32: return f_launch<TYPE, 1, 1, 1>(a, st);
        case 64: return f_launch<TYPE, 1, 2, 1>(a, st);
        default: return f_launch<TYPE, 2, 2, 2>(a, st);
    }
}

}  // namespace

bool prefill_f32_type(int type) { return type == kIQ4_NL || type == kQ5_0 || type == kIQ2_XS; }

size_t prefill_f32_act_bytes(uint32_t M, uint32_t K) { return size_t(M) * K * 6; }
size_t prefill_f32_workspace_bytes(uint32_t M, uint32_t N, uint32_t K, int num_cu) {
    const FGeom g = f_geom(M, N, K, num_cu);
    return size_t(g.G) * 2 * g.tt * kRows * 4;
}

hipError_t launch_prefill_f32(int type, const void *W, const float *x, float *out, uint32_t M, uint32_t N, uint32_t K,
                              int num_cu, void *act, void *workspace, hipStream_t st) {
    if (!prefill_f32_type(type) || M == 0 || N == 0 || K == 0 || K % 256 || act == nullptr || workspace == nullptr)
        return hipErrorInvalidValue;
    if (uint64_t(M) * K * 6 >= (uint64_t(1) << 32) || uint64_t(N) * (K / 256) * unit_bytes(type) >= (uint64_t(1) << 32))
        return hipErrorInvalidValue;
    const uint32_t ngroups = M * (K / 8);
    k_split_bf16<<<(ngroups + 255) / 256, 256, 0, st>>>(x, static_cast<unsigned char *>(act), M, K, ngroups);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const FGeom g = f_geom(M, N, K, num_cu);
    PfArgs a{};
    a.W = static_cast<const uint8_t *>(W);
    a.xs = static_cast<const int8_t *>(act);
    a.out = out;
    a.ws = static_cast<float *>(workspace);
    a.M = M;
    a.N = N;
    a.K = K;
    a.nblk = K / 256;
    a.row_bytes = a.nblk * unit_bytes(type);
    a.ntm = g.ntm;
    a.ntn = g.ntn;
    a.ntiles = g.ntiles;
    a.G = g.G;
    switch (type) {
        case kIQ4_NL: return f_launch_tt<kIQ4_NL>(g.tt, a, st);
        case kQ5_0: return f_launch_tt<kQ5_0>(g.tt, a, st);
        default: return f_launch_tt<kIQ2_XS>(g.tt, a, st);
    }
}

}  // namespace tc
