// tc_router.hip -- the qwen35moe MoE router on the device: the F32 router
// mat-vec (logits), the softmax over all experts, the top-k selection and the
// clamped renormalisation, bit-identical to the reference CPU router
// (src/cpp/core/ModelMoE.cpp:341-425, computeQwen35MoERouterOnly).
//
// The CPU router is the reference's exact path; its GPU kernel
// (include/gpu/GpuQwen35Kernels.hpp:931, kQ35MoeRouter) uses float exp and
// an insertion top-k and so differs from it on close and tied
// probabilities. Here every step follows the CPU's evaluation:
//  * logits: the AVX2 F32 kernel's order (SIMDMatMulVecAVX2.cpp:2982-3090):
//    32 FMA lanes (four 8-wide chains) over the 32-column steps, the leftover
//    8-column groups into chain 0, its fixed horizontal tree, then the
//    cols % 8 tail as serial FMAs;
//  * probabilities: float(exp(double(l) - maxL)), summed in double in expert
//    order, scaled by float(1 / sum) in float;
//  * selection: std::partial_sort's order, ties included (a k-entry binary
//    heap whose top is the smallest probability, replaced by each later entry
//    with a strictly larger one, then heap-sorted; the sift moves of the GNU
//    C++ library, whose tie order the result depends on);
//  * weights: p / float(max(double sum of the k, 6.103515625e-5)).
#include <type_traits>

#include "tc_kernels.hpp"

namespace tc {
namespace {

constexpr uint32_t kSelectMaxExperts = 4096;

// ---- logits -----------------------------------------------------------------
// out[s][r] = x[s] . W[r]. The evaluation order fixes 32 chains per output
// (column 32 i + j goes to chain j) and the tree that joins them, so a
// half-wave carries the 32 chains, one per lane, of a block of TS tokens x TE
// rows: per 32 columns TS + TE loads feed TS * TE FMAs.

template <int MASK>
__device__ __forceinline__ float from_xor(float v) {
    if constexpr (MASK == 1)
        return dpp_f<0xB1>(v);  // quad_perm [1,0,3,2]
    else if constexpr (MASK == 2)
        return dpp_f<0x4E>(v);  // quad_perm [2,3,0,1]
    else if constexpr (MASK == 8)
        return dpp_f<0x128>(v);  // row_ror:8
    else
        return __shfl_xor(v, MASK);
}
// One level of the joining tree over N outputs per lane: both lanes of a
// pair form the sum, so while a lane holds several outputs each keeps half of
// them (the lane with the mask's bit set the upper half); returns how many.
template <int MASK, int N, int NMAX>
__device__ __forceinline__ void join(float (&a)[NMAX], uint32_t lane) {
    if constexpr (N > 1) {
        const bool up = (lane & MASK) != 0;
#pragma unroll
        for (int o = 0; o < N / 2; ++o) {
            const float keep = up ? a[o + N / 2] : a[o], give = up ? a[o] : a[o + N / 2];
            a[o] = keep + from_xor<MASK>(give);
        }
    } else {
        a[0] += from_xor<MASK>(a[0]);
    }
}
constexpr int half_of(int n) { return n > 1 ? n / 2 : 1; }

// The joined outputs (chain 8k + j in lane 8k + j): (c_j + c_{8+j}) +
// (c_{16+j} + c_{24+j}) for j < 8, then j and j + 4, then pairs, then the two
// pairs; the cols % 8 tail as serial FMAs; and the stores. Tokens from s0,
// rows from r0; output o is token o / TE, row o % TE.
template <int TS, int TE>
__device__ __forceinline__ void finish(float (&a)[TS * TE], uint32_t lane, uint32_t s0, uint32_t r0, uint32_t S,
                                       uint32_t rows, uint32_t cols, const float *__restrict__ X,
                                       const float *__restrict__ W, float *__restrict__ out) {
    constexpr int N0 = TS * TE, N1 = half_of(N0), N2 = half_of(N1), N3 = half_of(N2), N4 = half_of(N3), N5 = half_of(N4);
    join<8, N0>(a, lane);
    join<16, N1>(a, lane);
    join<4, N2>(a, lane);
    join<1, N3>(a, lane);
    join<2, N4>(a, lane);
    // which outputs this lane holds: a level that halved them added its bit;
    // a level that did not left equal copies in both lanes
    uint32_t o0 = 0, dup = 0;
    auto level = [&](uint32_t mask, uint32_t n) __attribute__((always_inline)) {
        if (n > 1)
            o0 += (lane & mask) ? n / 2 : 0;
        else
            dup |= lane & mask;
    };
    level(8, N0);
    level(16, N1);
    level(4, N2);
    level(1, N3);
    level(2, N4);
    if (dup != 0) return;
#pragma unroll
    for (int o = 0; o < N5; ++o) {
        const uint32_t s = s0 + (o0 + o) / TE, r = r0 + (o0 + o) % TE;
        if (s >= S || r >= rows) continue;
        float v = a[o];
        for (uint32_t k = cols / 8 * 8; k < cols; ++k) v = fmaf(X[size_t(s) * cols + k], W[size_t(r) * cols + k], v);
        out[size_t(s) * rows + r] = v;
    }
}

// Whole 8-column groups left after the 32-column steps go to chains 0-7.
template <int TS, int TE>
__device__ __forceinline__ void leftover(float (&a)[TS * TE], uint32_t lane, uint32_t cols, const float *const (&x)[TS],
                                         const float *const (&w)[TE]) {
    if (lane >= 8) return;
    for (uint32_t i = cols / 32 * 32; i + 7 < cols; i += 8)
#pragma unroll
        for (int t = 0; t < TS; ++t)
#pragma unroll
            for (int e = 0; e < TE; ++e) a[t * TE + e] = fmaf(x[t][i + lane], w[e][i + lane], a[t * TE + e]);
}

// Straight from memory, U 32-column steps of loads in flight, one half-wave
// per TS x TE block: the launch is bound by load latency, so the blocks are
// small enough for two waves or more on most CUs. (The loop without loads in
// flight took 21 us at 1 token x 128 experts x 2048.)
template <int TS, int TE, int U>
__global__ __launch_bounds__(64) void k_router_logits(const float *__restrict__ W, const float *__restrict__ X, uint32_t S,
                                                      uint32_t rows, uint32_t cols, float *__restrict__ out) {
    const uint32_t lane = threadIdx.x & 31;
    const uint32_t r0 = (blockIdx.x * 2 + (threadIdx.x >> 5)) * TE, s0 = blockIdx.y * TS;
    const float *x[TS], *w[TE];
#pragma unroll
    for (int t = 0; t < TS; ++t) x[t] = X + size_t(min(s0 + t, S - 1)) * cols;
#pragma unroll
    for (int e = 0; e < TE; ++e) w[e] = W + size_t(min(r0 + e, rows - 1)) * cols;
    float a[TS * TE];
#pragma unroll
    for (int o = 0; o < TS * TE; ++o) a[o] = 0.0f;
    const uint32_t steps = cols / 32;
    uint32_t i = 0;
    auto batch = [&](auto n) __attribute__((always_inline)) {  // n steps from i
        constexpr int N = decltype(n)::value;
        float xv[N][TS], wv[N][TE];
#pragma unroll
        for (int k = 0; k < N; ++k) {
#pragma unroll
            for (int t = 0; t < TS; ++t) xv[k][t] = x[t][32 * (i + k) + lane];
#pragma unroll
            for (int e = 0; e < TE; ++e) wv[k][e] = w[e][32 * (i + k) + lane];
        }
        __builtin_amdgcn_sched_barrier(0);  // every load before the first FMA
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int t = 0; t < TS; ++t)
#pragma unroll
                for (int e = 0; e < TE; ++e) a[t * TE + e] = fmaf(xv[k][t], wv[k][e], a[t * TE + e]);
        i += N;
    };
    while (i + U <= steps) batch(std::integral_constant<int, U>{});
    while (i + 4 <= steps) batch(std::integral_constant<int, 4>{});
    while (i < steps) batch(std::integral_constant<int, 1>{});
    leftover<TS, TE>(a, lane, cols, x, w);
    finish<TS, TE>(a, lane, s0, r0, S, rows, cols, X, W, out);
}

// Many tokens: a workgroup of 8 half-waves (4 x 2 blocks of 4 x 8) computes
// 16 tokens x 16 rows from 128-column chunks in LDS, loaded one chunk ahead:
// 32 FMAs per 12 LDS reads (at a row stride that puts the two row blocks that
// a wave reads at once on different banks). cols % kChunk == 0. (8 x 8 blocks,
// half the waves: 25.0 against 20.5 us at 1024 tokens x 128 experts x 2048.)
constexpr uint32_t kTile = 16, kChunk = 128;
typedef float f4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_router_logits_tiled(const float *__restrict__ W, const float *__restrict__ X,
                                                             uint32_t S, uint32_t rows, uint32_t cols,
                                                             float *__restrict__ out) {
    __shared__ __align__(16) float lds[2][2 * kTile][kChunk + 4];  // tokens, then rows
    const uint32_t tid = threadIdx.x, lane = tid & 31, hw = tid >> 5;
    const uint32_t r0 = blockIdx.x * kTile, s0 = blockIdx.y * kTile;
    const uint32_t hs = 4 * (hw >> 1), hr = 8 * (hw & 1);
    constexpr int NL = 2 * kTile * kChunk / 4 / 256;  // float4 loads per thread and chunk
    f4 v[NL];
    // load k of this thread: columns 4 lane .. + 3 of row 8 k + hw of the chunk
    auto load = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const uint32_t q = 8 * k + hw;
            const float *p = q < kTile ? X + size_t(min(s0 + q, S - 1)) * cols : W + size_t(min(r0 + q - kTile, rows - 1)) * cols;
            v[k] = *reinterpret_cast<const f4 *>(p + c + 4 * lane);
        }
    };
    auto store = [&](uint32_t b) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NL; ++k) *reinterpret_cast<f4 *>(&lds[b][8 * k + hw][4 * lane]) = v[k];
    };
    float a[32];
#pragma unroll
    for (int o = 0; o < 32; ++o) a[o] = 0.0f;
    const uint32_t nchunk = cols / kChunk;
    load(0);
    store(0);
    for (uint32_t c = 0; c < nchunk; ++c) {
        __syncthreads();
        if (c + 1 < nchunk) load((c + 1) * kChunk);
        const uint32_t b = c & 1;
#pragma unroll
        for (int i = 0; i < int(kChunk / 32); ++i) {
            float xv[4], wv[8];
#pragma unroll
            for (int t = 0; t < 4; ++t) xv[t] = lds[b][hs + t][32 * i + lane];
#pragma unroll
            for (int e = 0; e < 8; ++e) wv[e] = lds[b][kTile + hr + e][32 * i + lane];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e) a[t * 8 + e] = fmaf(xv[t], wv[e], a[t * 8 + e]);
        }
        if (c + 1 < nchunk) store(b ^ 1);
    }
    finish<4, 8>(a, lane, s0 + hs, r0 + hr, S, rows, cols, X, W, out);
}

// ---- selection --------------------------------------------------------------

struct Scored {
    float p;
    uint32_t e;
};

__device__ __forceinline__ bool before(const Scored &a, const Scored &b) { return a.p > b.p; }

__device__ void heap_push_up(Scored *h, uint32_t hole, uint32_t top, Scored v) {
    uint32_t parent = (hole - 1) / 2;
    while (hole > top && before(h[parent], v)) {
        h[hole] = h[parent];
        hole = parent;
        parent = (hole - 1) / 2;
    }
    h[hole] = v;
}

// Sift-down of the hole to a leaf along the child not before its sibling,
// then sift-up of v.
__device__ void heap_adjust(Scored *h, uint32_t hole, uint32_t len, Scored v) {
    const uint32_t top = hole;
    uint32_t child = hole;
    while (child < (len - 1) / 2) {
        child = 2 * (child + 1);
        if (before(h[child], h[child - 1])) child--;
        h[hole] = h[child];
        hole = child;
    }
    if ((len & 1) == 0 && child == (len - 2) / 2) {
        child = 2 * (child + 1);
        h[hole] = h[child - 1];
        hole = child - 1;
    }
    heap_push_up(h, hole, top, v);
}

// Largest p of the wave in every lane (no NaN; p >= 0, whose bits order as
// integers).
__device__ __forceinline__ float wave_max_pos(float p) {
    uint32_t b = __builtin_bit_cast(uint32_t, p);
    auto mx = [&](uint32_t q) __attribute__((always_inline)) { b = b > q ? b : q; };
    mx(uint32_t(dpp_i<0xB1>(int(b))));
    mx(uint32_t(dpp_i<0x4E>(int(b))));
    mx(uint32_t(dpp_i<0x141>(int(b))));  // row_half_mirror
    mx(uint32_t(dpp_i<0x140>(int(b))));  // row_mirror
    uint32_t m = __builtin_amdgcn_readlane(b, 0);
#pragma unroll
    for (int l = 16; l < 64; l += 16) {
        const uint32_t q = __builtin_amdgcn_readlane(b, l);
        m = m > q ? m : q;
    }
    return __builtin_bit_cast(float, m);
}

// One wave per token: softmax, selection and weights. NV (E <= 64 NV, 0: any
// E): the probabilities stay in registers, and where nothing depends on the
// order of evaluation the wave works in parallel:
//  * the sum in double over the probabilities p = m 2^e (24-bit m, p <= 1) is
//    exact, so the same in any order, when the smallest nonzero p is at least
//    2^-28 E (every term is then a multiple of 2^-52 E, and no sum exceeds E);
//  * the K largest in descending order are what std::partial_sort gives when
//    they are distinct and distinct from all others.
// Otherwise (ties, tiny or NaN probabilities, K > 64) lane 0 evaluates the
// serial order below, whose dependent LDS round trips took 22 us at 1 token x
// 128 experts, top 8 and 32 us at 1024; in parallel 3.3 and 4.8.
template <int NV>
__global__ __launch_bounds__(64) void k_router_select(const float *__restrict__ logits, uint32_t E, uint32_t K,
                                                      int32_t *__restrict__ ids, float *__restrict__ wts) {
    extern __shared__ __align__(16) unsigned char smem[];
    float *prob = reinterpret_cast<float *>(smem);               // [E]
    Scored *heap = reinterpret_cast<Scored *>(smem + 4 * E);     // [K]
    const uint32_t s = blockIdx.x, lane = threadIdx.x;
    const float *l = logits + size_t(s) * E;
    float m = -__builtin_inff();
    for (uint32_t e = lane; e < E; e += 64) m = fmaxf(m, l[e]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    const double maxL = double(m);
    if constexpr (NV > 0) {
        float p[NV > 0 ? NV : 1];
        float least = 1.0f;
        bool odd = K > 64;  // needs the serial order
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const uint32_t e = lane + 64 * i;
            p[i] = -1.0f;  // past the end: below every probability
            if (e < E) {
                p[i] = float(exp(double(l[e]) - maxL));
                odd = odd || !(p[i] == p[i]);
                if (p[i] > 0.0f) least = fminf(least, p[i]);
                prob[e] = p[i];
            }
        }
        odd = odd || least < float(E) * 0x1p-28f;
        if (__ballot(odd) == 0) {
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < NV; ++i)
                if (p[i] > 0.0f) sum += double(p[i]);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
            const float inv = float(1.0 / sum);
#pragma unroll
            for (int i = 0; i < NV; ++i)
                if (p[i] >= 0.0f) p[i] *= inv;
            float rp = 0.0f;  // lane r: rank r's probability and expert
            uint32_t re = 0;
            double wsum = 0.0;
            bool tie = false;
            for (uint32_t r = 0; r < K && !tie; ++r) {
                float best = 0.0f;
#pragma unroll
                for (int i = 0; i < NV; ++i) best = fmaxf(best, p[i]);
                const float top = wave_max_pos(best);
                uint32_t hits = 0, at = 0;
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const uint64_t b = __ballot(p[i] == top);
                    hits += uint32_t(__builtin_popcountll(b));
                    if (b != 0) at = 64 * i + uint32_t(__builtin_ctzll(b));
                    if (p[i] == top) p[i] = -1.0f;
                }
                tie = hits != 1;
                if (lane == r) rp = top, re = at;
                wsum += double(top);
            }
            if (!tie) {
                const float wc = float(wsum > 6.103515625e-5 ? wsum : 6.103515625e-5);
                if (lane < K) {
                    ids[size_t(s) * K + lane] = int32_t(re);
                    wts[size_t(s) * K + lane] = __fdiv_rn(rp, wc);
                }
                return;
            }
        }
    } else {
        for (uint32_t e = lane; e < E; e += 64) prob[e] = float(exp(double(l[e]) - maxL));
    }
    __syncthreads();
    if (lane != 0) return;
    double sum = 0.0;
    for (uint32_t e = 0; e < E; ++e) sum += double(prob[e]);
    const float inv = float(1.0 / sum);
    // std::partial_sort over entries (prob[e] * inv, e): the heap of the first K,
    // each later strictly larger entry replacing the top, then the heap sort.
    for (uint32_t e = 0; e < K; ++e) heap[e] = Scored{prob[e] * inv, e};
    if (K > 1)
        for (uint32_t parent = (K - 2) / 2;; --parent) {
            heap_adjust(heap, parent, K, heap[parent]);
            if (parent == 0) break;
        }
    for (uint32_t e = K; e < E; ++e) {
        const Scored v{prob[e] * inv, e};
        if (before(v, heap[0])) heap_adjust(heap, 0, K, v);
    }
    for (uint32_t last = K; last > 1;) {
        --last;
        const Scored v = heap[last];
        heap[last] = heap[0];
        heap_adjust(heap, 0, last, v);
    }
    double wsum = 0.0;
    for (uint32_t r = 0; r < K; ++r) wsum += double(heap[r].p);
    const float wc = float(wsum > 6.103515625e-5 ? wsum : 6.103515625e-5);
    for (uint32_t r = 0; r < K; ++r) {
        ids[size_t(s) * K + r] = int32_t(heap[r].e);
        wts[size_t(s) * K + r] = __fdiv_rn(heap[r].p, wc);
    }
}

}  // namespace

hipError_t launch_router_logits(const float *W, const float *X, uint32_t S, uint32_t rows, uint32_t cols, float *out,
                                hipStream_t st) {
    if (S == 0 || rows == 0 || cols == 0 || S > 65535) return hipErrorInvalidValue;
    // The largest block that still gives 512 half-waves or more (128 experts x
    // 2048 against one token x 8 rows per workgroup: the launch takes 3.1 us
    // instead of 21 at 1 token, 20.5 instead of 182 at 1024); the tiled kernel
    // needs 16-byte aligned rows of whole chunks.
    const uint64_t outs = uint64_t(S) * rows;
    const bool vec4 = cols % kChunk == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0 &&
                      (reinterpret_cast<uintptr_t>(X) & 15) == 0;
    auto grid = [&](uint32_t ts, uint32_t te) { return dim3{(rows + 2 * te - 1) / (2 * te), (S + ts - 1) / ts, 1u}; };
    if (outs >= 512 * 64 && vec4)
        k_router_logits_tiled<<<dim3{(rows + kTile - 1) / kTile, (S + kTile - 1) / kTile, 1u}, 256, 0, st>>>(W, X, S, rows,
                                                                                                          cols, out);
    else if (outs >= 512 * 16)
        k_router_logits<4, 4, 4><<<grid(4, 4), 64, 0, st>>>(W, X, S, rows, cols, out);
    else if (outs >= 512 * 4)
        k_router_logits<2, 2, 8><<<grid(2, 2), 64, 0, st>>>(W, X, S, rows, cols, out);
    else
        k_router_logits<1, 1, 32><<<grid(1, 1), 64, 0, st>>>(W, X, S, rows, cols, out);
    return hipGetLastError();
}

hipError_t launch_router_select(const float *logits, uint32_t S, uint32_t E, uint32_t K, int32_t *ids, float *wts,
                                hipStream_t st) {
    if (S == 0 || E == 0 || K == 0 || K > E || E > kSelectMaxExperts) return hipErrorInvalidValue;
    const uint32_t lds = 4 * E + 8 * K;
    if (E <= 64)
        k_router_select<1><<<S, 64, lds, st>>>(logits, E, K, ids, wts);
    else if (E <= 128)
        k_router_select<2><<<S, 64, lds, st>>>(logits, E, K, ids, wts);
    else if (E <= 256)
        k_router_select<4><<<S, 64, lds, st>>>(logits, E, K, ids, wts);
    else if (E <= 512)
        k_router_select<8><<<S, 64, lds, st>>>(logits, E, K, ids, wts);
    else
        k_router_select<0><<<S, 64, lds, st>>>(logits, E, K, ids, wts);
    return hipGetLastError();
}

}  // namespace tc
