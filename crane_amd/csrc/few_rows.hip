// few_rows.hip -- the projections of a decode step of one sequence, with the
// residual add and RmsNorm in front of them in the same launch (gfx950); C ABI
// in include/crane_few.h.
//
// What bounds it: a small model's step is a chain of launches.  A launch in a
// replayed graph takes 2.3 us even when empty, and the add + norm and the
// SiLU * up between the projections are such launches.  With one row the norm
// is cheap enough for every wave to do itself:
//  - A wave owns a whole output: its weight row (GATED: a gate row and its up
//    row) is read in slices of 512 k, 1 KiB of consecutive bytes per load
//    instruction, non-temporal, one turn's slices all in flight before the
//    first is used.  No LDS, no barrier, no split of K: the sum ends in one
//    wave reduction, and the output is rounded once to T.
//  - Lane l holds elements 8 l .. 8 l + 7 of every slice, of the weight row and
//    of x alike, so the residual add, the sum of squares (a wave reduction) and
//    the normalised row stay in the registers the products read.  The weight
//    loads are issued first: HBM's latency runs beside the norm's.
//  - At most 512 workgroups, the turns evened out, so that the norm is not
//    repeated more than needed.
// Against the launches it replaces (add + norm, product and, gated, SiLU * up),
// one row, weights from HBM, us: Qwen3-0.6B qkv 6.2 -> 4.8, o 3.3 -> 3.2,
// gate_up 9.1 -> 5.1, down 4.5 -> 3.6; Qwen3-8B gate_up 37.2 -> 33.6, o 8.1 ->
// 7.5, down (few_long_kernel) 18.2 both; Qwen2.5-7B gate_up 49 -> 42.8.  Four rows
// do not pay (qkv 6.2 -> 8.5: the norm's arithmetic is repeated by every wave).
#include "few_merge.h"
#include "../../include/crane_few.h"

namespace crane {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kSlice = 512;    // k per slice: 64 lanes x 8
constexpr int kMaxWgs = 512;

enum Source { kFromRows, kFromNorm };

typedef unsigned int u32x4_v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint4 stream16(const bf16_t* p) {
    const u32x4_v v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_v*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_v, a), __builtin_bit_cast(bf16x2_v, b), c, false);
}

__device__ __forceinline__ void unpack8(const uint4& u, float (&v)[8]) {
    v[0] = bf16_lo(u.x); v[1] = bf16_hi(u.x); v[2] = bf16_lo(u.y); v[3] = bf16_hi(u.y);
    v[4] = bf16_lo(u.z); v[5] = bf16_hi(u.z); v[6] = bf16_lo(u.w); v[7] = bf16_hi(u.w);
}
__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
    return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                      pack_bf16x2(v[6], v[7]));
}

struct FewArgs {
    const bf16_t* x;         // the row [K]; norm: the residual stream
    const bf16_t* hidden;    // norm: added to the residual first, or null
    const bf16_t* norm_w;    // norm: [K]
    bf16_t* residual;        // norm: the new residual stream [K] when there is a hidden
    float eps;
    const bf16_t* w;         // [N, K]
    const bf16_t* bias;
    bf16_t* y;               // [N], or [N / 2] gated
    int N;
};

template <int NSL, bool GATED>
__device__ __forceinline__ void few_load(const FewArgs& p, uint4 (&wr)[NSL][GATED ? 2 : 1], int s, int row, int nout,
                                         int lane) {
    constexpr int K = kSlice * NSL;
#pragma unroll
    for (int f = 0; f < (GATED ? 2 : 1); ++f)
        wr[s][f] = stream16(p.w + (int64_t)(row + f * nout) * K + s * kSlice + 8 * lane);
}

// The products of a wave's outputs u, u + stride, ...: wr holds the slices of u,
// xv the row.
template <int NSL, bool GATED>
__device__ __forceinline__ void few_outputs(const FewArgs& p, uint4 (&wr)[NSL][GATED ? 2 : 1], const uint4 (&xv)[NSL],
                                            int u, int stride, int nout, int lane) {
    constexpr int F = GATED ? 2 : 1;
    for (; u < nout; u += stride) {
        float acc[F];
#pragma unroll
        for (int f = 0; f < F; ++f) acc[f] = 0.f;
        const int next = u + stride;
#pragma unroll
        for (int s = 0; s < NSL; ++s) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                acc[f] = dot2(wr[s][f].x, xv[s].x, acc[f]);
                acc[f] = dot2(wr[s][f].y, xv[s].y, acc[f]);
                acc[f] = dot2(wr[s][f].z, xv[s].z, acc[f]);
                acc[f] = dot2(wr[s][f].w, xv[s].w, acc[f]);
            }
            if (next < nout) few_load<NSL, GATED>(p, wr, s, next, nout, lane);
        }
        float v = wave_sum(acc[0]);
        if constexpr (GATED)
            v = silu(bf16_to_f32(f32_to_bf16(v))) * bf16_to_f32(f32_to_bf16(wave_sum(acc[F - 1])));
        else if (p.bias)
            v += bf16_to_f32(p.bias[u]);
        if (lane == 0) p.y[u] = f32_to_bf16(v);
    }
}

// One row, K = 512 NSL; wave u takes outputs u, u + waves, ...  Rounding as
// crane_hip_add_rms_norm, crane_gemm_linear and crane_hip_silu_mul: the new
// residual, m, x / m, the product with the norm weight, the projection (gated:
// each of the pair, then silu * up) are each rounded to T.
template <int NSL, int SRC, bool GATED>
__global__ __launch_bounds__(kThreads) void few_rows_kernel(FewArgs p) {
    constexpr int K = kSlice * NSL;
    constexpr int F = GATED ? 2 : 1;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nout = GATED ? p.N / 2 : p.N;
    const int stride = (int)gridDim.x * kWaves;
    int u = (int)blockIdx.x * kWaves + wave;
    if (u >= nout) return;
    const bool store_residual = SRC == kFromNorm && u == 0;
    uint4 wr[NSL][F];
#pragma unroll
    for (int s = 0; s < NSL; ++s) few_load<NSL, GATED>(p, wr, s, u, nout, lane);
    uint4 xv[NSL];
#pragma unroll
    for (int s = 0; s < NSL; ++s) xv[s] = *reinterpret_cast<const uint4*>(p.x + s * kSlice + 8 * lane);
    if constexpr (SRC == kFromNorm) {
        uint4 nw[NSL], hv[NSL];
#pragma unroll
        for (int s = 0; s < NSL; ++s) nw[s] = *reinterpret_cast<const uint4*>(p.norm_w + s * kSlice + 8 * lane);
        if (p.hidden) {
#pragma unroll
            for (int s = 0; s < NSL; ++s) hv[s] = *reinterpret_cast<const uint4*>(p.hidden + s * kSlice + 8 * lane);
        }
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < NSL; ++s) {
            float v[8];
            unpack8(xv[s], v);
            if (p.hidden) {
                float h[8];
                unpack8(hv[s], h);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += h[e];
                xv[s] = pack8(v);
                if (store_residual) *reinterpret_cast<uint4*>(p.residual + s * kSlice + 8 * lane) = xv[s];
                unpack8(xv[s], v);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(v[e], v[e], ss);
        }
        ss = wave_sum(ss);
        const float m = rt<bf16_t>(sqrtf(ss / (float)K + p.eps));
        const bool fast = m >= 0x1p-60f && m <= 0x1p60f;  // a normal, moderate divisor (div_by); else the division
        const float rm = 1.0f / m;
#pragma unroll
        for (int s = 0; s < NSL; ++s) {
            float v[8], wv[8];
            unpack8(xv[s], v);
            unpack8(nw[s], wv);
            if (fast) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = rt<bf16_t>(div_by(v[e], m, rm)) * wv[e];
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = rt<bf16_t>(v[e] / m) * wv[e];
            }
            xv[s] = pack8(v);
        }
    }
    few_outputs<NSL, GATED>(p, wr, xv, u, stride, nout, lane);
}

// One row, K past the registers (up to 32768): x in LDS, the weight slices
// through a ring of PD registers that runs on across a wave's outputs.
constexpr int kLongDepth = 8;
__global__ __launch_bounds__(kThreads) void few_long_kernel(FewArgs p, int K) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint4* xs = reinterpret_cast<uint4*>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nsl = K / kSlice, stride = (int)gridDim.x * kWaves, first = (int)blockIdx.x * kWaves + wave;
    const int steps = first < p.N ? ((p.N - first + stride - 1) / stride) * nsl : 0;
    uint4 wr[kLongDepth];
    int lrow = first, ls = 0;  // the next slice to load
    auto load = [&](int d) __attribute__((always_inline)) {
        wr[d] = stream16(p.w + (int64_t)lrow * K + ls * kSlice + 8 * lane);
        if (++ls == nsl) ls = 0, lrow += stride;
    };
#pragma unroll
    for (int d = 0; d < kLongDepth; ++d)
        if (d < steps) load(d);
    __builtin_amdgcn_sched_barrier(0);
    for (int c = threadIdx.x; c < K / 8; c += kThreads) xs[c] = reinterpret_cast<const uint4*>(p.x)[c];
    __syncthreads();
    float acc = 0.f;
    int s = 0, u = first;
    for (int i0 = 0; i0 < steps; i0 += kLongDepth) {
#pragma unroll
        for (int d = 0; d < kLongDepth; ++d) {
            if (i0 + d >= steps) break;  // uniform over the wave
            const uint4 xv = xs[s * (kSlice / 8) + lane];
            acc = dot2(wr[d].x, xv.x, acc);
            acc = dot2(wr[d].y, xv.y, acc);
            acc = dot2(wr[d].z, xv.z, acc);
            acc = dot2(wr[d].w, xv.w, acc);
            if (i0 + d + kLongDepth < steps) load(d);
            if (++s == nsl) {
                float v = wave_sum(acc);
                if (p.bias) v += bf16_to_f32(p.bias[u]);
                if (lane == 0) p.y[u] = f32_to_bf16(v);
                s = 0;
                acc = 0.f;
                u += stride;
            }
        }
    }
}

// o_proj of one sequence over its split-KV attention partials: the log-sum-exp
// merge (decode.hip's kernel 2, the same weights and roundings) runs in front
// of the product, its row in LDS: one launch less.  Each workgroup merges the
// whole row, the 16-byte pieces of up to 8 splits from L2, while its weights are
// in flight.  A sequence of one chunk has its row in p.x already.  Measured with
// the chunk kernel, 16 heads and 1024 outputs, us: 1000 keys 9.31 -> 8.76, 2000
// keys 9.25 -> 9.00, a Qwen3-0.6B step 838 -> 800.  The lines (kFewMergeSplits,
// kFewMergeOutputs, kFewMergeHeads): 12 splits 9.47 -> 10.10; 2048 outputs, with
// two workgroups a CU merging, 10.3 -> 9.9 at 1000 keys but 9.8 -> 10.4 at 2000;
// 32 heads, two pieces a thread, 12.2 -> 14.1, and 4096 outputs, where later
// turns' weights wait for the merge, 14.8 -> 17.0.
template <int NSL>
__global__ __launch_bounds__(kThreads) void few_merge_kernel(FewArgs p, const bf16_t* __restrict__ po,
                                                             const float* __restrict__ pml,
                                                             const int32_t* __restrict__ kv_len, int max_kv, int chunk,
                                                             int nsplit) {
    constexpr int S = kFewMergeSplits;
    constexpr int kPieces = NSL * kSlice / 8;
    static_assert(kPieces <= kThreads, "one piece of the row per thread");
    __shared__ uint4 xs[kPieces];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int stride = (int)gridDim.x * kWaves, u = (int)blockIdx.x * kWaves + wave;
    const bool live = u < p.N;  // uniform over the wave
    uint4 wr[NSL][1];
    if (live) {
#pragma unroll
        for (int s = 0; s < NSL; ++s) few_load<NSL, false>(p, wr, s, u, p.N, lane);
    }
    const int nc = (min(kv_len[0], max_kv) + chunk - 1) / chunk;  // chunks the sequence has, at most nsplit
    if (const int c = (int)threadIdx.x; c < kPieces) {  // piece c: dims 8 (c % 16) .. of head c / 16
        const int64_t row0 = (int64_t)(c >> 4) * nsplit;
        uint4 raw[S];
        float2 ml[S];
#pragma unroll
        for (int i = 0; i < S; ++i) {  // slots past the sequence's chunks hold stale values, dropped by selects
            const int64_t row = row0 + min(i, nsplit - 1);
            raw[i] = *reinterpret_cast<const uint4*>(po + row * kHeadDim + 8 * (c & 15));
            ml[i] = reinterpret_cast<const float2*>(pml)[row];
        }
        const uint4 one = reinterpret_cast<const uint4*>(p.x)[c];
        float M = -INFINITY;
#pragma unroll
        for (int i = 0; i < S; ++i) M = fmaxf(M, i < nc ? ml[i].x : -INFINITY);
        float den = 0.f, n[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) n[e] = 0.f;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const float w = fast_exp2(ml[i].x - M) * ml[i].y;  // a normalised partial weighs w l
            den += i < nc ? w : 0.f;
            float v[8];
            unpack8(raw[i], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) n[e] += i < nc ? w * v[e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) n[e] /= den;
        xs[c] = nc <= 1 ? one : pack8(n);
    }
    __syncthreads();
    if (!live) return;
    uint4 xv[NSL];
#pragma unroll
    for (int s = 0; s < NSL; ++s) xv[s] = xs[s * (kSlice / 8) + lane];
    few_outputs<NSL, false>(p, wr, xv, u, stride, p.N, lane);
}

// Workgroups for n outputs: at most kMaxWgs, every wave the same number of turns.
unsigned few_grid(int n) {
    const int turns = (n + kMaxWgs * kWaves - 1) / (kMaxWgs * kWaves);
    const int waves = (n + turns - 1) / turns;
    return (unsigned)((waves + kWaves - 1) / kWaves);
}

template <int SRC, bool GATED>
int launch_few(const FewArgs& a, int K, hipStream_t st) {
    const dim3 grid(few_grid(GATED ? a.N / 2 : a.N));
#define CRANE_FEW_CASE(n)                                                                                  \
    if (K == n * kSlice) {                                                                                 \
        hipLaunchKernelGGL((few_rows_kernel<n, SRC, GATED>), grid, dim3(kThreads), 0, st, a);              \
        return launch_status(hipGetLastError());                                                           \
    }
    CRANE_FEW_CASE(1) CRANE_FEW_CASE(2) CRANE_FEW_CASE(3) CRANE_FEW_CASE(4) CRANE_FEW_CASE(5) CRANE_FEW_CASE(6)
    CRANE_FEW_CASE(7) CRANE_FEW_CASE(8)
#undef CRANE_FEW_CASE
    return CRANE_HIP_E_INVALID;
}

int launch_merge(const FewArgs& a, int K, const FewMerge& m, hipStream_t st) {
    const dim3 grid(few_grid(a.N));
#define CRANE_MERGE_CASE(n)                                                                                       \
    if (K == n * kSlice) {                                                                                        \
        hipLaunchKernelGGL((few_merge_kernel<n>), grid, dim3(kThreads), 0, st, a, (const bf16_t*)m.rows, m.ml,    \
                           m.kv_len, m.max_kv, m.chunk, m.nsplit);                                                \
        return launch_status(hipGetLastError());                                                                  \
    }
    CRANE_MERGE_CASE(1) CRANE_MERGE_CASE(2) CRANE_MERGE_CASE(3) CRANE_MERGE_CASE(4)
#undef CRANE_MERGE_CASE
    return CRANE_HIP_E_INVALID;
}

bool few_takes(int64_t M, int64_t N, int64_t K, bool norm, bool gated, int dtype) {
    if (dtype != CRANE_HIP_BF16 || M != 1 || N < 1 || N > 0x3fffffff || K < kSlice || K % kSlice) return false;
    if (gated && N % 2) return false;
    return K <= (norm ? 8 * kSlice : 32768);
}

int check_few(const void* x, const void* w, const void* y, int64_t M, int64_t N, int64_t K, int dtype) {
    if (dtype != CRANE_HIP_F32 && dtype != CRANE_HIP_BF16) return CRANE_HIP_E_DTYPE;
    if (M < 0 || N <= 0 || K <= 0) return CRANE_HIP_E_INVALID;
    if (M == 0) return CRANE_HIP_OK;
    if (!x || !w || !y) return CRANE_HIP_E_INVALID;
    if (!aligned16(x) || !aligned16(w) || !aligned16(y)) return CRANE_HIP_E_ALIGN;
    return -1;  // go on
}

}  // namespace

int few_merge_linear(const FewMerge& m, const void* attn, const void* w, void* y, int N, int K, hipStream_t st) {
    FewArgs a{};
    a.x = (const bf16_t*)attn;
    a.w = (const bf16_t*)w;
    a.y = (bf16_t*)y;
    a.N = N;
    return launch_merge(a, K, m, st);
}

}  // namespace crane

using namespace crane;

extern "C" int crane_few_supported(int64_t M, int64_t N, int64_t K, int norm, int gated, int dtype) {
    return few_takes(M, N, K, norm != 0, gated != 0, dtype);
}

extern "C" int crane_few_linear(const void* x, const void* w, const void* bias, void* y, int64_t M, int64_t N,
                                int64_t K, int dtype, void* stream) {
    const int rc = check_few(x, w, y, M, N, K, dtype);
    if (rc >= 0) return rc;
    if (bias && !aligned16(bias)) return CRANE_HIP_E_ALIGN;
    if (!few_takes(M, N, K, false, false, dtype)) return CRANE_HIP_E_INVALID;
    FewArgs a{};
    a.x = (const bf16_t*)x;
    a.w = (const bf16_t*)w;
    a.bias = (const bf16_t*)bias;
    a.y = (bf16_t*)y;
    a.N = (int)N;
    if (K <= 8 * kSlice) return launch_few<kFromRows, false>(a, (int)K, (hipStream_t)stream);
    hipLaunchKernelGGL(few_long_kernel, dim3(few_grid((int)N)), dim3(kThreads), (size_t)K * 2, (hipStream_t)stream, a,
                       (int)K);
    return launch_status(hipGetLastError());
}

extern "C" int crane_few_norm_linear(const void* x, const void* hidden, const void* norm_w, void* residual, float eps,
                                     const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                                     int gated, int dtype, void* stream) {
    const int rc = check_few(x, w, y, M, N, K, dtype);
    if (rc >= 0) return rc;
    if (!(eps >= 0.0f) || !norm_w || (hidden && !residual) || (gated && bias)) return CRANE_HIP_E_INVALID;
    if (!aligned16(norm_w) || (hidden && (!aligned16(hidden) || !aligned16(residual))) || (bias && !aligned16(bias)))
        return CRANE_HIP_E_ALIGN;
    if (hidden && (residual == x || residual == hidden)) return CRANE_HIP_E_INVALID;
    if (!few_takes(M, N, K, true, gated != 0, dtype)) return CRANE_HIP_E_INVALID;
    FewArgs a{};
    a.x = (const bf16_t*)x;
    a.hidden = (const bf16_t*)hidden;
    a.norm_w = (const bf16_t*)norm_w;
    a.residual = (bf16_t*)residual;
    a.eps = eps;
    a.w = (const bf16_t*)w;
    a.bias = (const bf16_t*)bias;
    a.y = (bf16_t*)y;
    a.N = (int)N;
    return gated ? launch_few<kFromNorm, true>(a, (int)K, (hipStream_t)stream)
                 : launch_few<kFromNorm, false>(a, (int)K, (hipStream_t)stream);
}
