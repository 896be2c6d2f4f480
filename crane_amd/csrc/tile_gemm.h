// tile_gemm.h -- bf16 projections of a few to a few hundred token rows
// (y = x W^T) on LDS tiles and MFMA; instantiated by tile_rows.hip,
// tile_gated.hip and tile_parts.hip, dispatched by gemm.hip.
//
// What bounds it: the read of W.  A product of M rows does M flops per byte of
// W, against some 300 where the matrix cores would bound it (2.5 PFLOP/s over 8
// TB/s): up to a few hundred rows the kernel is a stream of W from HBM, with the
// token rows re-read from L2 by every workgroup.
//  - A workgroup of 4 waves owns 32 FT features x 32 MT token rows.  K is
//    walked in stages of 64 (128 bytes of every row): the W rows and the x rows
//    of a stage go to LDS by bounds-checked buffer_load ... lds (rows past N or
//    M read as zero), into a ring of up to 6 stages with all but one in flight
//    (40 KiB a workgroup for one tile by one, 112 to 128 for the wide forms).
//  - The waves split the stage's 64 k between them, 16 each: one
//    v_mfma_f32_32x32x16_bf16 per (feature tile, token tile) and stage, and
//    every byte of a stage is read from LDS exactly once.  The four k slices
//    meet once, at the end, through the freed ring (summed in wave order, so a
//    call's bits repeat).
//  - 16-byte chunk c of row r sits at slot c ^ (r / 2 % 8), so the 16 rows of
//    one ds_read_b128 cycle fall in 16 different bank groups.
//  - Workgroup `tile` starts its k walk at stage 5 tile % stages: rows of W
//    lie 2 K bytes apart, so workgroups that walk k in step read the same few
//    HBM channels at a time.  gate_up [24576 x 4096], 77 rows: 43.6 us started
//    in step or at stage `tile`, 39.5 us at 5 tile (3 tile: 51; the other odd
//    steps tried 39-41).
//  - W is read with the non-temporal policy when one block of token rows
//    covers M (each byte is used once: 41.1 -> 39.5 us on that shape), and by
//    the default one when several workgroups, placed on one XCD, share it.
//  - GATED: W is a merged gate_up [2 I, K].  Each 32-row tile holds 16 gate
//    rows and the 16 up rows of the same features, so accumulator e and e + 8
//    of a lane are one output's pair and the epilogue needs no exchange.
//  - PARTS: gridDim.y ranges of K, f32 sums to parts[split][M][N], unrounded.
// Time against hipBLASLt, us: gate_up with SiLU * up [24576 x 4096] at 77
// rows 53.3 -> 39.5 (5.1 TB/s of W), [37888 x 3584] 68.7 -> 54.7, at 32 rows
// 63.4 -> 44.2; down [4096 x 12288] at 77 rows 42.8 -> 28.8 (4 splits and
// their sum), [3584 x 18944] 95.8 -> 35.3; qkv [6144 x 4096] 23.6 -> 19.8;
// lm_head [151936 x 4096] at 33 rows 258.6 -> 205.1 (6.07 TB/s).
#pragma once

#include "common.h"

namespace crane {

enum TileOut { kTileRows = 0, kTileGated = 1, kTileParts = 2 };

// The form of a product: 32 ft features (GATED: 16 ft outputs) and 32 mt token
// rows per workgroup, K in `splits` ranges; ft == 0: not taken.
struct TileCfg {
    int ft, mt, splits;
};

struct TileArgs {
    const bf16_t* x;
    const bf16_t* w;
    const bf16_t* bias;  // rows only, or null
    bf16_t* y;           // rows, gated
    float* parts;        // parts
    int M, N, K;         // N: rows of W
};

// The fastest form of a product of M rows (gemm.hip), the splits' sums within
// ws_bytes; and that form where the kernel takes the product, else ft == 0.
TileCfg tile_cfg(int64_t M, int64_t N, int64_t K, bool gated, size_t ws_bytes);
TileCfg tile_route(int64_t M, int64_t N, int64_t K, bool gated, size_t ws_bytes);

// Launch one form; false when the form is not instantiated.
bool launch_tile_rows(const TileCfg& c, const TileArgs& a, hipStream_t st);
bool launch_tile_gated(const TileCfg& c, const TileArgs& a, hipStream_t st);
bool launch_tile_parts(const TileCfg& c, const TileArgs& a, hipStream_t st);

#ifdef CRANE_TILE_KERNEL

namespace {

__device__ __forceinline__ bf16x8_v tile_frag(uint4 u) { return __builtin_bit_cast(bf16x8_v, u); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

template <bool NT>
__device__ __forceinline__ void tile_copy(__amdgpu_buffer_rsrc_t src, uint8_t* dst, uint32_t vofs, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, dst, 16, vofs, soff, 0, NT ? 2 : 0);
}

template <int FT, int MT>
struct TileShape {
    static constexpr int kStage = 4096 * (FT + MT);                          // bytes: 32 rows x 128 per tile
    static constexpr int kDepth = 40 / (FT + MT) > 6 ? 6 : 40 / (FT + MT);   // stages within 160 KiB
};

// Workgroup ids congruent mod 8 run on one XCD: the token blocks of a feature
// tile follow each other there, so the second reads W from its L2.
template <int FT, int MT, int OUT, bool NTW>
__global__ __launch_bounds__(256) void tile_gemm_kernel(TileArgs p, int tiles, int tblocks) {
    constexpr int D = TileShape<FT, MT>::kDepth, kStage = TileShape<FT, MT>::kStage;
    constexpr int C = FT + MT;  // 1 KiB copies (8 rows) per wave and stage: the first FT of W, the others of x
    static_assert((D - 1) * C <= 63, "the copies in flight fit the 6-bit vmcnt");
    // one LDS object per stage: the compiler's wait-count pass then tells the
    // copies in flight apart from the stage being read
#define CRANE_TILE_SLOT(d) __shared__ __attribute__((aligned(1024))) uint8_t ring##d[D > d ? kStage : 16];
    CRANE_TILE_SLOT(0) CRANE_TILE_SLOT(1) CRANE_TILE_SLOT(2) CRANE_TILE_SLOT(3) CRANE_TILE_SLOT(4) CRANE_TILE_SLOT(5)
#undef CRANE_TILE_SLOT
    auto slot = [&](int d) -> uint8_t* {
        switch (d) {
            case 0: return ring0; case 1: return ring1; case 2: return ring2;
            case 3: return ring3; case 4: return ring4; default: return ring5;
        }
    };
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = (int)blockIdx.x / (8 * tblocks), rem = (int)blockIdx.x % (8 * tblocks);
    const int tile = grp * 8 + rem % 8, tb = rem / 8;
    if (tile >= tiles) return;  // padding ids, whole workgroups
    constexpr int kOutN = OUT == kTileGated ? 16 * FT : 32 * FT;
    const int M = p.M, K = p.K, nout = OUT == kTileGated ? p.N / 2 : p.N;
    const int kp = OUT == kTileParts ? K / (int)gridDim.y : K, k0 = OUT == kTileParts ? (int)blockIdx.y * kp : 0;
    const int nst = kp / 64;
    const int n0 = tile * kOutN, m0 = tb * 32 * MT;
    const uint32_t wbytes = (uint32_t)min(kOutN, nout - n0) * (uint32_t)K * 2u;
    const uint32_t xbytes = (uint32_t)min(32 * MT, M - m0) * (uint32_t)K * 2u;
    const bf16_t* wlo = p.w + (int64_t)n0 * K;
    const bf16_t* whi = OUT == kTileGated ? p.w + (int64_t)(nout + n0) * K : wlo;  // the up rows
    const bf16_t* xb = p.x + (int64_t)m0 * K;
    // copy i of a wave fills the 8 stage rows 8 (wave + 4 i) ..: lane l row l / 8, slot l % 8.  GATED: waves 0
    // and 1 copy gate rows (rows 0..15 of each tile), waves 2 and 3 the up rows
    uint32_t vofs[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int row = 8 * (wave + 4 * i) + (lane >> 3);
        const int src = i >= FT ? row - 32 * FT : OUT == kTileGated ? 16 * (row >> 5) + (row & 15) : row;
        vofs[i] = (uint32_t)src * (uint32_t)K * 2u + 16u * (uint32_t)((lane & 7) ^ ((row >> 1) & 7));
    }
    const int rot = tile * 5 % nst;
    // stage s into slot d; past the last stage the copies read zero bytes (a
    // resource of no bytes), so every step has the same count in flight
    auto issue = [&](int d, int s) __attribute__((always_inline)) {
        const bool live = s < nst;
        int st = s + rot;
        if (st >= nst) st -= nst;
        const int soff = live ? (k0 + 64 * st) * 2 : 0;
#pragma unroll
        for (int i = 0; i < C; ++i) {
            uint8_t* dst = slot(d) + (wave + 4 * i) * 1024;
            if (i >= FT)
                tile_copy<false>(tile_rsrc(xb, live ? xbytes : 0), dst, vofs[i], soff);
            else
                tile_copy<NTW>(tile_rsrc(OUT == kTileGated && wave >= 2 ? whi : wlo, live ? wbytes : 0), dst, vofs[i],
                               soff);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x16_v acc[FT][MT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[f][m][e] = 0.f;
    // fragments: lane l holds row l % 32 of a tile (W: the A operand, x: the B
    // operand), k 16 wave + 8 (l / 32) .. +7 of the stage
    const int r = lane & 31, h = lane >> 5;
    const int lofs = r * 128 + 16 * ((2 * wave + h) ^ ((r >> 1) & 7));
    constexpr int kFly = (D - 2) * C;
    auto step = [&](int d, int s) __attribute__((always_inline)) {
        // this wave's copies of stage s have landed (later ones fly on) and its
        // LDS reads of stage s - 1 are done; then every wave's: the slot of
        // stage s - 1 may be refilled.  A plain barrier: a release fence would
        // wait for the copies in flight.
        __builtin_amdgcn_s_waitcnt(0x0070 | (kFly & 15) | ((kFly >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        issue((d + D - 1) % D, s + D - 1);
        uint4 a[FT], b[MT];
#pragma unroll
        for (int f = 0; f < FT; ++f) a[f] = *reinterpret_cast<const uint4*>(slot(d) + f * 4096 + lofs);
#pragma unroll
        for (int m = 0; m < MT; ++m) b[m] = *reinterpret_cast<const uint4*>(slot(d) + (FT + m) * 4096 + lofs);
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                acc[f][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tile_frag(a[f]), tile_frag(b[m]), acc[f][m], 0, 0,
                                                                    0);
    };
#pragma unroll
    for (int d = 0; d < D - 1; ++d) issue(d, d);
    // whole turns of the ring, then the rest (kept apart: a branch inside the
    // turn makes the wait-count pass drain the ring at its first slot)
    int s0 = 0;
    for (; s0 + D <= nst; s0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) step(d, s0 + d);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (s0 + d < nst) step(d, s0 + d);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
    // The waves' k slices: tile u belongs to wave u % 4, the other three hand
    // theirs over through the ring (4 KiB cells, kBatch tiles a pass).
    constexpr int kBatch = C * D / 3;
    auto cell = [&](int c) -> f32x4_v* { return reinterpret_cast<f32x4_v*>(slot(c / C) + (c % C) * 4096) + lane; };
#pragma unroll
    for (int u0 = 0; u0 < FT * MT; u0 += kBatch) {
#pragma unroll
        for (int u = u0; u < (u0 + kBatch < FT * MT ? u0 + kBatch : FT * MT); ++u)
#pragma unroll
            for (int kk = 0; kk < 3; ++kk)
                if (wave == (kk < u % 4 ? kk : kk + 1)) {
                    f32x4_v* dst = cell((u - u0) * 3 + kk);
                    const f32x16_v& v = acc[u / MT][u % MT];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        dst[64 * e] = f32x4_v{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
                }
        __syncthreads();
#pragma unroll
        for (int u = u0; u < (u0 + kBatch < FT * MT ? u0 + kBatch : FT * MT); ++u) {
            if (wave != u % 4) continue;
            const int f = u / MT, m = u % MT;
            float v[16];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f32x4_v sum = {};
#pragma unroll
                for (int wv = 0; wv < 4; ++wv) {
                    if (wv == u % 4) {
                        const f32x16_v& o = acc[f][m];
                        sum += f32x4_v{o[4 * e], o[4 * e + 1], o[4 * e + 2], o[4 * e + 3]};
                    } else {
                        sum += cell((u - u0) * 3 + (wv < u % 4 ? wv : wv - 1))[64 * e];
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) v[4 * e + q] = sum[q];
            }
            // lane l holds token l % 32; element 4 e + q is feature 8 e + 4 (l / 32) + q of the tile
            const int t = m0 + 32 * m + r;
            if (t >= M) continue;
#pragma unroll
            for (int e = 0; e < (OUT == kTileGated ? 2 : 4); ++e) {
                const int n = n0 + (OUT == kTileGated ? 16 : 32) * f + 8 * e + 4 * h;
                if (n >= nout) continue;
                float o[4];
#pragma unroll
                for (int q = 0; q < 4; ++q)  // GATED: both rounded to T, then Crane's silu * up rounded once
                    o[q] = OUT == kTileGated ? silu(bf16_to_f32(f32_to_bf16(v[4 * e + q]))) *
                                                   bf16_to_f32(f32_to_bf16(v[8 + 4 * e + q]))
                                             : v[4 * e + q];
                if (OUT == kTileParts) {
                    store4(p.parts + ((int64_t)blockIdx.y * M + t) * nout + n, o);
                    continue;
                }
                if (OUT == kTileRows && p.bias) {
                    float bv[4];
                    load4(p.bias + n, bv);
#pragma unroll
                    for (int q = 0; q < 4; ++q) o[q] += bv[q];
                }
                store4(p.y + (int64_t)t * nout + n, o);
            }
        }
        if (u0 + kBatch < FT * MT) __syncthreads();
    }
}

template <int FT, int MT, int OUT>
bool launch_tile(const TileCfg& c, const TileArgs& a, hipStream_t st) {
    const int nout = OUT == kTileGated ? a.N / 2 : a.N, per = OUT == kTileGated ? 16 * FT : 32 * FT;
    const int tiles = (nout + per - 1) / per, tb = (a.M + 32 * MT - 1) / (32 * MT);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8 * tb), (unsigned)c.splits);
    if (tb == 1)
        hipLaunchKernelGGL((tile_gemm_kernel<FT, MT, OUT, true>), grid, dim3(256), 0, st, a, tiles, tb);
    else if constexpr (MT < 4)
        hipLaunchKernelGGL((tile_gemm_kernel<FT, MT, OUT, false>), grid, dim3(256), 0, st, a, tiles, tb);
    else
        return false;  // 4 token tiles only where they cover M
    return true;
}

template <int OUT>
bool launch_tile_form(const TileCfg& c, const TileArgs& a, hipStream_t st) {
#define CRANE_TILE_FORM(f, m) \
    if (c.ft == f && c.mt == m) return launch_tile<f, m, OUT>(c, a, st);
    CRANE_TILE_FORM(1, 1) CRANE_TILE_FORM(2, 1) CRANE_TILE_FORM(3, 1) CRANE_TILE_FORM(4, 1)
    CRANE_TILE_FORM(1, 2) CRANE_TILE_FORM(2, 2) CRANE_TILE_FORM(3, 2) CRANE_TILE_FORM(4, 2)
    CRANE_TILE_FORM(1, 3) CRANE_TILE_FORM(2, 3) CRANE_TILE_FORM(3, 3) CRANE_TILE_FORM(4, 3)
    CRANE_TILE_FORM(1, 4) CRANE_TILE_FORM(2, 4) CRANE_TILE_FORM(3, 4)
    if constexpr (OUT == kTileGated) {
        CRANE_TILE_FORM(5, 1) CRANE_TILE_FORM(5, 2) CRANE_TILE_FORM(5, 3)
    }
#undef CRANE_TILE_FORM
    return false;
}

}  // namespace

#endif  // CRANE_TILE_KERNEL

}  // namespace crane
