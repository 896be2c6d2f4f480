// prefill.hip -- causal GQA flash prefill over Crane's [B, Hkv, cap, D] cache (gfx950).
//
// Replaces the prefill SDPA of qwen3/modeling.rs:469-502 (K/V expanded to Hq
// heads, (q@K^T)*scale, + the causal -1e9 mask of :866-884, softmax_last_dim,
// @V, transpose to [B,S,Hq*D]); the same op chain is in
// hunyuan_dense/modeling.rs:610-645 and qwen2.rs:191-211 (-inf mask).  The
// [S, start+S] score matrix is never materialised: scores live in registers,
// the softmax is online (running max and sum per query row, log2 domain) and
// key tiles that lie entirely above the diagonal are never visited.
//
// bf16 kernel (MFMA): a workgroup owns 128 query rows of one q head (4 waves
// x 32 rows).  Each wave computes S^T = K Q^T with v_mfma_f32_32x32x16_bf16,
// so a lane holds 16 keys of ONE query row (lane%32) and the row max/sum need
// one cross-half exchange only.  The resulting P^T tile is already laid out as
// the B operand of O^T = V^T P^T: no data movement between the two products.
// K and V tiles are copied HBM -> LDS row-major, as Crane stores them, by
// bounds-checked buffer_load ... lds (no VGPRs, no VALU, zero rows past the
// cache end), double-buffered so tile t+1 is in flight while tile t is
// computed.  K rows are the A operand of the first product; the second
// product's A operand V^T comes from the same row-major tile through
// ds_read_b64_tr_b16 transposed reads.  16-byte chunks are XOR-swizzled per
// row so both read patterns avoid LDS bank conflicts.
// Workgroup ids are remapped so that heavy (late) query tiles start first and
// the q heads sharing a kv head run on the same XCD (shared L2).
//
// The key loop's step (one 64-key tile: the P V of the tile before, the
// scores of the tile after, the softmax of this one) is a single inline-asm
// statement generated by gen_prefill_step.py (prefill_step.inc) over a fixed
// register map, so that the MFMAs of one half interleave with the VALU work
// of the other at the hardware's wait states instead of where the compiler's
// scheduler leaves them.  The online softmax moves its reference max lazily:
// p = exp2(s * fac - m) is computed against the row's current m, and only
// when some lane's sum of p passes 256 (or is not finite) is the tile's max
// taken, O and l scaled and p computed again from the intact scores.  The
// output is the same function of the scores either way (m cancels between O
// and l), up to f32 rounding.
//
// Rounding points (bf16): candle's bf16 matmul returns Q K^T rounded to bf16,
// and its affine multiplies that by the scale converted to bf16 and rounds the
// product to bf16 again (qwen3/modeling.rs:488).  Every score reproduces both
// roundings by default: each rounding is a v_cvt_pk_bf16_f32 with a zero low
// half, read back as an f32, and the product of the two bf16 values is exact
// in f32 (a v_mul_f32).  With CRANE_HIP_PREFILL_LONG_ROWS_ONE_ROUNDING,
// workgroups whose first row sees at least kLongRowKeys keys keep the first
// rounding only and fold the scale into the exp2 argument's FMA (two VALU
// instructions fewer per score, about 7% of the time at config 4); over that
// many keys the second rounding's effect on an output averages out (1.3e-3
// more mean-relative distance from candle's chain on such rows).
// candle's softmax_last_dim then rounds s - max, exp, the row sum and the
// quotient p = e / sum to bf16 before the P V product (:493-494).  A one-pass
// kernel only has the row's max and sum at the end, so for rows with more than
// one 64-key tile these roundings are not reproduced: the online softmax keeps
// them in f32, P enters the P V product in bf16, and the row sum l adds the
// same bf16 p (v_dot2_f32_bf16 against (1, 1)), so numerator and denominator
// see the same weights.  A wave whose 32 rows all see keys of the first tile
// only (the first rows of a causal prefill, where few keys carry large
// weights and candle's roundings move the output most) runs candle's chain
// exactly: the row max, e = bf16(exp(bf16(s - max))), the bf16 sum, p =
// bf16(e / sum) (a correctly rounded division), and O = P V without a final
// division.
//
// f32 kernel: the same workgroup shape on v_mfma_f32_32x32x2_f32 with 32-key
// f32 tiles (see prefill_f32_kernel); candle's f32 path has no intermediate
// rounding to reproduce.  Crane serves prefill in bf16 on GPU
// (crane-serve/src/lib.rs:123-150); f32 is the operator's other dtype.
#include <atomic>
#include <type_traits>

#include "common.h"

namespace crane {
namespace {

#ifndef CRANE_PREFILL_WAVES
#define CRANE_PREFILL_WAVES 4
#endif
constexpr int kWaves = CRANE_PREFILL_WAVES;   // waves per workgroup, 32 query rows each
constexpr int kBM = 32 * kWaves;              // query rows per workgroup
constexpr int kCopies = 16 / kWaves;          // 1 KiB blocks of a 16 KiB tile each wave copies
constexpr int kBN = 64;                       // keys per tile
constexpr int kTileBytes = kBN * kHeadDim * 2;  // 16 KiB of K (or V) per tile
constexpr float kMaskRaw = -1.0e30f;          // raw score of a masked key (finite: see scores_bf16)
constexpr int kLongRowKeys = 1024;           // keys a workgroup's first row sees for its rows to be long

__device__ __forceinline__ f32x16_v mfma32(bf16x8_v a, bf16x8_v b, f32x16_v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8_v as_bf16x8(uint4 u) { return __builtin_bit_cast(bf16x8_v, u); }

// LDS tiles keep Crane's row-major rows (256 B per key, a full sweep of the 64
// banks) with the 16-byte chunks of row r XOR-permuted by swz(r), which swaps
// the two 2-bit halves of r mod 16.  Then 16 consecutive rows read at one chunk
// index (K fragments, 16 lanes per cycle) hit 16 different chunks, and a
// transposed V read (32 lanes per cycle: 4 rows x 4 consecutive chunks) hits
// 16 different chunks, so neither read pattern has bank conflicts.
__device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4_v;
typedef __attribute__((address_space(3))) s16x4_v lds_s16x4_v;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}

// Copy keys [64 t, 64 t + 64) of K (or V) into one 16 KiB LDS buffer with
// bounds-checked buffer_load ... lds (rows past the cache rows read as zero).
// Wave w copies the 1 KiB blocks kCopies*w .. +kCopies-1 of the tile; lane l of
// block blk fills row 4 blk + l/16, chunk l%16, with global chunk (l%16) ^ swz(row).
// NC: the blocks each wave copies (16 / waves of the workgroup).
template <int NC = kCopies>
__device__ __forceinline__ int copy_voffset(int i, int wave, int lane) {
    const int row = 4 * (wave * NC + i) + (lane >> 4);
    return row * (kHeadDim * 2) + 16 * ((lane & 15) ^ swz(row));
}
// vofs[i] = copy_voffset(i, ...): the lane part of the source offset, fixed per
// lane; the tile part (t * 16 KiB) is the wave-uniform soffset.
template <int NC>
__device__ __forceinline__ void issue_tile(__amdgpu_buffer_rsrc_t rsrc, int t, int wave, const uint32_t (&vofs)[NC],
                                           uint8_t* dst) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, dst + (wave * NC + i) * 1024, 16, vofs[i], t * kTileBytes,
                                                 0, 0);
}

// s_waitcnt with only vmcnt constrained (expcnt and lgkmcnt at their maxima).
#define CRANE_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))

// candle's bf16 rounding of an f32 (round to nearest even), read back as an
// f32: v_cvt_pk_bf16_f32 with a zero low half.  Written as an instruction
// because the compiler rounds into the low half and moves it up.  A masked
// key carries the finite raw score kMaskRaw, which stays a huge negative
// score through both roundings.
__device__ __forceinline__ float round_bf16(float x) {
    float r;
    asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r) : "v"(x));
    return r;
}
// candle's bf16 score of a raw f32 product: s = bf16(bf16(acc) * scale), with
// scale a bf16 value held as an f32.  The product of two bf16 values is exact
// in f32, so a plain v_mul_f32 forms it: no v_dot2_f32_bf16, which on gfx950
// does not run beside the MFMAs (a dot2 and an MFMA stream on one SIMD take
// longer together than one after the other).
__device__ __forceinline__ float score_bf16(float acc, float scale) { return round_bf16(round_bf16(acc) * scale); }

// Keep a value in a register as computed: the compiler may not split it into
// a base plus a per-use offset (which would cost an add per use in the loop).
__device__ __forceinline__ uint32_t pinned(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Map the 1-D workgroup id to (q tile, sequence, q head).  Groups of
// 8*n_rep consecutive ids hold 8 (qtile, b, kv head) units x n_rep heads, laid
// out so that ids congruent mod 8 (dispatched to the same XCD) share a unit.
// Units are ordered heaviest (last q tile) first.  Returns false for padding ids.
__device__ __forceinline__ bool map_block(int id, int n_qt, int B, int Hkv, int n_rep, int& qt, int& b, int& hq) {
    const int chunk = 8 * n_rep;
    const int c = id / chunk, rem = id % chunk;
    const int r = rem / 8, x = rem % 8;
    const int unit = c * 8 + x;
    const int n_units = n_qt * B * Hkv;
    if (unit >= n_units) return false;
    const int qt_rank = unit / (B * Hkv);
    const int rest = unit % (B * Hkv);
    b = rest / Hkv;
    const int kvh = rest % Hkv;
    qt = n_qt - 1 - qt_rank;
    hq = kvh * n_rep + r;
    return true;
}

typedef __attribute__((__vector_size__(16 * sizeof(int)))) int i32x16_v;
typedef __attribute__((__vector_size__(32 * sizeof(int)))) int i32x32_v;
typedef __attribute__((__vector_size__(8 * sizeof(uint32_t)))) uint32_t u32x8_v;

// The steady-state step as assembly (generated by gen_prefill_step.py).
#include "prefill_step.inc"

// LDS byte address of a __shared__ location, and reads at such an address.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_v;
__device__ __forceinline__ uint4 lds_read16(uint32_t a) {
    const u32x4_v v = *(const __attribute__((address_space(3))) u32x4_v*)(uintptr_t)a;
    return make_uint4(v[0], v[1], v[2], v[3]);
}
// ds_read_b64_tr_b16: within each 16-lane group, lane i supplies 4 consecutive
// bf16 x[i][0..3] and receives x[4k + i/4][i%4] for k = 0..3.  With lane i
// pointing at row base + i/4, columns c0 + 4(i%4) .. +3 of a row-major tile,
// lane i receives column c0 + i of rows base .. base + 3: a transposed read.
__device__ __forceinline__ uint2 lds_read_tr16(uint32_t a) {
    const s16x4_v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_v*)(uintptr_t)a);
    return __builtin_bit_cast(uint2, v);
}

// One step of the key loop as assembly (prefill_step.inc, written by
// gen_prefill_step.py, which documents the register map, the step's cases and
// the flags).  The O accumulators, Q fragments, score sets and LDS addresses
// are operands in the registers the assembly names, and the loop body is two
// such statements and nothing else touching them, so they stay there.
template <int PAR, int R>
__device__ __forceinline__ void pf_step(f32x16_v (&o)[4], const i32x16_v (&qq)[2], f32x16_v (&s)[4], i32x16_v& pb,
                                        u32x8_v ko, u32x8_v vo, float& m_run, float& l_run, int flags, int thr,
                                        int xaddr, float fac, float scale) {
    i32x32_v scratch;
#define CRANE_PF_ASM(TEXT)                                                                                            \
    asm volatile(TEXT                                                                                                 \
                 : "+{v[0:15]}"(o[0]), "+{v[16:31]}"(o[1]), "+{v[32:47]}"(o[2]), "+{v[48:63]}"(o[3]),                 \
                   "+{v[96:111]}"(s[0]), "+{v[112:127]}"(s[1]), "+{v[128:143]}"(s[2]), "+{v[144:159]}"(s[3]),         \
                   "+{v[208:223]}"(pb), "=&{v[176:207]}"(scratch), "+v"(m_run), "+v"(l_run)                           \
                 : "{v[64:79]}"(qq[0]), "{v[80:95]}"(qq[1]), "{v[160:167]}"(ko), "{v[168:175]}"(vo), "s"(flags),      \
                   "v"(thr), "v"(xaddr), "s"(fac), "s"(scale)                                                         \
                 : "vcc", "scc")
    if constexpr (PAR == 0 && R == 1) CRANE_PF_ASM(CRANE_PF_STEP_P0_R1);
    if constexpr (PAR == 0 && R == 2) CRANE_PF_ASM(CRANE_PF_STEP_P0_R2);
    if constexpr (PAR == 1 && R == 1) CRANE_PF_ASM(CRANE_PF_STEP_P1_R1);
    if constexpr (PAR == 1 && R == 2) CRANE_PF_ASM(CRANE_PF_STEP_P1_R2);
#undef CRANE_PF_ASM
    (void)scratch;
}

template <int X> using I = std::integral_constant<int, X>;

// O^T += V^T P^T over the V tile at LDS offset vt (from the lane's V^T
// addresses vo): 4 dim blocks x 4 key steps of 16; the A operand (dims x keys)
// comes straight from the row-major V tile by transposed reads, issued one
// key step ahead of the MFMAs that use them.
__device__ __forceinline__ void pv_from_lds(f32x16_v (&oacc)[4], const bf16x8_v (&pf)[4], u32x8_v vo, uint32_t vt) {
    uint4 cur[4], nxt[4];
#pragma unroll
    for (int db = 0; db < 4; ++db) {
        const uint2 lo = lds_read_tr16(vo[2 * db] + vt);
        const uint2 hi = lds_read_tr16(vo[2 * db + 1] + vt);
        cur[db] = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
#pragma unroll
    for (int st = 0; st < 4; ++st) {
        if (st + 1 < 4) {
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const uint2 lo = lds_read_tr16(vo[2 * db] + vt + (st + 1) * 4096);      // keys of slots 0..3
                const uint2 hi = lds_read_tr16(vo[2 * db + 1] + vt + (st + 1) * 4096);  // slots 4..7: 8 rows on
                nxt[db] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        }
#pragma unroll
        for (int db = 0; db < 4; ++db) oacc[db] = mfma32(as_bf16x8(cur[db]), pf[st], oacc[db]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int db = 0; db < 4; ++db) cur[db] = nxt[db];
    }
}

// P pair k (scores 2k, 2k+1 of a score set) packed in register k of the set's
// first block: key step st of the P V product takes registers 4st .. 4st+3.
__device__ __forceinline__ void p_tuples(const f32x16_v& p, bf16x8_v (&pf)[4]) {
#pragma unroll
    for (int st = 0; st < 4; ++st)
        pf[st] = as_bf16x8(make_uint4(__float_as_uint(p[4 * st]), __float_as_uint(p[4 * st + 1]),
                                      __float_as_uint(p[4 * st + 2]), __float_as_uint(p[4 * st + 3])));
}

// Rows whose keys all lie in tile 0 (the first rows of a causal prefill, or a
// short non-causal one): candle's softmax_last_dim chain in bf16 exactly, from
// the raw scores of tile 0 in s[0], s[1]: the row max of the rounded scores,
// e = bf16(exp(bf16(s - max))), the sum in f32 rounded to bf16, p = bf16(e /
// sum) (correctly rounded: one reciprocal, two FMAs), then O = P V over V
// tile 0 with no division at the end (l = 1, half in each lane half).
template <bool CAUSAL>
__device__ __forceinline__ void exact_rows(f32x16_v (&s)[4], f32x16_v (&oacc)[4], u32x8_v vo, int qpos, int L, int hh,
                                           float scale_f, float& m_run, float& l_run) {
    // key = 4 hh + e(nb, r) is masked when key >= L or, causal, key > qpos
    const int thr = (CAUSAL ? min(qpos, L - 1) : L - 1) - 4 * hh;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (nb * 32 + 8 * (r >> 2) + (r & 3) > thr) s[nb][r] = kMaskRaw;
    float mx = -INFINITY;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const float s0 = score_bf16(s[nb][r], scale_f), s1 = score_bf16(s[nb][r + 1], scale_f);
            const float s2 = score_bf16(s[nb][r + 2], scale_f), s3 = score_bf16(s[nb][r + 3], scale_f);
            s[nb][r] = s0;
            s[nb][r + 1] = s1;
            s[nb][r + 2] = s2;
            s[nb][r + 3] = s3;
            mx = fmaxf(mx, fmaxf(fmaxf(s0, s1), fmaxf(s2, s3)));
        }
    mx = fmaxf(mx, __shfl_xor(mx, 32));  // the row's other 32 keys sit in the other lane half
    float sum = 0.f;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[nb][r] = rt<bf16_t>(fast_exp2(rt<bf16_t>(s[nb][r] - mx) * kLog2e));
            sum += s[nb][r];
        }
    const float sum_r = rt<bf16_t>(sum + __shfl_xor(sum, 32));
    const float inv = 1.0f / sum_r;
    uint32_t pk[16];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; r += 2)
            pk[(16 * nb + r) >> 1] = pack_bf16x2(div_by(s[nb][r], sum_r, inv), div_by(s[nb][r + 1], sum_r, inv));
#pragma unroll
    for (int k = 0; k < 16; ++k) s[0][k] = __uint_as_float(pk[k]);
    bf16x8_v pf[4];
    p_tuples(s[0], pf);
    pv_from_lds(oacc, pf, vo, 0);
    m_run = 0.f;   // finite, so a key-split merge keeps these rows as they are
    l_run = 0.5f;  // each lane half holds half of the normalised row sum
}

// The kernel body (prefill_bf16_kernel below).  R: candle's score roundings
// that the workgroup reproduces (2: both, the default; 1: the first only, in
// long rows when the caller asks for it).
//
// A wave walks the key tiles of its rows.  Tile t's scores S(t) sit in the
// score set of parity t & 1; its softmax writes the packed bf16 p pairs over
// the first 16 registers of that set, and their P V product runs in the next
// step (P V deferred by one tile), beside the softmax of tile t+1 and the
// QK^T MFMAs of tile t+2.  Steps over full tiles whose scores do not move the
// reference max take the hand-scheduled assembly step; the first tile, masked
// (diagonal, last) tiles and steps that move the max take the same arithmetic
// in C++ (pending P V first, then the rescale, the softmax and the next QK^T).
template <bool CAUSAL, class ROWS, int SPLIT, int R>
__device__ __forceinline__ void prefill_bf16_body(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                  const bf16_t* __restrict__ vc, const ROWS& rows, int start, int S,
                                                  int Hq, int Hkv, uint32_t scale_bits, bf16_t* __restrict__ out,
                                                  int qt, int b, int hq, uint8_t (&kbufs)[SPLIT][2][kTileBytes],
                                                  uint8_t (&vbufs)[SPLIT][2][kTileBytes]) {
    const int n_rep = Hq / Hkv;
    const int kvh = hq / n_rep;
    const int m0 = qt * kBM;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS copy targets are scalar
    const int grp = SPLIT > 1 ? wave_all / kWaves : 0;              // key-range group
    const int wave = SPLIT > 1 ? wave_all % kWaves : wave_all;      // wave within the group: its query rows
    auto& kbuf = kbufs[grp];
    auto& vbuf = vbufs[grp];
    const int n = lane & 31, hh = lane >> 5;

    const int L = start + S;                                 // cache rows holding keys for this chunk
    const int kend = CAUSAL ? min(start + m0 + kBM, L) : L;  // keys any row of the tile can see
    const int n_all = (kend + kBN - 1) / kBN;
    const int half = (n_all + SPLIT - 1) / SPLIT;            // steps every group takes
    const int t0 = grp * half;                               // this group's first tile
    const int n_tiles = max(0, min(half, n_all - t0));       // ... and how many it has
    uint32_t vofs[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) vofs[i] = pinned(copy_voffset(i, wave, lane));
    // Tile x of K (or V) into LDS.  Dense: one resource over the sequence's L
    // rows, the tile picked by the scalar offset.  Paged: a resource over the
    // tile's rows inside its page (a page holds whole tiles); rows past L, and
    // a page id outside the pool, read as zero.
    const int64_t head0 = ROWS::kPaged ? 0 : rows.offset(b, Hkv, kvh, 0);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kc + head0, L * kHeadDim * 2);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vc + head0, L * kHeadDim * 2);
    auto issue = [&](const bf16_t* pool, const __amdgpu_buffer_rsrc_t& whole, int x, uint8_t* dst)
        __attribute__((always_inline)) {
        if constexpr (ROWS::kPaged) {
            const int key0 = x * kBN;
            const int64_t off = key0 < L ? rows.offset(b, Hkv, kvh, key0) : -1;
            const int bytes = off < 0 ? 0 : min(kBN, L - key0) * kHeadDim * 2;
            issue_tile(make_rsrc(pool + (off < 0 ? 0 : off), bytes), 0, wave, vofs, dst);
        } else {
            issue_tile(whole, x, wave, vofs, dst);
        }
    };
    // K(0) and V(0) into buffers 0, K(1) into buffer 1; step t copies K(t+2)
    // and (from t = 1) V(t) into the buffers of parity t & 1.
    if (n_tiles > 0) {
        issue(kc, rk, t0, kbuf[0]);
        issue(vc, rv, t0, vbuf[0]);
    }
    if (n_tiles > 1) issue(kc, rk, t0 + 1, kbuf[1]);

    // Q fragments (B operand of S^T = K Q^T): query row qrow, dims 16ks + 8hh
    // .. +7, fragment ks in elements 4(ks%4) .. +3 of qq[ks/4].
    const int qrow = m0 + wave * 32 + n;
    i32x16_v qq[2];
    {
        const bf16_t* qp = q + (((int64_t)b * Hq + hq) * S + min(qrow, S - 1)) * kHeadDim + 8 * hh;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            uint4 u = *reinterpret_cast<const uint4*>(qp + 16 * ks);
            if (qrow >= S) u = make_uint4(0, 0, 0, 0);
            qq[ks >> 2][4 * (ks & 3)] = (int)u.x;
            qq[ks >> 2][4 * (ks & 3) + 1] = (int)u.y;
            qq[ks >> 2][4 * (ks & 3) + 2] = (int)u.z;
            qq[ks >> 2][4 * (ks & 3) + 3] = (int)u.w;
        }
    }
    f32x16_v oacc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    f32x16_v s[4];  // score sets: s[2x], s[2x+1] hold key blocks 0 and 1 of a tile of parity x
    float m_run = -INFINITY, l_run = 0.f;
    const int qpos = start + qrow;                      // absolute position of my query
    const int wave_first = start + m0 + wave * 32;      // first position of this wave's rows
    // Every key this wave's rows see lies in tile 0: candle's softmax chain runs exactly.
    const bool exact = grp == 0 && (CAUSAL ? wave_first + 31 < kBN : L <= kBN);
    const float scale_f = __uint_as_float(scale_bits << 16);  // the bf16 scale as an f32
    const float scale_log2 = scale_f * kLog2e;                 // raw-score scale of the running max
    const float fac = R == 2 ? kLog2e : scale_log2;            // exp2 argument factor of a rounded score
    // transposed-read coordinates of this lane for the V^T fragments
    const int vg = lane >> 4, vi = lane & 15;
    const int v_h = vg >> 1;                            // key half of the A operand
    const int v_col = 16 * (vg & 1) + 4 * (vi & 3);     // column inside a 32-dim block
    const bf16x2_v ones = {(__bf16)1.f, (__bf16)1.f};
    // Per-lane LDS byte addresses (of the parity-0 tile buffers), fixed for the
    // whole loop.  K: chunk 2ks+hh of row n.  V (transposed reads): rows r =
    // 4 v_h + vi/4 (+8 for the high half) at column 32 db + v_col; key step st
    // adds 16 rows = 4 KiB, with the same swizzle (rows mod 16 are unchanged).
    const uint32_t kbase = lds_addr(&kbuf[0][0]), vbase = lds_addr(&vbuf[0][0]);
    u32x8_v ko, vo;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) ko[ks] = pinned(kbase + n * 256 + 16 * ((2 * ks + hh) ^ swz(n)));
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 4 * v_h + (vi >> 2) + 8 * h, col = 32 * db + v_col;
            vo[2 * db + h] = pinned(vbase + r * 256 + 16 * ((col >> 3) ^ swz(r)) + 2 * (col & 7));
        }

    auto qf_of = [&](int ks) __attribute__((always_inline)) {
        const uint4 u = make_uint4((uint32_t)qq[ks >> 2][4 * (ks & 3)], (uint32_t)qq[ks >> 2][4 * (ks & 3) + 1],
                                   (uint32_t)qq[ks >> 2][4 * (ks & 3) + 2], (uint32_t)qq[ks >> 2][4 * (ks & 3) + 3]);
        return as_bf16x8(u);
    };
    // S(x) = K(x) Q^T into the score set of parity X: two 32x32 blocks of 8
    // MFMAs.  Lane (n, hh) holds keys nb*32 + 8*(r/4) + 4*hh + r%4 of query
    // row n in s[2X+nb][r]; row 32+n has the same swizzle as row n, so block
    // nb adds nb * 8 KiB.
    auto qk = [&](auto X) __attribute__((always_inline)) {
        constexpr int x = decltype(X)::value;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[2 * x + nb][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                const uint4 ku = lds_read16(ko[ks] + x * kTileBytes + nb * 8192);
                s[2 * x + nb] = mfma32(as_bf16x8(ku), qf_of(ks), s[2 * x + nb]);
            }
    };
    // O^T += V^T P^T over the V tile and the P pairs of parity X
    auto pv = [&](auto X) __attribute__((always_inline)) {
        constexpr int x = decltype(X)::value;
        bf16x8_v pf[4];
        p_tuples(s[2 * x], pf);
        pv_from_lds(oacc, pf, vo, x * kTileBytes);
    };
    // Tile 0 is visible to every row (key 0 precedes every query position);
    // a later group's first tile need not be (see the -inf guards).
    if (n_tiles > 1) CRANE_WAIT_VMCNT(2 * kCopies); else CRANE_WAIT_VMCNT(kCopies);  // this wave's K(0) copies
    __syncthreads();                                                   // ... and every wave's
    qk(I<0>{});

    // Waves whose rows see keys of tile 0 only (the first rows of a causal
    // prefill, or a short non-causal one) run candle's softmax_last_dim chain
    // in bf16 exactly, before the loop: the row max, e = bf16(exp(bf16(s -
    // max))), the sum in f32 rounded to bf16, p = bf16(e / sum), then O = P V
    // with no division at the end.  Their workgroup waits for V(0) once more;
    // the loop leaves them alone.
    if (CAUSAL ? start + m0 + 31 < kBN : L <= kBN) {  // uniform: wave 0 of the workgroup is exact
        if (n_tiles > 1) CRANE_WAIT_VMCNT(kCopies); else CRANE_WAIT_VMCNT(0);  // this wave's V(0) copies
        __syncthreads();                                                     // ... and every wave's
        if (exact) exact_rows<CAUSAL>(s, oacc, vo, qpos, L, hh, scale_f, m_run, l_run);
    }

    // Step t (parity PAR = t & 1): tile t's softmax, tile t+1's QK^T, and the
    // P V of tile t-1 that the previous step left pending.  A wave with no
    // keys in tile t (above its diagonal, past its group's range, or an exact
    // wave) only finishes the pending P V; every wave passes every barrier
    // (a step past the last one does nothing but the barrier).
    const int xaddr = (lane ^ 32) << 2;  // ds_bpermute address of the other lane half
    // wave-uniform constants of the assembly, in scalar registers
    const float fac_s = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fac)));
    const float scale_s = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(scale_f)));
    // The loop's assembly reads S(0) and O, which compiler-issued MFMAs wrote:
    // the 12 wait states an MFMA result needs before a VALU read, with the
    // values as operands so the MFMAs stay before it.
    asm volatile("s_nop 11" : "+v"(s[0]), "+v"(s[1]), "+v"(oacc[0]), "+v"(oacc[1]), "+v"(oacc[2]), "+v"(oacc[3]));
    bool pending = false;
    i32x16_v pb;  // the P pairs of the last softmax (the assembly's P registers)
#pragma unroll
    for (int i = 0; i < 16; ++i) pb[i] = 0;
    auto step = [&](auto parity, int t) __attribute__((always_inline)) {
        constexpr int par = decltype(parity)::value;
        CRANE_WAIT_VMCNT(0);  // this wave's copies of K(t+1) and V(t-1) have landed
        __syncthreads();      // ... and every wave's; K(t) and V(t-2) are fully consumed
        if (t + 2 < n_tiles) issue(kc, rk, t0 + t + 2, kbuf[par]);
        if (t >= 1 && t < n_tiles) issue(vc, rv, t0 + t, vbuf[par]);
        const int kt = (t0 + t) * kBN;
        const bool live = t < n_tiles && !exact && !(CAUSAL && kt > wave_first + 31);
        const bool full = kt + kBN <= kend && !(CAUSAL && kt + kBN - 1 > wave_first);  // no key masked
        const int flags = __builtin_amdgcn_readfirstlane((live ? 1 : 0) | (full ? 2 : 0) | (pending ? 4 : 0));
        // key = kt + 4 hh + e(nb, r) is masked when e > thr
        const int thr = (CAUSAL ? min(qpos, kend - 1) : kend - 1) - kt - 4 * hh;
        pf_step<par, R>(oacc, qq, s, pb, ko, vo, m_run, l_run, flags, thr, xaddr, fac_s, scale_s);
        pending = live;
    };
    const int n_steps = SPLIT > 1 ? half : n_tiles;
    for (int t = 0; t <= n_steps; t += 2) {
        step(I<0>{}, t);
        step(I<1>{}, t + 1);
    }

    if constexpr (SPLIT > 1) {
        // Group 1's O (in the freed K tiles) and (m, l) (in the freed V tiles)
        // for each lane, lane-minor; group 0's wave w merges the same query
        // rows' values.
        static_assert(SPLIT == 2, "two key groups");
        static_assert(kWaves * 64 * 64 * 4 <= (int)sizeof(kbufs) && kWaves * 2 * 64 * 4 <= (int)sizeof(vbufs),
                      "exchange fits the tile space");
        float* xo = reinterpret_cast<float*>(&kbufs[0][0][0]) + wave * 64 * 64 + lane;
        float* xml = reinterpret_cast<float*>(&vbufs[0][0][0]) + wave * 2 * 64 + lane;
        __syncthreads();  // every wave is done with the tiles
        if (grp == 1) {
            xml[0] = m_run;
            xml[64] = l_run;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) xo[64 * (16 * i + r)] = oacc[i][r];
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = xml[0], l1 = xml[64];
        const float mm = fmaxf(m_run, m1);
        const float a0 = m_run == -INFINITY ? 0.f : fast_exp2(m_run - mm);
        const float a1 = m1 == -INFINITY ? 0.f : fast_exp2(m1 - mm);
        l_run = l_run * a0 + l1 * a1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] = oacc[i][r] * a0 + xo[64 * (16 * i + r)] * a1;
    }

    l_run += __shfl_xor(l_run, 32);  // the two lane halves hold different keys of the row (exact rows: 1)
    if (qrow < S) {
        const float inv = 1.0f / l_run;
        bf16_t* op = out + (((int64_t)b * S + qrow) * Hq + hq) * kHeadDim;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int dim = db * 32 + 8 * g + 4 * hh;
                const uint2 w = make_uint2(pack_bf16x2(oacc[db][4 * g] * inv, oacc[db][4 * g + 1] * inv),
                                           pack_bf16x2(oacc[db][4 * g + 2] * inv, oacc[db][4 * g + 3] * inv));
                *reinterpret_cast<uint2*>(op + dim) = w;
            }
    }
}

// SPLIT = 2 (a grid too small to fill the chip): 8 waves, two groups of 4 on
// the same 128 query rows; group g walks its half of the key tiles through its
// own LDS tiles, and group 1's running (max, sum, O) merge into group 0's
// through LDS at the end.  Every wave passes the same barriers: a step past a
// group's half does no copy and no work.
// flags: CRANE_HIP_PREFILL_CAUSAL | CRANE_HIP_PREFILL_LONG_ROWS_ONE_ROUNDING.
template <bool CAUSAL, class ROWS, int SPLIT>
__global__ __launch_bounds__(64 * kWaves * SPLIT) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_bf16_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc, ROWS rows,
    const int32_t* __restrict__ start_pos, int max_start, int S, int B, int Hq, int Hkv, uint32_t scale_bits,
    int one_rounding_long_rows, bf16_t* __restrict__ out) {
    const int n_rep = Hq / Hkv;
    const int n_qt = (S + kBM - 1) / kBM;
    int qt, b, hq;
    if (!map_block(blockIdx.x, n_qt, B, Hkv, n_rep, qt, b, hq)) return;
    const int start = min(max(start_pos[b], 0), max_start);
    // K tiles t+1 and t+2 and V tiles t-1 and t are resident or in flight
    // while tile t is computed.  One set per group.
    __shared__ __attribute__((aligned(1024))) uint8_t kbufs[SPLIT][2][kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t vbufs[SPLIT][2][kTileBytes];
    // The workgroup's first row sees at least kLongRowKeys keys (and so does every other row).
    const bool long_rows = CAUSAL ? start + qt * kBM + 1 >= kLongRowKeys : start + S >= kLongRowKeys;
    if (one_rounding_long_rows && long_rows)
        prefill_bf16_body<CAUSAL, ROWS, SPLIT, 1>(q, kc, vc, rows, start, S, Hq, Hkv, scale_bits, out, qt, b, hq,
                                                  kbufs, vbufs);
    else
        prefill_bf16_body<CAUSAL, ROWS, SPLIT, 2>(q, kc, vc, rows, start, S, Hq, Hkv, scale_bits, out, qt, b, hq,
                                                  kbufs, vbufs);
}

// ---- f32 kernel (MFMA, v_mfma_f32_32x32x2_f32) -----------------------------
//
// The bf16 kernel's shape in f32: a workgroup owns 128 query rows of one q
// head (4 waves of 32 rows); K and V tiles of 32 keys (16 KiB each, 512-byte
// rows) are copied HBM -> LDS by bounds-checked buffer_load ... lds, double-
// buffered.  S^T = K Q^T takes 64 MFMAs per 32-key tile: in step s lane half h
// multiplies dim 64 h + s (the dims of a dot product may pair in any order),
// so a lane's K fragments are 4 consecutive floats of its key row (one
// ds_read_b128 per 4 steps) and its Q fragments 64 consecutive floats of its
// query row, in registers.  The score accumulators hold S^T[key 8(r/4) + 4h +
// r%4][row l%32] in register r of lane l, which is exactly the B operand of
// O^T += V^T P^T for step r: P needs no data movement, and the A operand is
// one float of V per lane (the lane's output dim of the key the step takes).
// Online softmax in f32 (log2 domain), one rescale per tile; candle's f32
// path has no intermediate rounding to reproduce.
constexpr int kF32BN = 32;                             // keys per tile
constexpr int kF32Row = kHeadDim * 4;                  // bytes per key row
constexpr int kF32TileBytes = kF32BN * kF32Row;        // 16 KiB of K (or V) per tile
constexpr int kF32Copies = kF32TileBytes / 1024 / kWaves;  // 1 KiB blocks of a tile each wave copies
// f32 tiles keep 512-byte rows of 32 16-byte chunks; chunk c of row r sits at
// slot c ^ swz32(r), swz32 a permutation of the low 4 bits of r.  K reads (16
// lanes: rows r..r+15 at one chunk index) then hit 16 different chunks, and a
// V read (two rows 4 apart, bit 2 of the first clear, 32 consecutive floats
// each) puts the two rows 8 chunks apart, in disjoint banks.
__device__ __forceinline__ int swz32(int r) { return (r & 3) | (((r >> 2) & 1) << 3) | (((r >> 3) & 1) << 2); }

// Lane l of 1 KiB block blk fills row 2 blk + l/32, slot l%32, from global
// chunk (l%32) ^ swz32(row).
__device__ __forceinline__ int copy_voffset_f32(int i, int wave, int lane) {
    const int row = 2 * (wave * kF32Copies + i) + (lane >> 5);
    return row * kF32Row + 16 * ((lane & 31) ^ swz32(row));
}
__device__ __forceinline__ void issue_tile_f32(__amdgpu_buffer_rsrc_t rsrc, int t, int wave,
                                               const uint32_t (&vofs)[kF32Copies], uint8_t* dst) {
#pragma unroll
    for (int i = 0; i < kF32Copies; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, dst + (wave * kF32Copies + i) * 1024, 16, vofs[i],
                                                 t * kF32TileBytes, 0, 0);
}

template <bool CAUSAL, class ROWS>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, ROWS rows,
    const int32_t* __restrict__ start_pos, int max_start, int S, int B, int Hq, int Hkv, float scale_log2,
    float* __restrict__ out) {
    __shared__ __attribute__((aligned(1024))) uint8_t kbuf[2][kF32TileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t vbuf[2][kF32TileBytes];
    const int n_rep = Hq / Hkv;
    const int n_qt = (S + kBM - 1) / kBM;
    int qt, b, hq;
    if (!map_block(blockIdx.x, n_qt, B, Hkv, n_rep, qt, b, hq)) return;  // uniform: padding ids
    const int kvh = hq / n_rep;
    const int start = min(max(start_pos[b], 0), max_start);
    const int L = start + S;
    const int m0 = qt * kBM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: LDS copy targets are scalar
    const int n = lane & 31, h = lane >> 5;
    const int kend = CAUSAL ? min(start + m0 + kBM, L) : L;  // keys any row of the tile can see
    const int n_tiles = (kend + kF32BN - 1) / kF32BN;
    uint32_t vofs[kF32Copies];
#pragma unroll
    for (int i = 0; i < kF32Copies; ++i) vofs[i] = pinned(copy_voffset_f32(i, wave, lane));
    const int64_t head0 = ROWS::kPaged ? 0 : rows.offset(b, Hkv, kvh, 0);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kc + head0, L * kF32Row);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vc + head0, L * kF32Row);
    // Tile x into LDS (dense: the tile picked by the scalar offset; paged: a
    // resource over the tile's rows inside its page); rows past L, and a page
    // id outside the pool, read as zero.
    auto issue = [&](const float* pool, const __amdgpu_buffer_rsrc_t& whole, int x, uint8_t* dst)
        __attribute__((always_inline)) {
        if constexpr (ROWS::kPaged) {
            const int key0 = x * kF32BN;
            const int64_t off = key0 < L ? rows.offset(b, Hkv, kvh, key0) : -1;
            const int bytes = off < 0 ? 0 : min(kF32BN, L - key0) * kF32Row;
            issue_tile_f32(make_rsrc(pool + (off < 0 ? 0 : off), bytes), 0, wave, vofs, dst);
        } else {
            issue_tile_f32(whole, x, wave, vofs, dst);
        }
    };
    if (n_tiles > 0) {
        issue(kc, rk, 0, kbuf[0]);
        issue(vc, rv, 0, vbuf[0]);
    }
    // Q fragments: query row qrow, dims 64 h .. 64 h + 63 (rows past S read row S - 1, not stored)
    const int qrow = m0 + wave * 32 + n;
    float qf[64];
    {
        const float* qp = q + (((int64_t)b * Hq + hq) * S + min(qrow, S - 1)) * kHeadDim + 64 * h;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 v = *reinterpret_cast<const float4*>(qp + 4 * j);
            qf[4 * j] = v.x;
            qf[4 * j + 1] = v.y;
            qf[4 * j + 2] = v.z;
            qf[4 * j + 3] = v.w;
        }
    }
    f32x16_v oacc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const int qpos = start + qrow;
    const int lim = CAUSAL ? min(qpos, L - 1) : L - 1;  // the last key this row sees
    const int wave_first = start + m0 + wave * 32;      // first position of this wave's rows
    // per-lane LDS byte offsets inside a tile: K row n's chunks, V's dim column
    const int k_row = n * kF32Row;
    for (int t = 0; t < n_tiles; ++t) {
        const int par = t & 1;
        CRANE_WAIT_VMCNT(0);  // this wave's copies of tile t have landed
        __syncthreads();      // ... and every wave's; tile t - 1 is fully consumed
        if (t + 1 < n_tiles) {
            issue(kc, rk, t + 1, kbuf[par ^ 1]);
            issue(vc, rv, t + 1, vbuf[par ^ 1]);
        }
        const int kt = t * kF32BN;
        if (CAUSAL && kt > wave_first + 31) continue;  // uniform: no row of this wave sees the tile
        const uint8_t* kb = kbuf[par];
        f32x16_v acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 kk = *reinterpret_cast<const float4*>(kb + k_row + 16 * ((16 * h + j) ^ swz32(n)));
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.x, qf[4 * j], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.y, qf[4 * j + 1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.z, qf[4 * j + 2], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.w, qf[4 * j + 3], acc, 0, 0, 0);
        }
        // scores of keys kt + 8(r/4) + 4h + r%4 for this lane's row, log2 domain
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = kt + 8 * (r >> 2) + 4 * h + (r & 3);
            acc[r] = key > lim ? -INFINITY : acc[r] * scale_log2;
            mx = fmaxf(mx, acc[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a row with no key yet keeps p = 0
        const float alpha = fast_exp2(m_run - m_use);
        float rs = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[r] = fast_exp2(acc[r] - m_use);
            rs += acc[r];
        }
        rs += __shfl_xor(rs, 32);
        l_run = l_run * alpha + rs;
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
        // O^T += V^T P^T: step r takes key 8(r/4) + 4h + r%4 of the tile; lane
        // l reads that key's dim 32 db + n
        const uint8_t* vb = vbuf[par];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 8 * (r >> 2) + 4 * h + (r & 3);
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const int d = 32 * db + n;
                const float vv = *reinterpret_cast<const float*>(vb + row * kF32Row + 16 * ((d >> 2) ^ swz32(row)) +
                                                                 4 * (d & 3));
                oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, acc[r], oacc[db], 0, 0, 0);
            }
        }
    }
    if (qrow >= S) return;
    // register r of oacc[db] holds O^T[dim 32 db + 8(r/4) + 4h + r%4][this lane's row]
    const float inv = 1.f / l_run;
    float* op = out + (((int64_t)b * S + qrow) * Hq + hq) * kHeadDim;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(op + 32 * db + 8 * g + 4 * h) =
                make_float4(oacc[db][4 * g] * inv, oacc[db][4 * g + 1] * inv, oacc[db][4 * g + 2] * inv,
                            oacc[db][4 * g + 3] * inv);
}

// The same walk for grids too small to fill the chip (prefill_f32_split): a
// workgroup owns 32 query rows and its 4 waves split their key tiles, wave w
// taking tiles w, w + 4, ...  A wave runs at the f32 MFMA rate by itself (128
// MFMAs of 64 cycles a tile), so a short prompt is bound by how many SIMDs work:
// the 128-row form gives a 731-token prompt of 16 heads 96 workgroups, the
// longest walking all 23 tiles.  Each wave keeps a K and a V tile of its own in
// LDS (128 KiB in all): K(next) is copied while P V runs and V(next) while the
// scores do, each phase longer than the copy, and no barrier is needed until the
// waves' (max, sum, O) meet at the end.  Four times the K / V reads per flop, from
// L2.  Measured, us: 731 tokens of 16 heads 112 -> 38 (58 TFLOP/s), 2048 of 16 heads
// 315 -> 179 (96 TFLOP/s of 157), 100 tokens after 3000 453 -> 120.
template <bool CAUSAL, class ROWS>
__global__ __launch_bounds__(64 * kWaves) void prefill_f32_split_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, ROWS rows,
    const int32_t* __restrict__ start_pos, int max_start, int S, int B, int Hq, int Hkv, float scale_log2,
    float* __restrict__ out) {
    static_assert(kWaves == 4, "one output block of 32 dims per wave in the merge");
    __shared__ __attribute__((aligned(1024))) uint8_t kbuf[kWaves][kF32TileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t vbuf[kWaves][kF32TileBytes];
    __shared__ float2 ml[kWaves][32];
    const int n_rep = Hq / Hkv;
    const int n_qt = (S + 31) / 32;
    int qt, b, hq;
    if (!map_block(blockIdx.x, n_qt, B, Hkv, n_rep, qt, b, hq)) return;  // uniform: padding ids
    const int kvh = hq / n_rep;
    const int start = min(max(start_pos[b], 0), max_start);
    const int L = start + S;
    const int m0 = qt * 32;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int kend = CAUSAL ? min(start + m0 + 32, L) : L;  // keys any row of the tile can see
    const int n_tiles = (kend + kF32BN - 1) / kF32BN;
    constexpr int kTileCopies = kF32TileBytes / 1024;
    // copy i fills rows 2 i, 2 i + 1: the lane part of the source offset, and the rows swizzle alike mod 16
    uint32_t vofs[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = 2 * i + (lane >> 5);
        vofs[i] = pinned(row * kF32Row + 16 * ((lane & 31) ^ swz32(row)));
    }
    const int64_t head0 = ROWS::kPaged ? 0 : rows.offset(b, Hkv, kvh, 0);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kc + head0, L * kF32Row);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vc + head0, L * kF32Row);
    auto issue = [&](const float* pool, const __amdgpu_buffer_rsrc_t& whole, int x, uint8_t* dst)
        __attribute__((always_inline)) {
        __amdgpu_buffer_rsrc_t r = whole;
        int base = x * kF32TileBytes;
        if constexpr (ROWS::kPaged) {
            const int key0 = x * kF32BN;
            const int64_t off = key0 < L ? rows.offset(b, Hkv, kvh, key0) : -1;
            r = make_rsrc(pool + (off < 0 ? 0 : off), off < 0 ? 0 : min(kF32BN, L - key0) * kF32Row);
            base = 0;
        }
#pragma unroll
        for (int i = 0; i < kTileCopies; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst + i * 1024, 16, vofs[i & 7], base + (i >> 3) * 16 * kF32Row,
                                                     0, 0);
    };
    if (wave < n_tiles) {
        issue(kc, rk, wave, kbuf[wave]);
        issue(vc, rv, wave, vbuf[wave]);
    }
    const int qrow = m0 + n;
    float qf[64];
    {
        const float* qp = q + (((int64_t)b * Hq + hq) * S + min(qrow, S - 1)) * kHeadDim + 64 * h;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 v = *reinterpret_cast<const float4*>(qp + 4 * j);
            qf[4 * j] = v.x;
            qf[4 * j + 1] = v.y;
            qf[4 * j + 2] = v.z;
            qf[4 * j + 3] = v.w;
        }
    }
    f32x16_v oacc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    const int lim = CAUSAL ? min(start + qrow, L - 1) : L - 1;  // the last key this row sees
    const int k_row = n * kF32Row;
    const uint8_t* kb = kbuf[wave];
    const uint8_t* vb = vbuf[wave];
    // both halves of the wave hold keys of the same rows
    auto other = [&](float x) __attribute__((always_inline)) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
    };
    CRANE_WAIT_VMCNT(0);  // q, and the first tiles
    // q used here: the wait-count pass then does not wait for its loads inside
    // the loop, where the wait would be for the tile copies in flight
#pragma unroll
    for (int j = 0; j < 64; ++j) asm volatile("" : "+v"(qf[j]));
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    for (int t = wave; t < n_tiles; t += kWaves) {
        const bool more = t + kWaves < n_tiles;
        if (t != wave) {
            // K(t) has landed; V(t), issued after it, may fly
            CRANE_WAIT_VMCNT(kTileCopies);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
        const int kt = t * kF32BN;
        f32x16_v acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 kk = *reinterpret_cast<const float4*>(kb + k_row + 16 * ((16 * h + j) ^ swz32(n)));
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.x, qf[4 * j], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.y, qf[4 * j + 1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.z, qf[4 * j + 2], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.w, qf[4 * j + 3], acc, 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt 0: this tile's K reads are done
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue(kc, rk, t + kWaves, kbuf[wave]);
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = kt + 8 * (r >> 2) + 4 * h + (r & 3);
            acc[r] = key > lim ? -INFINITY : acc[r] * scale_log2;
            mx = fmaxf(mx, acc[r]);
        }
        const float2 mo = other(mx);
        const float m_new = fmaxf(m_run, fmaxf(mo.x, mo.y));
        const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a row with no key yet keeps p = 0
        const float alpha = fast_exp2(m_run - m_use);
        float rs = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[r] = fast_exp2(acc[r] - m_use);
            rs += acc[r];
        }
        const float2 so = other(rs);
        l_run = l_run * alpha + (so.x + so.y);
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
        if (more) CRANE_WAIT_VMCNT(kTileCopies); else CRANE_WAIT_VMCNT(0);  // V(t); K(next) may fly
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 8 * (r >> 2) + 4 * h + (r & 3);
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const int d = 32 * db + n;
                const float vv = *reinterpret_cast<const float*>(vb + row * kF32Row + 16 * ((d >> 2) ^ swz32(row)) +
                                                                 4 * (d & 3));
                oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, acc[r], oacc[db], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // this tile's V reads are done
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue(vc, rv, t + kWaves, vbuf[wave]);
    }
    // Merge: every wave leaves its O in its K tile, block db by block db, and
    // wave w sums block w of all four in wave order.
    float* xo = reinterpret_cast<float*>(kbuf[wave]) + lane;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) xo[64 * (16 * db + r)] = oacc[db][r];
    if (h == 0) ml[wave][n] = make_float2(m_run, l_run);
    __syncthreads();
    float mm = ml[0][n].x;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) mm = fmaxf(mm, ml[w][n].x);
    float a[kWaves], l = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        a[w] = ml[w][n].x == -INFINITY ? 0.f : fast_exp2(ml[w][n].x - mm);
        l += a[w] * ml[w][n].y;
    }
    if (qrow >= S) return;
    const float inv = 1.f / l;
    float* op = out + (((int64_t)b * S + qrow) * Hq + hq) * kHeadDim + 32 * wave + 4 * h;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] = 0.f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w)
                o[e] += a[w] * reinterpret_cast<const float*>(kbuf[w])[64 * (16 * wave + 4 * g + e) + lane];
        }
        *reinterpret_cast<float4*>(op + 8 * g) = make_float4(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
    }
}

}  // namespace

// Whether an f32 call of `blocks` 128-row workgroups takes the split form.
// Measured over 1 to 8 sequences of 17 to 2048 tokens, 4 to 32 heads, after 0 to
// 3000 cached keys, causal and not (1052 calls):
//   blocks <= 192:  always the faster one, 0.25 to 0.99 of the wide form's time;
//   blocks <= 384:  causal prompts of 500 tokens or more, where it also evens out
//                   their short and long rows (8 x 500 of 8 heads 0.81, 1500 of 32
//                   heads 276 -> 203 us; 4 x 333 of 32 heads 69.9 -> 77.4), and up
//                   to two row tiles, where the wide one's 128 rows are mostly
//                   padding (8 x 33 of 32 heads after 300 keys 0.67).  Between, both
//                   fill the chip and the wide one copies a quarter of the keys
//                   per row: 8 x 100 of 28 heads 23.9 us against 35.1, 500 tokens
//                   after 300, not causal, 120.7 against 145.1;
//   past that the wide one: 512 blocks (4 x 500 of 32 heads) 109 -> 130 us.
// Over two key tiles or fewer the split has too few tiles for its waves (17
// tokens 9.8 -> 11.4 us).
bool prefill_f32_split(int64_t blocks, int S, int64_t keys, bool causal) {
    if (keys <= 2 * kF32BN) return false;
    return blocks <= 192 || (blocks <= 384 && (S <= 64 || (causal && S >= 500)));
}

namespace {

// Compute units of the device that runs `stream` (cached per device; host
// threads may race to fill an entry, with the same value).
int device_cus(hipStream_t stream) {
    static std::atomic<int> cus[64];
    const int dev = stream_device(stream);
    if (dev < 0 || dev >= 64) return 256;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (!n) {
        n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Checks shared by both layouts, then the launch; `rows` addresses the cache.
template <class ROWS>
int attn_prefill(const void* q, const void* k_cache, const void* v_cache, const ROWS& rows, const int32_t* start_pos,
                 int64_t max_start, int B, int S, int Hq, int Hkv, int D, float scale, int flags, void* out,
                 int dtype, void* stream) {
    if (dtype != CRANE_HIP_F32 && dtype != CRANE_HIP_BF16) return CRANE_HIP_E_DTYPE;
    if (flags & ~(CRANE_HIP_PREFILL_CAUSAL | CRANE_HIP_PREFILL_LONG_ROWS_ONE_ROUNDING)) return CRANE_HIP_E_INVALID;
    const bool causal = flags & CRANE_HIP_PREFILL_CAUSAL;
    const int one_rounding = (flags & CRANE_HIP_PREFILL_LONG_ROWS_ONE_ROUNDING) ? 1 : 0;
    if (D != kHeadDim) return CRANE_HIP_E_HEAD_DIM;
    if (B < 0 || S < 0 || Hq <= 0 || Hkv <= 0 || max_start < 0) return CRANE_HIP_E_INVALID;
    if (Hq % Hkv != 0) return CRANE_HIP_E_GQA;
    if (!(scale > 0.0f) || !__builtin_isfinite(scale)) return CRANE_HIP_E_INVALID;
    if (B == 0 || S == 0) return CRANE_HIP_OK;
    if (!q || !k_cache || !v_cache || !start_pos || !out) return CRANE_HIP_E_INVALID;
    if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out)) return CRANE_HIP_E_ALIGN;
    if (max_start + (int64_t)S > 0x7fffffffLL / (kHeadDim * 4) || B > 65535 || Hq > 65535) return CRANE_HIP_E_INVALID;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == CRANE_HIP_BF16) {
        // candle scales the bf16 scores by the scale converted to bf16 (affine in T)
        const uint32_t sl = f32_bits(host_round_bf16(scale)) >> 16;
        const int n_rep = Hq / Hkv;
        const int64_t n_qt = (S + kBM - 1) / kBM;
        const int64_t units = n_qt * B * Hkv;
        const int64_t chunk = 8LL * n_rep;
        const int64_t blocks = ((units + 7) / 8) * chunk;
        if (blocks > 0x7fffffffLL) return CRANE_HIP_E_INVALID;
        // A grid of at most one workgroup per CU leaves each SIMD one wave and the
        // last query tiles' key walk as the critical path: split the keys of
        // each tile between two groups of waves instead.
        const int cus = device_cus(st);
        const bool split = blocks <= (int64_t)cus;
#define CRANE_PREFILL_LAUNCH(C, SP)                                                                              \
    hipLaunchKernelGGL((prefill_bf16_kernel<C, ROWS, SP>), dim3((unsigned)blocks), dim3(64 * kWaves * SP), 0, st, \
                       (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, rows, start_pos,        \
                       (int)max_start, S, B, Hq, Hkv, sl, one_rounding, (bf16_t*)out)
        if (causal) {
            if (split) CRANE_PREFILL_LAUNCH(true, 2); else CRANE_PREFILL_LAUNCH(true, 1);
        } else {
            if (split) CRANE_PREFILL_LAUNCH(false, 2); else CRANE_PREFILL_LAUNCH(false, 1);
        }
#undef CRANE_PREFILL_LAUNCH
    } else {
        const float sl = scale * kLog2e;
        const int n_rep = Hq / Hkv;
        const int64_t units = (int64_t)((S + kBM - 1) / kBM) * B * Hkv;
        const int64_t blocks = ((units + 7) / 8) * 8 * n_rep;
        if (blocks > 0x7fffffffLL) return CRANE_HIP_E_INVALID;
#define CRANE_PREFILL_F32(kernel, n)                                                                            \
    hipLaunchKernelGGL((kernel), dim3((unsigned)(n)), dim3(64 * kWaves), 0, st, (const float*)q,                  \
                       (const float*)k_cache, (const float*)v_cache, rows, start_pos, (int)max_start, S, B, Hq, Hkv, \
                       sl, (float*)out)
        const int64_t blocks32 = ((int64_t)((S + 31) / 32) * B * Hkv + 7) / 8 * 8 * n_rep;
        if (prefill_f32_split(blocks, S, max_start + S, causal)) {
            if (causal) CRANE_PREFILL_F32((prefill_f32_split_kernel<true, ROWS>), blocks32);
            else CRANE_PREFILL_F32((prefill_f32_split_kernel<false, ROWS>), blocks32);
        } else {
            if (causal) CRANE_PREFILL_F32((prefill_f32_kernel<true, ROWS>), blocks);
            else CRANE_PREFILL_F32((prefill_f32_kernel<false, ROWS>), blocks);
        }
#undef CRANE_PREFILL_F32
    }
    return launch_status(hipGetLastError());
}

}  // namespace
}  // namespace crane

using namespace crane;

extern "C" int crane_hip_attn_prefill(const void* q, const void* k_cache, const void* v_cache, int64_t cache_cap,
                                      const int32_t* start_pos, int64_t max_start, int B, int S, int Hq, int Hkv,
                                      int D, float scale, int flags, void* out, int dtype, void* stream) {
    if (dtype != CRANE_HIP_F32 && dtype != CRANE_HIP_BF16) return CRANE_HIP_E_DTYPE;
    if (D != kHeadDim) return CRANE_HIP_E_HEAD_DIM;
    if (max_start < 0 || S < 0) return CRANE_HIP_E_INVALID;
    if (cache_cap <= 0 || max_start + (int64_t)S > cache_cap) return CRANE_HIP_E_CAPACITY;
    if (cache_cap > 0x7fffffffLL) return CRANE_HIP_E_INVALID;
    return attn_prefill(q, k_cache, v_cache, DenseRows{cache_cap}, start_pos, max_start, B, S, Hq, Hkv, D, scale,
                        flags, out, dtype, stream);
}

extern "C" int crane_hip_attn_prefill_paged(const void* q, const void* k_pool, const void* v_pool, int64_t n_pages,
                                            int page_rows, const int32_t* block_table, int64_t table_stride,
                                            const int32_t* start_pos, int64_t max_start, int B, int S, int Hq, int Hkv,
                                            int D, float scale, int flags, void* out, int dtype, void* stream) {
    const int rc = check_paged(n_pages, page_rows, block_table, table_stride, Hkv);
    if (rc) return rc;
    if (max_start < 0 || S < 0) return CRANE_HIP_E_INVALID;
    if (max_start + (int64_t)S > table_stride * page_rows) return CRANE_HIP_E_CAPACITY;
    return attn_prefill(q, k_pool, v_pool, PagedRows{block_table, table_stride, n_pages, page_rows}, start_pos,
                        max_start, B, S, Hq, Hkv, D, scale, flags, out, dtype, stream);
}
