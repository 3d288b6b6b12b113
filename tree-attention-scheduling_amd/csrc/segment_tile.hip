// segment_tile.hip -- gfx950 kernels of the segment launches: work items of every kind.
//
// Replaces the reference's Triton _segment
// (src/tree_attention/kernels.py:8-55, launched at :158-165): grouped partial
// attention of one physical KV segment for all requests of a job, online
// softmax in fp32, P rounded to the input dtype before PV (kernels.py:49),
// output acc/z and the natural-log log-sum-exp m + ln z.
//
// One workgroup owns one (job, row tile, KV head) work item: NW waves of
// 16*NB query rows each (jobs with at most 16 rows: one wave, NB = 1).  The
// job's tokens are streamed in 64-token tiles.
//
//  * HBM -> LDS without registers: a tile is D/8 1-KiB blocks of K (8 d-rows
//    x 64 tokens each) and D/8 of V, each copied by one wave with one
//    global_load_lds_dwordx4 (lane i fills bytes 16i..16i+15 of the block).
//    Three LDS stages keep two tiles in flight while one is computed (one-wave
//    workgroups of small jobs use one stage, so that five fit a CU); each wave
//    waits for its own copies with s_waitcnt vmcnt and the waves meet at one
//    barrier per tile.
//  * The lane -> 16-byte-chunk assignment inside a block is chosen so that the
//    eight chunks one 16-lane group reads together are 128 contiguous bytes,
//    and odd blocks swap the two 128-byte halves of every 256 bytes so that
//    neighbouring groups land 128 bytes apart (no LDS bank conflicts; see
//    the LDS layout note above struct LdsOfs).
//  * MFMA operands are read with gfx950's transposing LDS load
//    ds_read_b64_tr_b16: within a group of 16 lanes, lane 4a+b receives
//    element b of the 8-byte chunks addressed by lanes a, a+4, a+8, a+12.
//    Lane (g, r) addresses contraction row r/4 (+4) of its group at column
//    4*(r%4), so every lane ends up with four consecutive contraction elements
//    of one output row or column -- the MFMA operand layout -- straight from
//    the pools' own layouts (K [d][token], V [token][d]).
//  * S^T = K Q^T with v_mfma_f32_16x16x32: the C layout gives each lane four
//    consecutive tokens of one query row, which is the B operand of the PV
//    product O^T = V^T P^T, so P never leaves registers.
//  * The softmax denominator is one more PV MFMA against an all-ones A
//    operand, so z sums exactly the rounded P that multiplies V (RowSum; pools of
//    other capacities sum the FP32 exponentials).
//  * Softmax in base 2 with log2(e)/sqrt(D) folded into one FMA; lazy
//    rescaling (the running maximum moves only by more than TAU).
// The kernels are templates over the layout of K and V (enum Layout): pools whose
// capacity is a multiple of 8 (every 8-token chunk of a K row is one aligned
// 16-byte copy), pools of any other capacity (K through registers) and
// token-major K and V (K's operand read without transposing) of a count that is a
// multiple of 8 or any other.  The text above describes the first; TileCopy,
// KTokens and RowSum say where the others differ.
#include "ta_common.h"
#include "tree_attn.h"

#ifndef TA_LAYOUT
#define TA_LAYOUT KV_POOL  // the layout this translation unit's kernels are compiled for
#endif

namespace ta {
namespace {

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const u16 lds_u16;

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding).
#define TA_VMCNT(n) ((((n)&15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14)))

// s_waitcnt lgkmcnt(0) alone
#define TA_LGKMCNT0 (15 | (7 << 4) | (0 << 8) | (3 << 14))

// A uniform load through the scalar unit (constant address space).
__device__ inline int sload(const int32_t *p, int i) {
    return ((const __attribute__((address_space(4))) int32_t *)p)[i];
}

// Wait until at most n tiles of this wave's copies (BPW each) are in flight
// (n = 0 .. 4; the immediate of s_waitcnt must be a constant).
template <int BPW>
__device__ inline void wait_tiles(int n) {
    static_assert(4 * BPW <= 63, "four tiles of copies fit the vmcnt counter");
    switch (n) {
        case 4: __builtin_amdgcn_s_waitcnt(TA_VMCNT(4 * BPW)); break;
        case 3: __builtin_amdgcn_s_waitcnt(TA_VMCNT(3 * BPW)); break;
        case 2: __builtin_amdgcn_s_waitcnt(TA_VMCNT(2 * BPW)); break;
        case 1: __builtin_amdgcn_s_waitcnt(TA_VMCNT(BPW)); break;
        default: __builtin_amdgcn_s_waitcnt(TA_VMCNT(0)); break;
    }
}

// Two transposing LDS loads -> one 8-element MFMA operand.
__device__ inline u32x4 tr_pair(const u16 *lo, const u16 *hi) {
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)hi);
    const u32x2 ua = __builtin_bit_cast(u32x2, a), ub = __builtin_bit_cast(u32x2, b);
    return u32x4{ua[0], ua[1], ub[0], ub[1]};
}

// LDS layout of one 64-token tile (16-bit elements): KBLK blocks of K, then
// VBLK blocks of V, each a 1 KiB copy unit of 64 16-byte slots.
//   K block b: d-rows 8b..8b+7; the 16-byte chunk c (tokens 8c..8c+7) of
//     d-row 8b+j has logical slot 16*(c>>1) + 8*(j>>2) + 4*(c&1) + (j&3).
//   V block b: token rows VROWS*b ..; chunk s (d = 8s..8s+7) of token row j
//     has logical slot SV*(s>>1) + 8*(j>>2) + 4*(s&1) + (j&3).
// Swizzle: in odd blocks (block index within the tile) logical slot l sits at
// physical slot l ^ 8, i.e. the two 128-byte halves of every 256 bytes are
// swapped.  The four 16-lane groups of a transposing read address blocks of
// alternating parity at equal logical offsets, so the groups land 128 bytes
// apart modulo 256 (disjoint LDS banks) without padding the blocks; a tile is
// 32 KiB and five of them fit the 160 KiB LDS.
struct LdsOfs {  // per-lane element offsets of the transposing reads (swizzle applied)
    int klo, khi;        // K: the two 8-byte halves of a lane's operand
    int kt[4];           // KV_TOKEN: K's 16-byte chunk of the lane's token, per 32-wide slice of d
    int vlo[2], vhi[2];  // V: same, by the parity of the 16-row block db of O^T
};

template <int D>
struct Tile {
    static constexpr int TT = 64;
    static constexpr int BLK = 512;         // 1 KiB block
    static constexpr int KBLK = D / 8;
    static constexpr int VROWS = 512 / D;   // token rows per V block
    static constexpr int VBLK = TT / VROWS;
    static constexpr int NBLK = KBLK + VBLK;
    static constexpr int ELEMS = NBLK * BLK;
    static constexpr int SV = 1024 / D;

    // physical element offset of logical in-block offset `e` in block `b`
    __device__ static int swz(int b, int e) { return e ^ (64 * (b & 1)); }

    // Lane (row, g4) of a transposing read addresses, within its block,
    // logical element 8 * (4 * ((row & 3) >> 1) + (row >> 2)) + 4 * (row & 1)
    // (< 64) of the chunk-slot group it reads; the K operand's two halves are
    // 64 elements apart in block 4 ks + g4 (a parity of g4 & 1 for every ks);
    // the V operand's halves are in blocks KBLK + base / VROWS + vb and
    // 16 / VROWS blocks further (base / VROWS is even), at in-block offset
    // 8 SV db + vin, whose bit 6 depends on db only through SV / 8 (odd for
    // D = 128).
    __device__ static LdsOfs offsets(int row, int g4) {
        const int lane_ofs = 8 * (4 * ((row & 3) >> 1) + (row >> 2)) + 4 * (row & 1);
        LdsOfs o;
        o.klo = BLK * g4 + swz(g4, lane_ofs);
        o.khi = BLK * g4 + swz(g4, lane_ofs + 64);
        const int vb = (4 * g4) / VROWS;
        const int vin = 64 * (((4 * g4) % VROWS) >> 2) + lane_ofs;
        const int blo = KBLK + vb, bhi = blo + 16 / VROWS;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int dbo = 8 * SV * e;  // representative db of parity e
            o.vlo[e] = BLK * vb + swz(blo, dbo + vin) - dbo;
            o.vhi[e] = BLK * (vb + 16 / VROWS) + swz(bhi, dbo + vin) - dbo;
        }
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) o.kt[ks] = row * D + 8 * ((4 * ks + g4) ^ ((row / (128 / D)) % (D / 8)));
        return o;
    }
};

// K of a KV_TOKEN tile: token rows of D elements, CPR 16-byte chunks each.  The
// QK operand is 16 contiguous bytes of one token, read without transposing;
// chunk c of token t sits at chunk c ^ flip(t) of its row, so that the 16 lanes
// (one chunk of 16 tokens) that read together cover 256 different bytes.
template <int D>
struct KTokens {
    static constexpr int CPR = D / 8;
    static constexpr int TPL = 16 / CPR;  // token rows of 256 bytes
    __device__ static int flip(int t) { return (t / TPL) % CPR; }
};

// Copies of one 64-token tile into an LDS stage by NW waves.  Inside the job
// (tokens [t0n, t0n + TT) all in [kst, kend)) no index is clamped; at its edges
// chunks past the pool end read its last chunk and V rows outside the job read
// a row inside it (finite values; their scores are masked, P = 0).
//
// KV_POOL and KV_TOKEN copy both operands by LDS DMA: issue() is all.  A KV_ODD
// pool's K rows start at any 2-byte address, which the DMA does not take: issue()
// loads each lane's 16 bytes into registers (unaligned global loads) and starts V's
// DMA, finish() waits for both and writes K to LDS at the slots the DMA would have
// filled.  The tile's compute runs between the two and hides the loads.  Moving both
// operands through registers with an 8 x 8 transpose took twice as long (24 ragged
// requests in two branches, 10,839 tokens, d = 128: layer 49.2 us, here 25.0 us; 32
// ragged requests, 1,745 tokens, d = 64: 14.4 us, here 8.4 us).
constexpr int SHORT_CAP = 1 << 28;
template <int D, int NW, int L, bool SHORT = false>
struct TileCopy {
    using T = Tile<D>;
    static constexpr int NK = (T::KBLK + NW - 1) / NW;  // K blocks of a wave, V likewise (D = 32: of some waves)
    u32x4 k[L == KV_ODD ? NK : 1];

    // SHORT (short_offsets): a copy's source is a scalar base per block plus a 32-bit lane offset
    // that all tiles of an item share; else a 64-bit address per lane.  In the one-wave kernel the
    // short form streams 128 x 8192 private tokens in 768 us against 782 us; in the mixed kernel,
    // whose scalar registers are full, it is the slower one (32 requests x 4096 tokens: 42.8 us
    // against 41.8 us).
    __device__ static void dma(u16 *dst, const u16 *base, u32 ofs) {
        __builtin_amdgcn_global_load_lds((const void *)((const char *)base + ofs), (lds_void *)dst, 16, 0, 0);
    }

    // Row t of head h of V (and of token-major K).
    __device__ static const u16 *row(const u16 *x, const SegParams &p, int h, int t) {
        return x + (token_major(L) ? (size_t)t * p.hk + h : (size_t)h * p.tcap + t) * D;
    }
    __device__ static u32 row_bytes(const SegParams &p) { return 2u * D * (token_major(L) ? p.hk : 1); }

    // Byte offsets of this lane's 16 bytes in a KV_POOL tile's copies of wave w from the first
    // row of the block copied: K block w + n NW, and V block w + n NW (NW and KBLK even, so
    // that a block's parity, which the swizzle follows, is w's).
    __device__ static u32 k_offset(const SegParams &p, int w, int lane) {
        const int l = lane ^ (8 * (w & 1));
        return 2u * ((u32)(4 * ((l >> 3) & 1) + (l & 3)) * (u32)p.tcap + 8 * (2 * (l >> 4) + ((l >> 2) & 1)));
    }
    __device__ static u32 v_offset(int w, int lane) {
        static_assert(NW % 2 == 0 || NW == 1, "one parity per wave");
        const int l = lane ^ (8 * (w & 1)), rem = l % T::SV;
        return 2u * ((4 * (rem >> 3) + (rem & 3)) * D + 8 * (2 * (l / T::SV) + ((rem >> 2) & 1)));
    }

    // Row t0n + t of a tile, chunk s; `base`: a row of the tile that is the same for all lanes.
    template <bool CLAMP>
    __device__ static void copy_row(u16 *dst, const u16 *x, const SegParams &p, int h, int t0n, int kst, int kend,
                                    int first, int j, int s) {
        if constexpr (SHORT) {
            const int from = CLAMP ? max(t0n, kst) : t0n + first;
            const int r = CLAMP ? min(max(t0n + first + j, kst), kend - 1) - from : j;
            dma(dst, row(x, p, h, from), r * row_bytes(p) + 16 * s);
        } else {
            const int t = t0n + first + j;
            dma(dst, row(x, p, h, CLAMP ? min(max(t, kst), kend - 1) : t) + 8 * s, 0);
        }
    }

    template <bool CLAMP>
    __device__ static void copy_v(u16 *st, const SegParams &p, int h, int t0n, int kst, int kend, int vb, int lane) {
        const int l = lane ^ (8 * ((T::KBLK + vb) & 1));  // logical slot filled by this lane (swizzle)
        const int rem = l % T::SV;
        copy_row<CLAMP>(st + (T::KBLK + vb) * T::BLK, p.vp, p, h, t0n, kst, kend, vb * T::VROWS,
                        4 * (rem >> 3) + (rem & 3), 2 * (l / T::SV) + ((rem >> 2) & 1));
    }

    template <bool CLAMP>
    __device__ static void copy_k(u16 *st, const SegParams &p, int h, int t0n, int kst, int kend, int blk, int lane) {
        u16 *dst = st + blk * T::BLK;
        if constexpr (token_major(L)) {
            // row-major tile: lane i fills slot i, chunk (i % CPR) ^ f of token row i / CPR (KTokens)
            const int j = lane / KTokens<D>::CPR;
            copy_row<CLAMP>(dst, p.kp, p, h, t0n, kst, kend, blk * T::VROWS, j,
                            (lane % KTokens<D>::CPR) ^ KTokens<D>::flip(blk * T::VROWS + j));
        } else {
            const int l = lane ^ (8 * (blk & 1));
            const int tok = 8 * (2 * (l >> 4) + ((l >> 2) & 1));
            const int j = 4 * ((l >> 3) & 1) + (l & 3);
            const int last = p.tcap - 8;  // (a tile starts inside the pool, at a multiple of 8 like its capacity)
            if constexpr (SHORT)
                dma(dst, p.kp + (size_t)(h * D + 8 * blk) * p.tcap + t0n,
                    2u * ((u32)j * (u32)p.tcap + (u32)(CLAMP ? min(tok, last - t0n) : tok)));
            else
                dma(dst, p.kp + (size_t)(h * D + 8 * blk + j) * p.tcap + (CLAMP ? min(t0n + tok, last) : t0n + tok), 0);
        }
    }

    template <bool CLAMP>
    __device__ static void copy_blocks(u16 *st, const SegParams &p, int h, int t0n, int kst, int kend, int w, int lane) {
#pragma unroll
        for (int n = 0; n < T::NBLK / NW; ++n) {
            // One wave alone alternates K (64 tokens of 8 rows, tcap apart) and V (one run of
            // 1 KiB): 16 strided blocks in a row, then 16 of a run, kept fewer HBM channels
            // busy (128 x 8192 private tokens, 4.3 GB: 818 us against 776 us).
            const int i = NW == 1 ? (n & 1) * T::KBLK + (n >> 1) : n;
            const int blk = w + i * NW;
            // with KBLK % NW == 0 every wave's i-th block is K for the same i
            const bool isk = T::KBLK % NW == 0 ? i * NW < T::KBLK : blk < T::KBLK;
            if (isk)
                copy_k<CLAMP>(st, p, h, t0n, kst, kend, blk, lane);
            else
                copy_v<CLAMP>(st, p, h, t0n, kst, kend, blk - T::KBLK, lane);
        }
    }

    // KV_ODD: this wave's K blocks of the tile into registers
    __device__ void load_k(const SegParams &p, int h, int t0n, int w, int lane) {
        const bool inside = t0n + T::TT <= p.tcap;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int blk = w + i * NW;
            if (T::KBLK % NW != 0 && blk >= T::KBLK) continue;
            const int l = lane ^ (8 * (blk & 1));
            const int tok = t0n + 8 * (2 * (l >> 4) + ((l >> 2) & 1));
            const int d = 8 * blk + 4 * ((l >> 3) & 1) + (l & 3);
            const u16 *src = p.kp + (size_t)(h * D + d) * p.tcap;
            if (inside) {
                __builtin_memcpy(&k[i], src + tok, 16);
            } else {  // the pool's last tile, element by element
                u32 e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = src[min(tok + j, p.tcap - 1)];
                k[i] = u32x4{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
            }
        }
    }

    __device__ void issue(u16 *st, const SegParams &p, int h, int t0n, int kst, int kend, int wave, int lane) {
        const int w = __builtin_amdgcn_readfirstlane(wave);
        const bool inner = t0n >= kst && t0n + T::TT <= kend;
        if constexpr (L == KV_ODD) {
            load_k(p, h, t0n, w, lane);
#pragma unroll
            for (int i = 0; i < NK; ++i) {
                const int vb = w + i * NW;
                if (T::VBLK % NW != 0 && vb >= T::VBLK) continue;
                if (inner)
                    copy_v<false>(st, p, h, t0n, kst, kend, vb, lane);
                else
                    copy_v<true>(st, p, h, t0n, kst, kend, vb, lane);
            }
        } else if (inner) {
            copy_blocks<false>(st, p, h, t0n, kst, kend, w, lane);
        } else {
            copy_blocks<true>(st, p, h, t0n, kst, kend, w, lane);
        }
    }

    // KV_ODD: everything issued has landed; K goes to the stage.  The LDS writes
    // are done when this returns (a barrier makes them the other waves').
    __device__ void finish(u16 *st, int wave, int lane) {
        if constexpr (L == KV_ODD) {
            const int w = __builtin_amdgcn_readfirstlane(wave);
            __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
#pragma unroll
            for (int i = 0; i < NK; ++i) {
                const int blk = w + i * NW;
                if (T::KBLK % NW != 0 && blk >= T::KBLK) continue;
                *(u32x4 *)(st + blk * T::BLK + 8 * lane) = k[i];
            }
            __builtin_amdgcn_s_waitcnt(TA_LGKMCNT0);
        }
    }
};

// The softmax denominator of a lane's row.  KV_POOL and KV_TOKEN: one more PV MFMA against
// an all-ones A operand, so that it sums exactly the rounded P that multiplies V.  The
// others (odd_count): the FP32 exponentials themselves, each lane its own tokens, added over the four lanes of
// the row at the end -- the log-sum-exp then carries no rounding of P.  Against the ones
// product: 24 ragged requests in two branches, 10,839 tokens, 25.7 us (25.5); 128 requests x
// 8192 in 256-row items 51.0 us (48.3, with the tails' merge fused).
template <int L>
struct RowSum {
    static constexpr bool FP32 = odd_count(L);
    f32x4 v;  // FP32: v[0] alone
    __device__ void reset() { v = f32x4{0.f, 0.f, 0.f, 0.f}; }
    __device__ void scale(float a) {
        if constexpr (FP32)
            v[0] *= a;
        else
            v *= a;
    }
    __device__ void add(const float (&p)[8]) {
        if constexpr (FP32) v[0] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    }
    template <class O>
    __device__ void add_rounded(u32x4 pb) {
        if constexpr (!FP32) v = O::mma_k32(u32x4{O::ONE2, O::ONE2, O::ONE2, O::ONE2}, pb, v);
    }
    __device__ float total() const {  // all four lanes of the row active
        if constexpr (FP32) {
            const float s = v[0] + __shfl_xor(v[0], 16);
            return s + __shfl_xor(s, 32);
        }
        return v[0];
    }
};

// odd_count layouts: V^T fragments of a step of which only the first n tokens are the job's, the others
// zero (the stage holds a row of the job there, which P = 0 would not cancel if it is infinite).
template <int DB>
__device__ inline void mask_v(u32x4 (&vf)[DB], int n, int g4) {
    u32x4 keep;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = 16 * (j >> 1) + 4 * g4 + 2 * (j & 1);
        keep[j] = (t < n ? 0xffffu : 0u) | (t + 1 < n ? 0xffff0000u : 0u);
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) vf[db] &= keep;
}

template <int D, bool FP16, int NB, int NW, int L>
struct TileMath {
    static constexpr int DB = D / 16;  // 16-row blocks of O^T
    static constexpr int KS = D / 32;  // 32-wide k slices of QK
    using O = Ops<FP16>;
    using T = Tile<D>;
    using Z = RowSum<L>;

    f32x4 o[NB][DB];
    Z z[NB];
    float m[NB];

    __device__ void reset() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            m[nb] = NEG_INF;
            z[nb].reset();
#pragma unroll
            for (int db = 0; db < DB; ++db) o[nb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }

    // One pipeline step: copy the tile at pool token t0n into stage `nxt` (if
    // `copy`), then compute the tile staged in `cur` (if `compute`).  The two
    // stages never alias; declaring them restrict in one function lets the
    // compiler keep the copies in flight across the reads of `cur`.
    __device__ void step(const u16 *__restrict__ cur, u16 *__restrict__ nxt, bool copy, bool compute,
                         const SegParams &p, int h, int t0n, int kst, int kend, int wave, int lane,
                         const u32x4 (&qf)[NB][KS], const LdsOfs &of, int lo, int hi, int g4, float c) {
        using C = TileCopy<D, NW, L>;
        C kr;
        if (copy) kr.issue(nxt, p, h, t0n, kst, kend, wave, lane);
        if (compute) tile(cur, qf, of, lo, hi, g4, c);
        if (copy) kr.finish(nxt, wave, lane);
    }

    // K fragments (A operand of QK) of the 32 tokens base .. base+31:
    // kf[b][ks] covers tokens base+16b .. +15, d = 32*ks .. +31.
    __device__ static void load_k(const u16 *__restrict__ cur, const LdsOfs &of, int base, u32x4 (&kf)[2][KS]) {
        if constexpr (token_major(L)) {
            u32 a[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) a[ks] = (u32)(uintptr_t)(lds_u16 *)(cur + of.kt[ks] + base * D);
            read_tokens(a, kf);
            return;
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kf[b][ks] = k_pair(cur, of, base, b, ks);
    }

    // one of them (not KV_TOKEN): block 4*ks + g4, chunk pair base/16 + b, block rows 0-3 / 4-7
    __device__ static u32x4 k_pair(const u16 *__restrict__ cur, const LdsOfs &of, int base, int b, int ks) {
        const int e = 4 * T::BLK * ks + 8 * (base + 16 * b);
        return tr_pair(cur + of.klo + e, cur + of.khi + e);
    }

    // KV_TOKEN: the chunks at LDS byte addresses a[ks] and 16 tokens further.  For
    // an ordinary LDS read the compiler waits for every LDS DMA in flight (it
    // cannot tell the stages apart), so these are written out, wait included.
    __device__ static void read_tokens(const u32 (&a)[KS], u32x4 (&kf)[2][KS]) {
        constexpr int N = 32 * D;  // bytes of 16 token rows
        if constexpr (KS == 4)
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
                         "ds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
                         "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\t"
                         "ds_read_b128 %6, %10 offset:%12\n\tds_read_b128 %7, %11 offset:%12\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(kf[0][0]), "=&v"(kf[0][1]), "=&v"(kf[0][2]), "=&v"(kf[0][3]), "=&v"(kf[1][0]),
                           "=&v"(kf[1][1]), "=&v"(kf[1][2]), "=&v"(kf[1][3])
                         : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "n"(N)
                         : "memory");
        else if constexpr (KS == 2)
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
                         "ds_read_b128 %2, %4 offset:%6\n\tds_read_b128 %3, %5 offset:%6\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(kf[0][0]), "=&v"(kf[0][1]), "=&v"(kf[1][0]), "=&v"(kf[1][1])
                         : "v"(a[0]), "v"(a[1]), "n"(N)
                         : "memory");
        else
            asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(kf[0][0]), "=&v"(kf[1][0])
                         : "v"(a[0]), "n"(N)
                         : "memory");
    }

    // V^T fragments (A operand of PV) of the 32 tokens base .. base+31: PV
    // k-slot j of lane group g4 is token 4*g4+j (j<4) or 16+4*g4+j-4 (j>=4),
    // where the QK output left P.
    __device__ static void load_v(const u16 *__restrict__ st, const LdsOfs &of, int base, u32x4 (&v)[DB]) {
        const u16 *vrow = st + T::BLK * (T::KBLK + base / T::VROWS);
#pragma unroll
        for (int db = 0; db < DB; ++db) v[db] = v_pair(vrow, of, db);
    }

    // one of them; vrow: the stage's first V block of the step
    __device__ static u32x4 v_pair(const u16 *__restrict__ vrow, const LdsOfs &of, int db) {
        const u16 *va = vrow + 8 * T::SV * db;
        return tr_pair(va + of.vlo[db & 1], va + of.vhi[db & 1]);
    }

    // S^T = K Q^T: s[nb][b] holds tokens base+16b+4*g4+i of row block nb.
    __device__ static void qk(const u32x4 (&kf)[2][KS], const u32x4 (&qf)[NB][KS], f32x4 (&s)[NB][2]) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s[nb][0] = s[nb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) s[nb][b] = O::mma_k32(kf[b][ks], qf[nb][ks], s[nb][b]);
    }

    // of: per-lane element offsets of the transposing loads;
    // tokens [lo, hi) of the tile belong to the job.  Software pipeline per
    // 32-token step k: the LDS loads of step k's V and step k+1's K are issued
    // before step k's softmax (which hides their latency), then PV of step k
    // and QK of step k+1 run back to back on the matrix cores.
    __device__ void tile(const u16 *__restrict__ cur, const u32x4 (&qf)[NB][KS], const LdsOfs &of, int lo,
                         int hi, int g4, float c) {
        constexpr int STEPS = T::TT / 32;
        f32x4 s[NB][2];
        {
            u32x4 kf[2][KS];
            load_k(cur, of, 0, kf);
            qk(kf, qf, s);
        }
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            const int base = 32 * k;
            if (base >= hi) break;
            u32x4 vf[DB];
            load_v(cur, of, base, vf);
            const bool more = k + 1 < STEPS && base + 32 < hi;
            u32x4 kf[2][KS];
            if (more) load_k(cur, of, base + 32, kf);
            if (lo > base || hi < base + 32) {  // wave-uniform: first or last step of the job
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int tok = base + 16 * b + 4 * g4 + i;
                            if (tok < lo || tok >= hi) s[nb][b][i] = NEG_INF;
                        }
                if constexpr (Z::FP32) mask_v(vf, hi - base, g4);
            }
            // ---- softmax of every row block -> P^T fragments (B operand of PV)
            u32x4 pb[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                float x[8];
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[4 * b + i] = s[nb][b][i];
                const float lm = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                                       fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
                const bool need = lm * c > m[nb] + TAU;
                if (__builtin_amdgcn_ballot_w64(need)) {  // wave-uniform, rare after the first step
                    const float mn = fmaxf(m[nb], xor_max(lm) * c);
                    const float alpha = fast_exp2(m[nb] - mn);
                    z[nb].scale(alpha);
#pragma unroll
                    for (int db = 0; db < DB; ++db) o[nb][db] *= alpha;
                    m[nb] = mn;
                }
                float pr[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) pr[i] = fast_exp2(__builtin_fmaf(x[i], c, -m[nb]));
                z[nb].add(pr);
                pb[nb] = u32x4{O::pack(pr[0], pr[1]), O::pack(pr[2], pr[3]), O::pack(pr[4], pr[5]),
                               O::pack(pr[6], pr[7])};
            }
            // ---- O^T += V^T P^T (each V^T fragment feeds NB MFMAs), then QK of step k+1
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) o[nb][db] = O::mma_k32(vf[db], pb[nb], o[nb][db]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) z[nb].template add_rounded<O>(pb[nb]);
            if (more) qk(kf, qf, s);
        }
    }
};

// Work item of linear block b of n: block b runs on XCD b % 8, and every XCD
// gets a contiguous range of items, so that row tiles of one (job, head)
// share its L2.
__device__ inline int xcd_item(int b, int n) {
    const int xcd = b & 7, slot = b >> 3;
    const int q8 = n >> 3, rm = n & 7;
    return xcd * q8 + min(xcd, rm) + slot;
}

// First token of the tiles of a job or segment that starts at token t: a KV_POOL
// K row is copied in aligned chunks of 8 tokens (KV_TOKEN follows it, so that both
// sum in the same order; the odd_count layouts start at the job's first token).
template <int L>
__device__ inline int tile_start(int t) {
    return odd_count(L) ? t : t & ~7;
}

// The waves of a work item meet at a barrier, unless one wave works alone on
// its own LDS stage (SOLO), where its own vmcnt wait orders copy and reads.
template <bool SOLO>
__device__ inline void item_barrier() {
    if constexpr (!SOLO) __builtin_amdgcn_s_barrier();
}

// One work item (job, first row, KV head) of the tile kernels: NW waves, NB
// 16-row blocks per wave, STAGES LDS stages at `lds`.  The item holds rows
// [row0, row0 + item_rows) of its job.  SOLO: one wave alone (tid = its lane).
template <int D, bool FP16, int NB, int NW, int STAGES, int L, bool SOLO = false, bool SHORT = false>
__device__ __forceinline__ void tile_item(const SegParams &p, const int32_t *__restrict__ items, int item,
                                          u16 *lds, int tid, int item_rows) {
    using T = Tile<D>;
    using M = TileMath<D, FP16, NB, NW, L>;
    using C = TileCopy<D, NW, L, SHORT>;
    constexpr int KS = M::KS;
    constexpr int BPW = T::NBLK / NW;  // copies per wave per tile
    static_assert(T::NBLK % NW == 0, "every wave copies the same number of blocks");
    static_assert(STAGES >= 1 && STAGES <= 3, "one to three LDS stages");
    static_assert(!SOLO || (NW == 1 && STAGES == 1), "a wave alone has one stage");
    const int job = items[3 * item], row0 = items[3 * item + 1], h = items[3 * item + 2];

    const int lane = tid & 63, wave = SOLO ? 0 : tid >> 6;
    const int row = lane & 15, g4 = lane >> 4;
    const int kst = p.kstart[job];
    const int ntok = max(0, min(p.klen[job], p.tcap - kst));
    const int kend = kst + ntok;
    const int nrows = min(p.qlen[job] * p.group, row0 + item_rows);
    const int wrow0 = row0 + 16 * NB * wave;
    const bool active = wrow0 < nrows;

    const int rb = sload(p.rowbase, job), qb = p.qbase ? sload(p.qbase, job) : -1;
    const int tb0 = tile_start<L>(kst);
    const int ntiles = ntok > 0 ? (kend - tb0 + T::TT - 1) / T::TT : 0;

    // Q^T fragments (B operand): lane (row, g4) holds d = 32*ks + 8*g4 .. +7 (rows
    // past the item repeat its last row and are never stored).  A job over
    // consecutive requests (qbase) needs no request-id loads.  The first tile's
    // copies go out behind the Q loads, so that one wait covers both.
    const int last = max(nrows, 1) - 1;  // (a job without requests reads a row and stores none)
    u32x4 qf[NB][KS];
    const u16 *qsrc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int rr = min(wrow0 + 16 * nb + row, last);
        const int lr = rr / p.group;
        int rq = qb + lr;
        if (qb < 0) {
            rq = nrows > 0 ? p.qids[(size_t)job * p.maxr + lr] : 0;
            asm volatile("" : "+v"(rq));  // waited for in this branch only
        }
        qsrc[nb] = p.q + ((size_t)rq * p.hq + h * p.group + (rr - lr * p.group)) * D + 8 * g4;
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[nb][ks] = *(const u32x4 *)(qsrc[nb] + 32 * ks);
    asm volatile("" ::: "memory");
    C first;
    if (ntiles > 0) first.issue(lds, p, h, tb0, kst, kend, wave, lane);
    // Pin the Q fragments: an empty asm that "redefines" them makes the wave
    // wait for the Q loads (and the first tile) once, here, and not inside the
    // tile loop behind the copies in flight.
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[nb][ks]));
    if (ntiles > 0) first.finish(lds, wave, lane);

    M acc;
    acc.reset();
    const LdsOfs of = T::offsets(row, g4);

    if (STAGES == 1) {
        // one stage (one-wave workgroups, five per CU): copy, wait, compute
        for (int it = 0; it < ntiles; ++it) {
            const int t0 = tb0 + it * T::TT;
            if (it > 0) {
                item_barrier<SOLO>();  // every wave is done with the previous tile
                C kr;
                kr.issue(lds, p, h, t0, kst, kend, wave, lane);
                __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
                kr.finish(lds, wave, lane);
            } else {
                __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
            }
            item_barrier<SOLO>();
            if (active) acc.tile(lds, qf, of, max(0, kst - t0), min(T::TT, kend - t0), g4, p.scale_log2);
        }
    } else {
    // Iteration it copies tile it+STAGES-1 and computes tile it (stage it %
    // STAGES); the first STAGES-2 iterations only copy (tile 0 is under way).
    constexpr int AHEAD = STAGES > 1 ? STAGES - 1 : 1;
    int cs = STAGES > 1 ? STAGES - AHEAD + 1 : 0;  // stage of tile it, starting at it = 1 - AHEAD
    if (cs == STAGES) cs = 0;
    for (int it = 1 - AHEAD; it < ntiles; ++it) {
        if (it >= 0) {
            // this wave's copies of tile it are done once at most those of the
            // tiles after it (issued, at most AHEAD-1 of them) are pending
            if (AHEAD == 2 && it + 1 < ntiles && L != KV_ODD)  // (KV_ODD: finish() waited for all)
                __builtin_amdgcn_s_waitcnt(TA_VMCNT(BPW));
            else
                __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
            item_barrier<SOLO>();  // every copy of tile it landed; stage of tile it-1 is free
        }
        const int ns = cs == 0 ? STAGES - 1 : cs - 1;  // stage of tile it+AHEAD (that of tile it-1)
        const int t0 = tb0 + it * T::TT;
        acc.step(lds + cs * T::ELEMS, lds + ns * T::ELEMS, it + AHEAD < ntiles, it >= 0 && active, p, h,
                 t0 + AHEAD * T::TT, kst, kend, wave, lane, qf, of, max(0, kst - t0), min(T::TT, kend - t0), g4,
                 p.scale_log2);
        cs = cs == STAGES - 1 ? 0 : cs + 1;
    }
    }

    if (!active) return;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int grow = wrow0 + 16 * nb + row;
        const float z = acc.z[nb].total();
        if (grow >= nrows) continue;
        const int lr = grow / p.group, gg = grow - lr * p.group;
        const size_t prow = (size_t)(rb + lr) * p.hq + h * p.group + gg;
        store_partial<M::DB>(p.part, p.lse, prow, acc.o[nb], acc.m[nb], z, g4);
    }
}

// One-wave items lie job by job with the KV heads inside.  Item i may go to XCD i % 8 ("by
// head": an XCD works on one head of 8 and translates and caches an eighth of the pools)
// or an XCD gets a range of jobs.  By head only where a head has four rows or more: items
// of fewer rows write neighbouring pieces of the same cache lines (a row's entry of `lse`
// is 8 bytes), and those then come from all XCDs, about 1.3 us a launch (32 requests x 128
// tokens, 8 heads of 32, one row each: 6.9 us by job, 8.2 by head; 8 requests, 1024 shared
// + 64 tokens, 8 heads of 128, four rows: 10.1 and 9.1).
//
// A launch of one-wave items alone goes by head only when they all run at once, five
// workgroups of 32 KiB per CU at d = 128 (128 x 8192 private tokens, several rounds: 781 us
// by job, 793 by head).  At d = 64 more of them do, but gain nothing (1,600 and 1,920 items
// 11.1 and 11.9 us by job, 11.0 and 11.8 by head; 4,096 items 24.0 and 24.9).
constexpr int ONE_ROUND = 5 * 256;
__device__ inline bool tile_by_head(const SegParams &p, int items) {
    return items <= ONE_ROUND && p.hk % 8 == 0 && p.group >= 4;
}
// Beside 64-row items also in several rounds (layers of 32 and 24 requests in two branches
// 43.3 -> 42.5 us and 26.2 -> 25.1; 96 requests x 64 tokens, eight rows a head 28.8 -> 27.4),
// and with fewer rows from two rounds of four a CU on at d = 128, whose 16-KiB runs then
// weigh more (3,072 items of one row, 16 heads: 36.4 -> 33.7 us; 768 of them 16.6 -> 17.8;
// d = 64 and 32 at 3,072 items 21.2 -> 22.0 and 13.5 -> 14.7).  Two heads gain nothing
// (0.0-0.15 us slower by head), four are even.  Beside 256-row items, which fill whole CUs
// by head already, four neighbours share a workgroup (by head 0.1-0.5 us slower).
inline bool mix_by_head(const SegParams &p, const int n[3], int d) {
    if (n[0] > 0 || p.hk % 4 != 0) return false;
    return p.group >= 4 || (d == 128 && p.hk % 8 == 0 && n[2] >= 2 * 4 * 256);
}
template <int D, bool FP16, int NB, int NW, int STAGES, int L, bool SHORT = false>
__global__ __launch_bounds__(64 * NW) void seg_tile_kernel(const int32_t *items, SegParams p) {
    __shared__ __attribute__((aligned(16))) u16 lds[STAGES * Tile<D>::ELEMS];
    const bool by_head = NW == 1 && tile_by_head(p, gridDim.x);
    const int item = by_head ? blockIdx.x : xcd_item(blockIdx.x, gridDim.x);
    tile_item<D, FP16, NB, NW, STAGES, L, false, SHORT>(p, items, item, lds, threadIdx.x, 16 * NB * NW);
}

// ------------------------------------------------------------------------
// Pipelined large-tile kernel.  The 32-token steps of a work item form one
// software pipeline that runs across tile boundaries; within a step the
// matrix cores and the VALU work on different steps:
//
//   block(g):  QK of step g+1 (MFMA)   || exponentials of step g (VALU),
//                                          LDS reads of V(g)
//              PV + row sums of step g  || LDS reads of K(g+2), masking and
//                                          row maxima of step g+1
//
// and the rare online-softmax rescale runs between blocks.  The order inside
// a block is written out so that MFMAs, LDS reads and VALU instructions
// alternate in each wave's instruction stream (see block()).  K/V tiles arrive
// by LDS DMA into five stages: tiles t and t+1 are read while t+2 .. t+4 are
// in flight, with one barrier per tile.
template <int D, bool FP16, int NW, int NB_, int L>
struct PipeMath {
    static constexpr int NB = NB_;
    static constexpr int DB = D / 16;
    static constexpr int KS = D / 32;
    using O = Ops<FP16>;
    using T = Tile<D>;
    using TM = TileMath<D, FP16, NB, NW, L>;
    using Z = RowSum<L>;

    f32x4 o[NB][DB];
    Z z[NB];
    float m[NB], lm[NB], thr[NB];  // running max (scaled), raw row max of the staged step, (m + TAU) / c
    f32x4 s[NB][2];      // scores of the step whose exponentials come next
    u32x4 kf[2][KS];     // K fragments of the next QK step
    u32x4 vf[DB];        // V^T fragments of the current PV step

    __device__ void reset() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            m[nb] = thr[nb] = NEG_INF;
            z[nb].reset();
#pragma unroll
            for (int db = 0; db < DB; ++db) o[nb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }

    // Scores of a step: mask tokens outside [lo, hi) (if MASK) and take the
    // lane-local row maxima.
    template <bool MASK>
    __device__ void finish_scores(f32x4 (&sn)[NB][2], int lo, int hi, int g4) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (MASK) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int tok = 16 * b + 4 * g4 + i;
                        if (tok < lo || tok >= hi) sn[nb][b][i] = NEG_INF;
                    }
            }
            float mx = sn[nb][0][0];  // a chain, so that it becomes three-input maxima
#pragma unroll
            for (int i = 1; i < 8; ++i) mx = fmaxf(mx, sn[nb][i >> 2][i & 3]);
            lm[nb] = mx;
            s[nb][0] = sn[nb][0];
            s[nb][1] = sn[nb][1];
        }
    }

    // The running maxima from the job's first scored step: O and z are still
    // zero, so the maxima are set without the pass over O that rescale makes
    // (the values equal rescale's from the initial state).
    __device__ void first_max(float c, float rc) {
        if constexpr (Z::FP32) return rescale(c, rc);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const float mn = xor_max(lm[nb]) * c;
            m[nb] = mn;
            thr[nb] = (mn + TAU) * rc;
        }
    }

    // Raise the running maxima where a score of the staged step exceeds them
    // by more than TAU (wave-uniform branch, rare after the first step).  odd_count
    // layouts decide it per row block as tile() does, so that a row's result does not
    // depend on the kind of item it is in.
    __device__ void rescale(float c, float rc) {  // rc = 1 / c
        if constexpr (Z::FP32) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if (!__builtin_amdgcn_ballot_w64(lm[nb] * c > m[nb] + TAU)) continue;
                const float mn = fmaxf(m[nb], xor_max(lm[nb]) * c);
                const float alpha = fast_exp2(m[nb] - mn);
                z[nb].scale(alpha);
#pragma unroll
                for (int db = 0; db < DB; ++db) o[nb][db] *= alpha;
                m[nb] = mn;
            }
            return;
        }
        bool need = false;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) need |= lm[nb] > thr[nb];
        if (__builtin_amdgcn_ballot_w64(need)) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const float mn = fmaxf(m[nb], xor_max(lm[nb]) * c);
                const float alpha = mn == NEG_INF ? 1.f : fast_exp2(m[nb] - mn);
                z[nb].scale(alpha);
#pragma unroll
                for (int db = 0; db < DB; ++db) o[nb][db] *= alpha;
                m[nb] = mn;
                thr[nb] = (mn + TAU) * rc;  // raw-score threshold of the next rescale
            }
        }
    }

    // One pipeline block (see above).  vs / vbase: stage and offset of V(g);
    // ks / kbase: of K(g+2) (any resident step when there is none); lo / hi:
    // valid tokens of step g+1 (without MORE: of step g, for odd_count layouts).  Every fragment register set is reloaded only
    // after its last reader: V(g) during QK(g+1), K(g+2) during PV(g).
    //
    // With MORE the order is written out, one matrix instruction per slot, and each
    // slot is closed by a sched_barrier: left to the compiler, sched_group_barrier
    // or not, all 16 K reads ended up behind the PV MFMAs and all V reads behind
    // half of QK's, so that every wave waited for LDS twice per step, all eight at
    // once (root kernel at 128 x 8192 28.1 -> 27.5 us by dispatch stamps).  What was
    // left per 64-token tile, 2.27 us on random data, was the matrix cores' own 1.36
    // us (that loop without copies, barrier, LDS reads and exponentials) plus about
    // 0.4 us each for the tile's copies, all sent behind the barrier, and the LDS
    // reads, 0.15 us each for the exponentials and the barrier.
    // `copy`, called with the slot's number, may start a copy of a later tile there.
    struct NoCopy {
        __device__ void operator()(int) const {}
    };
    template <bool MORE, bool MASKN, bool ROWMASK = false, class Copy = NoCopy>
    __device__ __forceinline__ void block(const u16 *__restrict__ vs, int vbase, const u16 *__restrict__ ks,
                                          int kbase, const u32x4 (&qf)[NB][KS], const LdsOfs &of, int lo,
                                          int hi, int g4, float c, unsigned keep = ~0u, Copy copy = Copy()) {
        u32x4 pb[NB];
        if constexpr (MORE) {
            constexpr int NQ = 2 * KS * NB;      // MFMAs of QK
            constexpr int EXPS = 8 * NB / NQ;    // exponentials per slot (1, 2, 4)
            f32x4 sn[NB][2];
            float pr[NB][8];
            const u16 *vrow = vs + T::BLK * (T::KBLK + vbase / T::VROWS);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                const int k = i / (2 * NB), b = i / NB % 2, nb = i % NB;
                sn[nb][b] = O::mma_k32(kf[b][k], qf[nb][k], k == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sn[nb][b]);
                if (i < DB) vf[i] = TM::v_pair(vrow, of, i);
                copy(i);
#pragma unroll
                for (int e = i * EXPS; e < (i + 1) * EXPS; ++e) {
                    const int n = e / 8, x = e % 8;
                    pr[n][x] = fast_exp2(__builtin_fmaf(s[n][x >> 2][x & 3], c, -m[n]));
                    if (x == 7) {
                        z[n].add(pr[n]);
                        pb[n] = u32x4{O::pack(pr[n][0], pr[n][1]), O::pack(pr[n][2], pr[n][3]),
                                      O::pack(pr[n][4], pr[n][5]), O::pack(pr[n][6], pr[n][7])};
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // V has landed by now; waited for here, the K reads below stay in flight behind PV
            __builtin_amdgcn_s_waitcnt(TA_LGKMCNT0);
            // the next step's maxima, two scores at a time, in the slots after the K reads
            constexpr int NP = DB * NB, FROM = NP > 4 * NB ? NP - 4 * NB : 0;
            float mx[NB];
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                const int db = j / NB, nb = j % NB;
                o[nb][db] = O::mma_k32(vf[db], pb[nb], o[nb][db]);
                if (token_major(L) ? j == 0 : j < 2 * KS) {
                    if constexpr (token_major(L))
                        TM::load_k(ks, of, kbase, kf);
                    else
                        kf[j % 2][j / 2] = TM::k_pair(ks, of, kbase, j % 2, j / 2);
                }
                if (!MASKN && j >= FROM) {
#pragma unroll
                    for (int u = (j - FROM) * 4 * NB / (NP - FROM); u < (j - FROM + 1) * 4 * NB / (NP - FROM); ++u) {
                        const int n = u % NB, x = 2 * (u / NB);
                        const float a0 = sn[n][x >> 2][x & 3], a1 = sn[n][x >> 2][(x & 3) + 1];
                        mx[n] = x == 0 ? fmaxf(a0, a1) : fmaxf(fmaxf(mx[n], a0), a1);
                        asm volatile("" : "+v"(mx[n]));  // in this slot, not at its last use
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) z[nb].template add_rounded<O>(pb[nb]);
            if constexpr (MASKN) {
                finish_scores<true>(sn, lo, hi, g4);
            } else {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    lm[nb] = mx[nb];
                    s[nb][0] = sn[nb][0];
                    s[nb][1] = sn[nb][1];
                }
            }
            return;
        }
        TM::load_v(vs, of, vbase, vf);
        if constexpr (Z::FP32)
            if (hi < 32) mask_v(vf, hi, g4);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float pr[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) pr[i] = fast_exp2(__builtin_fmaf(s[nb][i >> 2][i & 3], c, -m[nb]));
            z[nb].add(pr);
            pb[nb] = u32x4{O::pack(pr[0], pr[1]), O::pack(pr[2], pr[3]), O::pack(pr[4], pr[5]),
                           O::pack(pr[6], pr[7])};
            if (ROWMASK && !((keep >> nb) & 1)) pb[nb] = u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) o[nb][db] = O::mma_k32(vf[db], pb[nb], o[nb][db]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) z[nb].template add_rounded<O>(pb[nb]);
    }

    // One staged tile of an attached private segment (after the pipeline has
    // drained): tokens [lo, hi) of the tile, for this wave's rows [rlo, rhi)
    // only.  Other rows get P = 0 and keep their running maxima, so their
    // state is unchanged.
    __device__ void tail_tile(const u16 *__restrict__ st, const u32x4 (&qf)[NB][KS], const LdsOfs &of, int lo,
                              int hi, int rlo, int rhi, int row, int g4, float c, float rc) {
        unsigned keep = 0;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) keep |= (unsigned)(16 * nb + row >= rlo && 16 * nb + row < rhi) << nb;
#pragma unroll
        for (int k = 0; k < T::TT / 32; ++k) {
            const int base = 32 * k;
            if (base >= hi) break;
            f32x4 sn[NB][2];
            TM::load_k(st, of, base, kf);
            TM::qk(kf, qf, sn);
            if (lo <= base && hi >= base + 32)  // wave-uniform: every token of the step is the segment's
                finish_scores<false>(sn, 0, 32, g4);
            else
                finish_scores<true>(sn, lo - base, hi - base, g4);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                if (!((keep >> nb) & 1)) lm[nb] = NEG_INF;
            rescale(c, rc);
            block<false, false, true>(st, base, st, 0, qf, of, 0, 32, g4, c, keep);
        }
    }
};

#ifndef TA_PIPE_STAGES
#define TA_PIPE_STAGES 5
#endif
#ifndef TA_PIPE_PRO
#define TA_PIPE_PRO 3  // measured: 3 of 5 tiles in the prologue start the loop earliest
#endif

// STAGES LDS tiles; the waves meet at a barrier every SYNC tiles.  While the
// waves work on tiles t .. t+SYNC-1 they read those and the K of tile t+SYNC
// (the pipelined steps read one step ahead), so SYNC+1 tiles are resident
// and STAGES-SYNC-1 more can be in flight.  The prologue issues PRO tiles;
// the first loop barrier issues the rest of the ring.
// One 256-row work item of the pipelined kernel, with its attached segments
// (p.xtail, indexed by the item), STAGES LDS stages at `lds`.
template <int D, bool FP16, int NW, int NB, int L, int STAGES = TA_PIPE_STAGES, int SYNC = 1, int PRO = TA_PIPE_PRO>
__device__ __forceinline__ void pipe_item(const SegParams &p, const int32_t *__restrict__ items, int item, u16 *lds,
                                          int tid) {
    using T = Tile<D>;
    using M = PipeMath<D, FP16, NW, NB, L>;
    using TM = TileMath<D, FP16, NB, NW, L>;
    using C = TileCopy<D, NW, L>;
    constexpr int KS = M::KS;
    constexpr int BPW = T::NBLK / NW;  // copies per wave per tile
    static_assert(T::NBLK % NW == 0, "every wave copies the same number of blocks");
    static_assert(SYNC >= 1 && STAGES >= 2 * SYNC + 1 && STAGES <= 5,
                  "a group's tiles, the next K and the next group's copies fit the stages");
    static_assert(L != KV_ODD || SYNC == 1, "KV_ODD sends one tile per group");
    static_assert(PRO >= SYNC + 1 && PRO <= STAGES, "the prologue issues the tiles the first group reads");
    const int job = items[3 * item], row0 = items[3 * item + 1], h = items[3 * item + 2];

    const int lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, g4 = lane >> 4;
    const int kst = p.kstart[job];
    const int ntok = max(0, min(p.klen[job], p.tcap - kst));
    const int kend = kst + ntok;
    const int nrows = p.qlen[job] * p.group;
    if constexpr (odd_count(L))
        if (nrows <= row0) return;  // (a job without requests)
    const int wrow0 = row0 + 16 * NB * wave;
    const bool active = wrow0 < nrows;
    const float c = p.scale_log2, rc = 1.f / p.scale_log2;
    const int tb0 = tile_start<L>(kst);
    const int ntiles = ntok > 0 ? (kend - tb0 + T::TT - 1) / T::TT : 0;
    const int nsteps = ntok > 0 ? (kend - tb0 + 31) / 32 : 0;
    auto tile_stage = [&](int t) { return lds + (t % STAGES) * T::ELEMS; };
    auto stage = [&](int g) { return tile_stage(g >> 1); };  // stage of step g's tile

    // Attached segments (xtail record of this item: count, then (first token,
    // tokens, first job row, rows) for up to TA_XTAIL_MAX segments)
    // follow the job's own tiles in one tile sequence through the same LDS
    // stages.  The record is read at once (constant address space: one batch
    // of scalar loads, no chain of dependent loads) into per-segment values
    // that unrolled loops index with constants.
    constexpr int XM = TA_XTAIL_MAX;
    constexpr int XF = 4;  // fields per segment
    int rec[1 + XF * XM];
    if (p.xtail) {
        const __attribute__((address_space(4))) int32_t *xt =
            (const __attribute__((address_space(4))) int32_t *)(p.xtail + (size_t)item * p.xtail_stride);
#pragma unroll
        for (int i = 0; i < 1 + XF * XM; ++i) rec[i] = xt[i];
    } else {
#pragma unroll
        for (int i = 0; i < 1 + XF * XM; ++i) rec[i] = 0;
    }
    const int nx = min(max(rec[0], 0), XM);
    int xs[XM], xe[XM], xfirst[XM], xn[XM];  // clamped token range, first tile and tiles of each segment
    int ntot = ntiles;
#pragma unroll
    for (int k = 0; k < XM; ++k) {
        xs[k] = max(0, rec[1 + XF * k]);
        xe[k] = xs[k] + max(0, min(rec[2 + XF * k], p.tcap - xs[k]));
        xn[k] = k < nx && xe[k] > xs[k] ? (xe[k] - tile_start<L>(xs[k]) + T::TT - 1) / T::TT : 0;
        xfirst[k] = ntot;
        ntot += xn[k];
    }
    // start the copies of tile t of the sequence into stage st
    auto start_tile = [&](C &kr, int t, u16 *st) {
        if (t < ntiles) {
            kr.issue(st, p, h, tb0 + t * T::TT, kst, kend, wave, lane);
            return;
        }
        int t0n = 0, cs = 0, ce = 1;
#pragma unroll
        for (int k = 0; k < XM; ++k)
            if (t >= xfirst[k] && t < xfirst[k] + xn[k]) {
                t0n = tile_start<L>(xs[k]) + (t - xfirst[k]) * T::TT;
                cs = xs[k];
                ce = xe[k];
            }
        kr.issue(st, p, h, t0n, cs, ce, wave, lane);
    };
    // ... and, for KV_ODD, finish them
    auto copy_tile = [&](int t, u16 *st) {
        C kr;
        start_tile(kr, t, st);
        kr.finish(st, wave, lane);
    };

    int issued = 0;  // tiles of the sequence whose copies this wave has issued

    // Prologue.  Loads retire in order, and a wait for a load's result also
    // waits for every copy issued before it, so the dependent chain
    // (request ids -> Q rows) is kept short.  A job over consecutive requests
    // (qbase[job] >= 0, cf. the reference's contiguous-Q path,
    // kernels.py:23-26) addresses its Q rows from the first request id, a
    // scalar load beside the job's other metadata: the Q loads go out before
    // tile 0's copies.  Otherwise tile 0's copies go out with the request-id
    // loads (both are needed before the first step), then the Q loads.  Every
    // lane loads a valid row (rows past the job are zeroed afterwards); tiles
    // 1 .. PRO-1 follow.
    const int qb = p.qbase ? p.qbase[job] : -1;
    int rq[NB];
    C pro[L == KV_ODD ? PRO : 1];  // (KV_ODD: the first tiles' K, until all are on their way)
    if (qb < 0 && ntot > 0) start_tile(pro[0], 0, lds);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int rr = max(0, min(wrow0 + 16 * nb + row, nrows - 1));
        rq[nb] = qb >= 0 ? qb + rr / p.group : p.qids[(size_t)job * p.maxr + rr / p.group];
    }
    u32x4 qf[NB][KS];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int rr = max(0, min(wrow0 + 16 * nb + row, nrows - 1));
        const u16 *src = p.q + ((size_t)rq[nb] * p.hq + h * p.group + rr % p.group) * D + 8 * g4;
#pragma unroll
        for (int k = 0; k < KS; ++k) qf[nb][k] = *(const u32x4 *)(src + 32 * k);
    }
    if (qb >= 0 && ntot > 0) start_tile(pro[0], 0, lds);  // behind the Q loads: one wait covers both
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const bool valid = wrow0 + 16 * nb + row < nrows;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            if (!valid) qf[nb][k] = u32x4{0, 0, 0, 0};
            asm volatile("" : "+v"(qf[nb][k]));
        }
    }
    if constexpr (L == KV_ODD) {
#pragma unroll
        for (int t = 1; t < PRO; ++t)
            if (t < ntot) start_tile(pro[t], t, tile_stage(t));
#pragma unroll
        for (int t = 0; t < PRO; ++t)
            if (t < ntot) pro[t].finish(tile_stage(t), wave, lane);
    } else {
        for (int t = 1; t < PRO && t < ntot; ++t) copy_tile(t, tile_stage(t));
    }
    issued = min(PRO, ntot);

    M acc;
    acc.reset();
    const LdsOfs of = T::offsets(row, g4);

    wait_tiles<BPW>(issued - 1);  // tile 0 landed (tiles 1 .. PRO-1 may be in flight)
    __builtin_amdgcn_s_barrier();
    if (active && nsteps > 0) {
        f32x4 s0[NB][2];
        TM::load_k(lds, of, 0, acc.kf);
        TM::qk(acc.kf, qf, s0);
        acc.template finish_scores<true>(s0, kst - tb0, kend - tb0, g4);
        acc.first_max(c, rc);
        if (nsteps > 1) TM::load_k(lds, of, 32, acc.kf);
    }

    // Entering tile t (at step 2t): at the start of a group (t % SYNC == 0)
    // tiles t+1 .. t+SYNC must have landed (the earlier ones were waited for
    // at the previous group); the later issued ones may still be in flight.
    // Once every wave passed the barrier the stages of the previous group are
    // free for tiles up to t+STAGES-1.
    // KV_ODD: one tile per group is on its way, its K in registers (odd_k) since
    // the previous group; it goes to LDS before the barrier.
    C odd_k;
    int odd_tile = -1;
    auto sync_tile = [&](int t) {
        if (t % SYNC != 0 || t + 1 >= ntot) return;
        if constexpr (L == KV_ODD) {
            if (odd_tile >= 0) odd_k.finish(tile_stage(odd_tile), wave, lane);
            odd_tile = -1;
            __builtin_amdgcn_s_barrier();
            if (issued < min(t + STAGES, ntot)) {
                odd_tile = issued++;
                start_tile(odd_k, odd_tile, tile_stage(odd_tile));
            }
            return;
        }
        wait_tiles<BPW>(max(0, issued - 1 - (t + SYNC)));
        __builtin_amdgcn_s_barrier();
        for (; issued < min(t + STAGES, ntot); ++issued) copy_tile(issued, tile_stage(issued));
    };
    // steady state: steps whose successor is neither the last nor masked
    int g = 0;
    // ... and, while a whole tile is left to copy per tile attended, that tile's copies
    // spread over the two steps: K's in the slots of the first, V's in those of the second,
    // from a scalar base that the step selects and one lane offset each (8 K rows span
    // 14 tcap bytes, see SHORT_CAP).  All eight waves used to send their four copies at
    // once behind the barrier, with 64-bit lane addresses and the tests for a tile's place
    // in the sequence (128 requests x 8192: kernel 27.6 -> 26.7 us, layer 34.1 -> 33.2 us;
    // every 4th, 8th or 12th slot alike; the branch per tile instead of per loop spilled
    // 590 registers).  Items of fewer than STAGES whole tiles stay with the loop below.
    constexpr int NH = T::KBLK / NW;  // copies of K, and of V, of one wave
    if constexpr (L == KV_POOL && SYNC == 1 && T::KBLK % NW == 0 && NH * NW == T::VBLK) {
        // (readfirstlane: a lane-dependent branch here would move `issued` to vector registers)
        if (__builtin_amdgcn_readfirstlane(active) && p.tcap <= SHORT_CAP && (u32)tb0 + STAGES * T::TT <= (u32)kend) {
            constexpr int EVERY = 4;  // slots from one copy to the next
            static_assert(EVERY * NH <= 2 * KS * NB, "the copies fit the step's QK slots");
            const int w = __builtin_amdgcn_readfirstlane(wave);
            const u32 kofs = C::k_offset(p, w, lane), vofs = C::v_offset(w, lane);
            const u16 *kb = p.kp + (size_t)(h * D + 8 * w) * p.tcap + tb0;
            const u16 *vb = p.vp + ((size_t)h * p.tcap + tb0 + w * T::VROWS) * D;
            for (; issued < STAGES - 1; ++issued) copy_tile(issued, tile_stage(issued));
            for (; tb0 + ((g >> 1) + STAGES) * T::TT <= kend; ++g) {
                const int nt = (g >> 1) + STAGES - 1, odd = g & 1;  // nt: tile copied, inside the job
                if (!odd) {
                    wait_tiles<BPW>(STAGES - 3);  // tile (g >> 1) + 1 landed
                    __builtin_amdgcn_s_barrier();
                    ++issued;
                }
                const u16 *src = odd ? vb + (size_t)nt * (T::TT * D) : kb + nt * T::TT;
                const size_t next = odd ? (size_t)NW * T::VROWS * D : (size_t)8 * NW * p.tcap;
                const u32 ofs = odd ? vofs : kofs;
                u16 *dst = tile_stage(nt) + (odd ? T::KBLK + w : w) * T::BLK;
                acc.template block<true, false, false>(
                    stage(g), 32 * odd, stage(g + 2), 32 * odd, qf, of, 0, 32, g4, c, ~0u, [&](int slot) {
                        const int n = slot / EVERY;
                        if (slot % EVERY == EVERY / 2 && n < NH) C::dma(dst + n * NW * T::BLK, src + n * next, ofs);
                    });
                acc.rescale(c, rc);
            }
        }
    }
    for (; g + 2 < nsteps; ++g) {
        if (!(g & 1)) sync_tile(g >> 1);
        if (active) {
            const int gk = g + 2;
            acc.template block<true, false>(stage(g), 32 * (g & 1), stage(gk), 32 * (gk & 1), qf, of, 0, 32,
                                            g4, c);
            acc.rescale(c, rc);
        }
    }
    // the last two steps: the successor of step nsteps-2 may be masked at its end
    if (g + 1 < nsteps) {
        if (!(g & 1)) sync_tile(g >> 1);
        if (active) {  // one (masked) form for either end of the job keeps the register allocation simple
            acc.template block<true, true>(stage(g), 32 * (g & 1), stage(g + 1), 32 * ((g + 1) & 1), qf, of,
                                           0, kend - (tb0 + 32 * (g + 1)), g4, c);
            acc.rescale(c, rc);
        }
        ++g;
    }
    if (g < nsteps) {
        if (!(g & 1)) sync_tile(g >> 1);
        if (active)
            acc.template block<false, false>(stage(g), 32 * (g & 1), stage(g), 0, qf, of, 0, kend - (tb0 + 32 * g), g4,
                                             c);
    }

    // Attached segments, in rounds of up to STAGES tiles that are resident
    // together: one wait and one barrier per round, then every wave attends
    // the round's tiles of the segments holding its rows, side by side.  The
    // root loop (or the prologue) already issued the first tiles.
    if constexpr (!odd_count(L)) {  // (the launcher passes no attachments for the others)
        for (int r0 = ntiles; r0 < ntot; r0 += STAGES) {
            const int r1 = min(r0 + STAGES, ntot);
            __builtin_amdgcn_s_barrier();  // every wave is done with the tiles before r0
            for (; issued < r1; ++issued) copy_tile(issued, tile_stage(issued));
            __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
            __builtin_amdgcn_s_barrier();  // the round's tiles landed
#pragma unroll
            for (int k = 0; k < XM; ++k) {
                // segment rows relative to this wave's: [rlo, rlo + rows); with 16 rows per
                // wave (NB = 1) a segment may span two waves, each attends its own rows
                const int rlo = rec[3 + XF * k] - wrow0;
                if (xn[k] > 0 && active && rlo < 16 * NB && rlo + rec[4 + XF * k] > 0) {
                    for (int i = max(0, r0 - xfirst[k]); i < xn[k] && xfirst[k] + i < r1; ++i) {
                        const int t0 = tile_start<L>(xs[k]) + i * T::TT;
                        acc.tail_tile(tile_stage(xfirst[k] + i), qf, of, max(0, xs[k] - t0), min(T::TT, xe[k] - t0),
                                      rlo, rlo + rec[4 + XF * k], row, g4, c, rc);
                    }
                }
            }
        }
    }

    if (!active) return;
    const int rb = p.rowbase[job];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int grow = wrow0 + 16 * nb + row;
        const float z = acc.z[nb].total();
        if (grow >= nrows) continue;
        const int lr = grow / p.group, gg = grow - lr * p.group;
        const size_t prow = (size_t)(rb + lr) * p.hq + h * p.group + gg;
        store_partial<M::DB>(p.part, p.lse, prow, acc.o[nb], acc.m[nb], z, g4);
    }
}

// A 256-row work item whose job has at most 8 NW rows from the item's first
// row on runs 16 rows per wave, so that every wave computes (two per SIMD)
// instead of half of them 32 rows each; the arithmetic of every row is the same.
template <int D, bool FP16, int NW, int L>
__device__ __forceinline__ void pipe_item_rows(const SegParams &p, const int32_t *__restrict__ items, int item,
                                               u16 *lds, int tid) {
    const int job = items[3 * item], row0 = items[3 * item + 1];
    if (p.qlen[job] * p.group - row0 <= 16 * NW)
        pipe_item<D, FP16, NW, 1, L>(p, items, item, lds, tid);
    else
        pipe_item<D, FP16, NW, 2, L>(p, items, item, lds, tid);
}

template <int D, bool FP16, int NW, int L>
__global__ __launch_bounds__(64 * NW) void seg_pipe_kernel(const int32_t *items, SegParams p) {
    __shared__ __attribute__((aligned(16))) u16 lds[TA_PIPE_STAGES * Tile<D>::ELEMS];
    pipe_item_rows<D, FP16, NW, L>(p, items, xcd_item(blockIdx.x, gridDim.x), lds, threadIdx.x);
}

// Work items of several kinds of one layer in one launch of 512-thread
// workgroups: blocks [0, base[1]) run 256-row items (with their attached
// segments), blocks [base[1], base[2]) run 64-row items on eight waves (the
// upper four copy and meet at the barriers), and the blocks from base[2] on
// run four small items each, one per wave on its own stage (the upper four
// waves end at once).  The bases are multiples of 8, so that the row tiles map
// to XCDs as in their own kernels; blocks past a kind's item count end
// at once.  The kinds run side by side instead of one launch after another.
template <int D, bool FP16, int L>
__global__ __launch_bounds__(512) void seg_mix_kernel(const int32_t *items0, const int32_t *items1, const int32_t *items2,
                                                      MixParams mp) {
    using T = Tile<D>;
    __shared__ __attribute__((aligned(16))) u16 lds[TA_PIPE_STAGES * T::ELEMS];
    static_assert(TA_PIPE_STAGES >= 4 && 3 <= TA_PIPE_STAGES, "four small stages and three 64-row stages fit");
    const int b = blockIdx.x, tid = threadIdx.x;
    if (b < mp.base[1]) {
        if (b >= mp.n[0]) return;
        pipe_item_rows<D, FP16, 8, L>(mp.p, items0, xcd_item(b, mp.n[0]), lds, tid);
    } else if (b < mp.base[2]) {
        const int lb = b - mp.base[1];
        if (lb >= mp.n[1]) return;
        tile_item<D, FP16, 1, 8, 3, L>(mp.p, items1, xcd_item(lb, mp.n[1]), lds, tid, 64);
    } else {
        const int lb = b - mp.base[2], wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int it = mp.by_head ? 8 * (4 * (lb >> 3) + wave) + (lb & 7) : 4 * lb + wave;
        if (wave >= 4 || it >= mp.n[2]) return;
        tile_item<D, FP16, 1, 1, 1, L, true>(mp.p, items2, it, lds + wave * T::ELEMS, tid & 63, 16);
    }
}

// ------------------------------------------------------------------------
// Tail kernel with the merge fused in (TA_TAIL items with out given).  One
// two-wave workgroup per (tail job, KV head): the job's single request has
// G = hq/hk query rows for this head, and every other partial slot of the
// request was written by an earlier launch on the stream (the job's own slot
// is the request's last).  The two waves work side by side:
//   wave 0 attends the tail (the small-job tile loop) and leaves its
//          normalised partial and log-sum-exp in LDS;
//   wave 1 loads the other slots, PF float4 registers per round, and merges
//          them by the online log-sum-exp of the merge kernel; lane l owns
//          units u = l + 64k (k < UPL) of the G*D/4 float4 units, unit u =
//          (row u / (D/4), d = 4 (u % (D/4))).
// After one barrier wave 1 merges the own partial and writes the output rows.
template <int D, bool FP16, int UPL, int L>
__global__ __launch_bounds__(128) void seg_tail_kernel(SegParams p) {
    using T = Tile<D>;
    using M = TileMath<D, FP16, 1, 1, L>;
    using C = TileCopy<D, 1, L>;
    constexpr int KS = M::KS, DB = M::DB;
    constexpr int PF = 32;          // units of one merge round
    constexpr int CH = PF / UPL;    // slots per merge round
    constexpr int DU = D / 4;       // units per row
    constexpr float LOG2E = 1.44269504088896341f;
    __shared__ __attribute__((aligned(16))) u16 lds[T::ELEMS];
    float *opart = reinterpret_cast<float *>(lds);  // [G][D] own normalised partial, after the tile loop
    float *olse = opart + 16 * D;                   // [G] own log-sum-exp, log2 units

    const int item = blockIdx.x;
    const int job = p.items[3 * item], h = p.items[3 * item + 2];
    const int G = p.group;
    const int lane = threadIdx.x & 63;
    const int r = p.qids[(size_t)job * p.maxr];

    if (threadIdx.x < 64) {
        // ---- wave 0: the tail's attention
        const int row = lane & 15, g4 = lane >> 4;
        const int kst = p.kstart[job];
        const int ntok = max(0, min(p.klen[job], p.tcap - kst));
        const int kend = kst + ntok;
        const int tb0 = tile_start<L>(kst);
        const int ntiles = ntok > 0 ? (kend - tb0 + T::TT - 1) / T::TT : 0;
        C kr;
        if (ntiles > 0) kr.issue(lds, p, h, tb0, kst, kend, 0, lane);
        u32x4 qf[1][KS];
        {
            const int rr = row < G ? row : 0;  // rows past G repeat row 0 and are never stored
            const u16 *src = p.q + ((size_t)r * p.hq + h * G + rr) * D + 8 * g4;
#pragma unroll
            for (int k = 0; k < KS; ++k) qf[0][k] = *(const u32x4 *)(src + 32 * k);
        }
        M acc;
        acc.reset();
        const LdsOfs of = T::offsets(row, g4);
        for (int it = 0; it < ntiles; ++it) {
            const int t0 = tb0 + it * T::TT;
            if (it > 0) kr.issue(lds, p, h, t0, kst, kend, 0, lane);
            __builtin_amdgcn_s_waitcnt(TA_VMCNT(0));
            kr.finish(lds, 0, lane);
            acc.tile(lds, qf, of, max(0, kst - t0), min(T::TT, kend - t0), g4, p.scale_log2);
        }
        // the tile's reads fed the MFMAs above, so the stage is free for the partial
        const bool any = acc.m[0] != NEG_INF;
        const float zr = acc.z[0].total();
        const float inv = any ? 1.f / zr : 0.f;
        if (row < G) {
#pragma unroll
            for (int db = 0; db < DB; ++db)
                *(f32x4 *)(opart + row * D + 16 * db + 4 * g4) = acc.o[0][db] * inv;
            if (g4 == 0) olse[row] = any ? acc.m[0] + __builtin_amdgcn_logf(zr) : NEG_INF;
        }
        __syncthreads();
        return;
    }

    // ---- wave 1: merge the request's other slots
    const int own = p.rowbase[job];
    const int cnt = p.counts[r] - 1;
    const int32_t *slr = p.slots + (size_t)r * p.maxs;
    const int units = G * DU;
    float Mx[UPL], Z[UPL];
    f32x4 o[UPL];
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
        Mx[k] = NEG_INF;
        Z[k] = 0.f;
        o[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int s0 = 0; s0 < cnt; s0 += CH) {
        float l[CH][UPL];
        int e[CH][UPL];
        u32x2 v[CH][UPL];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int si = s0 + c;
            const int sl = slr[min(si, cnt - 1)];
            const bool use = si < cnt && sl != own;
#pragma unroll
            for (int k = 0; k < UPL; ++k) {
                const int u = min(lane + 64 * k, units - 1);
                const size_t prow = (size_t)sl * p.hq + h * G + u / DU;
                const u32x2 x = *(const u32x2 *)(p.part + prow * D + part_pos(u % DU));
                const float lx = p.lse[2 * prow], ex = p.lse[2 * prow + 1];
                l[c][k] = use ? lx * LOG2E : NEG_INF;
                e[c][k] = (int)ex;
                v[c][k] = use ? x : u32x2{0u, 0u};
            }
        }
#pragma unroll
        for (int k = 0; k < UPL; ++k) {
            float cm = Mx[k];
#pragma unroll
            for (int c = 0; c < CH; ++c) cm = fmaxf(cm, l[c][k]);
            const float alpha = Mx[k] == NEG_INF ? 0.f : fast_exp2(Mx[k] - cm);
            Z[k] *= alpha;
            o[k] *= alpha;
            Mx[k] = cm;
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const float w = l[c][k] == NEG_INF ? 0.f : fast_exp2(l[c][k] - cm);
                Z[k] += w;
                o[k] += __builtin_amdgcn_ldexpf(w, e[c][k]) * unpack_f16x4(v[c][k]);
            }
        }
    }
    __syncthreads();  // wave 0's partial is in LDS
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
        const int u = lane + 64 * k;
        if (u >= units) continue;
        const float lo = olse[u / DU];
        const f32x4 vo = *(const f32x4 *)(opart + (u / DU) * D + 4 * (u % DU));
        const float cm = fmaxf(Mx[k], lo);
        const float alpha = Mx[k] == NEG_INF ? 0.f : fast_exp2(Mx[k] - cm);
        const float w = lo == NEG_INF ? 0.f : fast_exp2(lo - cm);
        const float zt = Z[k] * alpha + w;
        const f32x4 a = (o[k] * alpha + w * vo) * (zt > 0.f ? 1.f / zt : 0.f);
        u16 *dst = p.out + ((size_t)r * p.hq + h * G + u / DU) * D + 4 * (u % DU);
        *(u32x2 *)dst = u32x2{Ops<FP16>::pack(a[0], a[1]), Ops<FP16>::pack(a[2], a[3])};
    }
}

template <int D, bool FP16, int L>
hipError_t launch_tail_merge(const SegParams &sp, hipStream_t stream) {
    // float4 units per lane: G*D/4 units over 64 lanes
    const int units = sp.group * (D / 4);
    if (units <= 64)
        TA_LAUNCH((seg_tail_kernel<D, FP16, 1, L>), dim3(sp.n_items), dim3(128), stream, sp);
    else if (units <= 128)
        TA_LAUNCH((seg_tail_kernel<D, FP16, 2, L>), dim3(sp.n_items), dim3(128), stream, sp);
    else if (units <= 256)
        TA_LAUNCH((seg_tail_kernel<D, FP16, 4, L>), dim3(sp.n_items), dim3(128), stream, sp);
    else if (units <= 512)
        TA_LAUNCH((seg_tail_kernel<D, FP16, 8, L>), dim3(sp.n_items), dim3(128), stream, sp);
    else
        return hipErrorNotSupported;
    return hipGetLastError();
}

// Whether the 32-bit lane offsets of TileCopy's short form cover a tile: 8 K rows of a pool span
// 14 tcap bytes; the 64 rows of token-major K and V 128 D hk, whatever their number.
template <int D, int L>
bool short_offsets(const SegParams &p) {
    return token_major(L) ? p.hk < (1 << 25) / D : L == KV_POOL && p.tcap <= SHORT_CAP;
}

template <int D, bool FP16, int L>
hipError_t launch_d(const SegParams &sp, int kind, hipStream_t stream) {
    switch (kind) {
        case TA_TAIL:  // as TA_SMALL, merging the request into out when out is given
            if (sp.out) {
                if constexpr (odd_count(L))
                    return (hipError_t)TA_ERR_ARG;
                else
                    return launch_tail_merge<D, FP16, L>(sp, stream);
            }
            [[fallthrough]];
        case TA_SMALL:  // one wave per (job, head); one stage so that five fit on a CU
            if (short_offsets<D, L>(sp))
                TA_LAUNCH((seg_tile_kernel<D, FP16, 1, 1, 1, L, L != KV_ODD>), dim3(sp.n_items), dim3(64), stream,
                          sp.items, sp);
            else
                TA_LAUNCH((seg_tile_kernel<D, FP16, 1, 1, 1, L>), dim3(sp.n_items), dim3(64), stream, sp.items, sp);
            break;
        case TA_LARGE64:
            TA_LAUNCH((seg_tile_kernel<D, FP16, 1, 4, 3, L>), dim3(sp.n_items), dim3(256), stream, sp.items, sp);
            break;
        case TA_LARGE128:
            TA_LAUNCH((seg_tile_kernel<D, FP16, 2, 4, 3, L>), dim3(sp.n_items), dim3(256), stream, sp.items, sp);
            break;
        case TA_LARGE256:
            TA_LAUNCH((seg_pipe_kernel<D, FP16, 8, L>), dim3(sp.n_items), dim3(512), stream, sp.items, sp);
            break;
        default:
            return (hipError_t)TA_ERR_ARG;
    }
    return hipGetLastError();
}

template <int D, bool FP16, int L>
hipError_t launch_mix_d(const MixParams &mp, int blocks, hipStream_t stream) {
    TA_LAUNCH((seg_mix_kernel<D, FP16, L>), dim3(blocks), dim3(512), stream, mp.items[0], mp.items[1], mp.items[2], mp);
    return hipGetLastError();
}

#define TA_BY_SHAPE(FN, L, ...)                                                               \
    switch (d) {                                                                              \
        case 128: return fp16 ? FN<128, true, L>(__VA_ARGS__) : FN<128, false, L>(__VA_ARGS__); \
        case 64: return fp16 ? FN<64, true, L>(__VA_ARGS__) : FN<64, false, L>(__VA_ARGS__);  \
        case 32: return fp16 ? FN<32, true, L>(__VA_ARGS__) : FN<32, false, L>(__VA_ARGS__);  \
        default: return hipErrorNotSupported;                                                 \
    }

}  // namespace

template <>
hipError_t launch_mix<TA_LAYOUT>(const SegParams &sp, const int32_t *const items[3], const int n[3], int d, bool fp16,
                                 hipStream_t stream) {
    MixParams mp;
    mp.p = sp;
    int base = 0;
    for (int k = 0; k < 3; ++k) {
        mp.items[k] = items[k];
        mp.n[k] = n[k] > 0 ? n[k] : 0;
        mp.base[k] = base;
        base += (mp.n[k] + 7) & ~7;  // (the last kind's is not needed)
    }
    mp.by_head = mix_by_head(sp, mp.n, d);
    const int small_blocks = mp.by_head ? (mp.n[2] + 31) / 32 * 8 : (mp.n[2] + 3) / 4;
    const int blocks = mp.base[2] + small_blocks;
    if (blocks <= 0) return hipSuccess;
    TA_BY_SHAPE(launch_mix_d, TA_LAYOUT, mp, blocks, stream)
}

template <>
hipError_t launch_kind<TA_LAYOUT>(const SegParams &sp, int kind, int d, bool fp16, hipStream_t stream) {
    TA_BY_SHAPE(launch_d, TA_LAYOUT, sp, kind, stream)
}

}  // namespace ta
