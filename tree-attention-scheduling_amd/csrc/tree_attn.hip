// tree_attn.hip -- gfx950 (CDNA4) kernels for tree-shared decode attention.
//
// Replaces the Triton kernels of the reference's src/tree_attention/kernels.py:
//   _segment (kernels.py:8-55): grouped partial attention of one physical KV
//     segment for every request of its job, online softmax in fp32, P rounded
//     to the input dtype before PV (kernels.py:49), writes acc/z and m + ln z.
//   _merge (kernels.py:58-83): per (request, query head) log-sum-exp merge of
//     the request's partial outputs, cast to the input dtype.
//
// This file holds the merge kernel, the read-ceiling stream and the C entry points; the
// segment kernels are in segment_tile.hip.
//   * Partial rows are stored as fp16 scaled by a power of two per row (the
//     exponent sits next to the log-sum-exp); the merge reads them with
//     16-byte loads, one thread per eight head-dim elements, and folds the
//     scale into each slot's weight.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "ta_common.h"
#include "tree_attn.h"

namespace {

using namespace ta;

// ------------------------------------------------------------------ merge
// One workgroup of NT threads per (request, group of MH query heads);
// thread (head, d8) owns eight head-dim elements of one query head.  The slot
// list is uniform per workgroup (scalar loads), and each thread reads, for
// MERGE_CHUNK slots at once, the 16-byte partial slice (eight fp16 values) and
// the 8-byte (log-sum-exp, exponent) pair, then merges them online in
// registers: slots -> (lse, partials) is the only chain of dependent memory
// round trips; no LDS and no barriers.  With an affine slot layout
// (slot_stride > 0: slot k of request r is r + k * slot_stride, maxs of them)
// the slots are computed and the partial loads are the first memory access.
constexpr int MERGE_CHUNK = 16;
constexpr int MERGE_NT = 128;
// Below this many workgroups of MERGE_NT threads the merge runs groups of
// MERGE_NT / 2 threads instead (half the heads per workgroup, twice the
// workgroups): one workgroup per CU of the 256 leaves the GPU half empty, and
// a small batch's merge is one round trip of loads per workgroup.
constexpr int MERGE_FILL_BLOCKS = 256;

// SPLIT groups of NT threads split a request's slots into SPLIT
// contiguous ranges, merge them side by side (one round trip of loads per
// MERGE_CHUNK slots each) and combine their running (max, sum, partial sums)
// through LDS; the first group writes the output.  SPLIT = 2 serves plans with
// more than MERGE_CHUNK slots per request: 32 slots wait for one round of loads
// instead of two.  SPLIT = 1 is the single-group kernel described above.
template <int D, bool FP16, int SPLIT, int NT = MERGE_NT>
__global__ __launch_bounds__(NT * SPLIT) void merge_kernel(const u16 *__restrict__ part,
                                                                 const float *__restrict__ lse,
                                                                 const int32_t *__restrict__ slots,
                                                                 const int32_t *__restrict__ counts,
                                                                 const int32_t *__restrict__ reqs,
                                                                 u16 *__restrict__ out, int hq, int maxs,
                                                                 int slot_stride) {
    constexpr int TPH = D / 8;          // threads per head
    constexpr int MH = NT / TPH;  // heads per workgroup
    constexpr float LOG2E = 1.44269504088896341f;
    const int r = reqs ? reqs[blockIdx.x] : blockIdx.x;
    // a group is whole waves: readfirstlane tells the compiler grp is uniform
    const int grp = SPLIT > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
    const int tid = threadIdx.x % NT;
    const int hl = tid / TPH, d8 = tid % TPH;
    const int head = blockIdx.y * MH + hl;
    const bool valid = head < hq;
    if (SPLIT == 1 && !valid) return;
    const int cnt = slot_stride > 0 ? maxs : counts[r];
    const int per = (cnt + SPLIT - 1) / SPLIT;
    const int beg = SPLIT > 1 ? min(cnt, grp * per) : 0, end = SPLIT > 1 ? min(cnt, beg + per) : cnt;
    const int hr = SPLIT > 1 ? min(head, hq - 1) : head;  // the head this lane reads
    const int32_t *slr = slots + (size_t)r * maxs;
    const u16 *src = part + (size_t)hr * D + 8 * d8;
    const float2 *lse2 = reinterpret_cast<const float2 *>(lse) + hr;
    const size_t srow = (size_t)hq * D;

    float M = NEG_INF, Z = 0.f;  // running max (log2 units) and weight sum
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    // the loop bounds stay uniform (so the slot list is read by scalar loads):
    // lanes past hq read head hq - 1 and store nothing
    for (int s0 = beg; s0 < end; s0 += MERGE_CHUNK) {
        float2 le[MERGE_CHUNK];
        u32x4 v[MERGE_CHUNK];
#pragma unroll
        for (int u = 0; u < MERGE_CHUNK; ++u) {
            const int k = min(s0 + u, end - 1);
            const int sl = slot_stride > 0 ? r + k * slot_stride : slr[k];
            // nontemporal: the partials are read once, and leaving them out of L2
            // keeps the next segment launch's metadata, Q and code there
            const f32x2 t = __builtin_nontemporal_load((const f32x2 *)(lse2 + (size_t)sl * hq));
            le[u] = float2(t[0], t[1]);
            v[u] = __builtin_nontemporal_load((const u32x4 *)(src + sl * srow));
        }
        float l[MERGE_CHUNK];
        float cm = M;
#pragma unroll
        for (int u = 0; u < MERGE_CHUNK; ++u) {
            l[u] = s0 + u < end ? le[u].x * LOG2E : NEG_INF;
            cm = fmaxf(cm, l[u]);
        }
        if (cm == NEG_INF) continue;  // every slot so far is empty
        if (cm > M) {
            const float alpha = fast_exp2(M - cm);  // 0 while M is -inf
            Z *= alpha;
            lo *= alpha;
            hi *= alpha;
            M = cm;
        }
#pragma unroll
        for (int u = 0; u < MERGE_CHUNK; ++u) {
            const float w = fast_exp2(l[u] - M);  // 0 for empty slots
            Z += w;
            const float ws = __builtin_amdgcn_ldexpf(w, (int)le[u].y);
            lo += ws * unpack_f16x4(u32x2{v[u][0], v[u][1]});
            hi += ws * unpack_f16x4(u32x2{v[u][2], v[u][3]});
        }
    }
    if constexpr (SPLIT > 1) {
        __shared__ float sh[SPLIT - 1][10][NT];
        if (grp > 0) {
            float *x = &sh[grp - 1][0][tid];
            x[0] = M;
            x[NT] = Z;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[(2 + i) * NT] = lo[i];
                x[(6 + i) * NT] = hi[i];
            }
        }
        __syncthreads();
        if (grp > 0 || !valid) return;
#pragma unroll
        for (int g = 0; g < SPLIT - 1; ++g) {
            const float *x = &sh[g][0][tid];
            const float Mg = x[0];
            if (Mg == NEG_INF) continue;  // an empty range
            const float cm = fmaxf(M, Mg);
            const float alpha = fast_exp2(M - cm), beta = fast_exp2(Mg - cm);  // alpha is 0 while M is -inf
            Z = Z * alpha + x[NT] * beta;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo[i] = lo[i] * alpha + x[(2 + i) * NT] * beta;
                hi[i] = hi[i] * alpha + x[(6 + i) * NT] * beta;
            }
            M = cm;
        }
    }
    if (Z > 0.f) {
        const float inv = 1.f / Z;
        lo *= inv;
        hi *= inv;
    }
    // the slice holds d = 32 (d8 / 4) + 4 (d8 % 4) + {0..3} (lo) and the same + 16 (hi)
    u16 *dst = out + ((size_t)r * hq + head) * D + 32 * (d8 >> 2) + 4 * (d8 & 3);
    *(u32x2 *)dst = u32x2{Ops<FP16>::pack(lo[0], lo[1]), Ops<FP16>::pack(lo[2], lo[3])};
    *(u32x2 *)(dst + 16) = u32x2{Ops<FP16>::pack(hi[0], hi[1]), Ops<FP16>::pack(hi[2], hi[3])};
}

// ------------------------------------------------------------------ read ceiling
// A read-only stream: every lane loads 16-byte chunks in a grid-stride loop
// and folds them into one word per wave, the ceiling against which the
// memory-bound segment kernels are measured (ta_read_stream).
constexpr int READ_NT = 256;

__global__ __launch_bounds__(READ_NT) void read_stream_kernel(const u32x4 *__restrict__ src, int64_t n,
                                                              uint32_t *__restrict__ sink) {
    u32x4 acc = {0u, 0u, 0u, 0u};
    const int64_t step = (int64_t)gridDim.x * READ_NT;
    int64_t i = (int64_t)blockIdx.x * READ_NT + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {
        const u32x4 a = src[i], b = src[i + step], c = src[i + 2 * step], d = src[i + 3 * step];
        acc ^= a ^ b ^ c ^ d;
    }
    for (; i < n; i += step) acc ^= src[i];
    uint32_t w = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
    for (int o = 32; o > 0; o >>= 1) w ^= __shfl_xor(w, o);
    if ((threadIdx.x & 63) == 0) sink[blockIdx.x * (READ_NT / 64) + threadIdx.x / 64] = w;
}

// ------------------------------------------------------------------ launch
// The layout of pools, and of token-major K and V, of `tcap` tokens.
int pool_layout(int32_t tcap) { return tcap % 8 == 0 ? KV_POOL : KV_ODD; }
int token_layout(int32_t tcap) { return tcap % 8 == 0 ? KV_TOKEN : KV_TOKEN_ODD; }

// nreq requests: reqs[0 .. nreq) when reqs is given, else 0 .. nreq-1
template <int D, bool FP16>
hipError_t launch_merge(const void *part, const float *lse, const int32_t *slots, const int32_t *counts,
                        const int32_t *reqs, void *out, int nreq, int hq, int maxs, hipStream_t stream,
                        int slot_stride = 0) {
    constexpr int MH = MERGE_NT / (D / 8), MH2 = MH / 2;
    const bool fill = (long)nreq * ((hq + MH - 1) / MH) < MERGE_FILL_BLOCKS;
    const dim3 grid(nreq, fill ? (hq + MH2 - 1) / MH2 : (hq + MH - 1) / MH);
    const u16 *p16 = static_cast<const u16 *>(part);
    u16 *o16 = static_cast<u16 *>(out);
    if (maxs > MERGE_CHUNK) {
        if (fill)
            TA_LAUNCH((merge_kernel<D, FP16, 2, MERGE_NT / 2>), grid, dim3(MERGE_NT), stream, p16, lse, slots,
                      counts, reqs, o16, hq, maxs, slot_stride);
        else
            TA_LAUNCH((merge_kernel<D, FP16, 2>), grid, dim3(2 * MERGE_NT), stream, p16, lse, slots, counts, reqs,
                      o16, hq, maxs, slot_stride);
    } else {
        if (fill)
            TA_LAUNCH((merge_kernel<D, FP16, 1, MERGE_NT / 2>), grid, dim3(MERGE_NT / 2), stream, p16, lse, slots,
                      counts, reqs, o16, hq, maxs, slot_stride);
        else
            TA_LAUNCH((merge_kernel<D, FP16, 1>), grid, dim3(MERGE_NT), stream, p16, lse, slots, counts, reqs, o16,
                      hq, maxs, slot_stride);
    }
    return hipGetLastError();
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check_common(int hq, int hk, int d, int dtype) {
    if (dtype != TA_BF16 && dtype != TA_FP16) return TA_ERR_DTYPE;
    if (hq <= 0 || hk <= 0 || hq % hk != 0) return TA_ERR_ARG;
    if (d != 32 && d != 64 && d != 128) return TA_ERR_ARG;
    return 0;
}

#define TA_DISPATCH(d, fp16, CALL)                                         \
    ((d) == 128 ? ((fp16) ? CALL(128, true) : CALL(128, false))           \
     : (d) == 64 ? ((fp16) ? CALL(64, true) : CALL(64, false))            \
                 : ((fp16) ? CALL(32, true) : CALL(32, false)))

}  // namespace

namespace ta {
thread_local LaunchEvents g_launch_events = {nullptr, nullptr};
}  // namespace ta

extern "C" {

const char *ta_version(void) { return "tree_attn gfx950 1.0"; }

const char *ta_error_string(int code) {
    switch (code) {
        case 0: return "success";
        case TA_ERR_ARG: return "tree_attn: invalid argument (null pointer, size or unsupported shape)";
        case TA_ERR_ALIGN: return "tree_attn: q/kp/vp/part/out must be 16-byte aligned, lse 8-byte aligned";
        case TA_ERR_DTYPE: return "tree_attn: dtype must be TA_BF16 or TA_FP16";
        case TA_ERR_SCRATCH:
            return "tree_attn: the plan's partials exceed TA_NOALLOC_SCRATCH_BYTES (use ta_attention_matrix)";
        default: return hipGetErrorString((hipError_t)code);
    }
}

}  // extern "C"

namespace {

void fill_params(SegParams &sp, const void *q, const void *kp, const void *vp, const int32_t *qids,
                 const int32_t *kstart, const int32_t *qlen, const int32_t *klen, const int32_t *rowbase,
                 const int32_t *items, int32_t n_items, void *part, float *lse, int32_t hq, int32_t hk, int32_t d,
                 int32_t tcap, int32_t maxr, const int32_t *slots, const int32_t *counts, void *out, int32_t maxs,
                 const int32_t *xtail, int32_t xtail_stride, const int32_t *qbase);

// One segment launch; with out given (TA_TAIL only) the items merge their
// requests into out.
int segment_launch(const void *q, const void *kp, const void *vp, const int32_t *qids, const int32_t *kstart,
                   const int32_t *qlen, const int32_t *klen, const int32_t *rowbase, const int32_t *items,
                   int32_t n_items, int32_t kind, void *part, float *lse, int32_t nreq, int32_t hq, int32_t hk,
                   int32_t d, int32_t tcap, int32_t maxr, int32_t dtype, const int32_t *slots,
                   const int32_t *counts, void *out, int32_t maxs, const int32_t *xtail, int32_t xtail_stride,
                   const int32_t *qbase, int layout, void *stream) {
    if (int e = check_common(hq, hk, d, dtype)) return e;
    if (n_items < 0 || nreq <= 0 || tcap <= 0 || maxr <= 0 || kind < TA_SMALL || kind > TA_TAIL) return TA_ERR_ARG;
    if (n_items == 0) return 0;
    if (!q || !kp || !vp || !qids || !kstart || !qlen || !klen || !rowbase || !items || !part || !lse)
        return TA_ERR_ARG;
    if (!aligned16(q) || !aligned16(kp) || !aligned16(vp) || !aligned16(part)) return TA_ERR_ALIGN;
    if (out) {
        if (kind != TA_TAIL || odd_count(layout) || !slots || !counts || maxs <= 0) return TA_ERR_ARG;
        if (!aligned16(out)) return TA_ERR_ALIGN;
    }
    if (xtail && (kind != TA_LARGE256 || odd_count(layout) || xtail_stride != TA_XTAIL_STRIDE)) return TA_ERR_ARG;
    SegParams sp;
    fill_params(sp, q, kp, vp, qids, kstart, qlen, klen, rowbase, items, n_items, part, lse, hq, hk, d, tcap, maxr,
                slots, counts, out, maxs, xtail, xtail_stride, qbase);
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const bool fp16 = dtype == TA_FP16;
    return (int)(layout == KV_POOL    ? ta::launch_kind<KV_POOL>(sp, kind, d, fp16, st)
                 : layout == KV_ODD   ? ta::launch_kind<KV_ODD>(sp, kind, d, fp16, st)
                 : layout == KV_TOKEN ? ta::launch_kind<KV_TOKEN>(sp, kind, d, fp16, st)
                                      : ta::launch_kind<KV_TOKEN_ODD>(sp, kind, d, fp16, st));
}

// The launch arguments every segment kernel shares.
void fill_params(SegParams &sp, const void *q, const void *kp, const void *vp, const int32_t *qids,
                 const int32_t *kstart, const int32_t *qlen, const int32_t *klen, const int32_t *rowbase,
                 const int32_t *items, int32_t n_items, void *part, float *lse, int32_t hq, int32_t hk, int32_t d,
                 int32_t tcap, int32_t maxr, const int32_t *slots, const int32_t *counts, void *out, int32_t maxs,
                 const int32_t *xtail, int32_t xtail_stride, const int32_t *qbase) {
    sp.q = static_cast<const u16 *>(q);
    sp.kp = static_cast<const u16 *>(kp);
    sp.vp = static_cast<const u16 *>(vp);
    sp.qids = qids;
    sp.kstart = kstart;
    sp.qlen = qlen;
    sp.klen = klen;
    sp.rowbase = rowbase;
    sp.items = items;
    sp.part = static_cast<u16 *>(part);
    sp.lse = lse;
    sp.n_items = n_items;
    sp.hq = hq;
    sp.hk = hk;
    sp.group = hq / hk;
    sp.tcap = tcap;
    sp.maxr = maxr;
    sp.scale_log2 = (float)(1.4426950408889634 / __builtin_sqrt((double)d));
    sp.slots = slots;
    sp.counts = counts;
    sp.out = static_cast<u16 *>(out);
    sp.maxs = maxs;
    sp.xtail = xtail;
    sp.xtail_stride = xtail_stride;
    sp.qbase = qbase;
}

int plan_segment(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan, int kind,
                 void *out, int layout, void *stream) {
    const bool xt = kind == TA_LARGE256 && plan->xtail;
    return segment_launch(q, kp, vp, plan->qids, plan->kstart, plan->qlen, plan->klen, plan->rowbase,
                          plan->items[kind], plan->n_items[kind], kind, plan->part, plan->lse, plan->nreq, plan->hq,
                          plan->hk, plan->d, tcap, plan->maxr, plan->dtype, plan->slots, plan->counts, out,
                          plan->maxs, xt ? plan->xtail : nullptr, xt ? plan->xtail_stride : 0, plan->qbase, layout,
                          stream);
}

// The merge of requests reqs[0 .. n) (reqs == NULL: 0 .. n-1) of a prepared
// plan into out, with the plan's affine slot layout when it has one.
int plan_merge(const ta_plan *plan, const int32_t *reqs, int32_t n, void *out, void *stream) {
    if (!plan->part || !plan->lse || !plan->slots || !plan->counts || n <= 0 || n > plan->nreq) return TA_ERR_ARG;
    if (plan->dtype != TA_BF16 && plan->dtype != TA_FP16) return TA_ERR_DTYPE;
    if (plan->maxs <= 0 || plan->hq <= 0 || (plan->d != 32 && plan->d != 64 && plan->d != 128)) return TA_ERR_ARG;
    if (!aligned16(plan->part) || !aligned16(out) || (reinterpret_cast<uintptr_t>(plan->lse) & 7)) return TA_ERR_ALIGN;
    // an affine slot layout must stay inside the partial slots
    if (plan->slot_stride < 0 ||
        (plan->slot_stride > 0 &&
         (int64_t)(plan->nreq - 1) + (int64_t)(plan->maxs - 1) * plan->slot_stride >= plan->nslot))
        return TA_ERR_ARG;
    const hipStream_t st = static_cast<hipStream_t>(stream);
#define TA_MRG(D, F) \
    launch_merge<D, F>(plan->part, plan->lse, plan->slots, plan->counts, reqs, out, n, plan->hq, plan->maxs, st, \
                       plan->slot_stride)
    return (int)TA_DISPATCH(plan->d, plan->dtype == TA_FP16, TA_MRG);
#undef TA_MRG
}

}  // namespace

extern "C" {

int ta_merge_plan(const ta_plan *plan, void *out, void *stream) {
    if (!plan || !out) return TA_ERR_ARG;
    return plan_merge(plan, nullptr, plan->nreq, out, stream);
}

int ta_segment(const void *q, const void *kp, const void *vp, const int32_t *qids, const int32_t *kstart,
               const int32_t *qlen, const int32_t *klen, const int32_t *rowbase, const int32_t *items,
               int32_t n_items, int32_t kind, void *part, float *lse, int32_t nreq, int32_t hq, int32_t hk,
               int32_t d, int32_t tcap, int32_t maxr, int32_t dtype, void *stream) {
    return segment_launch(q, kp, vp, qids, kstart, qlen, klen, rowbase, items, n_items, kind, part, lse, nreq, hq,
                          hk, d, tcap, maxr, dtype, nullptr, nullptr, nullptr, 0, nullptr, 0, nullptr, pool_layout(tcap), stream);
}

int ta_merge(const void *part, const float *lse, const int32_t *slots, const int32_t *counts, void *out,
             int32_t nreq, int32_t hq, int32_t d, int32_t maxs, int32_t dtype, void *stream) {
    if (dtype != TA_BF16 && dtype != TA_FP16) return TA_ERR_DTYPE;
    if (nreq <= 0 || hq <= 0 || maxs <= 0 || (d != 32 && d != 64 && d != 128)) return TA_ERR_ARG;
    if (!part || !lse || !slots || !counts || !out) return TA_ERR_ARG;
    if (!aligned16(part) || !aligned16(out) || (reinterpret_cast<uintptr_t>(lse) & 7)) return TA_ERR_ALIGN;
    const hipStream_t st = static_cast<hipStream_t>(stream);
#define TA_MRG(D, F) launch_merge<D, F>(part, lse, slots, counts, nullptr, out, nreq, hq, maxs, st)
    return (int)TA_DISPATCH(d, dtype == TA_FP16, TA_MRG);
#undef TA_MRG
}

int ta_segment_plan(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan, int32_t kind,
                    void *stream) {
    if (!plan || kind < TA_SMALL || kind > TA_TAIL) return TA_ERR_ARG;
    return plan_segment(q, kp, vp, tcap, plan, kind, nullptr, pool_layout(tcap), stream);
}

int ta_tail_merge(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan, void *out,
                  void *stream) {
    // (pools of other capacities store a tail's partial like any other and merge all requests alike)
    if (!plan || !out || tcap % 8 != 0) return TA_ERR_ARG;
    return plan_segment(q, kp, vp, tcap, plan, TA_TAIL, out, KV_POOL, stream);
}

}  // extern "C"

// Partial rows and log-sum-exp values of ta_attention_matrix_noalloc.  Each
// GPU the library runs on holds its own copy until the process ends.  In host
// code the name is a stand-in, not a device address: kernels get the address
// hipGetSymbolAddress returns for the current device (noalloc_scratch).
static __device__ __align__(256) unsigned char scratch[TA_NOALLOC_SCRATCH_BYTES];

namespace {

// The TA_LARGE256, TA_LARGE64 and small (TA_SMALL or TA_TAIL) items of a plan in
// one launch (seg_mix_kernel), when at least two of those kinds have items and
// TA_LARGE128 has none.  Returns -1 when the plan does not qualify.
int mix_launch(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan, int small,
               int layout, void *stream) {
    const int n[3] = {plan->n_items[TA_LARGE256], plan->n_items[TA_LARGE64], plan->n_items[small]};
    if ((n[0] > 0) + (n[1] > 0) + (n[2] > 0) < 2 || plan->n_items[TA_LARGE128] > 0) return -1;
    if (n[0] < 0 || n[1] < 0 || n[2] < 0) return TA_ERR_ARG;
    if (int e = check_common(plan->hq, plan->hk, plan->d, plan->dtype)) return e;
    if (plan->nreq <= 0 || tcap <= 0 || plan->maxr <= 0) return TA_ERR_ARG;
    if (!q || !kp || !vp || !plan->qids || !plan->kstart || !plan->qlen || !plan->klen || !plan->rowbase ||
        !plan->part || !plan->lse)
        return TA_ERR_ARG;
    for (int k : {(int)TA_LARGE256, (int)TA_LARGE64, small})
        if (plan->n_items[k] > 0 && !plan->items[k]) return TA_ERR_ARG;
    if (!aligned16(q) || !aligned16(kp) || !aligned16(vp) || !aligned16(plan->part)) return TA_ERR_ALIGN;
    const bool xt = n[0] > 0 && plan->xtail;
    if (xt && (plan->xtail_stride != TA_XTAIL_STRIDE || odd_count(layout))) return TA_ERR_ARG;
    SegParams sp;
    fill_params(sp, q, kp, vp, plan->qids, plan->kstart, plan->qlen, plan->klen, plan->rowbase, nullptr, 0,
                plan->part, plan->lse, plan->hq, plan->hk, plan->d, tcap, plan->maxr, plan->slots, plan->counts,
                nullptr, plan->maxs, xt ? plan->xtail : nullptr, xt ? plan->xtail_stride : 0, plan->qbase);
    const int32_t *const items[3] = {plan->items[TA_LARGE256], plan->items[TA_LARGE64], plan->items[small]};
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const bool fp16 = plan->dtype == TA_FP16;
    return (int)(layout == KV_POOL    ? ta::launch_mix<KV_POOL>(sp, items, n, plan->d, fp16, st)
                 : layout == KV_ODD   ? ta::launch_mix<KV_ODD>(sp, items, n, plan->d, fp16, st)
                 : layout == KV_TOKEN ? ta::launch_mix<KV_TOKEN>(sp, items, n, plan->d, fp16, st)
                                      : ta::launch_mix<KV_TOKEN_ODD>(sp, items, n, plan->d, fp16, st));
}

int attention_layer(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan, void *out,
                    int layout, void *stream) {
    if (!plan || !out) return TA_ERR_ARG;
    if (plan->xtail && odd_count(layout)) return TA_ERR_ARG;
    // the fused merge takes a tail's partial in FP32; other token counts than multiples of 8
    // store every partial and merge all requests alike, so that their tails are small items
    // like any other and run beside the large ones where nothing else does (128 requests x
    // 8192, capacity 8k + 3: 53.0 us with a launch of their own, 51.0 beside the root items;
    // 256 tails over 512 shared tokens 51.8 and 45.5; 128 x 8192 at d = 64 24.5 and 25.0)
    const bool fused = !odd_count(layout);
    const int small = !fused && plan->n_items[TA_SMALL] == 0 ? TA_TAIL : TA_SMALL;
    // the partials every merge reads come first: large jobs, then small jobs,
    // in one launch when the kinds allow it
    const int mixed = mix_launch(q, kp, vp, tcap, plan, small, layout, stream);
    if (mixed > 0) return mixed;
    const int order[] = {TA_LARGE256, TA_LARGE128, TA_LARGE64, small};
    for (int kind : order) {
        if (mixed == 0 && kind != TA_LARGE128) continue;
        if (plan->n_items[kind] == 0) continue;
        if (int e = plan_segment(q, kp, vp, tcap, plan, kind, nullptr, layout, stream)) return e;
    }
    if (plan->n_items[TA_TAIL] > 0 && small != TA_TAIL)
        if (int e = plan_segment(q, kp, vp, tcap, plan, TA_TAIL, fused ? out : nullptr, layout, stream)) return e;
    if (!fused) return plan_merge(plan, nullptr, plan->nreq, out, stream);
    if (plan->n_rest <= 0) return 0;
    // rest == NULL with n_rest == nreq: every request
    if (!plan->rest && plan->n_rest != plan->nreq) return TA_ERR_ARG;
    return plan_merge(plan, plan->rest, plan->n_rest, out, stream);
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char *g_scratch[kMaxDevices];  // per device: the device address of `scratch`

// The address of `scratch` on the current device, looked up once per device
// (with that device current) and kept.
int noalloc_scratch(unsigned char **ptr) {
    int dev = -1;
    if (hipError_t e = hipGetDevice(&dev)) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return TA_ERR_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) return (int)e;
        if (!p) return TA_ERR_ARG;
        g_scratch[dev] = static_cast<unsigned char *>(p);
    }
    *ptr = g_scratch[dev];
    return 0;
}

}  // namespace

extern "C" {

int ta_attention_matrix(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan,
                        void *out, void *stream) {
    return attention_layer(q, kp, vp, tcap, plan, out, pool_layout(tcap), stream);
}

int ta_attention_tokens(const void *q, const void *k, const void *v, int32_t tokens, const ta_plan *plan, void *out,
                        void *stream) {
    return attention_layer(q, k, v, tokens, plan, out, token_layout(tokens), stream);
}

int ta_attention_matrix_noalloc(const void *q, const void *kp, const void *vp, int32_t tcap, const ta_plan *plan,
                                void *out, void *stream) {
    if (!plan || !out) return TA_ERR_ARG;
    if (plan->nslot <= 0 || plan->hq <= 0 || plan->d <= 0) return TA_ERR_ARG;
    // partial rows (fp16) first, then the (lse, exponent) pairs at a 256-byte boundary
    const uint64_t part_bytes = (uint64_t)plan->nslot * (uint64_t)plan->hq * (uint64_t)plan->d * 2u;
    const uint64_t lse_offset = (part_bytes + 255u) & ~(uint64_t)255u;
    const uint64_t lse_bytes = (uint64_t)plan->nslot * (uint64_t)plan->hq * 2u * sizeof(float);
    if (lse_offset + lse_bytes > (uint64_t)TA_NOALLOC_SCRATCH_BYTES) return TA_ERR_SCRATCH;
    unsigned char *base = nullptr;
    if (int e = noalloc_scratch(&base)) return e;
    if (stream) {  // the scratch address belongs to the current device: the stream must be on it
        int cur = -1, sdev = -1;
        if (hipError_t e = hipGetDevice(&cur)) return (int)e;
        if (hipError_t e = hipStreamGetDevice(static_cast<hipStream_t>(stream), &sdev)) return (int)e;
        if (cur != sdev) return TA_ERR_ARG;
    }
    // every partial slot the merge reads is written by a segment launch of the
    // same call first, so nothing in the array needs clearing
    ta_plan local = *plan;
    local.part = base;
    local.lse = reinterpret_cast<float *>(base + lse_offset);
    return attention_layer(q, kp, vp, tcap, &local, out, pool_layout(tcap), stream);
}

int ta_read_stream(const void *src, int64_t bytes, uint32_t *sink, int32_t blocks, void *stream) {
    if (!src || !sink || bytes <= 0 || bytes % 16 != 0 || blocks <= 0) return TA_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(src) % 16 != 0) return TA_ERR_ALIGN;
    TA_LAUNCH(read_stream_kernel, dim3(blocks), dim3(READ_NT), static_cast<hipStream_t>(stream),
              static_cast<const u32x4 *>(src), bytes / 16, sink);
    return (int)hipGetLastError();
}

int ta_time_next_launch(void *start_event, void *stop_event) {
    if ((start_event == nullptr) != (stop_event == nullptr)) return TA_ERR_ARG;
    ta::g_launch_events = ta::LaunchEvents{static_cast<hipEvent_t>(start_event), static_cast<hipEvent_t>(stop_event)};
    return 0;
}

}  // extern "C"
