// GQA decode / prefill attention over an FP16 paged KV cache, for gfx950.
//
// Semantics follow attention_paged.cu:36-170: query token i of a sequence attends to
// positions 0 .. min(start_pos + i + 1, kv_len) - 1 (or seq_lens[i] in the batched form);
// position t lives in page block_table[t / 16], row (t % 16), as a [16][kv_heads][head_dim]
// fp16 block; score = dot(q, k) / sqrt(head_dim) with fp32 accumulation, softmax in fp32,
// out = half(sum_t p_t v_t). The reference keeps a kv_len-float score row in shared memory
// (attention_paged.cu:58-59, 176); here the context is split into 1024-position pieces with an
// online softmax each, merged by a second kernel: up to 1,048,576 positions per sequence.
//
// Work split: one workgroup per (query, kv head, block of up to 8 of its q heads, split). Each K
// row crosses HBM once per (query, kv head) for up to 8 q heads. In causal prefill at head_dim 256 with
// fewer than 8 q heads per kv head, it takes 8 / G consecutive queries instead, its columns
// being (query, head) pairs each masked to its own causal length, so that a K or V row is
// read once for all of them (head_dim 32, 64 and 128 have a prefill kernel of their own, below). Per
// 32-position chunk (16 when head_dim is 256):
//   QK on v_mfma_f32_16x16x32_f16: A = K rows (row = position, 8 consecutive dims per lane,
//      exactly their memory layout), B = Q^T (column = q head): fp16 x fp16 products are
//      exact in fp32, the sums are fp32;
//   online softmax per head in log2 units, weights to LDS;
//   PV on the VALU in fp32: lane (dim group of 8, position subset) loads 16 bytes of a V row
//      and accumulates p_h * v for the wave's heads. V needs no transpose this way, and the
//      fp32 weights need no fp16 rounding.
// The kernel streams 4 * head_dim bytes per (position, kv head) and is bound by HBM.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "fhip_common.h"
#include "fracture_hip.h"
#include "launch_rules.h"
#include "tq_attn_index.h"

using namespace fhip;

namespace {

constexpr int kPSplit = 1024;  // positions per split: 64 pages, one per lane of the page cache
constexpr int kHeadsMax = 8;   // q heads per wave
// Longest context a block table may describe (the combine kernel keeps one weight per
// split in LDS: 4 KiB at this bound).
constexpr int64_t kMaxTokens = (int64_t)kPSplit * 1024;

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// Page sources: per-block pointer arrays (the reference's interface) or contiguous pools.
struct F16PtrPages {
    const uint8_t* const* k;
    const uint8_t* const* v;
    int num_pages;
    __device__ bool valid(int p) const { return p >= 0 && p < num_pages; }
    // Wave-wide page cache: lane j holds the pointers of page j of the current split; the
    // `_at` accessors read them back from lane j.
    struct Lane {
        const uint8_t *k, *v;
    };
    __device__ Lane lane_load(int p) const {
        if (!valid(p)) return Lane{nullptr, nullptr};
        return Lane{k[p], v[p]};
    }
    static __device__ const uint8_t* rl(const uint8_t* x, int j) {
        const uint64_t u = (uint64_t)x;
        const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, j);
        const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), j);
        return (const uint8_t*)(((uint64_t)hi << 32) | lo);
    }
    __device__ const uint8_t* k_at(const Lane& l, int j, int) const { return rl(l.k, j); }
    __device__ const uint8_t* v_at(const Lane& l, int j, int) const { return rl(l.v, j); }
    // one lane's own page (any page id per lane)
    __device__ const uint8_t* k_page(int p) const { return k[p]; }
    __device__ const uint8_t* v_page(int p) const { return v[p]; }
};
struct F16PoolPages {
    const uint8_t* k;
    const uint8_t* v;
    int64_t sk, sv;  // bytes between pages
    int num_pages;
    __device__ bool valid(int p) const { return p >= 0 && p < num_pages; }
    struct Lane {};
    __device__ Lane lane_load(int) const { return Lane{}; }
    __device__ const uint8_t* k_at(const Lane&, int, int p) const { return k + p * sk; }
    __device__ const uint8_t* v_at(const Lane&, int, int p) const { return v + p * sv; }
    __device__ const uint8_t* k_page(int p) const { return k + p * sk; }
    __device__ const uint8_t* v_page(int p) const { return v + p * sv; }
};

// 16 bytes through a global pointer: page pointers read from memory are generic ones to the compiler,
// and flat loads would also be waited for with every LDS read.
typedef __attribute__((address_space(1))) const u32x4 g_u32x4;
__device__ __forceinline__ u32x4 gld16(const uint8_t* p) { return *(g_u32x4*)p; }

// Query i reads block-table row i (stride 0: one shared table) and attends to seq_lens[i]
// positions, or min(start_pos + i + 1, kv_len) when seq_lens is null; never more than the
// table holds.
struct PQueries {
    const int32_t* table;
    int64_t table_stride;
    int max_blocks;
    const int32_t* seq_lens;
    int kv_len, start_pos;
    int count;
    __device__ int causal_len(int qi) const {
        int c;
        if (seq_lens) {
            c = seq_lens[qi];
        } else {
            c = start_pos + qi + 1;
            if (c > kv_len) c = kv_len;
        }
        const int cap = max_blocks * FHIP_PAGE_TOKENS;
        if (c > cap) c = cap;
        return c < 0 ? 0 : c;
    }
};

// Split partials: per (query, q head, split) the running max m (natural log units), the sum
// l and the unnormalised accumulator acc[hd]. Splits at or past the causal length are not
// written; the combine kernel reads only the splits below it.
//
// A workgroup of W waves takes one (query, kv head, head block, split); wave w scores the
// split's positions [w, w + 1) * kPSplit / W and the waves' states are merged in LDS, so the
// partials stay one per split whatever W is (paged_waves in launch_rules.h). With a wave per split
// the chunk's loads had nothing beside them to hide behind: 16 sequences of 500 .. 8192
// positions (32 / 8 heads of 128, 285 MB) went from 136 to 72 us.
// W = 1 puts two splits of neighbouring kv heads, each a wave's own, in a workgroup instead.
template <int HD, int NH, int W, class Pages>
__global__ __launch_bounds__(64 * (W == 1 ? 2 : W)) __attribute__((amdgpu_waves_per_eu(2))) void
paged_attn_split_kernel(const uint16_t* __restrict__ q, PQueries qs, Pages pg, int qh, int kvh,
                        int nhb, float scale_log2, float* __restrict__ part_ml,
                        float* __restrict__ part_acc, int nsplit, int tok) {
    constexpr int kChunk = HD <= 128 ? 32 : 16;  // positions per chunk
    constexpr int kTiles = kChunk / 16;          // 16-position MFMA tiles (= pages) per chunk
    constexpr int kSteps = HD / 32;              // MFMA steps per tile
    constexpr int kDg = HD / 8;                  // lanes per V row, 8 dims each
    constexpr int kPpl = 64 / kDg;               // positions per V load
    constexpr int kVLoads = kChunk / kPpl;
    constexpr int kPiece = kPSplit / W;  // positions per wave
    static_assert(kPpl <= 16 && 16 % kPpl == 0, "a V load stays inside one page");
    static_assert(kPiece % kChunk == 0, "a wave's positions are whole chunks");
    // Every lane writes its own slot of these buffers (columns / entries past the wave's
    // heads are written and never read): a store guarded by the lane index followed by reads
    // of every lane lets the compiler sink the reads into the guarded block, where they run
    // with the other lanes switched off (seen in a variant of this loop at head_dim 32).
    constexpr int kWaves = W == 1 ? 2 : W;  // of the workgroup
    __shared__ __attribute__((aligned(16))) float pbuf[kWaves][kChunk][16];
    __shared__ __attribute__((aligned(16))) float abuf[kWaves][64];
    // the waves' states for the merge: (m, l) per column, and the accumulators
    __shared__ float mlbuf[kWaves][2][16];
    __shared__ __attribute__((aligned(16))) float sbuf[kWaves][NH][HD];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // W > 1: every exit before the merge's barrier is uniform over the workgroup
    const int64_t item = W == 1 ? (int64_t)blockIdx.x * 2 + wave : blockIdx.x;
    const int piece = W == 1 ? 0 : wave;  // of the split
    const int64_t per_q = (int64_t)kvh * nhb * nsplit;
    // queries tq0 .. tq0 + ntok - 1 (tok > 1 only in causal prefill over one shared table
    // with nhb == 1, where causal lengths grow with the query index)
    const int tq0 = (int)(item / per_q) * tok;
    if (tq0 >= qs.count) return;
    const int ntok = min(tok, qs.count - tq0);
    // kv head fastest: neighbouring workgroups read neighbouring rows of the same pages
    const int g = (int)(item % kvh);
    const int hb = (int)((item / kvh) % nhb);
    const int split = (int)((item / ((int64_t)kvh * nhb)) % nsplit);
    const int clen = qs.causal_len(tq0 + ntok - 1);
    if (split * kPSplit >= clen) return;
    const int t_begin = split * kPSplit + piece * kPiece;  // may lie past t_end: an empty piece
    const int t_end = min(clen, t_begin + kPiece);
    const int G = qh / kvh;
    const int h0 = g * G + hb * kHeadsMax;
    // MFMA columns (<= NH): with tok == 1 heads h0 .. h0 + ncols - 1 of query tq0, else
    // column c is head h0 + c % G of query tq0 + c / G
    const int ncols = tok > 1 ? ntok * G : min(kHeadsMax, G - hb * kHeadsMax);
    const int32_t* table = qs.table + (int64_t)tq0 * qs.table_stride;

    // the split's pages, one per lane, read once
    static_assert(kPSplit == 64 * FHIP_PAGE_TOKENS, "one cached page per lane");
    const int split_page =
        t_begin + FHIP_PAGE_TOKENS * lane < t_end ? table[t_begin / FHIP_PAGE_TOKENS + lane] : -1;
    const typename Pages::Lane pl = pg.lane_load(split_page);

    // Q^T as the QK B operand: lane (column n, k group kg) holds dims 32 s + 8 kg + 0..7 of
    // column n's query row at step s; columns n >= ncols are zero and fully masked.
    const int n = lane & 15, kg = lane >> 4;
    const bool col_ok = n < ncols;
    const int ct = col_ok ? n / G : 0;  // 0 whenever tok == 1 (n < ncols <= G)
    const int hn = col_ok ? n - ct * G : 0;
    const int col_len = !col_ok ? 0 : tok > 1 ? qs.causal_len(tq0 + ct) : clen;
    const int lim = min(t_end, col_len);  // column n scores positions below lim
    u32x4 bq[kSteps];
    {
        const uint16_t* qrow = q + ((int64_t)(tq0 + ct) * qh + h0 + hn) * HD + 8 * kg;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const u32x4 v = ld16(qrow + 32 * s);
            bq[s] = col_ok ? v : u32x4{0u, 0u, 0u, 0u};
        }
    }
    // lane offsets inside a page: K row (lane & 15) segment kg; V row of position subset ps,
    // dims 8 dg .. 8 dg + 7
    const int64_t k_off = ((int64_t)(lane & 15) * kvh + g) * (HD * 2) + 16 * kg;
    const int dg = lane % kDg, ps = lane / kDg;
    const uint8_t* dummy = (const uint8_t*)q;  // >= 2 HD readable bytes, finite values

    float m_run = -__builtin_inff(), l_run = 0.0f;  // lanes n (any kg): head n
    float acc[NH][8];
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[h][i] = 0.0f;

    for (int t0 = t_begin; t0 < t_end; t0 += kChunk) {
        const int j0 = (t0 - t_begin) / FHIP_PAGE_TOKENS;
        // ---- every load of the chunk first: K rows, then V rows. Loads of positions past
        // the end or in invalid pages read `dummy` and are masked below.
        bool pok[kTiles];
        const uint8_t* kb[kTiles];
        const uint8_t* vb[kTiles];
#pragma unroll
        for (int tt = 0; tt < kTiles; ++tt) {
            const int id = __builtin_amdgcn_readlane(split_page, j0 + tt);
            pok[tt] = pg.valid(id);
            kb[tt] = pok[tt] ? pg.k_at(pl, j0 + tt, id) : dummy;
            vb[tt] = pok[tt] ? pg.v_at(pl, j0 + tt, id) : dummy;
        }
        u32x4 kr[kTiles][kSteps];
#pragma unroll
        for (int tt = 0; tt < kTiles; ++tt) {
            const bool ok = pok[tt] && t0 + 16 * tt + (lane & 15) < t_end;
            const uint8_t* src = ok ? kb[tt] + k_off : dummy;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) kr[tt][s] = ld16(src + 64 * s);
        }
        u32x4 vr[kVLoads];
        bool vok[kVLoads];
#pragma unroll
        for (int j = 0; j < kVLoads; ++j) {
            const int pp = j * kPpl + ps;  // position in the chunk
            const int tt = (j * kPpl) / 16;
            vok[j] = pok[tt] && t0 + pp < t_end;
            const uint8_t* src =
                vok[j] ? vb[tt] + (((int64_t)(pp % 16) * kvh + g) * HD + 8 * dg) * 2 : dummy;
            vr[j] = ld16(src);
        }

        // ---- QK: lane (n, rg) gets positions 16 tt + 4 rg + e of head n
        float sc[kTiles][4];
#pragma unroll
        for (int tt = 0; tt < kTiles; ++tt) {
            f4_t d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, kr[tt][s]),
                                                           __builtin_bit_cast(h8_t, bq[s]), d,
                                                           0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int pos = t0 + 16 * tt + 4 * kg + e;
                sc[tt][e] = pok[tt] && pos < lim ? d[e] * scale_log2 : -__builtin_inff();
            }
        }
        // ---- online softmax per head (lanes n, n + 16, n + 32, n + 48 share head n)
        float cmax = -__builtin_inff();
#pragma unroll
        for (int tt = 0; tt < kTiles; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) cmax = fmaxf(cmax, sc[tt][e]);
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
        const float m_new = fmaxf(m_run, cmax);
        const float mref = m_new == -__builtin_inff() ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - mref);  // 0 while m_run is -inf
        float psum = 0.0f;
        // the previous chunk's reads of pbuf / abuf (other lanes' words) stay above these writes
        wave_lds_sync();
#pragma unroll
        for (int tt = 0; tt < kTiles; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float p = __builtin_amdgcn_exp2f(sc[tt][e] - mref);
                psum += p;
                pbuf[wave][16 * tt + 4 * kg + e][n] = p;
            }
        psum += __shfl_xor(psum, 16);
        psum += __shfl_xor(psum, 32);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        abuf[wave][lane] = alpha;
        // every lane's pbuf / abuf writes stay above the cross-lane reads below
        wave_lds_sync();

        // ---- PV
        float al[kHeadsMax];
        {
            const f4_t a0 = *(const f4_t*)&abuf[wave][0];
            const f4_t a1 = *(const f4_t*)&abuf[wave][4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                al[i] = a0[i];
                al[4 + i] = a1[i];
            }
        }
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] *= al[h];
#pragma unroll
        for (int j = 0; j < kVLoads; ++j) {
            const int pp = j * kPpl + ps;
            float pw[kHeadsMax];
            {
                const f4_t p0 = *(const f4_t*)&pbuf[wave][pp][0];
                const f4_t p1 = *(const f4_t*)&pbuf[wave][pp][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pw[i] = p0[i];
                    pw[4 + i] = p1[i];
                }
            }
            float v[8];
            unpack16<TrF16>(vok[j] ? vr[j] : u32x4{0u, 0u, 0u, 0u}, v);
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[h][i] = fmaf(pw[h], v[i], acc[h][i]);
        }
    }

    // ---- the wave's state: sum the position subsets (lanes with the same dim group), then
    // lanes of subset 0 leave dims 8 dg .. 8 dg + 7 of each column
#pragma unroll
    for (int o = kDg; o < 64; o <<= 1)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] += __shfl_xor(acc[h][i], o);
    // column c's vector is (query tq0 + c / G, head h0 + c % G)
    if constexpr (W == 1) {  // the split's state is the wave's
        if (lane < ncols) {  // lane == n here
            const int64_t v = (int64_t)(tq0 + ct) * qh + h0 + hn;
            part_ml[(v * nsplit + split) * 2 + 0] = m_run * 0.6931471805599453f;
            part_ml[(v * nsplit + split) * 2 + 1] = l_run;
        }
        if (ps == 0) {
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if (h >= ncols) break;
                const int cq = tok > 1 ? h / G : 0;
                const int64_t v = (int64_t)(tq0 + cq) * qh + h0 + (h - cq * G);
                float* dst = part_acc + (v * nsplit + split) * HD + 8 * dg;
                *(f4_t*)dst = f4_t{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
                *(f4_t*)(dst + 4) = f4_t{acc[h][4], acc[h][5], acc[h][6], acc[h][7]};
            }
        }
        return;
    }
    if (lane < 16) {
        mlbuf[wave][0][lane] = m_run;
        mlbuf[wave][1][lane] = l_run;
    }
    if (ps == 0) {
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            float* dst = &sbuf[wave][h][8 * dg];
            *(f4_t*)dst = f4_t{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
            *(f4_t*)(dst + 4) = f4_t{acc[h][4], acc[h][5], acc[h][6], acc[h][7]};
        }
    }
    __syncthreads();
    // ---- merge in wave order; a wave with m = -inf adds nothing (an empty or fully masked piece), or
    // the NaN that all its scores were
    for (int i = threadIdx.x; i < ncols * (HD / 4); i += 64 * W) {
        const int c = i / (HD / 4), d = 4 * (i - c * (HD / 4));
        const int cq = tok > 1 ? c / G : 0;
        float M = -__builtin_inff();
#pragma unroll
        for (int w = 0; w < W; ++w) M = fmaxf(M, mlbuf[w][0][c]);
        float L = 0.0f;
        f4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float mw = mlbuf[w][0][c];
            const float wt = mw == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
            L = fmaf(wt, mlbuf[w][1][c], L);
            const f4_t a = *(const f4_t*)&sbuf[w][c][d];
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = fmaf(wt, a[k], o[k]);
        }
        const int64_t v = (int64_t)(tq0 + cq) * qh + h0 + (c - cq * G);
        *(f4_t*)(part_acc + (v * nsplit + split) * HD + d) = o;
        if (d == 0) {
            part_ml[(v * nsplit + split) * 2 + 0] = M * 0.6931471805599453f;
            part_ml[(v * nsplit + split) * 2 + 1] = L;
        }
    }
}

// One wave's attention of one query row over positions [t_begin, t_end) of a kv head, any
// head_dim up to 256. Per 64-position chunk, lane l scores position t0 + l against the query (fp32
// dot over the dims in order, the query staged in `qv`, hd floats of LDS), the wave updates the
// online softmax (natural-log units), and each lane accumulates its dims l, l + 64, .. over the
// chunk's positions, their weights and row addresses broadcast from the lanes that scored them.
// A position outside [t_begin, t_end) or in a page outside the pool is never read.
template <class Pages>
__device__ __forceinline__ void wave_attend(const uint16_t* qrow, const int32_t* table, const Pages& pg,
                                            int t_begin, int t_end, int kvh, int g, int hd, float scale,
                                            int lane, float* qv, float& m_run, float& l_run,
                                            float (&acc)[4]) {
    wave_lds_sync();  // an earlier call's reads of qv stay above these writes
    for (int d = lane; d < hd; d += 64) qv[d] = h2f(qrow[d]);
    wave_lds_sync();  // every lane reads every dim below
    m_run = -__builtin_inff();
    l_run = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = 0.0f;  // dims lane + 64 i
    const int64_t row_bytes = (int64_t)hd * 2;
    for (int t0 = t_begin; t0 < t_end; t0 += 64) {
        const int pos = t0 + lane;
        const int id = pos < t_end ? table[pos / FHIP_PAGE_TOKENS] : -1;
        const bool ok = pos < t_end && pg.valid(id);
        const int64_t roff = ((int64_t)(pos % FHIP_PAGE_TOKENS) * kvh + g) * row_bytes;
        const uint16_t* krow = ok ? (const uint16_t*)(pg.k_page(id) + roff) : nullptr;
        const uint16_t* vrow = ok ? (const uint16_t*)(pg.v_page(id) + roff) : nullptr;
        float s = -__builtin_inff();
        if (ok) {
            float dot = 0.0f;
            for (int d = 0; d < hd; ++d) dot = fmaf(qv[d], h2f(krow[d]), dot);
            s = dot * scale;
        }
        const float cmax = wave_max(s);
        const float m_new = fmaxf(m_run, cmax);
        const float alpha = m_run == -__builtin_inff() ? 0.0f : expf(m_run - m_new);
        const float p = ok ? expf(s - m_new) : 0.0f;
        l_run = l_run * alpha + wave_sum(p);
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] *= alpha;
        const int n = min(64, t_end - t0);
        for (int j = 0; j < n; ++j) {
            const float pj = __shfl(p, j);
            const uint64_t vj = (uint64_t)__shfl((long long)(uintptr_t)vrow, j);
            if (vj == 0) continue;  // uniform: position j is masked
            const uint16_t* vr = (const uint16_t*)(uintptr_t)vj;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = lane + 64 * i;
                if (d < hd) acc[i] = fmaf(pj, h2f(vr[d]), acc[i]);
            }
        }
    }
}

// Causal prefill (head_dim 32 / 64 / 128, G <= 8 q heads per kv head): a workgroup of 4 waves takes
// kPfCols columns of one kv head, column c being head c % G of query q0 + c / G, each wave 32 of
// them, and walks a split of the positions in tiles of 64 that all its waves share.
//   S^T = K Q^T on v_mfma_f32_32x32x16_f16: row = position, column = (query, head); lane
//     (n, half) then holds 16 positions of column n per 32-position block, so the softmax of a
//     column needs one exchange between the two halves (the maximum) per tile.
//   out^T = V^T P^T on the same MFMA: slot j of lane half `half` in a 16-position step is
//     position 4 half + j (j < 4) or 8 + 4 half + j - 4, exactly what the lane holds after S^T,
//     so P goes into the B operand without moving between lanes. P = hi + lo in fp16, two
//     products into one accumulator: the exponent is biased by kPfBias, so that lo is a normal
//     fp16 number for every p above 2^-14 (p to ~2^-23; an absolute 2^-37 below that), and the
//     bias cancels in out = acc / l. V is exact. A = V^T comes from the row-major tile by
//     ds_read_b64_tr_b16.
//   The next tile's rows are loaded into registers before the tile's products and stored to the
//     other LDS buffer after them: one barrier per tile. Rows are padded so that the 16-byte
//     reads of 16 K rows, and the transposed reads of 4 V rows x 32 dims, cover all banks.
// Bound by the MFMA (48 products of 32 clocks per wave and tile at head_dim 128, a third of them
// the lo parts) and by the VALU work of the softmax (~1360 clocks), which two waves per SIMD
// overlap in part. 1000 queries at 3001 .. 4000, 32 / 8 heads of 128: 107 us (536 TFLOP/s of
// attention); waves of 16 columns over chunks of 32 positions with two barriers each took 214.
constexpr int kPfWaves = 4;                // waves per workgroup
constexpr int kPfCols = 32 * kPfWaves;     // (query, head) columns per workgroup
constexpr int kPfTile = 64;                // positions per tile
constexpr float kPfBias = 12.0f;           // log2 of the scale that P carries
constexpr float kPfScale = 4096.0f;        // 2^kPfBias
constexpr float kPfSlack = 3.75f;          // log2 that p may exceed it by (2^15.75 < fp16's largest)
constexpr int64_t kPfGroups = 512;         // workgroups wanted: the two per CU that fit at once
typedef float f16x_t __attribute__((ext_vector_type(16)));

template <int HD, class Pages>
__global__ __launch_bounds__(64 * kPfWaves) __attribute__((amdgpu_waves_per_eu(2))) void
paged_attn_prefill_mfma_kernel(const uint16_t* __restrict__ q, PQueries qs, Pages pg, int qh,
                               int kvh, float scale_log2, float* __restrict__ part_ml,
                               float* __restrict__ part_acc, uint16_t* __restrict__ out,
                               int nsplit, int split_pos, int nqb, int nblk) {
    constexpr int kSteps = HD / 16;     // S^T steps per 32-position block
    constexpr int kDt = HD / 32;        // 32-dim blocks of out^T
    constexpr int kRowK = HD * 2 + 16;  // bytes per staged K row
    constexpr int kRowV = HD * 2 + 64;  // bytes per staged V row
    constexpr int kPer = kPfTile * HD / 8 / (64 * kPfWaves);  // 16-byte pieces of K (of V) per thread
    constexpr int kSegs = HD / 8;                             // pieces per row
    static_assert(HD == 32 || HD == 64 || HD == 128, "a wave's pieces lie in one page");
    __shared__ __attribute__((aligned(16))) uint8_t kbuf[2][kPfTile * kRowK];
    __shared__ __attribute__((aligned(16))) uint8_t vbuf[2][kPfTile * kRowV];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // kv head fastest (one head's rows stay in one XCD's L2 at 8 kv heads), then the split, then
    // the query block from the last one down: the longest contexts start first
    const int g = (int)(blockIdx.x % kvh);
    const int rest = (int)(blockIdx.x / kvh);
    const int split = rest % nsplit;
    const int q0 = fhip_idx::prefill_block(rest / nsplit, nblk, 0) * nqb;  // the block's first query
    const int nq = min(nqb, qs.count - q0);
    const int G = qh / kvh;
    const int clen = qs.causal_len(q0 + nq - 1);  // the block's longest causal length
    const int clen0 = qs.causal_len(q0);          // and its shortest
    const int t_begin = split * split_pos;
    // uniform: of partials, a split past the block's length writes none
    if (!out && t_begin >= clen) return;
    const int t_end = min(clen, t_begin + split_pos);
    const int32_t* table = qs.table + (int64_t)q0 * qs.table_stride;

    // column n of the wave: head ch of query q0 + cq
    const int n = lane & 31, half = lane >> 5;
    const int ncols = nq * G;
    const int col = 32 * wave + n;
    const bool col_ok = col < ncols;
    const bool wave_live = 32 * wave < ncols;
    const int cq = col_ok ? col / G : 0;
    const int64_t vec = (int64_t)(q0 + cq) * qh + g * G + (col_ok ? col - cq * G : 0);
    const int lim = col_ok ? min(t_end, qs.causal_len(q0 + cq)) : 0;
    u32x4 bq[kSteps];  // dims 16 s + 8 half + 0..7 of the column's query row
#pragma unroll
    for (int s = 0; s < kSteps; ++s) bq[s] = ld16(q + vec * HD + 16 * s + 8 * half);
    // waited for here: left to the loop, the wait would also be for each next tile's loads
#pragma unroll
    for (int s = 0; s < kSteps; ++s) asm volatile("" : "+v"(bq[s]));

    // The pages of 1024 positions from `win`, one per lane, refreshed when a tile leaves them.
    const uint8_t* dummy = (const uint8_t*)q;  // >= 2 HD readable bytes
    int win = t_begin, win_page;
    typename Pages::Lane pl;
    auto load_window = [&](int t0) {
        win = t0;
        win_page = t0 + FHIP_PAGE_TOKENS * lane < t_end ? table[t0 / FHIP_PAGE_TOKENS + lane] : -1;
        pl = pg.lane_load(win_page);
    };
    // Piece u of a thread: row (threadIdx.x + 256 u) / kSegs of the tile, 16 bytes of it; the wave's
    // rows of one u lie in one page (4, 8 or 16 rows a wave), whose row and offset do not depend
    // on u. Pages outside the pool read `dummy`; their scores are masked. V rows past the end or
    // in such pages are staged as zeros.
    u32x4 kr[kPer], vr[kPer];
    const uint32_t row_off = (uint32_t)(((int)threadIdx.x / kSegs % FHIP_PAGE_TOKENS * kvh + g) * (HD * 2) +
                                        16 * ((int)threadIdx.x % kSegs));
    uint32_t pok = 0;  // bit j: page j of the tile in the registers is in the pool
    auto page_of = [&](int u) { return (64 * wave + 64 * kPfWaves * u) / kSegs / FHIP_PAGE_TOKENS; };
    auto load_tile = [&](int t0) {
        if (t0 >= win + 64 * FHIP_PAGE_TOKENS) load_window(t0);
        const int j0 = (t0 - win) / FHIP_PAGE_TOKENS;
        pok = (uint32_t)(__ballot(pg.valid(win_page)) >> j0) & 0xfu;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int j = page_of(u);
            const int id = __builtin_amdgcn_readlane(win_page, j0 + j);
            const bool ok = (pok >> j) & 1u;
            const uint8_t* kp = ok ? pg.k_at(pl, j0 + j, id) : dummy;
            const uint8_t* vp = ok ? pg.v_at(pl, j0 + j, id) : dummy;
            const uint32_t off = ok ? row_off : 0u;
            kr[u] = gld16(kp + off);
            vr[u] = gld16(vp + off);
        }
    };
    // Stores the tile of the registers. Where some column masks a position of the tile, also notes
    // a V value that is infinite or NaN: 0 x inf would carry it to that column.
    bool bad = false;
    auto store_tile = [&](int t0, int b) {
        const uint32_t off = ((uint32_t)threadIdx.x / kSegs) * kRowK + 16 * (threadIdx.x % kSegs);
        const uint32_t offv = ((uint32_t)threadIdx.x / kSegs) * kRowV + 16 * (threadIdx.x % kSegs);
        if (pok != 0xfu || t0 + kPfTile > t_end) {
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int r = ((int)threadIdx.x + 64 * kPfWaves * u) / kSegs;
                const bool rok = ((pok >> page_of(u)) & 1u) && t0 + r < t_end;
                if (!rok) vr[u] = u32x4{0u, 0u, 0u, 0u};
            }
        }
        if (t0 + kPfTile > clen0) {
#pragma unroll
            for (int u = 0; u < kPer; ++u)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    bad |= (vr[u][k] & 0x7c00u) == 0x7c00u || (vr[u][k] & 0x7c000000u) == 0x7c000000u;
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            *(u32x4*)(kbuf[b] + off + u * (64 * kPfWaves / kSegs) * kRowK) = kr[u];
            *(u32x4*)(vbuf[b] + offv + u * (64 * kPfWaves / kSegs) * kRowV) = vr[u];
        }
    };

    float m_run = -__builtin_inff(), l_run = 0.0f;  // l: the lane half's own positions
    f16x_t acc[kDt];
#pragma unroll
    for (int d = 0; d < kDt; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;

    uint32_t tile_pok = 0;
    if (t_begin < t_end) {
        load_window(t_begin);
        load_tile(t_begin);
        tile_pok = pok;
        store_tile(t_begin, 0);
        lds_barrier();
    }
    int b = 0;
    for (int t0 = t_begin; t0 < t_end; t0 += kPfTile, b ^= 1) {
        const bool more = t0 + kPfTile < t_end;
        if (more) load_tile(t0 + kPfTile);
        if (wave_live) {
            // ---- S^T: element i of block pt is position 32 pt + 8 (i / 4) + 4 half + i % 4
            // K reads run kSteps products ahead of their use, across the two blocks
            // (the priority lets this wave's products go first while the other wave of its SIMD is
            // in its softmax: 114 -> 107 us)
            __builtin_amdgcn_s_setprio(1);
            f16x_t sc[2];
            const uint8_t* ksrc = kbuf[b] + n * kRowK + 16 * half;
            u32x4 ka[kSteps];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) ka[s] = *(const u32x4*)(ksrc + 32 * s);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[pt][i] = 0.0f;
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    sc[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        __builtin_bit_cast(h8_t, ka[s]), __builtin_bit_cast(h8_t, bq[s]), sc[pt], 0, 0, 0);
                    if (pt == 0) {
                        ka[s] = *(const u32x4*)(ksrc + 32 * kRowK + 32 * s);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
            // a tile with every page in the pool and inside every column's length needs no mask
            if (!(tile_pok == 0xfu && t0 + kPfTile <= min(t_end, clen0))) {
#pragma unroll
                for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int pos = t0 + 32 * pt + 8 * (i / 4) + 4 * half + i % 4;
                        const bool ok = ((tile_pok >> (2 * pt + i / 8)) & 1u) && pos < lim;
                        sc[pt][i] = ok ? sc[pt][i] : -__builtin_inff();
                    }
            }
            // ---- online softmax in log2 units, one column per lane pair (n, n + 32)
            float cmax = sc[0][0];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i) cmax = fmaxf(cmax, sc[pt][i]);
            cmax = fmaxf(cmax, __shfl_xor(cmax, 32)) * scale_log2;
            const float m_new = fmaxf(m_run, cmax);
            // p may grow to 2^kPfSlack before the accumulators are rescaled: almost no tile after
            // the first rescales, where following the maximum would on most (32 columns a wave)
            if (__ballot(m_new > m_run + kPfSlack)) {
                const float mref = m_new == -__builtin_inff() ? 0.0f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run - mref);  // 0 while m_run is -inf
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < kDt; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[d][i] *= alpha;
                m_run = m_new;
            }
            const float ebias = kPfBias - (m_run == -__builtin_inff() ? 0.0f : m_run);
            float psum = 0.0f;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    sc[pt][i] = __builtin_amdgcn_exp2f(fmaf(sc[pt][i], scale_log2, ebias));
                    psum += sc[pt][i];
                }
            l_run += psum;
            __builtin_amdgcn_s_setprio(1);
            // ---- out^T: 4 steps of 16 positions
            const uint8_t* vsrc = vbuf[b] + (4 * half + ((lane & 15) >> 2)) * kRowV +
                                  2 * (16 * ((lane >> 4) & 1) + 4 * (lane & 3));
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                uint32_t ph[4], pl_[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    split_pair(sc[ks >> 1][8 * (ks & 1) + 2 * j], sc[ks >> 1][8 * (ks & 1) + 2 * j + 1],
                               ph[j], pl_[j]);
                const h8_t bh = __builtin_bit_cast(h8_t, u32x4{ph[0], ph[1], ph[2], ph[3]});
                const h8_t bl = __builtin_bit_cast(h8_t, u32x4{pl_[0], pl_[1], pl_[2], pl_[3]});
#pragma unroll
                for (int d = 0; d < kDt; ++d) {
                    typedef short v4s_t __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;
                    const uint8_t* src = vsrc + 16 * ks * kRowV + 64 * d;
                    const v4s_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_v4s_t*)(__attribute__((address_space(3))) uint8_t*)src);
                    const v4s_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_v4s_t*)(__attribute__((address_space(3))) uint8_t*)(src + 8 * kRowV));
                    const h8_t av = __builtin_bit_cast(
                        h8_t, (short __attribute__((ext_vector_type(8)))){
                                  lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]});
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bh, acc[d], 0, 0, 0);
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bl, acc[d], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        tile_pok = pok;
        if (more) store_tile(t0 + kPfTile, b ^ 1);
        lds_barrier();  // every wave is done with this tile's buffer, and the next one's is written
    }

    if (__syncthreads_or(bad)) {
        // Rare: a V value past some column's causal length is not finite. Every column again, one
        // at a time, its masked positions left out.
        float* qv = (float*)(kbuf[0]) + wave * HD;
        for (int c = 0; c < 32 && 32 * wave + c < ncols; ++c) {
            const int c2 = 32 * wave + c, cq2 = c2 / G;
            const int64_t v2 = (int64_t)(q0 + cq2) * qh + g * G + (c2 - cq2 * G);
            float m, l, a[4];
            wave_attend(q + v2 * HD, table, pg, t_begin, min(t_end, qs.causal_len(q0 + cq2)), kvh, g,
                        HD, scale_log2 * 0.6931471805599453f, lane, qv, m, l, a);
            if (lane == 0 && !out) {  // in the units of the other splits' partials
                part_ml[(v2 * nsplit + split) * 2 + 0] = m;
                part_ml[(v2 * nsplit + split) * 2 + 1] = l * kPfScale;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = lane + 64 * i;
                if (d >= HD) continue;
                if (out)
                    out[v2 * HD + d] = (uint16_t)f2h(l > 0.0f ? a[i] / l : 0.0f);
                else
                    part_acc[(v2 * nsplit + split) * HD + d] = a[i] * kPfScale;
            }
        }
        return;
    }

    l_run += __shfl_xor(l_run, 32);
    if (!col_ok) return;
    if (out) {
#pragma unroll
        for (int d = 0; d < kDt; ++d)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                u32x2 w;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const float a0 = acc[d][4 * j + 2 * k], a1 = acc[d][4 * j + 2 * k + 1];
                    w[k] = l_run > 0.0f ? f2h(a0 / l_run) | (f2h(a1 / l_run) << 16) : 0u;
                }
                *(u32x2*)(out + vec * HD + 32 * d + 8 * j + 4 * half) = w;
            }
        return;
    }
    if (half == 0) {
        part_ml[(vec * nsplit + split) * 2 + 0] = m_run * 0.6931471805599453f;
        part_ml[(vec * nsplit + split) * 2 + 1] = l_run;
    }
    float* dst = part_acc + (vec * nsplit + split) * HD + 4 * half;
#pragma unroll
    for (int d = 0; d < kDt; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *(f4_t*)(dst + 32 * d + 8 * j) =
                f4_t{acc[d][4 * j], acc[d][4 * j + 1], acc[d][4 * j + 2], acc[d][4 * j + 3]};
}

// Any other head_dim (1 .. 256; the reference kernel takes any width): one wave per (query,
// q head, 1024-position split), same partials as paged_attn_split_kernel. A fallback for widths no
// model on this path uses at scale (the tiny test models' 16, odd widths): no MFMA, no vector
// loads.
constexpr int kGenWaves = 4;
template <class Pages>
__global__ __launch_bounds__(64 * kGenWaves) void paged_attn_generic_kernel(
    const uint16_t* __restrict__ q, PQueries qs, Pages pg, int qh, int kvh, int hd,
    float scale, float* __restrict__ part_ml, float* __restrict__ part_acc, int nsplit,
    int64_t items) {
    __shared__ float qbuf[kGenWaves][256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t item = (int64_t)blockIdx.x * kGenWaves + wave;
    if (item >= items) return;
    const int split = (int)(item % nsplit);
    const int64_t vec = item / nsplit;  // query qi, q head h
    const int qi = (int)(vec / qh), h = (int)(vec % qh);
    const int clen = qs.causal_len(qi);
    const int t_begin = split * kPSplit;
    if (t_begin >= clen) return;  // not read by the combine (splits below the length only)
    float m_run, l_run, acc[4];
    wave_attend(q + vec * hd, qs.table + (int64_t)qi * qs.table_stride, pg, t_begin,
                min(clen, t_begin + kPSplit), kvh, h / (qh / kvh), hd, scale, lane, qbuf[wave], m_run,
                l_run, acc);
    if (lane == 0) {
        part_ml[(vec * nsplit + split) * 2 + 0] = m_run;
        part_ml[(vec * nsplit + split) * 2 + 1] = l_run;
    }
    float* dst = part_acc + (vec * nsplit + split) * hd;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (lane + 64 * i < hd) dst[lane + 64 * i] = acc[i];
}

// Merge of the splits of one (query, q head) vector per workgroup:
// out = (sum_s w_s acc_s) / (sum_s w_s l_s), w_s = exp(m_s - max m); zeros when the query
// attends to no position. The split weights are computed once, in parallel, into LDS; each
// thread then sums its output dims over the splits with eight loads in flight at a time.
constexpr int kCombThreads = 128;
__global__ __launch_bounds__(kCombThreads) void paged_attn_combine_kernel(
    PQueries qs, const float* __restrict__ ml, const float* __restrict__ acc,
    uint16_t* __restrict__ out, int qh, int hd, int nsplit, int split_pos) {
    extern __shared__ float wts[];  // nsplit weights
    __shared__ float red[2][kCombThreads / kWave];
    const int64_t vec = blockIdx.x;
    const int qi = (int)(vec / qh);
    const int clen = qs.causal_len(qi);
    const int ns = (clen + split_pos - 1) / split_pos;
    const float* m = ml + vec * nsplit * 2;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    constexpr int kW = kCombThreads / kWave;
    float mx = -__builtin_inff();
    for (int s = tid; s < ns; s += kCombThreads) mx = fmaxf(mx, m[2 * s]);
    mx = wave_max(mx);
    if (lane == 0) red[0][wv] = mx;
    __syncthreads();
    float M = red[0][0];
#pragma unroll
    for (int w = 1; w < kW; ++w) M = fmaxf(M, red[0][w]);
    float ls = 0.0f;
    for (int s = tid; s < ns; s += kCombThreads) {
        const float w = M == -__builtin_inff() ? 0.0f : expf(m[2 * s] - M);
        wts[s] = w;
        ls += w * m[2 * s + 1];
    }
    ls = wave_sum(ls);
    if (lane == 0) red[1][wv] = ls;
    __syncthreads();
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < kW; ++w) L += red[1][w];
    const float* a = acc + vec * nsplit * hd;
    for (int d = tid; d < hd; d += kCombThreads) {
        float o = 0.0f;
        int s = 0;
        for (; s + 8 <= ns; s += 8) {
            float av[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) av[j] = a[(int64_t)(s + j) * hd + d];
#pragma unroll
            for (int j = 0; j < 8; ++j) o = fmaf(wts[s + j], av[j], o);
        }
        for (; s < ns; ++s) o = fmaf(wts[s], a[(int64_t)s * hd + d], o);
        out[vec * hd + d] = (uint16_t)f2h(L > 0.0f ? o / L : 0.0f);
    }
}

// The same merge for launches with at most 8 splits per vector (contexts up to 8192 positions; causal
// prefill): kLanes lanes per vector, 256 / kLanes vectors per workgroup. Lane s of the group holds split
// s's (m, l), the weights reach the dim loop by lane broadcasts: no LDS, no barrier. A workgroup per vector
// spent most of its time being scheduled at prefill sizes. Half a wave per vector, every lane loading
// 16 bytes of each split, from head_dim 128 on (32000 vectors of 2 splits, 1000 queries at 3001: the call
// 103.8 us, 108.9 with a wave per vector and 4-byte loads); below, half of those lanes would be idle, and
// a whole wave is the faster one (64 sequences of 100, 16 / 8 heads of 64: 11.4 us and 11.0).
constexpr int kCombWaveMaxSplits = 8;
template <int kLanes, int kVec>
__global__ __launch_bounds__(256) void paged_attn_combine_wave_kernel(
    PQueries qs, const float* __restrict__ ml, const float* __restrict__ acc,
    uint16_t* __restrict__ out, int qh, int hd, int nsplit, int64_t nvec, int split_pos) {
    typedef float vec_t __attribute__((ext_vector_type(kVec)));
    const int gl = threadIdx.x & (kLanes - 1), g0 = threadIdx.x & 63 & ~(kLanes - 1);
    const int64_t vec = (int64_t)blockIdx.x * (256 / kLanes) + threadIdx.x / kLanes;
    const bool live = vec < nvec;  // dead groups join the shuffles on vector 0's numbers
    const int64_t v = live ? vec : 0;
    const int clen = qs.causal_len((int)(v / qh));
    const int ns = (clen + split_pos - 1) / split_pos;  // <= nsplit <= kCombWaveMaxSplits
    const float* m = ml + v * nsplit * 2;
    const float ms = gl < ns ? m[2 * gl] : -__builtin_inff();
    const float ls = gl < ns ? m[2 * gl + 1] : 0.0f;
    float M = ms, L = 0.0f;
    if constexpr (kLanes == 64) {
        M = wave_max(ms);
    } else {
#pragma unroll
        for (int o = 4; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));  // lanes 0..7 of the group
        M = __shfl(M, g0);
    }
    const float w = gl < ns && M != -__builtin_inff() ? expf(ms - M) : 0.0f;
    float ws[kCombWaveMaxSplits];
#pragma unroll
    for (int j = 0; j < kCombWaveMaxSplits; ++j) ws[j] = __shfl(w, g0 + j);
    if constexpr (kLanes == 64) {
        L = wave_sum(w * ls);
    } else {
#pragma unroll
        for (int j = 0; j < kCombWaveMaxSplits; ++j) L += ws[j] * __shfl(ls, g0 + j);
    }
    if (!live) return;
    const float* a = acc + v * nsplit * hd;
    for (int d = kVec * gl; d < hd; d += kVec * kLanes) {
        vec_t av[kCombWaveMaxSplits];
#pragma unroll
        for (int j = 0; j < kCombWaveMaxSplits; ++j) av[j] = j < ns ? *(const vec_t*)(a + (int64_t)j * hd + d) : (vec_t)0.0f;
        float o[kVec];
#pragma unroll
        for (int k = 0; k < kVec; ++k) {
            o[k] = 0.0f;
#pragma unroll
            for (int j = 0; j < kCombWaveMaxSplits; ++j) o[k] = fmaf(ws[j], av[j][k], o[k]);
            o[k] = L > 0.0f ? o[k] / L : 0.0f;
        }
        if constexpr (kVec == 1) {
            out[v * hd + d] = (uint16_t)f2h(o[0]);
        } else {
            *(u32x2*)(out + v * hd + d) =
                u32x2{f2h(o[0]) | (f2h(o[1]) << 16), f2h(o[2]) | (f2h(o[3]) << 16)};
        }
    }
}

size_t paged_ws_layout(int nq, int qh, int hd, int max_tokens, size_t* off_acc, int* nsplit) {
    const int ns = max_tokens > 0 ? (max_tokens + kPSplit - 1) / kPSplit : 1;
    const size_t ml = (size_t)nq * qh * ns * 2 * sizeof(float);
    const size_t acc = (size_t)nq * qh * ns * hd * sizeof(float);
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    if (off_acc) *off_acc = al(ml);
    if (nsplit) *nsplit = ns;
    return al(ml) + al(acc);
}

// head_dim 32 / 64 / 128 / 256 run the MFMA kernels, any other width up to 256 the generic one
bool paged_shape_ok(int qh, int kvh, int hd) {
    return kvh > 0 && qh > 0 && qh % kvh == 0 && hd >= 1 && hd <= 256;
}

template <int HD, int NH, int W, class Pages>
void launch_split_w(const uint16_t* q, const PQueries& qs, const Pages& pg, int qh, int kvh,
                    int nhb, float* ml, float* acc, int nsplit, int tok, int64_t items,
                    hipStream_t s) {
    const float scale_log2 = 1.4426950408889634f / sqrtf((float)HD);
    const int64_t wgs = W == 1 ? ceil_div(items, 2) : items;
    hipLaunchKernelGGL((paged_attn_split_kernel<HD, NH, W, Pages>), dim3((unsigned)wgs),
                       dim3(64 * (W == 1 ? 2 : W)), 0, s, q, qs, pg, qh, kvh, nhb, scale_log2, ml, acc, nsplit,
                       tok);
}
template <int HD, int NH, class Pages>
void launch_split_t(const uint16_t* q, const PQueries& qs, const Pages& pg, int qh, int kvh,
                    int nhb, float* ml, float* acc, int nsplit, int tok, int64_t items,
                    hipStream_t s) {
    switch (fhip_rules::paged_waves(items, HD, qs.max_blocks * FHIP_PAGE_TOKENS)) {
        case 8: return launch_split_w<HD, NH, 8>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
        case 4: return launch_split_w<HD, NH, 4>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
        case 2: return launch_split_w<HD, NH, 2>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
        default: return launch_split_w<HD, NH, 1>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
    }
}

template <int HD, class Pages>
void launch_split_hd(const uint16_t* q, const PQueries& qs, const Pages& pg, int qh, int kvh,
                     int nhb, float* ml, float* acc, int nsplit, int tok, int64_t items,
                     hipStream_t s) {
    if (qh / kvh * tok <= 4)
        launch_split_t<HD, 4>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
    else
        launch_split_t<HD, 8>(q, qs, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
}

template <int HD, class Pages>
void launch_prefill_t(const uint16_t* q, const PQueries& qs, const Pages& pg, int qh, int kvh,
                      float* ml, float* acc, uint16_t* out, const fhip_rules::PrefillSplit& ps,
                      hipStream_t s) {
    const float scale_log2 = 1.4426950408889634f / sqrtf((float)HD);
    hipLaunchKernelGGL((paged_attn_prefill_mfma_kernel<HD, Pages>), dim3((unsigned)ps.workgroups),
                       dim3(64 * kPfWaves), 0, s, q, qs, pg, qh, kvh, scale_log2, ml, acc, out, ps.nsplit,
                       ps.split_pos, ps.nqb, ps.nblk);
}

// The merge of nsplit splits of split_pos positions per vector.
void launch_combine(const PQueries& qs, const float* ml, const float* acc, void* out, int64_t nvec,
                    int qh, int hd, int nsplit, int split_pos, hipStream_t s) {
    if (nsplit <= kCombWaveMaxSplits && hd % 128 == 0 && fhip_host::aligned16(acc) &&
        ((uintptr_t)out & 7) == 0)
        hipLaunchKernelGGL((paged_attn_combine_wave_kernel<32, 4>), dim3((unsigned)ceil_div(nvec, 8)),
                           dim3(256), 0, s, qs, ml, acc, (uint16_t*)out, qh, hd, nsplit, nvec,
                           split_pos);
    else if (nsplit <= kCombWaveMaxSplits)
        hipLaunchKernelGGL((paged_attn_combine_wave_kernel<64, 1>), dim3((unsigned)ceil_div(nvec, 4)),
                           dim3(256), 0, s, qs, ml, acc, (uint16_t*)out, qh, hd, nsplit, nvec,
                           split_pos);
    else
        hipLaunchKernelGGL(paged_attn_combine_kernel, dim3((unsigned)nvec), dim3(kCombThreads),
                           (size_t)nsplit * sizeof(float), s, qs, ml, acc, (uint16_t*)out, qh, hd,
                           nsplit, split_pos);
}

template <class Pages>
int launch_paged(void* out, const void* q, const PQueries& qs, int nq, const Pages& pg, int qh,
                 int kvh, int hd, void* ws, hipStream_t s) {
    if (nq == 0) return hipSuccess;
    size_t off_acc;
    int nsplit;
    paged_ws_layout(nq, qh, hd, qs.max_blocks * FHIP_PAGE_TOKENS, &off_acc, &nsplit);
    float* ml = (float*)ws;
    float* acc = (float*)((char*)ws + off_acc);
    const int G = qh / kvh;
    const int nhb = (G + kHeadsMax - 1) / kHeadsMax;
    const int64_t nvec = (int64_t)nq * qh;
    PQueries q2 = qs;
    q2.count = nq;
    const uint16_t* qp = (const uint16_t*)q;
    // causal prefill over one shared table: kPfCols / G consecutive queries per workgroup on the
    // MFMA prefill kernel (head_dim <= 128, G <= 8), else 8 / G per wave (G < 8)
    const bool prefill = !qs.seq_lens && qs.table_stride == 0 && nq > 1;
    if (prefill && (hd == 32 || hd == 64 || hd == 128) && G <= kHeadsMax) {
        // Splits only as far as the workgroups need to fill the chip (kPfGroups: 768 or 1024
        // measured 129 and 120 us where 512 took 114), at most the
        // workspace's one per kPSplit positions: every split adds partials to write and merge. A single
        // split writes the output itself, 8 bytes a lane, where it is aligned to them.
        const int extent = (int)std::min<int64_t>(qs.kv_len, (int64_t)qs.max_blocks * FHIP_PAGE_TOKENS);
        const fhip_rules::PrefillSplit ps =
            fhip_rules::prefill_split(nq, G, kvh, kPfCols, kPfTile, kPfGroups, extent, nsplit);
        if (ps.workgroups > 0x7fffffff || nvec > 0x7fffffff) return hipErrorInvalidValue;
        uint16_t* direct = ps.nsplit == 1 && ((uintptr_t)out & 7) == 0 ? (uint16_t*)out : nullptr;
        switch (hd) {
            case 32:
                launch_prefill_t<32>(qp, q2, pg, qh, kvh, ml, acc, direct, ps, s);
                break;
            case 64:
                launch_prefill_t<64>(qp, q2, pg, qh, kvh, ml, acc, direct, ps, s);
                break;
            default:
                launch_prefill_t<128>(qp, q2, pg, qh, kvh, ml, acc, direct, ps, s);
                break;
        }
        if (!direct) launch_combine(q2, ml, acc, out, nvec, qh, hd, ps.nsplit, ps.split_pos, s);
        return hipGetLastError();
    }
    const int tok = prefill && G < kHeadsMax ? kHeadsMax / G : 1;
    const int64_t items = ceil_div((int64_t)nq, tok) * kvh * nhb * nsplit;
    if (items > 0x7fffffff || nvec > 0x7fffffff) return hipErrorInvalidValue;
    if (hd != 32 && hd != 64 && hd != 128 && hd != 256) {
        const int64_t gitems = (int64_t)nq * qh * nsplit;
        const int64_t gwgs = ceil_div(gitems, kGenWaves);
        if (gwgs > 0x7fffffff) return hipErrorInvalidValue;
        hipLaunchKernelGGL((paged_attn_generic_kernel<Pages>), dim3((unsigned)gwgs),
                           dim3(64 * kGenWaves), 0, s, qp, q2, pg, qh, kvh, hd,
                           1.0f / sqrtf((float)hd), ml, acc, nsplit, gitems);
    } else {
    switch (hd) {
        case 32:
            launch_split_hd<32>(qp, q2, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
            break;
        case 64:
            launch_split_hd<64>(qp, q2, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
            break;
        case 128:
            launch_split_hd<128>(qp, q2, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
            break;
        default:
            launch_split_hd<256>(qp, q2, pg, qh, kvh, nhb, ml, acc, nsplit, tok, items, s);
            break;
    }
    }
    launch_combine(q2, ml, acc, out, nvec, qh, hd, nsplit, kPSplit, s);
    return hipGetLastError();
}

}  // namespace

extern "C" {

size_t fhip_attention_paged_workspace_bytes(int batch, int num_q_heads, int head_dim,
                                            int max_blocks) {
    if (batch <= 0 || num_q_heads <= 0 || head_dim <= 0 || max_blocks <= 0) return 0;
    return paged_ws_layout(batch, num_q_heads, head_dim, max_blocks * FHIP_PAGE_TOKENS, nullptr,
                           nullptr);
}

int fhip_launch_attention_paged_decode(void* output, const void* q, const int32_t* block_table,
                                       const int32_t* seq_lens, int batch, int max_blocks,
                                       int num_pages, const void* k_pool, const void* v_pool,
                                       int64_t page_k_bytes, int64_t page_v_bytes,
                                       int num_q_heads, int num_kv_heads, int head_dim,
                                       void* workspace, fhip_stream_t stream) {
    if (batch < 0 || max_blocks <= 0 || num_pages < 0 || page_k_bytes < 0 || page_v_bytes < 0 ||
        !paged_shape_ok(num_q_heads, num_kv_heads, head_dim) ||
        (int64_t)max_blocks * FHIP_PAGE_TOKENS > kMaxTokens)
        return hipErrorInvalidValue;
    if (batch == 0) return hipSuccess;
    if (!output || !q || !block_table || !seq_lens || !k_pool || !v_pool || !workspace)
        return hipErrorInvalidValue;
    const PQueries qs{block_table, max_blocks, max_blocks, seq_lens, 0, 0, batch};
    const F16PoolPages pg{(const uint8_t*)k_pool, (const uint8_t*)v_pool, page_k_bytes,
                          page_v_bytes, num_pages};
    return launch_paged(output, q, qs, batch, pg, num_q_heads, num_kv_heads, head_dim, workspace,
                        fhip_host::as_stream(stream));
}

// The reference interface: one sequence, num_tokens queries at positions
// start_pos .. start_pos + num_tokens - 1, per-block pointer arrays indexed by the physical
// block ids of block_table[0 .. num_blocks_in_seq). `ws` holds the split partials
// (fhip_attention_paged_workspace_bytes(num_tokens, qh, hd, num_blocks_in_seq) bytes); null
// asks for a stream-ordered allocation freed on the same stream.
static int paged_attention_ref(void* output, const void* q, const int* block_table,
                               const void** k_block_ptrs, const void** v_block_ptrs,
                               int num_tokens, int num_q_heads, int num_kv_heads, int head_dim,
                               int kv_len, int start_pos, int num_blocks_in_seq, void* ws,
                               size_t ws_bytes, hipStream_t s) {
    if (num_tokens < 0 || kv_len < 0 || start_pos < 0 || num_blocks_in_seq < 0 ||
        !paged_shape_ok(num_q_heads, num_kv_heads, head_dim) ||
        (int64_t)num_blocks_in_seq * FHIP_PAGE_TOKENS > kMaxTokens)
        return hipErrorInvalidValue;
    if (num_tokens == 0) return hipSuccess;
    if (!output || !q) return hipErrorInvalidValue;
    if (num_blocks_in_seq > 0 && (!block_table || !k_block_ptrs || !v_block_ptrs))
        return hipErrorInvalidValue;
    const int mb = num_blocks_in_seq > 0 ? num_blocks_in_seq : 1;
    // with no blocks every query attends to nothing: the table is never read
    const PQueries qs{(const int32_t*)block_table, 0, num_blocks_in_seq, nullptr, kv_len,
                      start_pos, num_tokens};
    const size_t bytes = paged_ws_layout(num_tokens, num_q_heads, head_dim,
                                         mb * FHIP_PAGE_TOKENS, nullptr, nullptr);
    const bool own = ws == nullptr;
    if (!own && ws_bytes < bytes) return hipErrorInvalidValue;
    if (own) {
        hipError_t e = hipMallocAsync(&ws, bytes, s);
        if (e != hipSuccess) return e;
    }
    const F16PtrPages pg{(const uint8_t* const*)k_block_ptrs, (const uint8_t* const*)v_block_ptrs,
                         0x7fffffff};
    int r = launch_paged(output, q, qs, num_tokens, pg, num_q_heads, num_kv_heads, head_dim, ws,
                         s);
    if (own) {
        hipError_t e2 = hipFreeAsync(ws, s);
        if (r == hipSuccess) r = e2;
    }
    return r;
}

int fhip_launch_paged_attention(void* output, const void* q, const int* block_table,
                                const void** k_block_ptrs, const void** v_block_ptrs,
                                int num_tokens, int num_q_heads, int num_kv_heads, int head_dim,
                                int kv_len, int start_pos, int num_blocks_in_seq,
                                fhip_stream_t stream) {
    return paged_attention_ref(output, q, block_table, k_block_ptrs, v_block_ptrs, num_tokens,
                               num_q_heads, num_kv_heads, head_dim, kv_len, start_pos,
                               num_blocks_in_seq, nullptr, 0, fhip_host::as_stream(stream));
}

int fhip_launch_paged_attention_ws(void* output, const void* q, const int* block_table,
                                   const void** k_block_ptrs, const void** v_block_ptrs,
                                   int num_tokens, int num_q_heads, int num_kv_heads,
                                   int head_dim, int kv_len, int start_pos,
                                   int num_blocks_in_seq, void* workspace,
                                   size_t workspace_bytes, fhip_stream_t stream) {
    if (!workspace) return hipErrorInvalidValue;
    return paged_attention_ref(output, q, block_table, k_block_ptrs, v_block_ptrs, num_tokens,
                               num_q_heads, num_kv_heads, head_dim, kv_len, start_pos,
                               num_blocks_in_seq, workspace, workspace_bytes,
                               fhip_host::as_stream(stream));
}

// ffi.rs:172-184 `launch_attention`, attention over a contiguous KV cache: not supported. The
// engine's KV caches are paged (engine.rs:671-680 dispatches through the cache manager to the
// paged forms above), so this backend builds only those; the symbol exists so that a binding of
// the whole ffi.rs block links, and it launches nothing.
int fhip_launch_attention(void* output, const void* q, const void* k_cache, const void* v_cache,
                          int num_tokens, int num_q_heads, int num_kv_heads, int head_dim,
                          int kv_len, int start_pos, fhip_stream_t stream) {
    (void)output, (void)q, (void)k_cache, (void)v_cache, (void)num_tokens, (void)num_q_heads;
    (void)num_kv_heads, (void)head_dim, (void)kv_len, (void)start_pos, (void)stream;
    return hipErrorNotSupported;
}

}  // extern "C"
