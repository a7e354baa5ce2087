// GQA decode attention over a TurboQuant-compressed paged KV cache, for gfx950.
//
// Semantics follow attention_paged_tq.cu:56-257: the query is pre-rotated with Pi_k
// (scores in the rotated K space, dot(q, Pi_k^T y) = dot(Pi_k q, y)), the score of
// position t is (sum_d q_rot[d] * ck[idx_td]) * (norm_k * head_dim^-1/2), causal length
// min(start_pos + t + 1, kv_len), softmax over the positions, V accumulated in the rotated
// V space as sum p * cv[idx] * norm_v, and the output unrotated once with Pi_v^T.
//
// Layout on MI355X: the reference keeps a kv_len-float score row in shared memory
// (attention_paged_tq.cu:287-289), which caps the context; here each workgroup takes one
// (query, kv head, 1024-token split) and all q heads of the kv head's GQA group, so every
// K/V code byte crosses HBM once per group, and keeps an online (max, sum, acc) per head.
// A combine kernel merges the splits and applies Pi_v^T. Three launches in all:
//   1. q_rot = Pi_k q                  (per query head)
//   2. split partials                  (the HBM stream over the pages)
//   3. merge + unrotate -> fp16 output
#include <algorithm>
#include <type_traits>

#include "fhip_internal.h"
#include "launch_rules.h"
#include "tq_attn_index.h"
#include "tq_quant.h"

using namespace fhip;

namespace {

constexpr int kSplit = fhip_rules::kTqSplit;        // positions per split workgroup
constexpr int kFinePart = fhip_rules::kTqFinePart;  // and in small launches
constexpr int kSub = 256;      // positions per pass (one per lane in the score phase)
constexpr int kMaxG = 8;       // q heads per kv head
constexpr int kMaxHd = 256;
constexpr int kMaxPd = 256;    // packed bytes per head row (hd * bits / 8)

// Page sources: per-page pointer arrays (the reference's interface) or contiguous pools.
struct PtrPages {
    const uint8_t* const* kp;
    const uint8_t* const* kn;
    const uint8_t* const* vp;
    const uint8_t* const* vn;
    int num_pages;  // entries of the pointer arrays
    __device__ bool valid(int p) const { return p >= 0 && p < num_pages; }
    __device__ const uint8_t* kpage(int p) const { return kp[p]; }
    __device__ const uint8_t* knorm(int p) const { return kn[p]; }
    __device__ const uint8_t* vpage(int p) const { return vp[p]; }
    __device__ const uint8_t* vnorm(int p) const { return vn[p]; }
    // The four part addresses of page p (p valid).
    __device__ void addrs(int p, const uint8_t*& k, const uint8_t*& knp, const uint8_t*& v,
                          const uint8_t*& vnp) const {
        k = kp[p];
        knp = kn[p];
        v = vp[p];
        vnp = vn[p];
    }
};
struct PoolPages {
    const uint8_t* kp;
    const uint8_t* kn;
    const uint8_t* vp;
    const uint8_t* vn;
    int64_t skp, skn, svp, svn;
    int num_pages;
    __device__ bool valid(int p) const { return p >= 0 && p < num_pages; }
    __device__ const uint8_t* kpage(int p) const { return kp + p * skp; }
    __device__ const uint8_t* knorm(int p) const { return kn + p * skn; }
    __device__ const uint8_t* vpage(int p) const { return vp + p * svp; }
    __device__ const uint8_t* vnorm(int p) const { return vn + p * svn; }
    __device__ void addrs(int p, const uint8_t*& k, const uint8_t*& knp, const uint8_t*& v,
                          const uint8_t*& vnp) const {
        k = kpage(p);
        knp = knorm(p);
        v = vpage(p);
        vnp = vnorm(p);
    }
};

// Query q_i reads block-table row i (stride 0: one shared table) and attends to
// seq_lens[i] positions, or min(start_pos + i + 1, kv_len) when seq_lens is null.
struct Queries {
    const int32_t* table;
    int64_t table_stride;
    int max_blocks;
    const int32_t* seq_lens;
    int kv_len, start_pos;
    int seq_lens_count;  // number of queries (set by the MFMA launcher)
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

// Byte k of a row held as little-endian 32-bit words.
__device__ __forceinline__ uint32_t row_byte(const uint32_t* w, int k) {
    return (w[k >> 2] >> (8 * (k & 3))) & 0xffu;
}
template <int B>
__device__ __forceinline__ void row_group(const uint32_t* w, int g, int bits_rt, int (&codes)[8]) {
    const int bits = B > 0 ? B : bits_rt;
    uint64_t word;
    if (B == 4) {
        word = __builtin_bswap32(w[g]);
    } else if (B == 8) {
        word = ((uint64_t)__builtin_bswap32(w[2 * g]) << 32) | __builtin_bswap32(w[2 * g + 1]);
    } else {
        word = 0;
        for (int k = 0; k < bits; ++k) word = (word << 8) | row_byte(w, g * bits + k);
    }
    const uint32_t mask = (1u << bits) - 1u;
#pragma unroll
    for (int i = 0; i < 8; ++i) codes[i] = (int)((word >> (bits * (7 - i))) & mask);
}

// 1. q_rot[v, :] = Pi_k q[v, :] (fp32 dots in coordinate order, attention_paged_tq.cu:102-113).
// A workgroup rotates kRotVecs vectors so Pi_k is read once per workgroup: work unit
// (row i, half) computes row i of vectors 4 half .. 4 half + 3.
constexpr int kRotVecs = 8;
constexpr int kMfmaRotVecs = fhip_rules::kRotBatch;  // from this many query vectors on, batched MFMA rotations
__global__ __launch_bounds__(256) void tq_attn_prerotate_kernel(const uint16_t* __restrict__ q,
                                                                const float* __restrict__ rot,
                                                                float* __restrict__ qrot, int hd,
                                                                int nvec) {
    __shared__ float qs[kRotVecs][kMaxHd];
    const int v0 = blockIdx.x * kRotVecs;
    {
        // every load is issued before the first is waited for: vectors past nvec read
        // vector 0 (in bounds) and are zeroed
        constexpr int kPer = kRotVecs * kMaxHd / 256;
        uint16_t raw[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int e = threadIdx.x + k * 256;
            const int v = e / hd, j = e - v * hd;
            const int64_t src = e < kRotVecs * hd && v0 + v < nvec ? (int64_t)(v0 + v) * hd + j : 0;
            raw[k] = q[src];
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int e = threadIdx.x + k * 256;
            const int v = e / hd, j = e - v * hd;
            if (e < kRotVecs * hd) qs[v][j] = v0 + v < nvec ? h2f(raw[k]) : 0.0f;
        }
    }
    __syncthreads();
    for (int r = threadIdx.x; r < 2 * hd; r += blockDim.x) {
        const int i = r % hd, vb = 4 * (r / hd);
        const float* pr = rot + (int64_t)i * hd;
        float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int j = 0; j < hd; ++j) {
            const float rv = pr[j];
#pragma unroll
            for (int k = 0; k < 4; ++k) dot[k] += rv * qs[vb + k][j];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (v0 + vb + k < nvec) qrot[(int64_t)(v0 + vb + k) * hd + i] = dot[k];
    }
}

// The same at head_dim 128: 4 vectors per workgroup of 512 lanes, lane (row i, quarter jq) holding 32
// coordinates of Pi_k's row i, read as eight 16-byte loads that are all in flight with the vectors'
// own; the quarters are summed by DPP. The general kernel walks a row of 128 loads a lane, one
// latency after another, over half the workgroups: 6.4 us for 32 vectors and 9.9 for 2048 against
// 4.5 and 8.4 here (kernel trace; a kernel that does nothing takes 2).
constexpr int kRot128Vecs = 4;
__global__ __launch_bounds__(512) void tq_attn_prerotate128_kernel(const uint16_t* __restrict__ q,
                                                                   const float* __restrict__ rot,
                                                                   float* __restrict__ qrot, int nvec) {
    __shared__ __attribute__((aligned(16))) float qs[kRot128Vecs][4][36];  // quarters on distinct banks
    const int v0 = blockIdx.x * kRot128Vecs;
    const int tid = threadIdx.x, i = tid >> 2, jq = tid & 3;
    f32x4 r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = *(const f32x4*)(rot + 128 * i + 32 * jq + 4 * k);
    const int lv = tid >> 7, lj = tid & 127;
    const uint16_t raw = v0 + lv < nvec ? q[(int64_t)(v0 + lv) * 128 + lj] : 0;
    qs[lv][lj >> 5][lj & 31] = h2f(raw);
    __syncthreads();
    float mine = 0.0f;
#pragma unroll
    for (int v = 0; v < kRot128Vecs; ++v) {
        float dot = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const f32x4 x = *(const f32x4*)&qs[v][jq][4 * k];
#pragma unroll
            for (int e = 0; e < 4; ++e) dot = fmaf(r[k][e], x[e], dot);
        }
        dot += __builtin_amdgcn_update_dpp(0.0f, dot, 0xB1, 0xF, 0xF, true);  // lane ^ 1
        dot += __builtin_amdgcn_update_dpp(0.0f, dot, 0x4E, 0xF, 0xF, true);  // lane ^ 2
        mine = v == jq ? dot : mine;
    }
    if (v0 + jq < nvec) qrot[(int64_t)(v0 + jq) * 128 + i] = mine;
}

// 2. One (split, kv head, query) per workgroup of 256 lanes. Each pass of 256 positions
// stages the positions' packed K and V rows in LDS (row stride padded to an odd number of
// words, so lanes reading different rows hit different banks), scores them one position per
// lane against the group's rotated queries, updates the online softmax, then accumulates V
// with lanes mapped to (8-coordinate code group, position slice).
template <int KB, int VB, class Pages>
__global__ __launch_bounds__(256) void tq_attn_split_kernel(
    const float* __restrict__ qrot, Queries qs, Pages pg, const float* __restrict__ kcent,
    const float* __restrict__ vcent, int kbits_rt, int vbits_rt, int qh, int kvh, int hd,
    float scale, float* __restrict__ part_ml, float* __restrict__ part_acc, int nsplit) {
    int split, kvhead, qi;  // grid (nsplit, kvh, queries), placed on the XCDs by split_grid_item
    fhip_idx::split_grid_item(
        blockIdx.x + (int64_t)gridDim.x * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z),
        (int64_t)gridDim.x * gridDim.y * gridDim.z, nsplit, kvh, split, kvhead, qi);
    const int clen = qs.causal_len(qi);
    const int t0 = split * kSplit;
    if (t0 >= clen) return;
    const int t1 = min(clen, t0 + kSplit);
    const int kbits = KB > 0 ? KB : kbits_rt, vbits = VB > 0 ? VB : vbits_rt;
    const int G = qh / kvh;
    const int pdk = (hd * kbits + 7) / 8, pdv = (hd * vbits + 7) / 8;
    const int kwords = (pdk + 3) / 4, vwords = (pdv + 3) / 4;
    const int ks = kwords | 1, vs = vwords | 1;  // odd LDS row strides
    const int NG = hd / 8;          // code groups per row
    const int NS = 256 / NG;        // position slices in the PV phase
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    __shared__ float kc[kMaxLevels], vc[kMaxLevels];
    __shared__ float qr[kMaxG * kMaxHd];
    __shared__ float w[kSub * kMaxG];            // p * norm_v, [pos][head]
    __shared__ float red[4][kMaxG];
    __shared__ float accbuf[kMaxG * kMaxHd];
    extern __shared__ uint32_t dyn[];
    uint32_t* krows = dyn;                        // [kSub][ks]
    uint32_t* vrows = dyn + kSub * ks;            // [kSub][vs]

    for (int i = tid; i < (1 << kbits); i += 256) kc[i] = kcent[i];
    for (int i = tid; i < (1 << vbits); i += 256) vc[i] = vcent[i];
    const float* qsrc = qrot + ((int64_t)qi * qh + (int64_t)kvhead * G) * hd;
    for (int i = tid; i < G * hd; i += 256) qr[i] = qsrc[i];
    const int32_t* table = qs.table + (int64_t)qi * qs.table_stride;

    float m_run[kMaxG], l_run[kMaxG];
    float acc[kMaxG][8];
#pragma unroll
    for (int h = 0; h < kMaxG; ++h) {
        m_run[h] = -__builtin_inff();
        l_run[h] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = 0.0f;
    }
    const int my_group = tid % NG, my_slice = tid / NG;
    __syncthreads();

    for (int sub = t0; sub < t1; sub += kSub) {
        // ---- stage this lane's position: packed K / V rows into LDS
        const int pos = sub + tid;
        bool valid = pos < t1;
        const int page = valid ? table[pos / FHIP_PAGE_TOKENS] : -1;
        valid = valid && pg.valid(page);
        const int slot = pos % FHIP_PAGE_TOKENS;
        const int64_t row = (int64_t)slot * kvh + kvhead;
        float knorm = 0.0f, vnorm = 0.0f;
        uint32_t* kdst = krows + tid * ks;
        uint32_t* vdst = vrows + tid * vs;
        if (valid) {
            const uint8_t* kr = pg.kpage(page) + row * pdk;
            const uint8_t* vr = pg.vpage(page) + row * pdv;
            if ((pdk & 15) == 0 && (((uintptr_t)kr) & 15u) == 0) {
                for (int i = 0; i < kwords; i += 4) {
                    const u32x4 x = ld16(kr + 4 * i);
                    kdst[i] = x[0]; kdst[i + 1] = x[1]; kdst[i + 2] = x[2]; kdst[i + 3] = x[3];
                }
            } else {
                for (int i = 0; i < kwords; ++i) {
                    uint32_t x = 0;
                    for (int b = 0; b < 4; ++b)
                        if (4 * i + b < pdk) x |= (uint32_t)kr[4 * i + b] << (8 * b);
                    kdst[i] = x;
                }
            }
            if ((pdv & 15) == 0 && (((uintptr_t)vr) & 15u) == 0) {
                for (int i = 0; i < vwords; i += 4) {
                    const u32x4 x = ld16(vr + 4 * i);
                    vdst[i] = x[0]; vdst[i + 1] = x[1]; vdst[i + 2] = x[2]; vdst[i + 3] = x[3];
                }
            } else {
                for (int i = 0; i < vwords; ++i) {
                    uint32_t x = 0;
                    for (int b = 0; b < 4; ++b)
                        if (4 * i + b < pdv) x |= (uint32_t)vr[4 * i + b] << (8 * b);
                    vdst[i] = x;
                }
            }
            knorm = h2f(((const uint16_t*)pg.knorm(page))[row]);
            vnorm = h2f(((const uint16_t*)pg.vnorm(page))[row]);
        } else {
            for (int i = 0; i < vwords; ++i) vdst[i] = 0u;
        }

        // ---- scores: lane = position (its own K row, so no barrier needed yet)
        float s[kMaxG];
#pragma unroll
        for (int h = 0; h < kMaxG; ++h) s[h] = -__builtin_inff();
        if (valid) {
            float dot[kMaxG];
#pragma unroll
            for (int h = 0; h < kMaxG; ++h) dot[h] = 0.0f;
            for (int g = 0; g < NG; ++g) {
                int codes[8];
                row_group<KB>(kdst, g, kbits, codes);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float cv = kc[codes[e]];
                    const int d = 8 * g + e;
#pragma unroll
                    for (int h = 0; h < kMaxG; ++h)
                        if (h < G) dot[h] += qr[h * hd + d] * cv;
                }
            }
            const float f = knorm * scale;
#pragma unroll
            for (int h = 0; h < kMaxG; ++h) s[h] = dot[h] * f;
        }

        // ---- online softmax update per head
        float alpha[kMaxG], mnew[kMaxG];
#pragma unroll
        for (int h = 0; h < kMaxG; ++h) {
            if (h >= G) break;
            const float mx = wave_max(s[h]);
            if (lane == 0) red[wave][h] = mx;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < kMaxG; ++h) {
            if (h >= G) break;
            const float cm = fmaxf(fmaxf(red[0][h], red[1][h]), fmaxf(red[2][h], red[3][h]));
            mnew[h] = fmaxf(m_run[h], cm);
            alpha[h] = m_run[h] == -__builtin_inff() ? 0.0f : expf(m_run[h] - mnew[h]);
        }
        __syncthreads();  // red[] reused below
#pragma unroll
        for (int h = 0; h < kMaxG; ++h) {
            if (h >= G) break;
            const float p = valid ? expf(s[h] - mnew[h]) : 0.0f;
            w[tid * kMaxG + h] = p * vnorm;
            const float ps = wave_sum(p);
            if (lane == 0) red[wave][h] = ps;
        }
        __syncthreads();  // also publishes w[] and vrows[]
#pragma unroll
        for (int h = 0; h < kMaxG; ++h) {
            if (h >= G) break;
            l_run[h] = l_run[h] * alpha[h] + (red[0][h] + red[1][h] + red[2][h] + red[3][h]);
            m_run[h] = mnew[h];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[h][e] *= alpha[h];
        }

        // ---- PV: lane = (code group, position slice)
        const int npos = min(kSub, t1 - sub);
        for (int tk = my_slice; tk < npos; tk += NS) {
            int codes[8];
            row_group<VB>(vrows + tk * vs, my_group, vbits, codes);
            float cv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) cv[e] = vc[codes[e]];
#pragma unroll
            for (int h = 0; h < kMaxG; ++h) {
                if (h >= G) break;
                const float wv = w[tk * kMaxG + h];
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[h][e] += wv * cv[e];
            }
        }
        __syncthreads();  // w / rows / red reused by the next pass
    }

    // ---- merge the position slices in a fixed order, write the split's partials
    for (int i = tid; i < G * hd; i += 256) accbuf[i] = 0.0f;
    __syncthreads();
    for (int sl = 0; sl < NS; ++sl) {
        if (my_slice == sl) {
#pragma unroll
            for (int h = 0; h < kMaxG; ++h) {
                if (h >= G) break;
#pragma unroll
                for (int e = 0; e < 8; ++e) accbuf[h * hd + 8 * my_group + e] += acc[h][e];
            }
        }
        __syncthreads();
    }
    const int64_t head0 = (int64_t)qi * qh + (int64_t)kvhead * G;
    for (int i = tid; i < G * hd; i += 256) {
        const int h = i / hd, d = i - h * hd;
        part_acc[((head0 + h) * nsplit + split) * hd + d] = accbuf[i];
    }
    if (tid < G) {
        part_ml[((head0 + tid) * nsplit + split) * 2 + 0] = m_run[tid];
        part_ml[((head0 + tid) * nsplit + split) * 2 + 1] = l_run[tid];
    }
}

// Merge the splits of kCombHeads consecutive (query, head) vectors per workgroup and apply
// Pi_v^T: out = Pi_v^T (sum_s w_s acc_s) / (sum_s w_s l_s), w_s = exp(m_s - max m). The work
// is a few dependent memory round trips, so each phase issues its loads together:
//   the rotation (hd x hd fp32) is staged in LDS first, overlapping the rest (kRotLds; for
//            head_dim above kRotLdsMaxHd it does not fit LDS and phase 3 reads it from L2);
//   phase 1: a half-wave per vector loads its splits' (m, l) once and folds them into
//            weights (LDS) and 1 / L;
//   phase 2: the weighted split sums, four (vector, coordinate) items per thread, sixteen
//            splits per step, each item summed in split order;
//   phase 3: the matvec, one output coordinate for 4 vectors per thread and step.
// Dynamic LDS: hd * hd rotation floats (kRotLds), then kCombHeads * nsplit weights.
constexpr int kCombHeads = 4;  // two workgroups per CU at the decode workload's 2048 vectors
constexpr int kRotLdsMaxHd = 128;
constexpr int kMaxTokensTq = kSplit * kSplit;  // 1024 splits: 32 KB of combine weights
size_t combine_lds_bytes(int hd, int nsplit, bool merge_only = false) {
    return ((hd <= kRotLdsMaxHd && !merge_only ? (size_t)hd * hd : 0) + (size_t)kCombHeads * nsplit) *
           sizeof(float);
}
// The merge alone with one wave per vector, four vectors per workgroup, when a vector has at
// most 8 splits (contexts up to 8192 positions; causal prefill): lane s holds split s's
// (m, l), the weights reach the dim loop by lane broadcasts, and each merged vector (fp32,
// divided by its sum) goes to merged[vector]. The combine kernel's 16-split load batches
// would be mostly clamped repeats at these sizes.
constexpr int kMergeWaveMaxSplits = fhip_rules::kMergeSplits;
__global__ __launch_bounds__(256) void tq_attn_merge_wave_kernel(
    Queries qs, const float* __restrict__ part_ml, const float* __restrict__ part_acc, int qh,
    int hd, int nsplit, int64_t nvec, float* __restrict__ merged, int split_pos) {
    const int lane = threadIdx.x & 63;
    const int64_t vec = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (vec >= nvec) return;
    const int clen = qs.causal_len((int)(vec / qh));
    const int ns = (clen + split_pos - 1) / split_pos;  // <= nsplit <= kMergeWaveMaxSplits
    const float* ml = part_ml + vec * nsplit * 2;
    const float ms = lane < ns ? ml[2 * lane] : -__builtin_inff();
    const float ls = lane < ns ? ml[2 * lane + 1] : 0.0f;
    const float M = wave_max(ms);
    const float w = lane < ns && ms != -__builtin_inff() ? expf(ms - M) : 0.0f;
    const float L = wave_sum(w * ls);
    const float linv = L > 0.0f ? 1.0f / L : 0.0f;
    float ws[kMergeWaveMaxSplits];
#pragma unroll
    for (int j = 0; j < kMergeWaveMaxSplits; ++j) ws[j] = __shfl(w, j);
    const float* a = part_acc + vec * nsplit * hd;
    for (int d = lane; d < hd; d += 64) {
        float av[kMergeWaveMaxSplits];
#pragma unroll
        for (int j = 0; j < kMergeWaveMaxSplits; ++j) av[j] = j < ns ? a[(int64_t)j * hd + d] : 0.0f;
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < kMergeWaveMaxSplits; ++j) sum = fmaf(av[j], ws[j], sum);
        merged[vec * hd + d] = sum * linv;
    }
}

// kMergeOnly: phase 2 writes each merged vector (fp32, already divided by its sum) to
// merged[vector] and the kernel ends; the unrotation then runs as a batched MFMA product.
template <bool kRotLds, bool kMergeOnly = false>
__global__ __launch_bounds__(256) void tq_attn_combine_kernel(
    Queries qs, const float* __restrict__ part_ml, const float* __restrict__ part_acc,
    const float* __restrict__ vrot, uint16_t* __restrict__ out, int qh, int hd, int nsplit,
    int64_t nvec, float* __restrict__ merged, int split_pos) {
    __shared__ float o[kCombHeads][kMaxHd];
    __shared__ float linv[kCombHeads];
    __shared__ int nsv[kCombHeads];
    extern __shared__ uint32_t dyn[];
    float* rl = (float*)dyn;                                  // [hd][hd] (kRotLds)
    float* wts = (float*)dyn + (kRotLds && !kMergeOnly ? hd * hd : 0);  // [kCombHeads][nsplit]
    const float* rot = kRotLds ? (const float*)rl : vrot;
    const int tid = threadIdx.x;
    const int64_t h0 = (int64_t)blockIdx.x * kCombHeads;
    if (kRotLds && !kMergeOnly) {   // the rotation into LDS: hd * hd / 4 16-byte chunks, all loads first
        const int n16 = hd * hd / 4;
        for (int c0 = tid; c0 < n16; c0 += 16 * 256) {
            u32x4 v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = ld16(vrot + 4 * min(c0 + u * 256, n16 - 1));
#pragma unroll
            for (int u = 0; u < 16; ++u) *(u32x4*)&rl[4 * min(c0 + u * 256, n16 - 1)] = v[u];
        }
    }
    {
        // a half-wave per vector (the half-waves past kCombHeads only join the shuffles)
        const int hh = min(tid >> 5, kCombHeads - 1), l32 = tid & 31;
        const bool mine = (tid >> 5) < kCombHeads;
        const int64_t head = h0 + hh;
        int ns = 0;
        if (mine && head < nvec) {
            const int clen = qs.causal_len((int)(head / qh));
            ns = (clen + split_pos - 1) / split_pos;
        }
        const float* ml = part_ml + head * nsplit * 2;
        float M = -__builtin_inff();
        for (int sp = l32; sp < ns; sp += 32) M = fmaxf(M, ml[2 * sp]);
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
        float L = 0.0f;
        for (int sp = l32; sp < ns; sp += 32) {
            const float m = ml[2 * sp];
            const float w = (m == -__builtin_inff()) ? 0.0f : expf(m - M);
            wts[hh * nsplit + sp] = w;
            L += ml[2 * sp + 1] * w;
        }
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) L += __shfl_xor(L, off);
        if (mine && l32 == 0) {
            linv[hh] = L > 0.0f ? 1.0f / L : 0.0f;
            nsv[hh] = ns;
        }
    }
    __syncthreads();
    for (int idx0 = tid; idx0 < kCombHeads * hd; idx0 += 4 * 256) {
        const float* a[4];
        int hh[4], ns[4];
        float sum[4];
        int nsmax = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int idx = min(idx0 + k * 256, kCombHeads * hd - 1);
            hh[k] = idx / hd;
            const int d = idx - hh[k] * hd;
            ns[k] = idx0 + k * 256 < kCombHeads * hd ? nsv[hh[k]] : 0;
            nsmax = max(nsmax, ns[k]);
            // vectors past nvec (last workgroup) read vector 0's row: in bounds, unused
            a[k] = part_acc + (h0 + hh[k] < nvec ? (h0 + hh[k]) * nsplit * hd : 0) + d;
            sum[k] = 0.0f;
        }
        for (int sp = 0; sp < nsmax; sp += 16) {
            float v[4][16];
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int u = 0; u < 16; ++u)  // clamped: every load is in bounds, unused ones ignored
                    v[k][u] = a[k][(int64_t)min(sp + u, max(ns[k] - 1, 0)) * hd];
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    if (sp + u < ns[k]) sum[k] = fmaf(v[k][u], wts[hh[k] * nsplit + sp + u], sum[k]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (idx0 + k * 256 >= kCombHeads * hd) continue;
            const float v = sum[k] * linv[hh[k]];
            if constexpr (kMergeOnly) {
                if (h0 + hh[k] < nvec) merged[(h0 + hh[k]) * hd + idx0 + k * 256 - hh[k] * hd] = v;
            } else {
                o[hh[k]][idx0 + k * 256 - hh[k] * hd] = v;
            }
        }
    }
    if constexpr (kMergeOnly) return;
    __syncthreads();
    for (int idx = tid; idx < 2 * hd; idx += 256) {
        const int hg = idx / hd, i = idx - hg * hd;
        float dot[kCombHeads / 2] = {};
        for (int j = 0; j < hd; ++j) {
            const float v = rot[j * hd + i];
#pragma unroll
            for (int k = 0; k < kCombHeads / 2; ++k) dot[k] += v * o[hg + 2 * k][j];
        }
#pragma unroll
        for (int k = 0; k < kCombHeads / 2; ++k) {
            const int64_t head = h0 + hg + 2 * k;
            if (head < nvec) out[head * hd + i] = (uint16_t)f2h(dot[k]);
        }
    }
}

// Merge and unrotation at head_dim 128: 4 vectors per workgroup of 512 lanes. Everything that does not
// depend on the rest is loaded at once: lane (i, quarter jq) its 32 entries of Pi_v's column i, lane
// (vector, d) up to kChunk splits' (m, l) and accumulator d, folded as an online softmax over chunks of
// kChunk splits, 16 or, where there are no more, 4 (32 vectors of one split: 5.4 us and 3.9; 2048: 6.9
// and 4.6). The merged vectors cross LDS once, then each lane sums its 32 products for the 4
// vectors and the quarters meet in LDS. The general kernel above stages Pi_v in LDS, then waits for
// (m, l), for the accumulators and for 128 LDS reads in turn: 8.3 us for 32 vectors of 4 splits and
// 19.9 for 2048 of up to 32 against 4.6 (of 16 parts) and 13.7 here (kernel trace, as above).
constexpr int kComb128Vecs = 4;
template <int kChunk>
__global__ __launch_bounds__(512) void tq_attn_combine128_kernel(
    Queries qs, const float* __restrict__ part_ml, const float* __restrict__ part_acc,
    const float* __restrict__ vrot, uint16_t* __restrict__ out, int qh, int nsplit, int64_t nvec,
    int split_pos) {
    __shared__ __attribute__((aligned(16))) float o[kComb128Vecs][128];
    __shared__ float red[4][kComb128Vecs][128];
    const int tid = threadIdx.x, i = tid & 127;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 7);  // the lane's vector, then its quarter
    float r[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) r[k] = vrot[(32 * w + k) * 128 + i];
    const int64_t vec = (int64_t)blockIdx.x * kComb128Vecs + w;
    float M = -__builtin_inff(), L = 0.0f, sum = 0.0f;
    if (vec < nvec) {
        const float* ml = part_ml + vec * nsplit * 2;
        const float* a = part_acc + vec * nsplit * 128 + i;
        const int ns = (qs.causal_len((int)(vec / qh)) + split_pos - 1) / split_pos;
        for (int s0 = 0; s0 < (s0 == 0 ? nsplit : ns); s0 += kChunk) {
            // the first chunk goes by the layout, so that its loads need not wait for the length;
            // what lies past the length is not used
            const int top = s0 == 0 ? nsplit : ns;
            float m[kChunk], l[kChunk], av[kChunk];
#pragma unroll
            for (int u = 0; u < kChunk; ++u) {
                const int sp = min(s0 + u, top - 1);
                m[u] = ml[2 * sp];
                l[u] = ml[2 * sp + 1];
                av[u] = a[(int64_t)sp * 128];
            }
            float mx = M;
#pragma unroll
            for (int u = 0; u < kChunk; ++u) {
                const bool live = s0 + u < ns;
                m[u] = live ? m[u] : -__builtin_inff();
                l[u] = live ? l[u] : 0.0f;
                av[u] = live ? av[u] : 0.0f;
                mx = fmaxf(mx, m[u]);
            }
            const float old = M == -__builtin_inff() ? 0.0f : expf(M - mx);
            L *= old;
            sum *= old;
#pragma unroll
            for (int u = 0; u < kChunk; ++u) {
                const float wt = m[u] == -__builtin_inff() ? 0.0f : expf(m[u] - mx);  // NaN sums stay
                L = fmaf(wt, l[u], L);
                sum = fmaf(wt, av[u], sum);
            }
            M = mx;
        }
    }
    o[w][i] = sum * (L > 0.0f ? 1.0f / L : 0.0f);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kComb128Vecs; ++v) {
        float dot = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const f32x4 x = *(const f32x4*)&o[v][32 * w + 4 * k];
#pragma unroll
            for (int e = 0; e < 4; ++e) dot = fmaf(r[4 * k + e], x[e], dot);
        }
        red[w][v][i] = dot;
    }
    __syncthreads();
    if (vec < nvec)
        out[vec * 128 + i] =
            (uint16_t)f2h((red[0][w][i] + red[1][w][i]) + (red[2][w][i] + red[3][w][i]));
}

// ---------------------------------------------------------------------------------------
// 2'. MFMA split kernel: head_dim 128, K and V codes of 2, 3, 4 or 8 bits (the pairs that
//     launch_mfma_split lists), G <= 8 query heads per kv head. Codes of 2 and 3 bits are widened to
//     4 on their way into registers (K) or LDS (V); 8-bit codes have one table entry each.
//
// A workgroup owns one (query, kv head, 1024-position block); each of its W waves walks an
// equal split of it in 64-position chunks (two waves of 512 positions, four of 256 where a launch
// has few workgroups, or four of 64 over a block of 256 positions where it has very few; tq_route
// in launch_rules.h):
//   QK  D[pos][col] = sum_k A[pos][k] B[k][col] on v_mfma_f32_16x16x32_f16. The K slots come
//       in (hi, lo') pairs per coordinate: A = (c_hi, c_lo*2^12) of the position's centroid,
//       B = (q_hi, 0) in column h and (q_lo*2^12, q_hi) in column 8+h, so one MFMA gives
//       D[h] = sum c_hi q_hi and D[8+h] = 2^12 (sum c_hi q_lo + c_lo q_hi), and the score is
//       (D[h] + 2^-12 D[8+h]) * norm_k / sqrt(128): fp16 operands, ~fp32 accuracy, no fp16
//       subnormals. A fragments come from an LDS table indexed by a code byte (two
//       coordinates): byte -> the (c_hi | c_lo' << 16) words of its two codes, one
//       ds_read_b64 and one address op per two codes.
//   PV  out[h][d] accumulates W[h][pos] V[pos][d] the same way: B = (v_hi, v_lo') of the V
//       code, A = (w_hi, 0) in row h and (w_lo*2^12, w_hi) in row 8+h, w = p * norm_v.
//       The B operand needs 4 positions of one coordinate per lane; ds_read_b64_tr_b4 reads
//       them transposed out of the chunk's V code rows staged in LDS in their page layout.
// Chunk position order: QK tile pt (16 rows) holds positions 4i + pt, so the 4 scores a lane
// ends up with for tile pt (rows 4rg..4rg+3) are positions 16rg + 4e + pt, and the PV
// K slots of lane group rg in tile pt are those same positions: no score shuffling.
// Online softmax per head (lanes n = h), lazily rescaling the accumulators.
// ---------------------------------------------------------------------------------------
constexpr int kChunkM = 64;     // positions per chunk
constexpr int kXcds = 8;         // MI355X: accelerator complex dies, each with its own L2
constexpr int kWavesM = 2;      // waves per workgroup, large launches
constexpr int kWavesWide = 4;   // and small ones
static_assert(kChunkM == fhip_idx::kChunk && kXcds == fhip_idx::kXcdCount && kXcds == fhip_rules::kXcds &&
                  FHIP_PAGE_TOKENS == fhip_idx::kPageTokens,
              "tq_attn_index.h and launch_rules.h describe this kernel");

typedef int v2i_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ uint32_t hi_lo_pair(float v, float& hi_f) {
    const _Float16 hi = (_Float16)v;
    hi_f = (float)hi;
    const _Float16 lo = (_Float16)((v - hi_f) * 4096.0f);
    return (uint32_t)__builtin_bit_cast(uint16_t, hi) |
           ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
}
// e with |x| < 2^e (and >= 2^(e-1)) for normal x; infinities and NaN give 129, 0 gives -126.
__device__ __forceinline__ int exponent_above(float x) {
    return (int)((__float_as_uint(x) >> 23) & 0xffu) - 126;
}
__device__ __forceinline__ float exp2i(int e) { return ldexpf(1.0f, e); }
// The power of two that brings magnitudes up to x below 2^kScaleExp, so that an fp16 hi + lo pair of a
// scaled value holds 22 bits whatever range the fp32 values come in.
constexpr int kScaleExp = 8;
__device__ __forceinline__ int scale_exponent(float x) { return kScaleExp - max(exponent_above(x), -100); }
// A table of 2^B centroids in a wave's registers (centroid 64 k + lane, the last one repeated), and the
// exponent that scales it.
template <int B>
struct Centroids {
    float v[B == 8 ? 4 : 1];
    int e;
    __device__ void load(const float* cent) {
        const int lane = threadIdx.x & 63;
        for (int k = 0; k < (B == 8 ? 4 : 1); ++k) v[k] = cent[min(64 * k + lane, (1 << B) - 1)];
    }
    __device__ void find_exponent() {
        float m = 0.0f;
        for (int k = 0; k < (B == 8 ? 4 : 1); ++k) m = fmaxf(m, fabsf(v[k]));
        e = __builtin_amdgcn_readfirstlane(scale_exponent(wave_max(m)));
    }
};
__device__ __forceinline__ float ror8(float v) {  // lane n of each 16-lane row gets lane n^8
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true));
}
// Row-local DPP moves (rotations within each 16-lane row: lane n takes lane (n - kRor) mod 16)
// that write only the lanes of the 4-lane banks in kBank; other lanes keep `old`.
template <int kRor, int kBank>
__device__ __forceinline__ float dpp_into(float old, float src) {
    constexpr int kCtrl = kRor == 0 ? 0xE4 : 0x120 + kRor;  // identity quad_perm, or row_ror
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src),
                                                      kCtrl, 0xF, kBank, false));
}
template <int kRor, int kBank>
__device__ __forceinline__ uint32_t dpp_into_u(uint32_t old, uint32_t src) {
    constexpr int kCtrl = kRor == 0 ? 0xE4 : 0x120 + kRor;
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, kCtrl, 0xF, kBank, false);
}
// acc += 2^-12 * (lane (n - kRor) mod 16's src), in the lanes of bank kBank only
// (v_fmac_f32_dpp; `c` holds 2^-12).
template <int kRor, int kBank>
__device__ __forceinline__ void dpp_fmac_lo(float& acc, float src, float c) {
    static_assert(kBank == 1 || kBank == 2 || kBank == 4 || kBank == 8, "one bank");
#define FHIP_FMAC_DPP(CTRL, BANK) \
    asm("v_fmac_f32_dpp %0, %1, %2 " CTRL " row_mask:0xf bank_mask:" BANK : "+v"(acc) : "v"(src), "v"(c))
    if constexpr (kBank == 1) {
        static_assert(kRor == 8, "tile 0");
        FHIP_FMAC_DPP("row_ror:8", "0x1");
    } else if constexpr (kBank == 2) {
        static_assert(kRor == 12, "tile 1");
        FHIP_FMAC_DPP("row_ror:12", "0x2");
    } else if constexpr (kBank == 4) {
        static_assert(kRor == 0, "tile 2");
        FHIP_FMAC_DPP("quad_perm:[0,1,2,3]", "0x4");
    } else {
        static_assert(kRor == 4, "tile 3");
        FHIP_FMAC_DPP("row_ror:4", "0x8");
    }
#undef FHIP_FMAC_DPP
}
// Max / sum over the 4 banks of each row (lanes n, n ^ 4, n ^ 8, n ^ 12 hold one head).
// A DPP read of a VGPR that a VALU instruction has just written needs two wait states, which
// the compiler does not insert for inline asm: each DPP instruction here follows an s_nop 1.
__device__ __forceinline__ float bank_max(float v) {
    asm("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf" : "+v"(v));
    asm("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(v));
    return v;
}
__device__ __forceinline__ float bank_sum(float v) {
    asm("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf" : "+v"(v));
    asm("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(v));
    return v;
}

// 8 * (byte kByte of x), the byte offset of a pair-table entry, in one v_lshlrev_b32_sdwa.
// Written as asm: the compiler turns the extract-and-shift into two instructions for most
// byte positions.
template <int kByte>
__device__ __forceinline__ uint32_t byte_x8(uint32_t x) {
    uint32_t r;
    if constexpr (kByte == 0)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
            : "=v"(r) : "s"(3u), "v"(x));
    else if constexpr (kByte == 1)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_1"
            : "=v"(r) : "s"(3u), "v"(x));
    else if constexpr (kByte == 2)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2"
            : "=v"(r) : "s"(3u), "v"(x));
    else
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_3"
            : "=v"(r) : "s"(3u), "v"(x));
    return r;
}
// Pair-table entries of bytes kB and kB + 1 of a code word w: the (c_hi | c_lo' << 16) words
// of those bytes' four codes, in the order the table holds each byte's two.
template <int kB>
__device__ __forceinline__ u32x4 pair2(const u32x2* tab, uint32_t w) {
    const u32x2 e0 = *(const u32x2*)((const char*)tab + byte_x8<kB>(w));
    const u32x2 e1 = *(const u32x2*)((const char*)tab + byte_x8<kB + 1>(w));
    return u32x4{e0[0], e0[1], e1[0], e1[1]};
}

// 8-bit codes: the words of the four codes of w (one table entry per code).
__device__ __forceinline__ u32x4 quad8(const uint32_t* tab, uint32_t w) {
    return u32x4{tab[w & 0xffu], tab[(w >> 8) & 0xffu], tab[(w >> 16) & 0xffu], tab[w >> 24]};
}

// The split's pages, read once per split into a per-wave LDS table: entry j holds the four
// part addresses (K codes, V codes, K norms, V norms) of the split's page j. Where page j holds
// no position of the split, or its table entry is outside the pool, the entry holds the split's
// first valid page instead, so every chunk load below reads a real page; the positions of such
// pages are masked in the scores (bit j of the returned mask clear) and their norms zeroed.
// With no valid page at all (mask 0) the split reads nothing.
struct PageAddrs {
    const uint8_t *k, *v, *kn, *vn;
};
template <int kPages, class Pages>
__device__ __forceinline__ uint64_t split_pages(const Pages& pg, const int32_t* table, int t_begin,
                                                int t_end, int lane, PageAddrs* pages) {
    int column;
    const bool in = fhip_idx::split_page_column(t_begin, t_end, lane, column);
    const int id = in ? table[column] : -1;
    const bool ok = in && pg.valid(id);
    const uint64_t vmask = __ballot(ok);
    if (vmask == 0) return 0;
    const int first = __builtin_amdgcn_readlane(id, (int)__builtin_ctzll(vmask));
    PageAddrs a;
    pg.addrs(ok ? id : first, a.k, a.kn, a.v, a.vn);
    if (lane < kPages) pages[lane] = a;
    wave_lds_sync();  // the wave reads other lanes' entries next
    return vmask;
}
// Loads through global-address-space pointers: addresses read back from LDS lose their
// address space, and generic (flat) loads would also count against the LDS counter, so every
// table-read wait would wait for them too.
typedef __attribute__((address_space(1))) const u32x4 g_u32x4;
typedef __attribute__((address_space(1))) const uint16_t g_u16;
__device__ __forceinline__ u32x4 gld16(const uint8_t* p) { return *(g_u32x4*)p; }
__device__ __forceinline__ uint32_t gld2(const uint8_t* p) { return *(g_u16*)p; }

// Lane j's address as a wave-uniform value (v_readlane into SGPRs).
__device__ __forceinline__ const uint8_t* addr_of_lane(const uint8_t* p, int j) {
    const uint64_t u = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), j);
    return (const uint8_t*)(((uint64_t)hi << 32) | lo);
}

// One 16-byte LDS DMA copy per lane from sbase + voff (sbase wave-uniform, in SGPRs): lane L
// writes lds + 16 L (lds wave-uniform). Issued as asm so that the compiler, which counts
// pending LDS DMA against the LDS counter as well, keeps exact LDS waits for the table lookups
// that run while copies are in flight (the hardware tracks these copies on the vector memory
// counter only). Every read of the DMA buffers waits for them explicitly.
__device__ __forceinline__ void dma16(const uint8_t* sbase, uint32_t voff, uint8_t* lds) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
    // m0 is saved and restored around the copy: the compiler may keep a value in it
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(voff), "s"(sbase), "s"(m)
        : "memory");
}

// Chunk loads. The chunk starts at split page j0 (positions t0 .. t0 + 63 = pages j0 .. j0 + 3);
// every address comes from the split's page lanes, so no load needs a per-position check.
//
// K codes, straight into the registers QK uses (LDS DMA streams markedly slower than vector
// loads, and K needs no LDS stage): tile pt is position 4n + pt, the 4 KB bytes of coordinates
// [32rg, 32rg + 32) for lane (n, rg); the lane's page is j0 + n / 4 and the four tiles are 4 rows
// apart. Pages of other widths than 4 may lie at any address: their loads assume no alignment.
typedef u32x4 u32x4_any __attribute__((aligned(1)));
typedef u32x2 u32x2_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef __attribute__((address_space(1))) const u32x4_any g_u32x4_any;
typedef __attribute__((address_space(1))) const u32x2_any g_u32x2_any;
typedef __attribute__((address_space(1))) const u32_any g_u32_any;
template <int KB>
struct KCodes {
    u32x4 w[4][KB == 8 ? 2 : 1];  // [pt]: KB words
};
template <int KB>
__device__ __forceinline__ void load_k(const PageAddrs* pages, int j0, int kvh, int g, int lane,
                                       KCodes<KB>& kc) {
    const uint8_t* src = pages[j0 + fhip_idx::k_page(lane)].k + fhip_idx::k_offset(lane, kvh, g, KB);
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
        const uint8_t* p = src + pt * fhip_idx::k_tile_stride(kvh, KB);
        if constexpr (KB == 4) {
            kc.w[pt][0] = gld16(p);
        } else if constexpr (KB == 8) {
            kc.w[pt][0] = *(g_u32x4_any*)p;
            kc.w[pt][1] = *(g_u32x4_any*)(p + 16);
        } else {
            const u32x2 v = *(g_u32x2_any*)p;
            kc.w[pt][0] = u32x4{v[0], v[1], KB == 3 ? *(g_u32_any*)(p + 8) : 0u, 0u};
        }
    }
}
// V codes by LDS DMA: copy i moves page j0 + i (positions 16i .. 16i + 15); lane L takes
// position p = 16i + L / 4 and stores 16 bytes at 64p + 16(L % 4). The 16-byte segment it
// copies is (L % 4) ^ ((p / 2) % 4): rows are XOR-swizzled so the transposed reads of one
// dim range from 16 rows spread over the banks. `voff` is that segment's offset in the page.
__device__ __forceinline__ void dma_v(const PageAddrs* pages, int j0, uint32_t voff, uint8_t* vb,
                                      int lane) {
    const uint8_t* v4 = pages[j0 + (lane & 3)].v;  // lane i < 4: page j0 + i
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(addr_of_lane(v4, i), voff, vb + 1024 * i);
}
// 2-bit V codes: the same segments as dma_v, from rows of 32 bytes. Lane L takes 8 bytes of
// position 16i + L / 4 of page j0 + i (v2_offset), and once they have arrived store_v2 widens
// each 2-bit code to a 4-bit one and writes the 16 bytes that dma_v would have copied, so the
// transposed reads and the pair table serve both widths (its V entries map codes 0..3).
__device__ __forceinline__ void load_v2(const PageAddrs* pages, int j0, uint32_t voff,
                                        u32x2 (&r)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = *(g_u32x2_any*)(pages[j0 + i].v + voff);
}
// Bytes sel of w (two code bytes, four codes each, the first in the top bits) as four bytes
// of 4-bit codes, the first in the high nibble: byte b -> (c0 << 4 | c1), (c2 << 4 | c3).
__device__ __forceinline__ uint32_t widen2(uint32_t w, uint32_t sel) {
    const uint32_t x = __builtin_amdgcn_perm(w, w, sel);  // b0, b0, b1, b1
    return ((x & 0x00C000C0u) >> 2) | ((x & 0x00300030u) >> 4) | ((x & 0x0C000C00u) << 2) |
           (x & 0x03000300u);
}
// Eight 3-bit codes of the three bytes sel picks from (hi, lo), the first in the top bits of the
// first byte, as four bytes of 4-bit codes, the first in the high nibble.
__device__ __forceinline__ uint32_t widen3(uint32_t hi, uint32_t lo, uint32_t sel) {
    uint32_t x = __builtin_amdgcn_perm(hi, lo, sel);          // 24 bits, the first code on top
    x = ((x & 0x00FFF000u) << 4) | (x & 0x00000FFFu);         // 4 codes a half
    x = ((x & 0x0FC00FC0u) << 2) | (x & 0x003F003Fu);         // 2 codes a byte
    x = ((x & 0x38383838u) << 1) | (x & 0x07070707u);
    return __builtin_amdgcn_perm(x, x, 0x00010203u);          // first byte lowest
}
// 32 codes of 2 or 3 bits (B words) as 4 words of 4-bit codes.
template <int B, class Words>
__device__ __forceinline__ u32x4 widen32(const Words& w) {
    if constexpr (B == 2)
        return u32x4{widen2(w[0], 0x01010000u), widen2(w[0], 0x03030202u), widen2(w[1], 0x01010000u),
                     widen2(w[1], 0x03030202u)};
    else  // bytes 3j .. 3j + 2 of the twelve, byte 3j on top
        return u32x4{widen3(w[0], w[0], 0x0C000102u), widen3(w[1], w[0], 0x0C030405u),
                     widen3(w[2], w[1], 0x0C020304u), widen3(w[2], w[2], 0x0C010203u)};
}
__device__ __forceinline__ void store_v2(const u32x2 (&r)[4], uint8_t* vb, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *(u32x4*)(vb + 1024 * i + 16 * lane) =
            u32x4{widen2(r[i][0], 0x01010000u), widen2(r[i][0], 0x03030202u),
                  widen2(r[i][1], 0x01010000u), widen2(r[i][1], 0x03030202u)};
}

// 3-bit V codes: the same with 12 bytes of rows of 48.
struct V3Codes {
    uint32_t w[4][3];
};
__device__ __forceinline__ void load_v3(const PageAddrs* pages, int j0, uint32_t voff, V3Codes& r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint8_t* p = pages[j0 + i].v + voff;
        const u32x2 v = *(g_u32x2_any*)p;
        r.w[i][0] = v[0];
        r.w[i][1] = v[1];
        r.w[i][2] = *(g_u32_any*)(p + 8);
    }
}
__device__ __forceinline__ void store_v3(const V3Codes& r, uint8_t* vb, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *(u32x4*)(vb + 1024 * i + 16 * lane) = widen32<3>(r.w[i]);
}
// 8-bit V codes: eight 16-byte loads of rows of 128 bytes, swizzled as v8_offset says.
__device__ __forceinline__ void load_v8(const PageAddrs* pages, int j0, int kvh, int g, int lane,
                                        u32x4 (&r)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
        r[i] = *(g_u32x4_any*)(pages[j0 + fhip_idx::v8_page(i)].v + fhip_idx::v8_offset(lane, i, kvh, g));
}
__device__ __forceinline__ void store_v8(const u32x4 (&r)[8], uint8_t* vb, int lane) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *(u32x4*)(vb + 1024 * i + 16 * lane) = r[i];
}

// Value norms enter the weights as quarters: a weight's w_hi, rounded toward zero, then leaves less than
// 8, and lo' = 2^12 of that stays in fp16's range up to the largest norm.
constexpr float kNormVUnit = 0.25f;
constexpr int kNormVExp = 2;  // 1 / kNormVUnit = 2^kNormVExp
// Norms of position t0 + lane, loaded raw (fp16 bits): pack() gives (knorm, vnorm kNormVUnit) in fp32
// once they are needed (0 where there is none), so each norm is converted once, by the lane
// that loaded it. Packing later keeps the wait for them away from the copies issued after them.
struct NormRegs {
    uint32_t k, v;
    bool ok;
    __device__ float2 pack() const {
        uint32_t a = k, b = v;
        // pins the pack here: the compiler would otherwise pack right after the loads
        asm volatile("" : "+v"(a), "+v"(b));
        const float fk = (float)__builtin_bit_cast(_Float16, (uint16_t)a);
        const float fv = (float)__builtin_bit_cast(_Float16, (uint16_t)b) * kNormVUnit;
        return ok ? float2{fk, fv} : float2{0.0f, 0.0f};
    }
};
__device__ __forceinline__ NormRegs load_norms(const PageAddrs* pages, int j0, uint32_t pm, int t0,
                                               int t_end, int kvh, int g, int lane) {
    const int k = fhip_idx::norm_page(lane);
    const uint32_t row = fhip_idx::norm_offset(lane, kvh, g);
    const bool ok = ((pm >> k) & 1u) && t0 + lane < t_end;
    const PageAddrs& pa = pages[j0 + k];
    return NormRegs{gld2(pa.kn + row), gld2(pa.vn + row), ok};
}

// Loads of chunk i + 1 (V codes by LDS DMA, then norms and K codes into registers) are issued
// together right after chunk i's QK, and chunk i + 1 starts by waiting for all of them
// (vmcnt(0)), so its PV reads the V buffer with no further wait. The transposed V reads are
// asm: the compiler's own wait counting would also hold PV back for the loads issued after QK.
// The "memory" clobber keeps every copy on its side of these reads.
// Transposed V reads of dim tiles 0..7 (tile c at row segment (c / 2) ^ sw, half c % 2):
// seg[s] is the lane's address of its row's segment s ^ sw.
__device__ __forceinline__ void read_v_codes(const uint32_t (&seg)[4], v2i_t (&tv)[8]) {
    asm volatile(
        "ds_read_b64_tr_b4 %0, %8\n"
        "ds_read_b64_tr_b4 %1, %8 offset:8\n"
        "ds_read_b64_tr_b4 %2, %9\n"
        "ds_read_b64_tr_b4 %3, %9 offset:8\n"
        "ds_read_b64_tr_b4 %4, %10\n"
        "ds_read_b64_tr_b4 %5, %10 offset:8\n"
        "ds_read_b64_tr_b4 %6, %11\n"
        "ds_read_b64_tr_b4 %7, %11 offset:8\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(tv[0]), "=&v"(tv[1]), "=&v"(tv[2]), "=&v"(tv[3]), "=&v"(tv[4]), "=&v"(tv[5]),
          "=&v"(tv[6]), "=&v"(tv[7])
        : "v"(seg[0]), "v"(seg[1]), "v"(seg[2]), "v"(seg[3])
        : "memory");
}

// The same for 8-bit codes: dim tile c of position tiles 2 half, 2 half + 1; addr[c] is the lane's
// address of segment c ^ swizzle of its row. ds_read_b64_tr_b8 gives lane n of each 16-lane group
// byte n % 8 of source lanes 2 k + n / 8 (k = 0..7): word pt % 2 holds the four positions of tile pt.
template <int kHalf>
__device__ __forceinline__ void read_v_codes8(const uint32_t (&addr)[8], v2i_t (&tv)[8]) {
#define FHIP_TR8(OFF)                                                                              \
    asm volatile(                                                                                  \
        "ds_read_b64_tr_b8 %0, %8" OFF "\n"                                                        \
        "ds_read_b64_tr_b8 %1, %9" OFF "\n"                                                        \
        "ds_read_b64_tr_b8 %2, %10" OFF "\n"                                                       \
        "ds_read_b64_tr_b8 %3, %11" OFF "\n"                                                       \
        "ds_read_b64_tr_b8 %4, %12" OFF "\n"                                                       \
        "ds_read_b64_tr_b8 %5, %13" OFF "\n"                                                       \
        "ds_read_b64_tr_b8 %6, %14" OFF "\n"                                                       \
        "ds_read_b64_tr_b8 %7, %15" OFF "\n"                                                       \
        "s_waitcnt lgkmcnt(0)"                                                                     \
        : "=&v"(tv[0]), "=&v"(tv[1]), "=&v"(tv[2]), "=&v"(tv[3]), "=&v"(tv[4]), "=&v"(tv[5]),      \
          "=&v"(tv[6]), "=&v"(tv[7])                                                               \
        : "v"(addr[0]), "v"(addr[1]), "v"(addr[2]), "v"(addr[3]), "v"(addr[4]), "v"(addr[5]),      \
          "v"(addr[6]), "v"(addr[7])                                                               \
        : "memory")
    if constexpr (kHalf == 0)
        FHIP_TR8("");
    else
        FHIP_TR8(" offset:256");
#undef FHIP_TR8
}

// kG4 score compaction: tile kPt's head-h score D[h] + 2^-12 D[8 + h] (MFMA columns h and 8 + h
// of the lane's row) into lane 4 kPt + h, elements e = 0..3; the other banks keep theirs.
template <int kPt>
__device__ __forceinline__ void compact_scores(float (&S)[4], const f32x4_t& d, float c12) {
    constexpr int kBank = 1 << kPt;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        S[e] = dpp_into<(4 * kPt) & 15, kBank>(S[e], d[e]);
        dpp_fmac_lo<(4 * kPt + 8) & 15, kBank>(S[e], d[e], c12);
    }
}
// kG4 PV operand of tile kPt: column h (lanes h < 4) takes (w_hi, 0) and column 8 + h takes
// (w_lo', w_hi) of lane 4 kPt + h; banks 1 and 3 are not written (they stay 0).
template <int kPt>
__device__ __forceinline__ void expand_weights(uint32_t (&b)[4], const uint32_t (&x)[4],
                                               const uint32_t (&y)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        b[e] = dpp_into_u<(16 - 4 * kPt) & 15, 0x1>(b[e], x[e]);
        b[e] = dpp_into_u<(24 - 4 * kPt) & 15, 0x4>(b[e], y[e]);
    }
}

// 8-bit codes hold twice the registers in flight, so two waves per SIMD instead of three.
template <class Pages, bool kG4, int KB, int VB, int W, int kPart>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(KB == 8 || VB == 8 ? 2 : 3))) void
tq_attn_mfma_kernel(const float* __restrict__ qrot, Queries qs, Pages pg,
                    const float* __restrict__ kcent, const float* __restrict__ vcent, int qh,
                    int kvh, float scale, float* __restrict__ part_ml,
                    float* __restrict__ part_acc, int nsplit, int nblk, int tok) {
    constexpr int hd = 128;
    constexpr int kSwap = VB == 8 ? 0 : 1;  // element e of a dim tile holds dim e ^ kSwap
    // Code-byte tables: byte b -> the (c_hi | c_lo' << 16) words of its two codes, K as
    // {high nibble, low nibble} (the QK A operand's order), V as {low, high} (the PV B
    // operand's). One ds_read_b64 serves two codes: lookups at random entries of 2 KB tables
    // cost some bank conflicts, but half the LDS instructions and under half the address
    // arithmetic of per-code lookups in a 16-word table. The DMA
    // targets are separate objects: table reads never wait for DMA traffic.
    __shared__ u32x2 pk[256], pv[256];  // 8-bit codes: 256 words, one per code
    // two chunks of 4-bit V codes, by chunk parity, or one of 8-bit codes
    __shared__ __attribute__((aligned(64))) uint8_t vbuf[W][2][kChunkM * 64];
    __shared__ __attribute__((aligned(16))) float2 nbuf[W][kChunkM];  // (knorm, vnorm)
    __shared__ PageAddrs pagebuf[W][kPart / W / FHIP_PAGE_TOKENS];  // the wave's split pages
    __shared__ int waves_done;  // waves that have left their state for the merge
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, rg = lane >> 4;  // MFMA column / row group
    static_assert(kPart / W % kChunkM == 0 && kPart / W <= 64 * FHIP_PAGE_TOKENS,
                  "a wave's split is whole chunks, its pages one per lane");

    // Workgroup (query, kv head, block of W consecutive splits); wave w takes split
    // W * blk + w. Workgroups go to the 8 XCDs round-robin (workgroup b on XCD b % 8),
    // and the kv heads of one token row share 128-byte lines, so the index puts every kv head
    // of one (query, block) item on the same XCD: item i = (query, block) and kv head g run
    // as workgroup (i / 8) (8 kvh) + 8 g + i % 8, and each line is filled into one L2 only.
    // A workgroup whose block holds no position leaves before the tables are built (the exit
    // is uniform, so no wave misses the barriers below).
    int64_t item;
    int g;
    fhip_idx::wg_item(blockIdx.x, kvh, item, g);
    // Item (token group, block): a group is `tok` consecutive queries of one sequence (causal
    // prefill; 1 in decode), whose G query heads each fill MFMA columns h = G t + head.
    const int qg = (int)(item / nblk);
    const int tq0 = qg * tok;
    if (tq0 >= qs.seq_lens_count) return;
    const int tq_last = min(tq0 + tok, qs.seq_lens_count) - 1;
    const int blk = (int)(item % nblk);
    const int clen = qs.causal_len(tq_last);  // the group's longest causal length
    if (blk * kPart >= clen) return;
    int ek, ev;
    {
        Centroids<KB> ck;
        Centroids<VB> cv;
        ck.load(kcent);
        cv.load(vcent);
        ck.find_exponent();
        cv.find_exponent();
        ek = ck.e;
        ev = cv.e;
        // each wave fills its share of the entries 64 k + lane
        auto fill = [&](auto& c, u32x2* tab, int bits, bool high_first) {
            float hf;
            if (bits == 8) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k % W == wave)
                        ((uint32_t*)tab)[64 * k + lane] = hi_lo_pair(ldexpf(c.v[k % (sizeof(c.v) / 4)], c.e), hf);
            } else {
                const int word = (int)hi_lo_pair(ldexpf(c.v[0], c.e), hf);  // lane: its code's
                const int low = __shfl(word, lane & 15);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int high = __shfl(word, 4 * k + (lane >> 4));
                    if (k % W == wave)
                        tab[64 * k + lane] = high_first ? u32x2{(uint32_t)high, (uint32_t)low}
                                                        : u32x2{(uint32_t)low, (uint32_t)high};
                }
            }
        };
        fill(ck, pk, KB, true);
        fill(cv, pv, VB, false);
        if (threadIdx.x == 0) waves_done = 0;
    }
    __syncthreads();

    // (a constant where it can only be one chunk: the loop below is then straight code. Two waves of 8-bit
    // codes keep halves of the block: with two waves per SIMD a large launch is bound by the waves' fixed
    // part, 128 sequences of 400, 8 / 8 heads 40.4 us and 43.2 in halves of their positions)
    const int span = kPart / W == kChunkM || (KB == 8 && W == 2)
                         ? kPart / W
                         : fhip_idx::wave_span(min(kPart, clen - blk * kPart), W);
    const int t_begin = fhip_idx::split_begin(blk, wave, kPart, span);
    const int t_end = min(clen, t_begin + span);
    const int G = qh / kvh;
    const int32_t* table = qs.table + (int64_t)tq0 * qs.table_stride;
    uint8_t* vb = vbuf[wave][0];
    float2* nb = nbuf[wave];
    const int ncols = tok * G;  // live head columns (at most 8)
    // this lane's column: token tq0 + ct, head ch; its causal length (0 for a column past the
    // queries, so that every position is masked for it)
    const int ct = (n & 7) / G;
    bool col_ok;  // the column is head (n & 7) % G of a query of the group
    const int64_t qvec = fhip_idx::q_vector(lane, tq0, tok, G, qs.seq_lens_count, qh, g, col_ok);
    const int col_len = col_ok ? qs.causal_len(tq0 + ct) : 0;
    // the shortest length of the group (its first query's): chunks below it need no mask
    const int min_len = tok > 1 ? qs.causal_len(tq0) : clen;

    float m_run = -__builtin_inff(), l_run = 0.0f;  // log2 units; lanes n, n ^ 8: head n & 7
    // PV accumulators out^T, dim tile c: lane (n, rg) holds head slot n (n < 8: head n, hi
    // part; n >= 8: head n - 8, lo' part) at dims 16c + ((4rg + e) ^ 1), e = 0..3
    f32x4_t acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // The split's pages, read once: the chunk loop then issues no memory
    // instruction besides its loads and copies. A wave with no position to read (its split
    // starts past the end, or no page is in the pool) keeps the empty state.
    PageAddrs* pages = pagebuf[wave];
    const uint64_t vmask = t_begin < clen ? split_pages<kPart / W / FHIP_PAGE_TOKENS>(pg, table, t_begin, t_end, lane, pages) : 0;
    if (vmask != 0) {
    // first chunk's copies go out before the Q set-up
    const uint32_t v_lane_off = VB == 2   ? fhip_idx::v2_offset(lane, kvh, g)
                                : VB == 3 ? fhip_idx::v3_offset(lane, kvh, g)
                                          : fhip_idx::v_offset(lane, kvh, g);
    uint32_t pmask = (uint32_t)vmask & 0xfu;  // pages of the current chunk to read
    // the next chunk's V codes where they go through registers into LDS when it starts (all
    // widths but 4)
    u32x2 v2reg[VB == 2 ? 4 : 1];
    V3Codes v3reg;
    u32x4 v8reg[VB == 8 ? 8 : 1];
    auto load_v = [&](int j0, uint8_t* dst) {
        if constexpr (VB == 2)
            load_v2(pages, j0, v_lane_off, v2reg);
        else if constexpr (VB == 3)
            load_v3(pages, j0, v_lane_off, v3reg);
        else if constexpr (VB == 8)
            load_v8(pages, j0, kvh, g, lane, v8reg);
        else
            dma_v(pages, j0, v_lane_off, dst, lane);
    };
    load_v(0, vb);  // chunk 0: buffer 0
    NormRegs nreg = load_norms(pages, 0, pmask, t_begin, t_end, kvh, g, lane);
    KCodes<KB> kreg;
    load_k<KB>(pages, 0, kvh, g, lane, kreg);

    // Q as the QK B operand, scaled like the tables: step s, lane (n, rg) holds coordinates
    // 32rg + 4s + c4. What a score is then multiplied by, with the key's norm, to be in log2 units
    // (never 0: a masked score stays -inf):
    float colscale;
    uint32_t bq[8][4];
    {
        // columns past the group's heads read the group's first vector and are zeroed
        const float* qsrc = qrot + qvec * hd;
        f32x4_t qv[8];
#pragma unroll
        for (int s8 = 0; s8 < 8; ++s8) qv[s8] = *(const f32x4_t*)(qsrc + fhip_idx::q_lane_offset(lane, s8));
        float qmax = 0.0f;
#pragma unroll
        for (int s8 = 0; s8 < 8; ++s8)
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) qmax = fmaxf(qmax, fabsf(qv[s8][c4]));
        qmax = fmaxf(qmax, __shfl_xor(qmax, 16));
        qmax = fmaxf(qmax, __shfl_xor(qmax, 32));
        const int eq = scale_exponent(qmax);
        const float qmul = col_ok ? exp2i(eq) : 0.0f;
        colscale = fmaxf(ldexpf(scale * 1.4426950408889634f, -eq - ek), 0x1p-126f);
        // kG4: lane 4 pt + h holds head h's scores
        if constexpr (kG4) colscale = __shfl(colscale, (lane & 48) | (lane & 3));
#pragma unroll
        for (int s8 = 0; s8 < 8; ++s8) {
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) {
                const float q = qv[s8][c4] * qmul;
                float qhf;
                const uint32_t pr = hi_lo_pair(q, qhf);  // q_hi | q_lo' << 16
                // column h: (q_hi, 0); column 8 + h: (q_lo', q_hi)
                bq[s8][c4] = n < 8 ? (pr & 0xffffu) : ((pr >> 16) | (pr << 16));
            }
        }
    }
    // Score of head n & 7 in both lanes n and n ^ 8: D[h] + 2^-12 D[8 + h].
    const float ca = n < 8 ? 1.0f : 1.0f / 4096.0f, cb = n < 8 ? 1.0f / 4096.0f : 1.0f;
    // PV A operand of weight w: row h (lanes n < 8) takes (w_hi, 0), row 8 + h takes
    // (w_lo', w_hi), w_hi = w rounded toward zero. r = pkrtz(w, w) = (w_hi, w_hi), then
    // r.lo = f16(r.lo * wb + w * wc) in place (lanes n < 8: w_hi; n >= 8: 2^12 (w - w_hi)),
    // then lanes n < 8 clear r.hi.
    const float wb = n < 8 ? 1.0f : -4096.0f, wc = n < 8 ? 0.0f : 4096.0f;
    const uint32_t hmask = n < 8 ? 0xffffu : 0xffffffffu;
    // cross-row exchanges (lane ^ 16, lane ^ 32) as ds_bpermute byte addresses
    const int bp16 = (lane ^ 16) << 2, bp32 = (lane ^ 32) << 2;
    auto xrow = [](int bp, float v) {
        return __int_as_float(__builtin_amdgcn_ds_bpermute(bp, __float_as_int(v)));
    };
    // transposed V reads: source lane m of group rg reads position 16rg + 4(m % 4) + m / 4;
    // segment s of that row sits at vrow[s ^ sw]. 8-bit codes: lane m reads half m % 2 of the
    // 16 dims of a tile at position 16rg + 4(k % 4) + k / 4 (+ 2 for tiles 2, 3), k = m / 2.
    uint32_t vseg[VB == 8 ? 8 : 1];
    const uint32_t vb32 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)vb;
    if constexpr (VB == 8) {
        const int k = n >> 1, srow = 16 * rg + 4 * (k & 3) + (k >> 2);
#pragma unroll
        for (int c = 0; c < 8; ++c)
            vseg[c] = vb32 + 128 * srow + 16 * (c ^ fhip_idx::v8_swizzle(srow)) + 8 * (n & 1);
    } else {
        const int srow = 16 * rg + 4 * (n & 3) + (n >> 2);
        const int sw = (srow >> 1) & 3;
        vseg[0] = vb32 + 64 * srow + 16 * sw;  // segment s: exclusive or with 16 s (rows are aligned)
    }

    // kG4 (at most 4 query heads per kv head): scores, probabilities and weights are held
    // compactly, lane (n, rg) with n = 4 pt + h holding head h's 4 positions 16rg + 4e + pt of
    // tile pt (one distinct value per lane and element, where the MFMA layout repeats each
    // four times); the tiles' weights are moved back into the PV operand layout per tile.
    // Norm records are stored in that order (nb index 16 rg + 4 pt + e), so a lane's four come
    // in two 16-byte reads.
    const int ptc = n >> 2;  // kG4: the lane's position tile
    const int nb_idx = kG4 ? (lane & 0x30) | ((lane & 3) << 2) | ((lane >> 2) & 3) : lane;
    const float c12 = 1.0f / 4096.0f;
    uint32_t awz[4] = {0u, 0u, 0u, 0u};  // kG4 PV operand: banks 1 and 3 (heads 4-7) stay 0

    for (int t0 = t_begin, par = 0; t0 < t_end; t0 += kChunkM, par ^= 1) {
        const int tn = t0 + kChunkM;  // next chunk
        const int jn = fhip_idx::chunk_first_page(tn, t_begin);  // its first split page
        const uint32_t pmask_n = tn < t_end ? (uint32_t)(vmask >> jn) & 0xfu : 0u;
        const bool full = pmask == 0xfu && tn <= t_end && tn <= min_len;

        // ---- QK: 4 tiles x 8 steps
        float sc[4][4];  // !kG4 [pt][e]: position 16rg + 4e + pt, head n & 7
        float scc[4];    // kG4 [e]: position 16rg + 4e + ptc, head n & 3
        // all loads of this chunk are in (the V copies included)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // the V buffer PV reads below (the sync after the norm records orders these writes
        // before the transposed reads)
        if constexpr (VB == 2) store_v2(v2reg, vb + par * (kChunkM * 64), lane);
        if constexpr (VB == 3) store_v3(v3reg, vb + par * (kChunkM * 64), lane);
        if constexpr (VB == 8) store_v8(v8reg, vb, lane);
        u32x4 kcs[4][KB == 8 ? 2 : 1];
#pragma unroll
        for (int pt = 0; pt < 4; ++pt) {
            if constexpr (KB == 2 || KB == 3) {
                kcs[pt][0] = widen32<KB>(kreg.w[pt][0]);
            } else {
#pragma unroll
                for (int k = 0; k < KB / 4; ++k) kcs[pt][k] = kreg.w[pt][k];
            }
        }
        // 32 MFMA steps t = (tile pt, word s2, half): the A operand of step t holds the table
        // entries of bytes 2 half, 2 half + 1 of word s2 (coordinates 8 s2 + 4 half + 0..3; 8-bit
        // codes: of word t % 8).
        // Table reads run kLookAhead steps ahead of their MFMA, so their LDS latency is
        // covered by the MFMAs in between.
        constexpr int kLookAhead = 2;
        auto qk_a = [&](int t) -> u32x4 {
            if constexpr (KB == 8) {
                return quad8((const uint32_t*)pk, kcs[t >> 3][(t & 7) >> 2][t & 3]);
            } else {
                const uint32_t w = kcs[t >> 3][0][(t >> 1) & 3];
                return (t & 1) ? pair2<2>(pk, w) : pair2<0>(pk, w);
            }
        };
        {
            u32x4 ahead[kLookAhead + 1];
#pragma unroll
            for (int t = 0; t < kLookAhead; ++t) ahead[t] = qk_a(t);
            f32x4_t d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 32; ++t) {
                if (t + kLookAhead < 32) ahead[(t + kLookAhead) % (kLookAhead + 1)] = qk_a(t + kLookAhead);
                const int s8 = t & 7;  // Q step 2 s2 + half
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(f16x8_t, ahead[t % (kLookAhead + 1)]),
                    __builtin_bit_cast(f16x8_t, u32x4{bq[s8][0], bq[s8][1], bq[s8][2], bq[s8][3]}),
                    d, 0, 0, 0);
                if ((t & 7) == 7) {
                    if constexpr (kG4) {
                        // tile pt's head-h score D[h] + 2^-12 D[8 + h] into lanes 4 pt + h
                        switch (t >> 3) {
                            case 0: compact_scores<0>(scc, d, c12); break;
                            case 1: compact_scores<1>(scc, d, c12); break;
                            case 2: compact_scores<2>(scc, d, c12); break;
                            default: compact_scores<3>(scc, d, c12); break;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            // fma(ror8(d), cb, d * ca) with the row rotation folded into the
                            // fmac (the multiply reads d first, after the MFMA result is ready)
                            float v = d[e] * ca;
                            asm("v_fmac_f32_dpp %0, %1, %2 row_ror:8 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                                : "+v"(v)
                                : "v"(d[e]), "v"(cb));
                            sc[t >> 3][e] = v;
                        }
                    }
                    d = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
                // keeps the scheduler from sinking the look-ahead reads to their MFMAs
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- K norms; then the K and norm registers are free: all loads of the next chunk,
        // its V codes into the other V buffer. The previous chunk's nb reads are above the
        // transposed V reads' asm (a compiler barrier); the sync after the write keeps the
        // cross-lane reads below it also when no copy asm follows (the last chunk).
        nb[nb_idx] = nreg.pack();
        wave_lds_sync();
        uint8_t* vnext = vb + (par ^ 1) * (kChunkM * 64);
        if (tn < t_end) {
            load_v(jn, vnext);
            nreg = load_norms(pages, jn, pmask_n, tn, t_end, kvh, g, lane);
            load_k<KB>(pages, jn, kvh, g, lane, kreg);
        }
        float m_new, alpha;
        uint32_t aw[4][4];  // !kG4 [pt][e]
        uint32_t xw[4], yw[4];  // kG4: (w_hi, 0) and (w_lo', w_hi) of the lane's 4 weights
        if constexpr (kG4) {
            const f32x4_t n0 = *(const f32x4_t*)&nb[16 * rg + 4 * ptc];
            const f32x4_t n1 = *(const f32x4_t*)&nb[16 * rg + 4 * ptc + 2];
            const float kn[4] = {n0[0], n0[2], n1[0], n1[2]};
            const float vn[4] = {n0[1], n0[3], n1[1], n1[3]};
#pragma unroll
            for (int e = 0; e < 4; ++e) scc[e] *= kn[e];
            if (!full) {
                const bool row_ok = (pmask >> rg) & 1u;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (!(row_ok && t0 + 16 * rg + 4 * e + ptc < t_end)) scc[e] = -__builtin_inff();
            }
            float cmax = fmaxf(fmaxf(scc[0], scc[1]), fmaxf(scc[2], scc[3]));
            cmax = bank_max(cmax);
            cmax = fmaxf(cmax, xrow(bp16, cmax));
            cmax = fmaxf(cmax, xrow(bp32, cmax));
            m_new = fmaxf(m_run, cmax * colscale);
            alpha = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            float psum = 0.0f;
            const float mref = m_new == -__builtin_inff() ? 0.0f : m_new;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float pr = __builtin_amdgcn_exp2f(fmaf(scc[e], colscale, -mref));
                psum += pr;
                const float w = pr * vn[e];
                // w_hi = w rounded toward zero; lo' = f16(2^12 (w - w_hi)) in place of r.lo
                uint32_t r = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(w, w));
                xw[e] = r & 0xffffu;
                asm("v_fma_mixlo_f16 %0, %0, %1, %2 op_sel_hi:[1,0,0]"
                    : "+v"(r)
                    : "v"(-4096.0f), "v"(w * 4096.0f));
                yw[e] = r;
            }
            psum = bank_sum(psum);
            psum += xrow(bp16, psum);
            psum += xrow(bp32, psum);
            l_run = l_run * alpha + psum;
        } else {
            float kn[16], vn[16];  // positions 16rg + j
#pragma unroll
            for (int j2 = 0; j2 < 8; ++j2) {
                const f32x4_t v = *(const f32x4_t*)&nb[16 * rg + 2 * j2];
                kn[2 * j2] = v[0];
                vn[2 * j2] = v[1];
                kn[2 * j2 + 1] = v[2];
                vn[2 * j2 + 1] = v[3];
            }
#pragma unroll
            for (int pt = 0; pt < 4; ++pt)
#pragma unroll
                for (int e = 0; e < 4; ++e) sc[pt][e] *= kn[4 * e + pt];
            if (!full) {
                const bool row_ok = (pmask >> rg) & 1u;
                const int lim = min(t_end, col_len);
#pragma unroll
                for (int pt = 0; pt < 4; ++pt)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!(row_ok && t0 + 16 * rg + 4 * e + pt < lim)) {
                            sc[pt][e] = -__builtin_inff();
                            vn[4 * e + pt] = 0.0f;  // an infinite or NaN norm past the column's length
                        }
            }
            float cmax = -__builtin_inff();
#pragma unroll
            for (int pt = 0; pt < 4; ++pt)
#pragma unroll
                for (int e = 0; e < 4; ++e) cmax = fmaxf(cmax, sc[pt][e]);
            cmax = fmaxf(cmax, xrow(bp16, cmax));
            cmax = fmaxf(cmax, xrow(bp32, cmax));
            m_new = fmaxf(m_run, cmax * colscale);
            alpha = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            // ---- probabilities, weights, B operands of PV
            float psum = 0.0f;
            const float mref = m_new == -__builtin_inff() ? 0.0f : m_new;
#pragma unroll
            for (int pt = 0; pt < 4; ++pt) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float pr = __builtin_amdgcn_exp2f(fmaf(sc[pt][e], colscale, -mref));
                    psum += pr;
                    const float w = pr * vn[4 * e + pt];
                    uint32_t r = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(w, w));
                    // in place: written in C, the compiler merges the halves with an extra v_bfi
                    asm("v_fma_mixlo_f16 %0, %0, %1, %2 op_sel_hi:[1,0,0]"
                        : "+v"(r)
                        : "v"(wb), "v"(w * wc));
                    aw[pt][e] = r & hmask;
                }
            }
            psum += xrow(bp16, psum);
            psum += xrow(bp32, psum);
            l_run = l_run * alpha + psum;
        }
        // rescale the accumulators when some head's max moved (each lane's alpha is that of
        // its accumulator slot's head)
        const bool moved_any =
            __ballot((n < ncols) && (!kG4 || n < 4) && (rg == 0) && (m_new > m_run)) != 0;
        if (moved_any) {
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[c][e] *= alpha;
        }
        m_run = m_new;

        // ---- PV: 8 dim tiles x 4 position tiles
        v2i_t tvs[8];
        if constexpr (VB == 8) {
            read_v_codes8<0>(vseg, tvs);
        } else {
            const uint32_t vo = (uint32_t)par * (kChunkM * 64);
            const uint32_t s0 = vseg[0] + vo;
            const uint32_t seg[4] = {s0, s0 ^ 16, s0 ^ 32, s0 ^ 48};
            read_v_codes(seg, tvs);
        }
        // out^T = V^T W^T: the V entries are the A operand (row m: dim 16c + (m ^ 1)), the
        // weights the B operand (column n: head slot n). 32 MFMA steps t = (position tile pt,
        // dim tile c): nibble 4pt + c4 of dim tile c's transposed read is the code of position
        // (pt, c4) at dim 16c + (n ^ 1) (8-bit codes: a byte, at dim 16c + n); tile pt sits in word pt / 2, bytes 2 (pt % 2),
        // 2 (pt % 2) + 1. Table reads run kLookAhead steps ahead as in QK.
        auto pv_b = [&](int t) -> u32x4 {
            const int pt = t >> 3, c = t & 7;
            if constexpr (VB == 8) {
                // the codes of tiles 2, 3 are read once tiles 0, 1 have used theirs
                if (t == 16) read_v_codes8<1>(vseg, tvs);
                return quad8((const uint32_t*)pv, (uint32_t)tvs[c][pt & 1]);
            } else {
                const uint32_t w = (uint32_t)tvs[c][pt >> 1];
                return (pt & 1) ? pair2<2>(pv, w) : pair2<0>(pv, w);
            }
        };
        {
            constexpr int kAheadPv = kLookAhead;
            u32x4 ahead[kAheadPv + 1];
#pragma unroll
            for (int t = 0; t < kAheadPv; ++t) ahead[t] = pv_b(t);
#pragma unroll
            for (int t = 0; t < 32; ++t) {
                if (t + kAheadPv < 32) ahead[(t + kAheadPv) % (kAheadPv + 1)] = pv_b(t + kAheadPv);
                const int pt = t >> 3, c = t & 7;
                if constexpr (kG4) {
                    if (c == 0) {  // tile pt's weights into the operand layout
                        switch (pt) {
                            case 0: expand_weights<0>(awz, xw, yw); break;
                            case 1: expand_weights<1>(awz, xw, yw); break;
                            case 2: expand_weights<2>(awz, xw, yw); break;
                            default: expand_weights<3>(awz, xw, yw); break;
                        }
                    }
                }
                const u32x4 bw = kG4 ? u32x4{awz[0], awz[1], awz[2], awz[3]}
                                     : u32x4{aw[pt][0], aw[pt][1], aw[pt][2], aw[pt][3]};
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(f16x8_t, ahead[t % (kAheadPv + 1)]),
                    __builtin_bit_cast(f16x8_t, bw), acc[c], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        pmask = pmask_n;
    }

    }  // vmask != 0

    // no copy may land in LDS after this point: the V buffers hold the merge state next
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- merge the workgroup's splits into the block's partial. Each wave leaves its state
    // in its own V buffer: acc[h][d] = slot h (hi) + 2^-12 slot 8 + h (lo'), lanes n and n ^ 8,
    // then m (log2 units) and l per head, and counts itself done; the last wave to finish
    // merges (no barrier: the others leave at once and free their slots). Each output (h, d)
    // sums the waves in wave order, weighted by exp2(m_w - max m) (0 for a wave with
    // m = -inf: one with nothing to add, or with nothing but NaN scores, which stay NaN), whichever
    // wave merges.
    // Head rows are kStRow floats apart (144: the 16 writing lanes of a 16-byte store, 4 heads
    // x 4 row groups, land in distinct banks); a lane's 4 values of dim tile c are dims
    // 16c + 4rg + 0..3 (element e holds dim e ^ 1), one 16-byte store.
    constexpr int kStRow = hd + 16;
    constexpr int kStM = kMaxG * kStRow, kStL = kStM + kMaxG;
    float* st = (float*)vb;
    static_assert(sizeof(vbuf[0]) >= (kStL + kMaxG) * sizeof(float), "merge state");
    const float vunit = exp2i(kNormVExp - ev), vunit_lo = vunit * (1.0f / 4096.0f);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        f32x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e ^ kSwap] = fmaf(ror8(acc[c][e]), vunit_lo, acc[c][e] * vunit);
        if (n < ncols) *(f32x4_t*)&st[n * kStRow + 16 * c + 4 * rg] = v;
    }
    if (n < ncols && rg == 0) {
        st[kStM + n] = m_run;
        st[kStL + n] = l_run;
    }
    // the state writes complete before the count (workgroup-scope release), and the merging
    // wave reads the others' states after it (acquire)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    int arrived = 0;
    if (lane == 0) arrived = atomicAdd(&waves_done, 1);
    arrived = __builtin_amdgcn_readfirstlane(arrived);
    if (arrived != W - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    // one (head, 8-coordinate group) per lane and step: the head's wave weights once, then two
    // 16-byte reads per wave state and two 16-byte stores
    for (int it = lane; it < ncols * (hd / 8); it += 64) {
        const int h = it / (hd / 8), d0 = 8 * (it % (hd / 8));
        if (tq0 + h / G >= qs.seq_lens_count) continue;  // a column past the queries
        const int64_t vec = fhip_idx::partial_vector(h, tq0, G, qh, g);
        const int64_t prow = fhip_idx::partial_row(vec, nsplit, blk);
        float mw[W], M = -__builtin_inff();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            mw[w] = ((const float*)vbuf[w][0])[kStM + h];
            M = fmaxf(M, mw[w]);
        }
        float L = 0.0f;
        f32x4_t A0 = {0.0f, 0.0f, 0.0f, 0.0f}, A1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float* sw = (const float*)vbuf[w][0];
            const float wt = mw[w] == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mw[w] - M);
            L = fmaf(wt, sw[kStL + h], L);
            const f32x4_t a0 = *(const f32x4_t*)&sw[h * kStRow + d0];
            const f32x4_t a1 = *(const f32x4_t*)&sw[h * kStRow + d0 + 4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                A0[k] = fmaf(wt, a0[k], A0[k]);
                A1[k] = fmaf(wt, a1[k], A1[k]);
            }
        }
        float* pa = part_acc + prow * hd + d0;
        *(f32x4_t*)pa = A0;
        *(f32x4_t*)(pa + 4) = A1;
        if (d0 == 0) {  // m back in natural units
            part_ml[prow * 2 + 0] = M == -__builtin_inff() ? M : M * 0.6931471805599453f;
            part_ml[prow * 2 + 1] = L;
        }
    }
}

// ---------------------------------------------------------------------------------------
// 2''. Causal prefill (many queries of one sequence over one block table; head_dim 128, the MFMA
//      kernel's width pairs, G <= 8). The decode kernel would look every code up again for each 8
//      columns; here a workgroup of 4 waves takes kPqCols (query, head) columns of one kv head,
//      32 per wave, and expands each tile of 64 positions once, into fp16 hi and lo rows of K and
//      V centroids in LDS, which all its waves read:
//   S^T = K Q^T and out^T = V^T W^T on v_mfma_f32_32x32x16_f16, each product as hi hi + hi lo +
//   lo hi into one accumulator (what is left out is 2^-22 of the product). lo = x - hi stays a
//   normal fp16 number because every factor is scaled by a power of two first: the centroids by
//   their table's largest magnitude, a query by its own, the weights w = p norm_v by the largest
//   value norm that the column has seen (e_run, for which the accumulators are rescaled like for
//   the running maximum) and by 2^kPqBias: an absolute 2^-38 of the largest w, in fp16 pairs. The
//   scales are exact and leave with the score or the output.
//   Lane layouts are those of the FP16 prefill kernel: lane (n, half) holds 16 positions of column n
//   per 32-position block, which are its own slots of W^T.
// Bound by the MFMA (96 products of 32 clocks per wave and tile) with the lookups (16 8-byte LDS
// reads a thread and tile at 4 bits) and the softmax beside it. 2048 queries from
// position 0, 32 / 8 heads, K4/V2: 177 us in all (194 TFLOP/s of attention, three products each),
// 324 with the decode kernel; 1500 at 1000: 246 and 389 us.
// ---------------------------------------------------------------------------------------
constexpr int kPqWaves = 4;
constexpr int kPqCols = fhip_rules::kPqCols;
constexpr int kPqTile = fhip_rules::kPqTile;
static_assert(kPqCols == 32 * kPqWaves, "a wave has the 32 columns of its MFMA");
constexpr int kPqRowK = 256 + 16;       // bytes per K row in LDS: 16 rows' 16-byte reads on all banks
constexpr int kPqRowV = 256 + 64;       // per V row: the transposed reads of 4 rows x 32 dims
constexpr float kPqBias = 13.0f;        // log2 of the scale that p carries
// log2 that p may exceed it by before a rescale: w < 2^16 (1 - 2^-11) (an fp16 norm's largest share of
// its power of two), which fp16 holds
constexpr float kPqSlack = 3.0f;
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// Codes of one thread's quarter row (32 codes) of a tile: 4 B bytes.
template <int B>
struct Codes32 {
    u32x4 w[B == 8 ? 2 : 1];
};
template <int B>
__device__ __forceinline__ void load_codes32(const uint8_t* p, Codes32<B>& c) {
    if constexpr (B == 8) {
        c.w[0] = *(g_u32x4_any*)p;
        c.w[1] = *(g_u32x4_any*)(p + 16);
    } else if constexpr (B == 4) {
        c.w[0] = *(g_u32x4_any*)p;
    } else {
        const u32x2 v = *(g_u32x2_any*)p;
        c.w[0] = u32x4{v[0], v[1], B == 3 ? *(g_u32_any*)(p + 8) : 0u, 0u};
    }
}
// Expands them: 32 fp16 hi parts at `hi`, lo parts at `lo` (64 bytes each). Tables: B == 8, one
// (hi | lo << 16) word per code; else per byte of two 4-bit codes the words (hi, hi) and (lo, lo).
template <int B>
__device__ __forceinline__ void expand_codes32(const Codes32<B>& c, const u32x2* tab, uint8_t* hi,
                                               uint8_t* lo) {
    u32x4 w = c.w[0];
    if constexpr (B == 2 || B == 3) w = widen32<B>(c.w[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // 8 codes
        u32x4 h, l;
        if constexpr (B == 8) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4 v = quad8((const uint32_t*)tab, c.w[j >> 1][2 * (j & 1) + k]);
                h[2 * k] = __builtin_amdgcn_perm(v[1], v[0], 0x05040100u);
                h[2 * k + 1] = __builtin_amdgcn_perm(v[3], v[2], 0x05040100u);
                l[2 * k] = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
                l[2 * k + 1] = __builtin_amdgcn_perm(v[3], v[2], 0x07060302u);
            }
        } else {
            const u32x4 a = pair2<0>(tab, w[j]), b = pair2<2>(tab, w[j]);
            h = u32x4{a[0], a[2], b[0], b[2]};
            l = u32x4{a[1], a[3], b[1], b[3]};
        }
        *(u32x4*)(hi + 16 * j) = h;
        *(u32x4*)(lo + 16 * j) = l;
    }
}

template <int KB, int VB>
__global__ __launch_bounds__(64 * kPqWaves) __attribute__((amdgpu_waves_per_eu(2))) void
tq_attn_prefill_kernel(float* __restrict__ qrot, Queries qs, PtrPages pg,
                       const float* __restrict__ kcent, const float* __restrict__ vcent, int qh,
                       int kvh, float scale_log2, float* __restrict__ part_ml,
                       float* __restrict__ part_acc, int nsplit, int split_pos, int nqb, int nblk,
                       int fold, bool merged) {
    constexpr int hd = 128;
    __shared__ u32x2 tabs[2][256];
    __shared__ __attribute__((aligned(16))) uint8_t kbuf[2][kPqTile * kPqRowK];  // hi, lo
    __shared__ __attribute__((aligned(16))) uint8_t vbuf[2][kPqTile * kPqRowV];
    __shared__ __attribute__((aligned(16))) float nbuf[2][kPqTile];  // norm_k scale log2(e), norm_v
    __shared__ float tmax;  // the tile's largest norm_v

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // kv head fastest, then the split, then the query block: see the launcher for its order
    const int g = (int)(blockIdx.x % kvh);
    const int rest = (int)(blockIdx.x / kvh);
    const int split = rest % nsplit;
    const int bi = rest / nsplit;
    const int q0 = fhip_idx::prefill_block(bi, nblk, fold) * nqb;
    const int nq = min(nqb, qs.seq_lens_count - q0);
    const int G = qh / kvh;
    const int clen = qs.causal_len(q0 + nq - 1), clen0 = qs.causal_len(q0);
    const int t_begin = split * split_pos;
    // uniform; merged (a single split): every column is written, also one that attends to nothing
    if (!merged && t_begin >= clen) return;
    const int t_end = min(clen, t_begin + split_pos);
    const int32_t* table = qs.table + (int64_t)q0 * qs.table_stride;

    // ---- centroid tables, scaled
    Centroids<KB> ck;
    Centroids<VB> cv;
    ck.load(kcent);
    cv.load(vcent);
    ck.find_exponent();
    cv.find_exponent();
    const int ek = ck.e, ev = cv.e;
    {
        auto fill = [&](u32x2* tab, const float* cent, int bits, int e) {
            for (int b = threadIdx.x; b < 256; b += 64 * kPqWaves) {
                uint32_t h, l;
                if (bits == 8) {
                    split_pair(ldexpf(cent[b], e), 0.0f, h, l);
                    ((uint32_t*)tab)[b] = (h & 0xffffu) | (l << 16);
                } else {
                    const int top = (1 << bits) - 1;
                    split_pair(ldexpf(cent[min(b >> 4, top)], e), ldexpf(cent[min(b & 15, top)], e), h, l);
                    tab[b] = u32x2{h, l};
                }
            }
        };
        fill(tabs[0], kcent, KB, ek);
        fill(tabs[1], vcent, VB, ev);
    }

    // ---- column n of the wave: head col % G of query q0 + col / G
    const int n = lane & 31, half = lane >> 5;
    const int ncols = nq * G;
    const int col = 32 * wave + n;
    const bool col_ok = col < ncols;
    const bool wave_live = 32 * wave < ncols;
    const int cq = col_ok ? col / G : 0;
    const int64_t vec = (int64_t)(q0 + cq) * qh + g * G + (col_ok ? col - cq * G : 0);
    const int lim = col_ok ? min(t_end, qs.causal_len(q0 + cq)) : 0;
    u32x4 bh[8], bl[8];  // the query's hi and lo, dims 16 s + 8 half + 0..7, scaled to below 2^8
    float colscale;      // what a score is multiplied by, with norm_k's factor
    {
        f32x4_t v[8][2];
        const float* src = qrot + vec * hd + 8 * half;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            v[s][0] = *(const f32x4_t*)(src + 16 * s);
            v[s][1] = *(const f32x4_t*)(src + 16 * s + 4);
        }
        float m = 0.0f;
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int k = 0; k < 8; ++k) m = fmaxf(m, fabsf(v[s][k >> 2][k & 3]));
        m = fmaxf(m, __shfl_xor(m, 32));
        const int eq = scale_exponent(m);
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t h, l;
                split_pair(ldexpf(v[s][k >> 1][2 * (k & 1)], eq), ldexpf(v[s][k >> 1][2 * (k & 1) + 1], eq), h, l);
                bh[s][k] = h;
                bl[s][k] = l;
            }
        colscale = exp2i(-eq - ek);
    }

    // ---- tile loads: thread -> row tid / 4, quarter tid % 4 (32 codes); threads of wave 0 the norms.
    // The row's page is looked up per thread (a wave's 16 rows are one page).
    const int row = threadIdx.x >> 2, quarter = threadIdx.x & 3;
    const uint32_t koff = fhip_idx::prefill_code_offset(row, quarter, kvh, g, KB);
    const uint32_t voff = fhip_idx::prefill_code_offset(row, quarter, kvh, g, VB);
    const uint32_t noff = fhip_idx::norm_offset(lane, kvh, g);
    Codes32<KB> kc;
    Codes32<VB> vc;
    uint32_t kn = 0, vn = 0;
    bool nok = false;
    // pages of the next tile (lane j < 4: page j), read one tile ahead of their rows
    int page_next = -1;
    auto load_pages = [&](int t0) {
        page_next = lane < 4 && t0 + FHIP_PAGE_TOKENS * lane < t_end ? table[t0 / FHIP_PAGE_TOKENS + lane] : -1;
    };
    uint32_t pok = 0, pages_ok = 0;
    const uint8_t *pk_ = nullptr, *pkn = nullptr, *pv_ = nullptr, *pvn = nullptr;  // lane j < 4: page j
    auto load_addrs = [&]() {
        const bool ok = lane < 4 && pg.valid(page_next);
        pages_ok = (uint32_t)__ballot(ok) & 0xfu;
        if (ok) pg.addrs(page_next, pk_, pkn, pv_, pvn);
    };
    auto load_tile = [&](int t0) {
        pok = pages_ok;
        if ((pok >> wave) & 1u) {  // the wave's rows: page `wave` of the tile
            load_codes32<KB>(addr_of_lane(pk_, wave) + koff, kc);
            load_codes32<VB>(addr_of_lane(pv_, wave) + voff, vc);
        } else {  // any codes: the scores are masked
#pragma unroll
            for (int k = 0; k < (KB == 8 ? 2 : 1); ++k) kc.w[k] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int k = 0; k < (VB == 8 ? 2 : 1); ++k) vc.w[k] = u32x4{0u, 0u, 0u, 0u};
        }
        if (wave == 0) {
            const int j = lane >> 4;
            const uint8_t* a = (const uint8_t*)__shfl((long long)(uintptr_t)pkn, j);
            const uint8_t* b = (const uint8_t*)__shfl((long long)(uintptr_t)pvn, j);
            nok = ((pok >> j) & 1u) && t0 + lane < t_end;
            if (nok) {
                kn = gld2(a + noff);
                vn = gld2(b + noff);
            }
        }
    };
    auto store_tile = [&]() {
        expand_codes32<KB>(kc, tabs[0], kbuf[0] + row * kPqRowK + 64 * quarter, kbuf[1] + row * kPqRowK + 64 * quarter);
        expand_codes32<VB>(vc, tabs[1], vbuf[0] + row * kPqRowV + 64 * quarter, vbuf[1] + row * kPqRowV + 64 * quarter);
        if (wave == 0) {
            const float a = nok ? h2f(kn) * scale_log2 : 0.0f, b = nok ? h2f(vn) : 0.0f;
            nbuf[0][lane] = a;
            nbuf[1][lane] = b;
            const float m = wave_max(fabsf(b));
            if (lane == 0) tmax = m;
        }
    };

    float m_run = -__builtin_inff(), l_run = 0.0f;  // l: the lane half's own positions
    int e_run = -100;  // the column's accumulators are in units of 2^e_run (norm_v below it)
    f32x16_t acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;

    if (t_begin < t_end) {
        load_pages(t_begin);
        load_addrs();
        load_tile(t_begin);
        if (t_begin + kPqTile < t_end) {
            load_pages(t_begin + kPqTile);
            load_addrs();
        }
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) asm volatile("" : "+v"(bh[s]), "+v"(bl[s]));
    for (int t0 = t_begin; t0 < t_end; t0 += kPqTile) {
        __syncthreads();  // the tables are written; every wave is done with the previous tile
        store_tile();
        const uint32_t tile_pok = pok;
        lds_barrier();
        if (t0 + kPqTile < t_end) {
            load_tile(t0 + kPqTile);
            if (t0 + 2 * kPqTile < t_end) load_pages(t0 + 2 * kPqTile);
        }
        if (wave_live) {
            __builtin_amdgcn_s_setprio(1);
            // ---- S^T: element i of block pt is position 32 pt + 8 (i / 4) + 4 half + i % 4
            f32x16_t sc[2];
            const uint8_t* ksrc = kbuf[0] + n * kPqRowK + 16 * half;
            constexpr int kLoPart = kPqTile * kPqRowK;
            constexpr int kAhead = 3;
            auto k_hi = [&](int t) { return *(const u32x4*)(ksrc + (t >> 3) * 32 * kPqRowK + 32 * (t & 7)); };
            auto k_lo = [&](int t) { return *(const u32x4*)(ksrc + kLoPart + (t >> 3) * 32 * kPqRowK + 32 * (t & 7)); };
            u32x4 kh[kAhead + 1], kl[kAhead + 1];
#pragma unroll
            for (int t = 0; t < kAhead; ++t) {
                kh[t] = k_hi(t);
                kl[t] = k_lo(t);
            }
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[pt][i] = 0.0f;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                if (t + kAhead < 16) {
                    kh[(t + kAhead) % (kAhead + 1)] = k_hi(t + kAhead);
                    kl[(t + kAhead) % (kAhead + 1)] = k_lo(t + kAhead);
                }
                const f16x8_t h = __builtin_bit_cast(f16x8_t, kh[t % (kAhead + 1)]);
                const f16x8_t l = __builtin_bit_cast(f16x8_t, kl[t % (kAhead + 1)]);
                const f16x8_t qhi = __builtin_bit_cast(f16x8_t, bh[t & 7]), qlo = __builtin_bit_cast(f16x8_t, bl[t & 7]);
                sc[t >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(l, qhi, sc[t >> 3], 0, 0, 0);
                sc[t >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h, qlo, sc[t >> 3], 0, 0, 0);
                sc[t >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h, qhi, sc[t >> 3], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            const bool masked = !(tile_pok == 0xfu && t0 + kPqTile <= min(t_end, clen0));
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4_t nk = *(const f32x4_t*)&nbuf[0][32 * pt + 8 * j + 4 * half];
#pragma unroll
                    for (int k = 0; k < 4; ++k) sc[pt][4 * j + k] *= nk[k];
                }
            float vmax = tmax;
            if (masked) {
                vmax = 0.0f;  // of the positions that the column sees
#pragma unroll
                for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int p = 32 * pt + 8 * j + 4 * half;
                        const f32x4_t nv = *(const f32x4_t*)&nbuf[1][p];
                        const int end = (tile_pok >> (2 * pt + j / 2)) & 1u ? lim - t0 - p : 0;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            sc[pt][4 * j + k] = k < end ? sc[pt][4 * j + k] : -__builtin_inff();
                            vmax = fmaxf(vmax, k < end ? fabsf(nv[k]) : 0.0f);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                vmax = fmaxf(vmax, __shfl_xor(vmax, 32));
            }
            // ---- online softmax in log2 units
            float cmax = sc[0][0];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i) cmax = fmaxf(cmax, sc[pt][i]);
            cmax = fmaxf(cmax, __shfl_xor(cmax, 32)) * colscale;
            const float m_new = fmaxf(m_run, cmax);
            const int e_new = max(e_run, min(exponent_above(vmax), 17));
            if (__ballot(m_new > m_run + kPqSlack || e_new > e_run) != 0) {
                const float mref = m_new == -__builtin_inff() ? 0.0f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run - mref);  // 0 while m_run is -inf
                l_run *= alpha;
                const float beta = alpha * exp2i(e_run - e_new);
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[d][i] *= beta;
                m_run = m_new;
                e_run = e_new;
            }
            const float ebias = kPqBias - (m_run == -__builtin_inff() ? 0.0f : m_run);
            const float nscale = exp2i(-e_run);
            float psum = 0.0f;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    f32x4_t nv = *(const f32x4_t*)&nbuf[1][32 * pt + 8 * j + 4 * half];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float p = __builtin_amdgcn_exp2f(fmaf(sc[pt][4 * j + k], colscale, ebias));
                        psum += p;
                        const float w = p * (nv[k] * nscale);
                        // a masked position's norm may be infinite or NaN
                        sc[pt][4 * j + k] = masked && p == 0.0f ? 0.0f : w;
                    }
                }
            l_run += psum;
            __builtin_amdgcn_s_setprio(1);
            // ---- out^T: 4 steps of 16 positions
            const uint8_t* vsrc = vbuf[0] + (4 * half + ((lane & 15) >> 2)) * kPqRowV +
                                  2 * (16 * ((lane >> 4) & 1) + 4 * (lane & 3));
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                uint32_t ph[4], pl[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    split_pair(sc[ks >> 1][8 * (ks & 1) + 2 * j], sc[ks >> 1][8 * (ks & 1) + 2 * j + 1], ph[j], pl[j]);
                const f16x8_t wh = __builtin_bit_cast(f16x8_t, u32x4{ph[0], ph[1], ph[2], ph[3]});
                const f16x8_t wl = __builtin_bit_cast(f16x8_t, u32x4{pl[0], pl[1], pl[2], pl[3]});
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    auto tr = [&](const uint8_t* src) -> f16x8_t {
                        typedef short v4s_t __attribute__((ext_vector_type(4)));
                        typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;
                        const v4s_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (lds_v4s_t*)(__attribute__((address_space(3))) uint8_t*)src);
                        const v4s_t b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (lds_v4s_t*)(__attribute__((address_space(3))) uint8_t*)(src + 8 * kPqRowV));
                        return __builtin_bit_cast(f16x8_t, (short __attribute__((ext_vector_type(8)))){
                                                               a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]});
                    };
                    const uint8_t* src = vsrc + 16 * ks * kPqRowV + 64 * d;
                    const f16x8_t vh = tr(src), vl = tr(src + kPqTile * kPqRowV);
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, wh, acc[d], 0, 0, 0);
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, wl, acc[d], 0, 0, 0);
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, wh, acc[d], 0, 0, 0);
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        if (t0 + 2 * kPqTile < t_end) load_addrs();
    }

    l_run += __shfl_xor(l_run, 32);
    if (!col_ok) return;
    // merged: acc / l replaces the query in q_rot, which only this column's lanes have read
    const float unit = exp2i(e_run - ev) * (merged ? (l_run > 0.0f ? 1.0f / l_run : 0.0f) : 1.0f);
    float* dst = merged ? qrot + vec * hd : part_acc + (vec * nsplit + split) * hd;
    if (!merged && half == 0) {
        part_ml[(vec * nsplit + split) * 2 + 0] = m_run * 0.6931471805599453f;
        part_ml[(vec * nsplit + split) * 2 + 1] = l_run;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *(f32x4_t*)(dst + 32 * d + 8 * j + 4 * half) =
                f32x4_t{acc[d][4 * j] * unit, acc[d][4 * j + 1] * unit, acc[d][4 * j + 2] * unit,
                        acc[d][4 * j + 3] * unit};
}

template <class Pages, int KB, int VB>
void launch_mfma_t(const float* qrot, const Queries& q2, const Pages& pg, const float* kcent,
                   const float* vcent, int qh, int kvh, int nsplit, const fhip_rules::TqRoute& route,
                   int64_t wgs, float* ml, float* acc, hipStream_t s) {
    const int tok = route.tok;
    const bool g4 = qh / kvh <= 4 && tok == 1;
    auto go = [&](auto kern, int waves) {
        hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * waves), 0, s, qrot, q2, pg, kcent, vcent,
                           qh, kvh, 1.0f / sqrtf(128.0f), ml, acc, nsplit, nsplit, tok);
    };
    if (route.part == kFinePart)
        go(g4 ? tq_attn_mfma_kernel<Pages, true, KB, VB, 4, kFinePart>
              : tq_attn_mfma_kernel<Pages, false, KB, VB, 4, kFinePart>, 4);
    else if (route.waves == kWavesWide)
        go(g4 ? tq_attn_mfma_kernel<Pages, true, KB, VB, kWavesWide, kSplit>
              : tq_attn_mfma_kernel<Pages, false, KB, VB, kWavesWide, kSplit>, kWavesWide);
    else
        go(g4 ? tq_attn_mfma_kernel<Pages, true, KB, VB, kWavesM, kSplit>
              : tq_attn_mfma_kernel<Pages, false, KB, VB, kWavesM, kSplit>, kWavesM);
}

template <class Pages>
void launch_mfma_split(const float* qrot, const Queries& qsv, const Pages& pg,
                       const float* kcent, const float* vcent, int nq, int qh, int kvh,
                       int nsplit, const fhip_rules::TqRoute& route, int kbits, int vbits, float* ml,
                       float* acc, hipStream_t s) {
    // Causal prefill (queries at consecutive positions of one sequence: one shared block table,
    // lengths from start_pos) groups 8 / G consecutive queries per item so that they share the
    // MFMA columns and every code lookup; decode keeps one query per item.
    // one workgroup per (item, kv head, part-position block): the block count is the
    // partial layout's split count; the (item, block) pairs are padded to a multiple of the
    // XCD count (the kernel's index spreads them, not heads, over the XCDs)
    const int64_t wgs = fhip_rules::tq_decode_workgroups(nq, route.tok, kvh, nsplit);
    Queries q2 = qsv;
    q2.seq_lens_count = nq;
    if (kbits == 8)
        launch_mfma_t<Pages, 8, 8>(qrot, q2, pg, kcent, vcent, qh, kvh, nsplit, route, wgs, ml, acc, s);
    else if (kbits == 3)
        launch_mfma_t<Pages, 3, 3>(qrot, q2, pg, kcent, vcent, qh, kvh, nsplit, route, wgs, ml, acc, s);
    else if (kbits == 2)
        launch_mfma_t<Pages, 2, 2>(qrot, q2, pg, kcent, vcent, qh, kvh, nsplit, route, wgs, ml, acc, s);
    else if (vbits == 2)
        launch_mfma_t<Pages, 4, 2>(qrot, q2, pg, kcent, vcent, qh, kvh, nsplit, route, wgs, ml, acc, s);
    else
        launch_mfma_t<Pages, 4, 4>(qrot, q2, pg, kcent, vcent, qh, kvh, nsplit, route, wgs, ml, acc, s);
}

struct AttnArgs {
    void* out;
    const void* q;
    Queries qs;
    int nq;
    const float *krot, *vrot, *kcent, *vcent;
    int qh, kvh, hd, kbits, vbits;
    void* ws;
    size_t ws_bytes = 0;  // what `ws` holds; 0: what the workspace size function asks for this call
};

template <int KB, int VB, class Pages>
void launch_split(const AttnArgs& a, const Pages& pg, int nsplit, float* ml, float* acc,
                  hipStream_t s) {
    dim3 grid(nsplit, a.kvh, a.nq);
    const int kwords = ((a.hd * a.kbits + 7) / 8 + 3) / 4, vwords = ((a.hd * a.vbits + 7) / 8 + 3) / 4;
    const size_t lds = (size_t)kSub * ((kwords | 1) + (vwords | 1)) * sizeof(uint32_t);
    hipLaunchKernelGGL((tq_attn_split_kernel<KB, VB, Pages>), grid, dim3(256), lds, s,
                       (const float*)a.ws, a.qs, pg, a.kcent, a.vcent, a.kbits, a.vbits, a.qh,
                       a.kvh, a.hd, 1.0f / sqrtf((float)a.hd), ml, acc, nsplit);
}

// Launches the prefill kernel; `merged`: it leaves merged vectors in qrot.
void launch_prefill(float* qrot, const AttnArgs& a, const PtrPages& pg, const fhip_rules::PrefillSplit& ps,
                    bool merged, float* ml, float* acc, hipStream_t s) {
    const int fold = fhip_rules::prefill_fold(ps, a.kvh, fhip_host::cu_count());
    Queries q2 = a.qs;
    q2.seq_lens_count = a.nq;
    auto kern = a.kbits == 8   ? tq_attn_prefill_kernel<8, 8>
                : a.kbits == 3 ? tq_attn_prefill_kernel<3, 3>
                : a.kbits == 2 ? tq_attn_prefill_kernel<2, 2>
                : a.vbits == 2 ? tq_attn_prefill_kernel<4, 2>
                               : tq_attn_prefill_kernel<4, 4>;
    hipLaunchKernelGGL(kern, dim3((unsigned)ps.workgroups), dim3(64 * kPqWaves), 0, s, qrot, q2, pg, a.kcent,
                       a.vcent, a.qh, a.kvh, 1.4426950408889634f / sqrtf(128.0f), ml, acc, ps.nsplit,
                       ps.split_pos, ps.nqb, ps.nblk, fold, merged);
}

template <class Pages>
int launch_attention(const AttnArgs& a, const Pages& pg, hipStream_t s) {
    if (a.nq == 0) return hipSuccess;
    const int max_tokens = a.qs.max_blocks * FHIP_PAGE_TOKENS;
    const bool causal = std::is_same_v<Pages, PtrPages> && !a.qs.seq_lens && a.qs.table_stride == 0;
    const size_t ws_bytes = a.ws_bytes ? a.ws_bytes : fhip_rules::tq_workspace_bytes(a.nq, a.qh, a.hd, max_tokens);
    const fhip_rules::TqRoute route = fhip_rules::tq_route({a.nq, a.qh, a.kvh, a.hd, a.kbits, a.vbits, max_tokens,
                                                            a.qs.kv_len, causal, ws_bytes});
    const fhip_rules::TqLayout layout = fhip_rules::tq_layout(a.nq, a.qh, a.hd, max_tokens, route.part);
    int nsplit = layout.nsplit, split_pos = route.part;
    if (route.kind == fhip_rules::TqRoute::kPrefill) {
        nsplit = route.prefill.nsplit;
        split_pos = route.prefill.split_pos;
    }
    float* qrot = (float*)a.ws;
    float* ml = (float*)((char*)a.ws + layout.off_ml);
    float* acc = (float*)((char*)a.ws + layout.off_acc);
    const int nvec = a.nq * a.qh;
    // Many vectors (prefill): both rotations as batched MFMA products (the VALU kernels'
    // per-workgroup copies of Pi would cross L2 once per 8 vectors); the merged outputs reuse
    // the q_rot buffer, which the split kernel has finished with.
    const bool batched_rot = nvec >= kMfmaRotVecs && a.hd == 128 &&
                             fhip_host::aligned16(a.q) && fhip_host::aligned16(a.out);
    if (batched_rot) {
        const int e = fhip_internal::tq_rotate_rows(a.q, a.krot, qrot, nvec, s);
        if (e != hipSuccess) return e;
    } else if (a.hd == 128 && fhip_host::aligned16(a.krot)) {
        hipLaunchKernelGGL(tq_attn_prerotate128_kernel, dim3((unsigned)ceil_div(nvec, kRot128Vecs)),
                           dim3(512), 0, s, (const uint16_t*)a.q, a.krot, qrot, nvec);
    } else {
        const unsigned rot_groups = (unsigned)ceil_div(nvec, kRotVecs);
        hipLaunchKernelGGL(tq_attn_prerotate_kernel, dim3(rot_groups), dim3(256), 0, s,
                           (const uint16_t*)a.q, a.krot, qrot, a.hd, nvec);
    }
    // one split: the prefill kernel leaves the merged vectors in q_rot
    const bool merged = route.kind == fhip_rules::TqRoute::kPrefill && nsplit == 1 && batched_rot;
    if (route.kind == fhip_rules::TqRoute::kPrefill) {
        if constexpr (std::is_same_v<Pages, PtrPages>)
            launch_prefill(qrot, a, pg, route.prefill, merged, ml, acc, s);
    } else if (route.kind == fhip_rules::TqRoute::kDecode)
        launch_mfma_split(qrot, a.qs, pg, a.kcent, a.vcent, a.nq, a.qh, a.kvh, nsplit, route,
                          a.kbits, a.vbits, ml, acc, s);
    else if (a.kbits == 4 && a.vbits == 4)
        launch_split<4, 4>(a, pg, nsplit, ml, acc, s);
    else if (a.kbits == 4 && a.vbits == 2)
        launch_split<4, 2>(a, pg, nsplit, ml, acc, s);
    else
        launch_split<0, 0>(a, pg, nsplit, ml, acc, s);
    if (batched_rot) {
        if (merged)
            ;
        else if (nsplit <= kMergeWaveMaxSplits)
            hipLaunchKernelGGL(tq_attn_merge_wave_kernel, dim3((unsigned)ceil_div(nvec, 4)),
                               dim3(256), 0, s, a.qs, ml, acc, a.qh, a.hd, nsplit, (int64_t)nvec,
                               qrot, split_pos);
        else
            hipLaunchKernelGGL((tq_attn_combine_kernel<true, true>),
                               dim3((unsigned)ceil_div(nvec, kCombHeads)), dim3(256),
                               combine_lds_bytes(a.hd, nsplit, true), s, a.qs, ml, acc, a.vrot,
                               (uint16_t*)a.out, a.qh, a.hd, nsplit, (int64_t)nvec, qrot, split_pos);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        return fhip_internal::tq_rotate_back_rows(qrot, a.vrot, a.out, nvec, s);
    }
    if (a.hd == 128) {
        auto merge = nsplit <= 4 ? tq_attn_combine128_kernel<4> : tq_attn_combine128_kernel<16>;
        hipLaunchKernelGGL(merge, dim3((unsigned)ceil_div(nvec, kComb128Vecs)),
                           dim3(512), 0, s, a.qs, ml, acc, a.vrot, (uint16_t*)a.out, a.qh, nsplit,
                           (int64_t)nvec, split_pos);
        return hipGetLastError();
    }
    auto comb = a.hd <= kRotLdsMaxHd ? tq_attn_combine_kernel<true> : tq_attn_combine_kernel<false>;
    hipLaunchKernelGGL(comb, dim3((unsigned)ceil_div(nvec, kCombHeads)), dim3(256),
                       combine_lds_bytes(a.hd, nsplit), s, a.qs, ml, acc, a.vrot,
                       (uint16_t*)a.out, a.qh, a.hd, nsplit, (int64_t)nvec, nullptr, split_pos);
    return hipGetLastError();
}

// Split-partial scratch of fhip_launch_attention_paged_tq_noalloc: one copy per device, held
// until the process ends. Host code never passes the name `scratch` to a kernel (on the host
// it is a stand-in, not a device address); it resolves each device's address once with
// hipGetSymbolAddress and passes that.
constexpr size_t kNoAllocScratchBytes = FHIP_TQ_ATTN_SCRATCH_BYTES;
__device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];

// The scratch address on `dev`, looked up on the first call for that device (made current for
// the lookup, then restored).
hipError_t scratch_on_device(int dev, void** out) {
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return e;
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (cur != dev) {
            hipError_t e2 = hipSetDevice(cur);
            if (e == hipSuccess) e = e2;
        }
        if (e != hipSuccess) return e;
        if (!ptr) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

bool attn_shape_ok(int qh, int kvh, int hd, int kbits, int vbits) {
    return kvh > 0 && qh > 0 && qh % kvh == 0 && qh / kvh <= kMaxG && hd % 8 == 0 && hd > 0 &&
           hd <= kMaxHd && kbits >= 1 && kbits <= 8 && vbits >= 1 && vbits <= 8 &&
           (hd * kbits + 7) / 8 <= kMaxPd && (hd * vbits + 7) / 8 <= kMaxPd && 256 % (hd / 8) == 0;
}

}  // namespace

extern "C" {

size_t fhip_attention_tq_workspace_bytes(int batch, int num_q_heads, int head_dim,
                                         int max_blocks) {
    if (batch <= 0 || num_q_heads <= 0 || head_dim <= 0 || max_blocks <= 0) return 0;
    return fhip_rules::tq_workspace_bytes(batch, num_q_heads, head_dim, max_blocks * FHIP_PAGE_TOKENS);
}

int fhip_launch_attention_tq_decode(void* output, const void* q, const int32_t* block_table,
                                    const int32_t* seq_lens, int batch, int max_blocks,
                                    int num_pages, const void* k_packed_pool,
                                    const void* k_norms_pool, const void* v_packed_pool,
                                    const void* v_norms_pool, int64_t page_k_packed_bytes,
                                    int64_t page_k_norm_bytes, int64_t page_v_packed_bytes,
                                    int64_t page_v_norm_bytes, const float* k_rotation,
                                    const float* v_rotation, const float* k_centroids,
                                    const float* v_centroids, int num_q_heads, int num_kv_heads,
                                    int head_dim, int key_bits, int value_bits, void* workspace,
                                    fhip_stream_t stream) {
    if (batch < 0 || max_blocks <= 0 || num_pages < 0 ||
        !attn_shape_ok(num_q_heads, num_kv_heads, head_dim, key_bits, value_bits))
        return hipErrorInvalidValue;
    if ((int64_t)batch * num_q_heads > (int64_t)1 << 30 || batch > 65535 ||
        max_blocks * (int64_t)FHIP_PAGE_TOKENS > kMaxTokensTq)
        return hipErrorInvalidValue;
    // each page stride must cover a page: the kernels read rows [0, 16) of every page
    const int64_t pdk = (head_dim * key_bits + 7) / 8, pdv = (head_dim * value_bits + 7) / 8;
    if (page_k_packed_bytes < (int64_t)FHIP_PAGE_TOKENS * num_kv_heads * pdk ||
        page_v_packed_bytes < (int64_t)FHIP_PAGE_TOKENS * num_kv_heads * pdv ||
        page_k_norm_bytes < (int64_t)FHIP_PAGE_TOKENS * num_kv_heads * 2 ||
        page_v_norm_bytes < (int64_t)FHIP_PAGE_TOKENS * num_kv_heads * 2)
        return hipErrorInvalidValue;
    if (batch == 0) return hipSuccess;
    if (!output || !q || !block_table || !seq_lens || !k_packed_pool || !k_norms_pool ||
        !v_packed_pool || !v_norms_pool || !k_rotation || !v_rotation || !k_centroids ||
        !v_centroids || !workspace)
        return hipErrorInvalidValue;
    AttnArgs a;
    a.out = output;
    a.q = q;
    a.qs = Queries{block_table, max_blocks, max_blocks, seq_lens, 0, 0, batch};
    a.nq = batch;
    a.krot = k_rotation;
    a.vrot = v_rotation;
    a.kcent = k_centroids;
    a.vcent = v_centroids;
    a.qh = num_q_heads;
    a.kvh = num_kv_heads;
    a.hd = head_dim;
    a.kbits = key_bits;
    a.vbits = value_bits;
    a.ws = workspace;
    PoolPages pg{(const uint8_t*)k_packed_pool, (const uint8_t*)k_norms_pool,
                 (const uint8_t*)v_packed_pool, (const uint8_t*)v_norms_pool,
                 page_k_packed_bytes, page_k_norm_bytes, page_v_packed_bytes, page_v_norm_bytes,
                 num_pages};
    return launch_attention(a, pg, fhip_host::as_stream(stream));
}

int fhip_launch_attention_tq_decode_ptrs(void* output, const void* q, const int32_t* block_table,
                                         const int32_t* seq_lens, int batch, int max_blocks,
                                         int num_pages, const void** k_packed_ptrs,
                                         const void** k_norms_ptrs, const void** v_packed_ptrs,
                                         const void** v_norms_ptrs, const float* k_rotation,
                                         const float* v_rotation, const float* k_centroids,
                                         const float* v_centroids, int num_q_heads,
                                         int num_kv_heads, int head_dim, int key_bits,
                                         int value_bits, void* workspace,
                                         fhip_stream_t stream) {
    if (batch < 0 || max_blocks <= 0 || num_pages < 0 ||
        !attn_shape_ok(num_q_heads, num_kv_heads, head_dim, key_bits, value_bits))
        return hipErrorInvalidValue;
    if ((int64_t)batch * num_q_heads > (int64_t)1 << 30 || batch > 65535 ||
        max_blocks * (int64_t)FHIP_PAGE_TOKENS > kMaxTokensTq)
        return hipErrorInvalidValue;
    if (batch == 0) return hipSuccess;
    if (!output || !q || !block_table || !seq_lens || (num_pages > 0 && (!k_packed_ptrs ||
        !k_norms_ptrs || !v_packed_ptrs || !v_norms_ptrs)) || !k_rotation || !v_rotation ||
        !k_centroids || !v_centroids || !workspace)
        return hipErrorInvalidValue;
    AttnArgs a;
    a.out = output;
    a.q = q;
    a.qs = Queries{block_table, max_blocks, max_blocks, seq_lens, 0, 0, batch};
    a.nq = batch;
    a.krot = k_rotation;
    a.vrot = v_rotation;
    a.kcent = k_centroids;
    a.vcent = v_centroids;
    a.qh = num_q_heads;
    a.kvh = num_kv_heads;
    a.hd = head_dim;
    a.kbits = key_bits;
    a.vbits = value_bits;
    a.ws = workspace;
    PtrPages pg{(const uint8_t* const*)k_packed_ptrs, (const uint8_t* const*)k_norms_ptrs,
                (const uint8_t* const*)v_packed_ptrs, (const uint8_t* const*)v_norms_ptrs,
                num_pages};
    return launch_attention(a, pg, fhip_host::as_stream(stream));
}

}  // extern "C"

namespace fhip_internal {

int attention_tq_decode_ptrs_staged(void* output, const void* q, const int32_t* block_table,
                                    const int32_t* seq_lens, int batch, int max_blocks,
                                    int table_stride, int num_pages, const void** k_packed_ptrs,
                                    const void** k_norms_ptrs, const void** v_packed_ptrs,
                                    const void** v_norms_ptrs, const float* k_rotation,
                                    const float* v_rotation, const float* k_centroids,
                                    const float* v_centroids, int num_q_heads, int num_kv_heads,
                                    int head_dim, int key_bits, int value_bits, void* workspace,
                                    hipStream_t stream) {
    if (batch < 0 || max_blocks <= 0 || num_pages < 0 || table_stride < max_blocks ||
        !attn_shape_ok(num_q_heads, num_kv_heads, head_dim, key_bits, value_bits))
        return hipErrorInvalidValue;
    if ((int64_t)batch * num_q_heads > (int64_t)1 << 30 || batch > 65535 ||
        max_blocks * (int64_t)FHIP_PAGE_TOKENS > kMaxTokensTq)
        return hipErrorInvalidValue;
    if (batch == 0) return hipSuccess;
    if (!output || !q || !block_table || !seq_lens || (num_pages > 0 && (!k_packed_ptrs ||
        !k_norms_ptrs || !v_packed_ptrs || !v_norms_ptrs)) || !k_rotation || !v_rotation ||
        !k_centroids || !v_centroids || !workspace)
        return hipErrorInvalidValue;
    AttnArgs a;
    a.out = output;
    a.q = q;
    a.qs = Queries{block_table, table_stride, max_blocks, seq_lens, 0, 0, batch};
    a.nq = batch;
    a.krot = k_rotation;
    a.vrot = v_rotation;
    a.kcent = k_centroids;
    a.vcent = v_centroids;
    a.qh = num_q_heads;
    a.kvh = num_kv_heads;
    a.hd = head_dim;
    a.kbits = key_bits;
    a.vbits = value_bits;
    a.ws = workspace;
    PtrPages pg{(const uint8_t* const*)k_packed_ptrs, (const uint8_t* const*)k_norms_ptrs,
                (const uint8_t* const*)v_packed_ptrs, (const uint8_t* const*)v_norms_ptrs,
                num_pages};
    return launch_attention(a, pg, stream);
}

}  // namespace fhip_internal

extern "C" {

// The reference interface: one sequence, num_tokens queries at positions
// start_pos .. start_pos + num_tokens - 1, per-block pointer arrays. `ws` holds the split
// partials (fhip_attention_tq_workspace_bytes(num_tokens, qh, hd, ceil(kv_len / 16)) bytes);
// null asks for a stream-ordered allocation freed on the same stream.
static int attention_paged_tq_ref(void* output, const void* q, const int* block_table,
                                  const void** k_packed_ptrs, const void** k_norms_ptrs,
                                  const void** v_packed_ptrs, const void** v_norms_ptrs,
                                  const float* k_rotation, const float* v_rotation,
                                  const float* k_centroids, const float* v_centroids,
                                  int num_tokens, int num_q_heads, int num_kv_heads, int head_dim,
                                  int kv_len, int start_pos, int key_bits, int value_bits,
                                  int k_packed_dim_per_head, int v_packed_dim_per_head,
                                  void* ws, size_t ws_bytes, hipStream_t s) {
    if (num_tokens < 0 || kv_len < 0 || start_pos < 0 || kv_len > kMaxTokensTq ||
        !attn_shape_ok(num_q_heads, num_kv_heads, head_dim, key_bits, value_bits) ||
        k_packed_dim_per_head != (head_dim * key_bits + 7) / 8 ||
        v_packed_dim_per_head != (head_dim * value_bits + 7) / 8 || num_tokens > 65535)
        return hipErrorInvalidValue;
    if (num_tokens == 0) return hipSuccess;
    if (!output || !q || !k_rotation || !v_rotation || !k_centroids || !v_centroids)
        return hipErrorInvalidValue;
    const int nblocks = (kv_len + FHIP_PAGE_TOKENS - 1) / FHIP_PAGE_TOKENS;
    if (nblocks > 0 && (!block_table || !k_packed_ptrs || !k_norms_ptrs || !v_packed_ptrs ||
                        !v_norms_ptrs))
        return hipErrorInvalidValue;
    const int mb = nblocks > 0 ? nblocks : 1;
    const size_t need = fhip_rules::tq_workspace_bytes(num_tokens, num_q_heads, head_dim, mb * FHIP_PAGE_TOKENS);
    const bool own = ws == nullptr;
    if (!own && ws_bytes < need) return hipErrorInvalidValue;
    if (own) {
        ws_bytes = need;
        hipError_t e = hipMallocAsync(&ws, ws_bytes, s);
        if (e != hipSuccess) return e;
    }
    AttnArgs a;
    a.out = output;
    a.q = q;
    a.qs = Queries{(const int32_t*)block_table, 0, mb, nullptr, kv_len, start_pos, num_tokens};
    a.nq = num_tokens;
    a.krot = k_rotation;
    a.vrot = v_rotation;
    a.kcent = k_centroids;
    a.vcent = v_centroids;
    a.qh = num_q_heads;
    a.kvh = num_kv_heads;
    a.hd = head_dim;
    a.kbits = key_bits;
    a.vbits = value_bits;
    a.ws = ws;
    a.ws_bytes = ws_bytes;
    PtrPages pg{(const uint8_t* const*)k_packed_ptrs, (const uint8_t* const*)k_norms_ptrs,
                (const uint8_t* const*)v_packed_ptrs, (const uint8_t* const*)v_norms_ptrs,
                0x7fffffff};
    int r = launch_attention(a, pg, s);
    if (own) {
        hipError_t e2 = hipFreeAsync(ws, s);
        if (r == hipSuccess) r = e2;
    }
    return r;
}

int fhip_launch_attention_paged_tq(void* output, const void* q, const int* block_table,
                                   const void** k_packed_ptrs, const void** k_norms_ptrs,
                                   const void** v_packed_ptrs, const void** v_norms_ptrs,
                                   const float* k_rotation, const float* v_rotation,
                                   const float* k_centroids, const float* v_centroids,
                                   int num_tokens, int num_q_heads, int num_kv_heads,
                                   int head_dim, int kv_len, int start_pos, int key_bits,
                                   int value_bits, int k_packed_dim_per_head,
                                   int v_packed_dim_per_head, fhip_stream_t stream) {
    return attention_paged_tq_ref(output, q, block_table, k_packed_ptrs, k_norms_ptrs,
                                  v_packed_ptrs, v_norms_ptrs, k_rotation, v_rotation,
                                  k_centroids, v_centroids, num_tokens, num_q_heads,
                                  num_kv_heads, head_dim, kv_len, start_pos, key_bits,
                                  value_bits, k_packed_dim_per_head, v_packed_dim_per_head,
                                  nullptr, 0, fhip_host::as_stream(stream));
}

int fhip_launch_attention_paged_tq_noalloc(void* output, const void* q, const int* block_table,
                                           const void** k_packed_ptrs, const void** k_norms_ptrs,
                                           const void** v_packed_ptrs, const void** v_norms_ptrs,
                                           const float* k_rotation, const float* v_rotation,
                                           const float* k_centroids, const float* v_centroids,
                                           int num_tokens, int num_q_heads, int num_kv_heads,
                                           int head_dim, int kv_len, int start_pos, int key_bits,
                                           int value_bits, int k_packed_dim_per_head,
                                           int v_packed_dim_per_head, fhip_stream_t stream) {
    if (num_tokens < 0 || kv_len < 0 || num_q_heads <= 0 || head_dim <= 0)
        return hipErrorInvalidValue;
    if (num_tokens == 0) return hipSuccess;
    const int nblocks = (kv_len + FHIP_PAGE_TOKENS - 1) / FHIP_PAGE_TOKENS;
    const size_t need = fhip_rules::tq_workspace_bytes(num_tokens, num_q_heads, head_dim,
                                     (nblocks > 0 ? nblocks : 1) * FHIP_PAGE_TOKENS);
    static_assert(fhip_rules::kTqFineBytes <= kNoAllocScratchBytes, "finer splits never make a call too large");
    if (need > kNoAllocScratchBytes) return hipErrorOutOfMemory;
    hipStream_t s = fhip_host::as_stream(stream);
    int dev = -1;
    hipError_t e = hipStreamGetDevice(s, &dev);
    if (e != hipSuccess) return e;
    void* ws = nullptr;
    if ((e = scratch_on_device(dev, &ws)) != hipSuccess) return e;
    return attention_paged_tq_ref(output, q, block_table, k_packed_ptrs, k_norms_ptrs,
                                  v_packed_ptrs, v_norms_ptrs, k_rotation, v_rotation,
                                  k_centroids, v_centroids, num_tokens, num_q_heads,
                                  num_kv_heads, head_dim, kv_len, start_pos, key_bits,
                                  value_bits, k_packed_dim_per_head, v_packed_dim_per_head, ws,
                                  kNoAllocScratchBytes, s);
}

int fhip_launch_attention_paged_tq_ws(void* output, const void* q, const int* block_table,
                                      const void** k_packed_ptrs, const void** k_norms_ptrs,
                                      const void** v_packed_ptrs, const void** v_norms_ptrs,
                                      const float* k_rotation, const float* v_rotation,
                                      const float* k_centroids, const float* v_centroids,
                                      int num_tokens, int num_q_heads, int num_kv_heads,
                                      int head_dim, int kv_len, int start_pos, int key_bits,
                                      int value_bits, int k_packed_dim_per_head,
                                      int v_packed_dim_per_head, void* workspace,
                                      size_t workspace_bytes, fhip_stream_t stream) {
    if (!workspace) return hipErrorInvalidValue;
    return attention_paged_tq_ref(output, q, block_table, k_packed_ptrs, k_norms_ptrs,
                                  v_packed_ptrs, v_norms_ptrs, k_rotation, v_rotation,
                                  k_centroids, v_centroids, num_tokens, num_q_heads,
                                  num_kv_heads, head_dim, kv_len, start_pos, key_bits,
                                  value_bits, k_packed_dim_per_head, v_packed_dim_per_head,
                                  workspace, workspace_bytes, fhip_host::as_stream(stream));
}

}  // extern "C"
