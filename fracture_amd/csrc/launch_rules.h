// Which kernel, split and workspace a launch takes, from its sizes alone: called by the launchers and,
// through tq_attn_index_host.cpp, by the CPU tests. Host code.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace fhip_rules {

inline int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------------------
// FP16 decode: waves per 1024-position split, of `items` splits (splits x kv heads x head blocks x query
// groups) over block tables of max_tokens positions. Times in us, 1 / 2 / 4 / 8 waves, 32 / 8 heads of
// 128 unless said otherwise; one wave is what there was before waves shared a split.
//   Up to 256 items eight waves hide one another's memory latency (one sequence of 1000: 67 / 31 / 23 /
//     19), up to 512 four (64 of 1000: 109 / 51 / 45 / 48), up to 1024 two (64 of 2000: 145 / 99 / 109 /
//     106; of 250 .. 2000: 130 / 66 / 83 / 76). Far beyond, one wave per split fills the chip, and more only
//     add merges and idle waves (64 of 4000: 185 / 214 / 199 / 202; 256 of 200: 40 / 48 / 58 / 83).
//   Between, to 1536 items, one wave is a second turn that is half empty, or emptier where the batch is ragged.
//     Four waves: 48 of 3000 160 / 124 / 121, of 375 .. 3000 134 / 72 / 79; 64 / 8 heads, 64 of 3000 154 / 175
//     / 162, of 375 .. 3000 137 / 112 / 110. At head_dim 64 two: 96 of 2000, 16 / 8 heads, 96 / 86 / 95, of
//     250 .. 2000 74 / 54 / 58. Not on tables below half a split (192 of 300, 64 / 8 heads).
//   Head_dim 256 takes two waves to 1024 items (64 of 4000, 16 / 4 heads: 194 / 195 / 218, of 500 .. 4000 176 /
//     133 / 170), head_dim 32 to 768 (8 / 8 heads, 32 of 3000: 41 / 36 / 40, of 375 .. 3000 40 / 27 / 28; 64
//     of 2000, 1024 items: 41 / 48 / 50).
//   A wave takes 1024 / W positions of the split, so waves past the end of a short table are idle. At
//     head_dim 128 they cost less than two splits sharing a workgroup, as one wave per split has them
//     (64 of 100: 16.9 with one, 14.1 with two or four): halved while one wave would hold the table, not
//     below two. Elsewhere they lose from about two thirds of the table on (64 of 16, 16 / 8 heads of 64: 7.5
//     / 8.3 / 8.6 / 11.0; of 300, 8 / 8 heads of 32: 15.2 / 18.5 / 17.3 / 15.1; of 400: 18.2 / 21.7 /
//     17.9 / 16.4), but for two waves of head_dim 64 and 256 (128 of 300, 16 / 8 heads of 64: 26.6 / 26.5;
//     of 700 49 / 41).
inline int paged_waves(int64_t items, int hd, int max_tokens) {
    const int span = std::min(max_tokens, 1024);
    if (items > 1024) return items <= 1536 && span > 512 ? (hd == 128 ? 4 : hd == 64 ? 2 : 1) : 1;
    int w = items <= 256 ? 8 : items <= 512 ? 4 : 2;
    if (hd == 128) {
        while (w > 2 && span * w <= 1024) w /= 2;
        return w;
    }
    if (w == 2) return hd == 32 ? (items <= 768 && span >= 768 ? 2 : 1) : span > 128 ? 2 : 1;
    return span * w >= 1536 ? w : 1;
}

// ---------------------------------------------------------------------------------------
// Causal prefill on the tiled kernels: query blocks of `cols` (query, head) columns, and as many splits of
// the positions as bring the launch to `groups` workgroups, of whole tiles each.
// ---------------------------------------------------------------------------------------
struct PrefillSplit {
    int nqb, nblk;          // queries per block, blocks
    int nsplit, split_pos;  // splits, positions of each
    int64_t workgroups;
};
inline PrefillSplit prefill_split(int nq, int G, int kvh, int cols, int tile, int64_t groups, int extent,
                                  int max_splits) {
    PrefillSplit p;
    p.nqb = cols / G;
    p.nblk = (int)div_up(nq, p.nqb);
    const int64_t base = (int64_t)p.nblk * kvh;
    extent = std::max(extent, 1);
    const int64_t want = std::min<int64_t>(std::max<int64_t>(div_up(groups, base), 1), max_splits);
    p.split_pos = (int)(div_up(div_up(extent, want), tile) * tile);
    p.nsplit = (int)div_up(extent, p.split_pos);
    p.workgroups = base * p.nsplit;
    return p;
}

// Blocks start from the last (the longest contexts) down. Where all of a single split's fit at once, two to a
// CU, those of the second half go up from the first instead (their index from this one on), so that a
// long block shares its CU with a short one.
inline int prefill_fold(const PrefillSplit& p, int kvh, int cus) {
    return p.nsplit == 1 && p.workgroups > cus && p.workgroups <= 2 * (int64_t)cus ? cus / kvh : 0;
}

// ---------------------------------------------------------------------------------------
// TurboQuant attention
// ---------------------------------------------------------------------------------------
constexpr int kTqSplit = 1024;     // positions per split partial
constexpr int kTqFinePart = 256;   // and in launches too small to fill the chip with those
constexpr size_t kTqFineBytes = (size_t)24 << 20;  // the largest workspace that finer splits may ask for

// The workspace: q_rot, then (m, l) and the accumulators of the split partials, one split per `part`
// positions.
struct TqLayout {
    size_t off_ml, off_acc, bytes;
    int nsplit;
};
inline TqLayout tq_layout(int nq, int qh, int hd, int max_tokens, int part) {
    TqLayout l;
    l.nsplit = max_tokens > 0 ? (max_tokens + part - 1) / part : 1;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t qrot = (size_t)nq * qh * hd * sizeof(float);
    const size_t ml = (size_t)nq * qh * l.nsplit * 2 * sizeof(float);
    const size_t acc = (size_t)nq * qh * l.nsplit * hd * sizeof(float);
    l.off_ml = al(qrot);
    l.off_acc = l.off_ml + al(ml);
    l.bytes = l.off_acc + al(acc);
    return l;
}
// Small launches may split finer, where the layout of kTqFinePart positions stays within kTqFineBytes. The
// size a caller is asked for covers that layout too, of every table with as many kTqSplit-position splits,
// and at every smaller size (it never falls as an argument grows): a workspace serves the tables that it
// would serve if no launch split finer, and one warmed up at the largest call the smaller ones.
inline size_t tq_workspace_bytes(int nq, int qh, int hd, int max_tokens) {
    const int whole = (int)(div_up(std::max(max_tokens, 1), kTqSplit) * kTqSplit);
    return std::max(tq_layout(nq, qh, hd, whole, kTqSplit).bytes,
                    std::min(tq_layout(nq, qh, hd, whole, kTqFinePart).bytes, kTqFineBytes));
}

// The (K, V) code widths that the MFMA kernels are built for: the default cache, equal widths, and the
// protected layers' 8 bits. On the VALU split kernel, which takes any other pair, 8 sequences of 1000
// .. 8000 measured 438 us at 8 bits, 200 at 3 and 191 at 2, against 50, 43 and 44 on the MFMA kernel.
inline bool tq_mfma_widths(int kbits, int vbits) {
    return (kbits == 4 && (vbits == 4 || vbits == 2)) ||
           (kbits == vbits && (kbits == 2 || kbits == 3 || kbits == 8));
}

struct TqCall {
    int nq, qh, kvh, hd, kbits, vbits;
    int max_tokens;   // positions that the block table describes
    int kv_len;       // causal: positions of the sequence
    bool causal;      // consecutive queries of one sequence over one table
    size_t ws_bytes;  // of the workspace, at least tq_layout's at kTqSplit
};
struct TqRoute {
    enum Kind { kValu, kDecode, kPrefill } kind;
    int part;   // positions per partial of the layout
    int waves;  // kDecode: per workgroup
    int tok;    // kDecode: queries per workgroup (its MFMA columns are tok x G)
    PrefillSplit prefill;
};
constexpr int kXcds = 8;
inline int64_t tq_decode_workgroups(int nq, int tok, int kvh, int nsplit) {
    return div_up(div_up(nq, tok) * nsplit, kXcds) * kXcds * kvh;
}
constexpr int kPqCols = 128;        // prefill kernel: columns per workgroup
constexpr int kPqTile = 64;         // positions per tile
constexpr int64_t kPqGroups = 512;  // workgroups wanted: the two per CU that fit at once
constexpr int kRotBatch = 4096;     // vectors from which both rotations are batched MFMA products ...
constexpr int kMergeSplits = 8;     // ... and the splits that the merge before the second takes in one wave

// The prefill kernel's splits, at most `most`: the shortest of those that fill kPqGroups, those that stay
// within it and those of the wave merge. A tile takes a workgroup 4.3 us alone on its CU and 6.3 beside another;
// more than kMergeSplits splits of a batch are merged in LDS, 25 us slower. 32 / 8 heads unless said otherwise:
// 64 queries at 3000 of 64 / 8 heads 8 splits (96 us in 12), at 30000 16 (223 us, 269 in 8), 130 at 30000 12
// (264; 288 in 13, 299 in 8), 200 at 30000 8 or 9 (359; 475 in 10).
inline PrefillSplit tq_prefill_split(int nq, int G, int kvh, int extent, int most, bool batch) {
    const int64_t base = div_up(nq, kPqCols / G) * kvh;
    PrefillSplit best = {};
    int64_t least = 0;
    for (const int64_t limit : {(int64_t)most, kPqGroups / base, batch ? (int64_t)kMergeSplits : (int64_t)most}) {
        const PrefillSplit p = prefill_split(nq, G, kvh, kPqCols, kPqTile, kPqGroups, extent,
                                             (int)std::max<int64_t>(std::min<int64_t>(limit, most), 1));
        const int64_t rest = p.workgroups % kPqGroups;
        const int64_t ns = p.split_pos / kPqTile * (p.workgroups / kPqGroups * 6300 + (rest > 256 ? 6300 : rest ? 4300 : 0)) +
                           (batch && p.nsplit > kMergeSplits ? 25000 : 0);
        if (!least || ns < least) best = p, least = ns;
    }
    return best;
}

// The route of a call. Times in us at K4/V2 unless said otherwise.
//   The decode kernel in 256-position parts, four waves of one chunk each, where that makes at most three
//   workgroups per CU and 48 parts: four times the workgroups of 1024-position parts (one sequence of
//   1000, 32 / 8 heads: 16.5 us; 23.3 in 1024-position blocks of four waves, 31.2 of two). More
//   parts make the merge the larger half (one sequence of 20000, 79 parts: 28.3 and 25.6; 32000: 37.3 and
//   26.8). More workgroups run in turns; up to 1536 of them are still the shorter way where the
//   1024-position parts are more than one per CU, whose second turn is nearly empty or short: with up to 384 of
//   those, or 512 where some hold only a sequence's rest (K4/V4, 32 / 8 heads: 20 sequences of 1200 23.9 and
//   29.7, 40 of 1000 32.3 and 34.8, 32 of 1400 32.0 and 32.0, of 175 .. 1400 25.1 and 30.3; but 64 of 378
//   28.4 and 26.8, 28 of 1000 25.2 and 25.2).
//   Else 1024-position parts: four waves up to 512 workgroups (64 sequences of 1000: 35.4 us, with two
//   42.4, with eight 38.7; 32 of 2000 32.5, 39.7, 35.7), two beyond (64 of 3000, 1536 workgroups: 62.6 us,
//   with four 64.8).
//   Causal calls of more workgroups than that (than 256 where the codes' expansion is dearer, at 3 and 8
//   bits) go to the prefill kernel where it is the shorter one: a tile takes a workgroup 4.3 us, with up to
//   one workgroup per CU, and a decode workgroup of 1024 positions 0.042 us of the whole chip, twice that at
//   3 and 8 bits. It also has to have 96 workgroups, 128 at 4 and 2 bits where its partials are merged by a
//   kernel of their own (130 queries at 3000, 120 workgroups: 88 us decoded and 95, at 8 bits 122 and 101).
//   32 / 8 heads, decoded and tiled: 8 queries at 8000 26.6 and 31.9, 32 at 3000 33.2 and 32.9, 32 at 8000 52
//   and 40, 8 at 30000 51 and 59, 200 at 1000 of 64 / 8 heads (104 workgroups of 16 tiles) 90 and 92.
inline TqRoute tq_route(const TqCall& c) {
    TqRoute r;
    const int G = c.qh / c.kvh;
    r.kind = TqRoute::kValu;
    r.part = kTqSplit;
    r.waves = 0;
    r.tok = 1;
    r.prefill = {};
    if (!tq_mfma_widths(c.kbits, c.vbits) || c.hd != 128 || G > 8) return r;
    r.kind = TqRoute::kDecode;
    r.tok = c.causal && c.nq > 1 && G < 8 ? 8 / G : 1;
    const TqLayout fine = tq_layout(c.nq, c.qh, c.hd, c.max_tokens, kTqFinePart);
    const bool fits = fine.bytes <= std::min(c.ws_bytes, kTqFineBytes);
    const int nsplit = tq_layout(c.nq, c.qh, c.hd, c.max_tokens, kTqSplit).nsplit;
    const int64_t wgs = tq_decode_workgroups(c.nq, r.tok, c.kvh, nsplit);
    // decode in a second turn of 1024-position parts
    const bool second = wgs > 256 && wgs <= (nsplit > 1 ? 512 : 384) && !(c.causal && c.nq > 1);
    if (fits && fine.nsplit <= 48 &&
        tq_decode_workgroups(c.nq, r.tok, c.kvh, fine.nsplit) <= (second ? 1536 : 768)) {
        r.part = kTqFinePart;
        r.waves = 4;
        return r;
    }
    r.waves = wgs <= 512 ? 4 : 2;
    const bool dear = c.kbits == 3 || c.kbits == 8;
    if (c.causal && c.nq > 1 && wgs > (dear ? 256 : 512)) {
        const bool batch = (int64_t)c.nq * c.qh >= kRotBatch;
        r.prefill = tq_prefill_split(c.nq, G, c.kvh, std::min(c.kv_len, c.max_tokens),
                                     fits ? fine.nsplit : nsplit, batch);
        const int64_t tiles = r.prefill.split_pos / kPqTile * div_up(r.prefill.workgroups, 256);
        if (r.prefill.workgroups >= (batch && !dear && r.prefill.nsplit > 1 ? 128 : 96) &&
            tiles * (dear ? 50 : 105) < wgs) {
            r.kind = TqRoute::kPrefill;
            r.part = fits ? kTqFinePart : kTqSplit;
        }
    }
    return r;
}

// ---------------------------------------------------------------------------------------
// Matmul: whether C[M, N] = A[M, K] B[N, K]^T takes the streaming kernel of matmul_skinny.hip instead of the
// library. Two times count: the kernel's, and a call's among others, where the library's host path takes
// 23 us and this one's 9. A decode step between graph launches is bound by the second: 2 layers and a head at
// batch 16, 987 us with it for the 4096-wide projections and 1094 without, at batch 1, 358 with it for
// all of them, 376 for up to 2^25 elements, 433 without.
//   A workgroup's 8 waves share a row's K, so K bounds the kernel: N = 1024, M = 1 / 4 / 16, us of this one and
//   of the library, K = 2048 5.1 / 5.5 / 6.6 and 10.6 / 8.0 / 7.9, 4096 8.3 / 8.5 / 10.4 and 11.0 / 8.3 /
//   8.2, 8192 13.1 / 14.2 / 18.1 and 11.6 / 9.2 / 9.3, 2^18 on N = 16 315 / 351 / 475 and 94 / 80 / 80. It is
//   taken while it stays below the library's call: to 8192 with up to 4 rows, to 4096 with up to 16.
//   Up to 2^25 elements (M = 16, 8192 x 4096: 19.5, the library 15.9, its call 23), and 2^27 with one or two
//   rows, whose product is bound by B's stream either way (14336 x 4096 25.4 and 24.8, 4096 x 14336 25.4 and
//   24.1, 32000 x 4096 48.5 and 54.5; in the step 1.8 us a product faster for all three).
//   Up to 65536 rows of B: beyond, its many short workgroups are the longer way (524288 x 64: 38 and 29).
inline bool matmul_skinny(int m, int n, int k) {
    const int64_t elems = (int64_t)n * k;
    if (m < 1 || m > 16 || n > 65536 || k < 8 || k % 8 != 0) return false;
    if (elems <= (int64_t)1 << 25 && k <= (m <= 4 ? 8192 : 4096)) return true;
    return m <= 2 && elems <= (int64_t)1 << 27 && n >= 4096 && k <= 16384;
}

}  // namespace fhip_rules
