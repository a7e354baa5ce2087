// Host build of the MFMA decode-attention kernel's index arithmetic (tq_attn_index.h), for the
// CPU bounds check of the kernel's global accesses, and of the launchers' rules (launch_rules.h). Each entry evaluates the same inline
// functions the kernel calls, over all 64 lanes where an index depends on the lane.
#include <stdint.h>

#include <algorithm>

#include "launch_rules.h"
#include "tq_attn_index.h"

extern "C" {

// Per-lane tables for kv head g of kvh: K code offsets k_off[pt][lane] (pt = 0..3) and split
// page slots k_page[lane]; V copy offsets v_off[lane]; norm offsets n_off[lane] and slots
// n_page[lane]; query coordinate offsets q_off[s8][lane] (floats, s8 = 0..7).
int fhip_idx_lane_tables(int kvh, int g, uint32_t* k_off, int32_t* k_page, uint32_t* v_off,
                         uint32_t* n_off, int32_t* n_page, int32_t* q_off) {
    if (kvh < 1 || g < 0 || g >= kvh || !k_off || !k_page || !v_off || !n_off || !n_page || !q_off)
        return -1;
    for (int lane = 0; lane < 64; ++lane) {
        for (int pt = 0; pt < 4; ++pt)
            k_off[pt * 64 + lane] = fhip_idx::k_offset(lane, kvh, g, 4) + pt * fhip_idx::k_tile_stride(kvh, 4);
        k_page[lane] = fhip_idx::k_page(lane);
        v_off[lane] = fhip_idx::v_offset(lane, kvh, g);
        n_off[lane] = fhip_idx::norm_offset(lane, kvh, g);
        n_page[lane] = fhip_idx::norm_page(lane);
        for (int s8 = 0; s8 < 8; ++s8) q_off[s8 * 64 + lane] = fhip_idx::q_lane_offset(lane, s8);
    }
    return 0;
}

// 2-bit V codes: the per-lane load offsets v2_off[lane] for kv head g of kvh.
int fhip_idx_v2_offsets(int kvh, int g, uint32_t* v2_off) {
    if (kvh < 1 || g < 0 || g >= kvh || !v2_off) return -1;
    for (int lane = 0; lane < 64; ++lane) v2_off[lane] = fhip_idx::v2_offset(lane, kvh, g);
    return 0;
}

// Codes of 2, 3, 4 or 8 bits: K offsets k_off[pt][lane] (pt = 0..3) and V load offsets
// v_off[i][lane] with their split page slots v_page[i] (i < 4, or i < 8 at 8 bits); kw and vw are
// the bytes of one K and one V load.
int fhip_idx_code_tables(int kvh, int g, int kbits, int vbits, uint32_t* k_off, uint32_t* v_off,
                         int32_t* v_page, int32_t* kw, int32_t* vw) {
    if (kvh < 1 || g < 0 || g >= kvh || !k_off || !v_off || !v_page || !kw || !vw) return -1;
    if ((kbits != 2 && kbits != 3 && kbits != 4 && kbits != 8) ||
        (vbits != 2 && vbits != 3 && vbits != 4 && vbits != 8))
        return -1;
    *kw = 4 * kbits;
    *vw = vbits == 8 ? 16 : 4 * vbits;
    for (int lane = 0; lane < 64; ++lane) {
        for (int pt = 0; pt < 4; ++pt)
            k_off[pt * 64 + lane] =
                fhip_idx::k_offset(lane, kvh, g, kbits) + pt * fhip_idx::k_tile_stride(kvh, kbits);
        for (int i = 0; i < (vbits == 8 ? 8 : 4); ++i)
            v_off[i * 64 + lane] = vbits == 8   ? fhip_idx::v8_offset(lane, i, kvh, g)
                                   : vbits == 4 ? fhip_idx::v_offset(lane, kvh, g)
                                   : vbits == 3 ? fhip_idx::v3_offset(lane, kvh, g)
                                                : fhip_idx::v2_offset(lane, kvh, g);
    }
    for (int i = 0; i < 8; ++i) v_page[i] = vbits == 8 ? fhip_idx::v8_page(i) : i;
    return 0;
}

// First position of wave `wave` of `waves` in block blk of `part` positions, all of them live.
int32_t fhip_idx_split_begin(int blk, int wave, int waves, int part) {
    return fhip_idx::split_begin(blk, wave, part, fhip_idx::wave_span(part, waves));
}

// Workgroup wg of a launch with kvh kv heads -> its item and kv head.
int fhip_idx_wg_item(int64_t wg, int kvh, int64_t* item, int32_t* g) {
    if (kvh < 1 || wg < 0 || !item || !g) return -1;
    int gg;
    fhip_idx::wg_item(wg, kvh, *item, gg);
    *g = gg;
    return 0;
}

// Workgroup lin of the VALU split kernel's grid (nsplit, kvh, nq) -> (split, kv head, query).
int fhip_idx_split_grid_item(int64_t lin, int nsplit, int kvh, int nq, int32_t* split,
                             int32_t* kvhead, int32_t* qi) {
    const int64_t total = (int64_t)nsplit * kvh * nq;
    if (nsplit < 1 || kvh < 1 || nq < 1 || lin < 0 || lin >= total || !split || !kvhead || !qi)
        return -1;
    int s, h, q;
    fhip_idx::split_grid_item(lin, total, nsplit, kvh, s, h, q);
    *split = s;
    *kvhead = h;
    *qi = q;
    return 0;
}

// Wave `wave` of `waves` in block blk of `part` positions, `clen` the longest causal length that it sees: its
// split [t_begin, t_end), and per lane the block-table column of split page `lane` and whether that page holds
// positions of the split.
int fhip_idx_wave_split(int blk, int wave, int waves, int part, int clen, int32_t* t_begin, int32_t* t_end,
                        int32_t* column, uint8_t* in_split) {
    if (blk < 0 || wave < 0 || waves < 1 || part < waves || clen <= blk * part || !t_begin || !t_end || !column ||
        !in_split)
        return -1;
    const int span = fhip_idx::wave_span(std::min(part, clen - blk * part), waves);
    *t_begin = fhip_idx::split_begin(blk, wave, part, span);
    *t_end = std::min(clen, *t_begin + span);
    for (int lane = 0; lane < 64; ++lane) {
        int c;
        in_split[lane] = fhip_idx::split_page_column(*t_begin, *t_end, lane, c) ? 1 : 0;
        column[lane] = c;
    }
    return 0;
}

// A whole 1024-position block's two waves, the split ending at t_end.
int fhip_idx_split(int blk, int wave, int t_end, int32_t* t_begin, int32_t* column, uint8_t* in_split) {
    if (blk < 0 || wave < 0 || !t_begin || !column || !in_split) return -1;
    *t_begin = fhip_idx_split_begin(blk, wave, 2, 1024);
    for (int lane = 0; lane < 64; ++lane) {
        int c;
        in_split[lane] = fhip_idx::split_page_column(*t_begin, t_end, lane, c) ? 1 : 0;
        column[lane] = c;
    }
    return 0;
}

// The first split page of the chunk starting at t0.
int32_t fhip_idx_chunk_first_page(int t0, int t_begin) {
    return fhip_idx::chunk_first_page(t0, t_begin);
}

// Per lane: the rotated-query vector its MFMA column reads, and whether the column is live.
int fhip_idx_q_vectors(int tq0, int tok, int G, int nq, int qh, int g, int64_t* vec, uint8_t* live) {
    if (G < 1 || tok < 1 || !vec || !live) return -1;
    for (int lane = 0; lane < 64; ++lane) {
        bool l;
        vec[lane] = fhip_idx::q_vector(lane, tq0, tok, G, nq, qh, g, l);
        live[lane] = l ? 1 : 0;
    }
    return 0;
}

// The partial row the merge writes for head column h of the item (query group tq0, kv head g,
// block blk).
int64_t fhip_idx_partial_row(int h, int tq0, int G, int qh, int g, int nsplit, int blk) {
    return fhip_idx::partial_row(fhip_idx::partial_vector(h, tq0, G, qh, g), nsplit, blk);
}

// Route of a TurboQuant attention call (launch_rules.h): out[0..5] = kind (0 VALU, 1 decode, 2 prefill), positions per
// partial, waves, queries per workgroup, splits, positions per split; returns the workspace bytes of its
// layout.
int64_t fhip_rule_tq_route(int nq, int qh, int kvh, int hd, int kbits, int vbits, int max_tokens, int kv_len,
                           int causal, int64_t ws_bytes, int32_t* out) {
    const fhip_rules::TqRoute r = fhip_rules::tq_route(
        {nq, qh, kvh, hd, kbits, vbits, max_tokens, kv_len, causal != 0, (size_t)ws_bytes});
    const fhip_rules::TqLayout l = fhip_rules::tq_layout(nq, qh, hd, max_tokens, r.part);
    const bool prefill = r.kind == fhip_rules::TqRoute::kPrefill;
    out[0] = r.kind;
    out[1] = r.part;
    out[2] = r.waves;
    out[3] = r.tok;
    out[4] = prefill ? r.prefill.nsplit : l.nsplit;
    out[5] = prefill ? r.prefill.split_pos : r.part;
    return (int64_t)l.bytes;
}
// The workspace size a caller is asked for.
int64_t fhip_rule_tq_workspace(int nq, int qh, int hd, int max_tokens) {
    return (int64_t)fhip_rules::tq_workspace_bytes(nq, qh, hd, max_tokens);
}

// Waves per split of an FP16 decode launch (launch_rules.h).
int fhip_rule_paged_waves(int64_t items, int hd, int max_tokens) {
    return fhip_rules::paged_waves(items, hd, max_tokens);
}

// Whether a matmul takes the streaming kernel (launch_rules.h).
int fhip_rule_matmul_skinny(int m, int n, int k) { return fhip_rules::matmul_skinny(m, n, k); }

// Split of a tiled prefill (launch_rules.h): out[0..4] = queries per block, blocks, splits, positions per split,
// workgroups.
void fhip_rule_prefill_split(int nq, int G, int kvh, int cols, int tile, int64_t groups, int extent, int max_splits,
                             int64_t* out) {
    const fhip_rules::PrefillSplit p = fhip_rules::prefill_split(nq, G, kvh, cols, tile, groups, extent, max_splits);
    out[0] = p.nqb;
    out[1] = p.nblk;
    out[2] = p.nsplit;
    out[3] = p.split_pos;
    out[4] = p.workgroups;
}
int fhip_rule_prefill_fold(int nsplit, int64_t workgroups, int kvh, int cus) {
    fhip_rules::PrefillSplit p{};
    p.nsplit = nsplit;
    p.workgroups = workgroups;
    return fhip_rules::prefill_fold(p, kvh, cus);
}
int fhip_idx_prefill_block(int bi, int nblk, int fold) { return fhip_idx::prefill_block(bi, nblk, fold); }
uint32_t fhip_idx_prefill_code_offset(int row, int quarter, int kvh, int g, int bits) {
    return fhip_idx::prefill_code_offset(row, quarter, kvh, g, bits);
}

}  // extern "C"
