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
//     106; of 250 .. 2000: 130 / 66 / 83 / 76). Beyond, one wave per split fills the chip, and more only
//     add merges and idle waves (64 of 4000: 185 / 214 / 199 / 202; 256 of 200: 40 / 48 / 58 / 83).
//   A wave takes 1024 / W positions of the split, so waves past the end of a short table are idle. At
//     head_dim 128 they cost less than two splits sharing a workgroup, as one wave per split has them
//     (64 of 100: 16.9 with one, 14.1 with two or four): halved while one wave would hold the table, not
//     below two. Elsewhere they lose from about two thirds of the table on (64 of 16, 16 / 8 heads of 64: 7.5
//     / 8.3 / 8.6 / 11.0; of 300, 8 / 8 heads of 32: 15.2 / 18.5 / 17.3 / 15.1; of 400: 18.2 / 21.7 /
//     17.9 / 16.4).
//   Head_dim 32 and 256 take one wave from 513 items: uniform batches lose (64 of 2000, 8 / 8 heads of
//     32: 41 / 47; of 4000, 16 / 4 heads of 256: 186 / 196).
inline int paged_waves(int64_t items, int hd, int max_tokens) {
    if (items > 1024) return 1;
    int w = items <= 256 ? 8 : items <= 512 ? 4 : hd == 64 || hd == 128 ? 2 : 1;
    const int span = std::min(max_tokens, 1024);
    if (hd == 128) {
        while (w > 2 && span * w <= 1024) w /= 2;
        return w;
    }
    return span * w >= 1536 ? w : 1;
}

}  // namespace fhip_rules
