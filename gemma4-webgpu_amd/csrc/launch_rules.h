// Launch rules that are plain functions of a call's sizes, apart from the
// kernels so that they can be checked without a GPU.
#pragma once

#include <stdint.h>

namespace g4 {

// The prefill's merge launches 2^shift workgroup columns per cut query tile;
// shift covers the largest token count among those tiles (at most 128). A
// tile's columns without a token leave at once, but launching them is not free:
// 4 tokens after 100000 cached rows (209 parts, 8 heads) with 16 columns for the
// one tile 28.4 us, with 4 columns 27.0.
inline unsigned token_merge_shift(uint32_t tile_tokens) {
    unsigned s = 0;
    while ((1u << s) < tile_tokens) s++;
    return s;
}

// Scores per thread of softmax's register form (4 or 16), or 0 for the loop
// form. The register form's 1024 threads a head pay for their launch and their
// exchange through LDS from 513 scores on (us in a replayed graph, loop / register:
// 8 heads of 64 scores 3.2 / 3.9, of 400 4.5 / 4.6, of 513 5.0 / 4.7, of 2048
// 7.3 / 4.9), and two such workgroups fill a CU where the loop form's 256 threads
// run eight deep: above 256 heads the line is at 11/4 scores for each head of the launch
// (512 heads of 1024 5.8 / 6.8, of 1500 7.9 / 7.2; 1024 heads of 2048 9.6 / 11.7, of 3000
// 13.3 / 12.8), at 6 with 16 scores a thread, where one workgroup fills a CU (1024
// heads of 5000 23.2 / 26.1, of 7000 32.4 / 26.7; 2048 heads of 7000 48.2 / 47.7).
// Past 16384 scores LDS and the registers hold no more.
inline unsigned softmax_scores_per_thread(uint32_t heads, uint32_t seq_len) {
    if (seq_len <= 512 || seq_len > 16384) return 0;
    const bool few = heads <= 256;
    if (seq_len <= 4096) return few || 4ull * seq_len >= 11ull * heads ? 4 : 0;
    return few || seq_len >= 6ull * heads ? 16 : 0;
}

// attnOutput: whether its chain form takes `workgroups` (64 columns of a head
// each) over seq_len rows on `cus` compute units. The form's products fill 129 KB of LDS,
// so one workgroup runs per CU, and a round of them takes ~1.6 us + 4.4 ns a
// row; the general form's dependent loads take ~107 ns a row whatever the
// number of workgroups. Both meet near 16, 33, 74, 187 and 640 rows at 1, 2, 4, 8
// and 16 rounds, and by 1024 rows at 32 (V then leaves the L2, and the general form
// doubles). Measured (us in a replayed graph, general / chain), 8 heads of 256: 4 rows
// 2.3 / 3.1, 12 rows 3.0 / 3.2, 16 rows 3.4 / 3.1, 2048 rows 206 / 11.8; 256 heads of 256
// (4 rounds): 48 rows 8.6 / 10.3, 96 rows 13.3 / 11.0; 256 of 512 (8): 128 rows 16.5 / 19.8,
// 256 rows 29.2 / 25.0; 512 of 512 (16): 512 rows 59.6 / 64.0, 768 rows 93.9 / 81.6; 1024
// of 512 (32): 768 rows 138 / 166, 1024 rows 250 / 206.
inline bool attn_output_chain(uint64_t workgroups, uint32_t seq_len, uint32_t cus) {
    const uint64_t rounds = (workgroups + cus - 1) / cus;
    return seq_len >= 1024 || seq_len >= 14 * rounds + 2 * rounds * rounds;
}

// argmax over few logits takes 256 threads of 4-byte loads: a 1024-thread
// workgroup's launch and its sixteen candidates cost more than three more loads
// in turn (us in a replayed graph, 1024 threads / 256: 1 logit 2.5 / 2.2, 255
// logits 2.7 / 2.2, 768 logits 2.7 / 2.3).
inline bool argmax_small(uint32_t size) { return size <= 768; }

}  // namespace g4
