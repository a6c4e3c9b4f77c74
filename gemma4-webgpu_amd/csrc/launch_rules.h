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

}  // namespace g4
