// Which attention calls run query-tiled, shared by the launcher and a host-side check.
#pragma once

#include <algorithm>

namespace uocr_hip {

// Query-tiled from this many (row, head, key) triples on, with as many keys per row as the
// call has rows (a prompt's rows see each other; the capacity of the cache says nothing
// about them, and a few rows over many keys give too few tiles) and no more than
// max_len (0: unknown). Below, the row kernel's shorter start wins. us by rows / tiled, 10
// heads of 128: prompts of 52 rows 8.8 / 12.6, 60 9.5 / 12.7, 80 12.0 / 12.7, 100 14.4 /
// 12.7, 200 29.9 / 16.7; 64 rows at position 936 41 / 49. 8 heads of 64: 100 rows 7.5 /
// 12.8, 200 13.6 / 12.9.
inline bool rswa_call_tiled(long long rows, int heads, int head_dim, int max_len) {
    if (rows * heads < 512 || (head_dim != 64 && head_dim != 128)) return false;
    const long long pairs = rows * heads, keys = max_len > 0 ? std::min<long long>(rows, max_len) : rows;
    const long long least = head_dim == 128 ? 98304 : 262144;
    return pairs >= (least + keys - 1) / keys;
}

}  // namespace uocr_hip
