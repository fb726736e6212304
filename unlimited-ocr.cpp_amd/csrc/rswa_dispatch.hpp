// Which attention calls run query-tiled, shared by the launcher and a host-side check.
#pragma once

#include <algorithm>

namespace uocr_hip {

#ifdef __HIP__
#define UOCR_HD __host__ __device__
#else
#define UOCR_HD
#endif

// Time of a tile whose rows see up to `keys` keys, in `passes` requests one after the
// other: 128 keys per step of a workgroup. Tiles run side by side, so this is also a
// call's time until they fill the chip. ns, fitted to: one pass of 64..1156 keys 11..60 us
// at head_dim 128, 11.5..36 at 64; 8 passes of 4 keys 51 and 34.
UOCR_HD inline float rswa_tile_ns(int head_dim, int keys, int passes) {
    const float steps = (float)((keys + 127u) / 128u);
    return head_dim == 128 ? 6600.0f + passes * (400.0f + 5200.0f * steps) : 5000.0f + passes * (800.0f + 3000.0f * steps);
}

// n times the time of `pairs` (row, head) pairs walked one by one, side by side, where n
// rows have `keys` keys together. Rows of one request share its keys in L2, and the
// less the more other requests there are among 32 rows and the fewer heads share a
// KV head (`apart`: others x kv_heads / heads, 5 others at most). ns, fitted to: chunks of 52..256
// rows 43 ps per pair and key (19 at head_dim 64), 2 requests of 60 rows 52, 6 of 20 64, 10 of 12
// 88, 128 of 4 126; 10 of 12 with 16 heads over 4 58.
UOCR_HD inline float rswa_rows_ns(int head_dim, float pairs, int n, float keys, float apart) {
    const float row = head_dim == 128 ? 9.5f : 4.2f;
    const float key = head_dim == 128 ? 0.043f + 0.015f * apart : 0.019f + 0.007f * apart;
    return n * 3000.0f + pairs * (n * row + key * keys);
}

// Query-tiled where the tiles' time is below the row kernel's. `last` keys are
// seen by the last row, `mean` by a row on average: known for one cache of known length.
// Elsewhere a prompt from position 0 is assumed, as many keys as the call has rows (the
// capacity of the cache says nothing about them); near the line a longer cache adds about
// the same to both sides. us by rows / tiled, rows at position p:
//   10 heads of 128: 64 rows at 0 9.7 / 10.0, at 900 40 / 50; 80 at 0 11.5 / 11.9, at 216 22.2 /
//   22.0; 98 at 0 13.5 / 11.4, at 216 24.0 / 22.3; 128 at 0 17.5 / 11.3, at 900 65 / 55
//   32 heads over 8 of 128: 52 rows at 100 26.2 / 16.8, at 450 52 / 29
//   12 heads of 64: 98 rows at 0 9.2 / 15.5, at 450 21.0 / 20.8; 128 at 100 14.7 / 11.6, at 216 18.2 /
//   14.8, at 900 39 / 33
//   8 heads over 2 of 64: 128 rows at 900 24 / 33; 160 at 0 10.3 / 11.0, at 216 16.7 / 14.8, at 900 30.8 / 32.9
inline bool rswa_tiles_win(long long rows, int heads, int head_dim, int last, int mean) {
    if (rows * heads < 512 || (head_dim != 64 && head_dim != 128)) return false;
    return rswa_tile_ns(head_dim, head_dim == 64 ? std::max(last, 256) : last, 1) <
           rswa_rows_ns(head_dim, (float)rows * heads, 1, (float)mean, 0.0f);
}

// ... for a call whose rows' positions the host does not know: max_len bounds them (0:
// unknown)
inline bool rswa_call_tiled(long long rows, int heads, int head_dim, int max_len) {
    const int last = (int)std::min<long long>(rows, max_len > 0 ? max_len : 0x7fffffff);
    return rswa_tiles_win(rows, heads, head_dim, last, last - last / 2);
}

// ... and for rows q_start .. of one cache with kv_len keys
inline bool rswa_one_cache_tiled(long long rows, int heads, int head_dim, int kv_len, int q_start, bool causal) {
    if (!causal) return rswa_tiles_win(rows, heads, head_dim, kv_len, kv_len);
    const long long last = std::max(0ll, std::min<long long>(kv_len, q_start + rows));
    const long long first = std::max(0ll, std::min<long long>(kv_len, q_start + 1ll));
    return rswa_tiles_win(rows, heads, head_dim, (int)last, (int)((first + last) / 2));
}

}  // namespace uocr_hip
