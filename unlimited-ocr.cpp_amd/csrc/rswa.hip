// R-SWA attention and KV-cache writes (the step after the MoE path):
// counterparts of src/kernels/cuda/rswa_attention.cu and the host cache
// semantics of src/scheduler/kv_cache.cpp. Cache layout as the reference's:
// [capacity, kv_heads, head_dim] f32 per request (a batch of requests: slot s
// at base + s * batch_cap * kv_heads * head_dim); rows 0..P-1 hold the first
// prefill ("reference tokens"), rows P..P+W-1 a ring of the last W decoded
// tokens.
//
// Attention, row kernel: one workgroup per (query row, head), 8 waves splitting the keys.
// A wave takes groups of 8 consecutive keys (groups w, w + 8, ...): lane
// (j, p) = (lane / 8, lane % 8) holds key j's dims 4p + 32i .. + 3 (i < HDP / 32)
// of K and V (each load: the 8 lanes of a key read one contiguous 128-byte run),
// with the next two groups' K and V loads (one for head_dim > 128) issued
// before the current group is used. Scores reduce over the 8 lanes of a key, the online softmax runs per
// wave (max, rescale, sum over the group's keys), and each lane accumulates
// p * V for its own key slot; the 8 key slots and then the 8 waves are
// combined at the end (flash-decoding). Decode is HBM-bound: every (row, head)
// streams kv_len * head_dim * 8 bytes of K and V.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <initializer_list>
#include <mutex>
#include <string>

#include "common.hpp"
#include "launch.hpp"
#include "rswa_dispatch.hpp"
#include "xcd_order.hpp"
#include "uocr_hip/moe_capi.h"

namespace uocr_hip {
namespace {

constexpr int kRswaWaves = 8;

struct RswaArgs {
    const float* q;
    const float* kc;
    const float* vc;
    float* out;
    int heads, kv_heads, head_dim;
    float scale;
    int mode;  // 0: one cache, kv_len (causal: q_start); 1: same, kv_len = *d_len;
               // 2: batch (slot d_slots[b], length d_len[slot]); 3: ragged (slot d_slots[t], rows 0..d_pos[t])
    int kv_len, q_start, causal;
    const int* d_len;
    const int* d_slots;
    const int* d_pos;
    int batch_cap;
    int n_chunks;  // > 1: keys split over blockIdx.z, partial (m, l, o) records to part
    float* part;   // [rows][heads][n_chunks][kRswaRec]
    float pairs, kv_share;  // (tiles) rows * heads, kv_heads / heads
    bool full;  // (tiles) they take most of the chip
};

// one partial record: m, l, (pad), then o[head_dim]
constexpr int kRswaRec = 256 + 4;

// LDS of one row's wave results
template <int HDP, int WAVES>
struct RowLds {
    float m[WAVES], l[WAVES];
    __attribute__((aligned(16))) float acc[WAVES][HDP];
};

template <int HDP, int WAVES>
__device__ __forceinline__ void row_attention(const RswaArgs& a, int row, int head, int chunk, RowLds<HDP, WAVES>& s) {
#include "rswa_row_body.hpp"
}

template <int HDP>
__global__ __launch_bounds__(kRswaWaves * 64) void rswa_kernel(RswaArgs a) {
    constexpr int WAVES = kRswaWaves;
    __shared__ RowLds<HDP, WAVES> s;
    const int row = blockIdx.x, head = blockIdx.y, chunk = blockIdx.z;
#include "rswa_row_body.hpp"
}

// ---------------------------------------------------------------------------
// Query-tiled attention (prefill): a workgroup of 4 waves takes 32 consecutive
// query rows of one head on v_mfma_f32_32x32x2_f32; the waves split the keys
// in blocks of 32 (block w, w + 4, ...) with an online softmax per wave and
// are combined at the end, as in the row kernel. f32 throughout.
//   * S^T = K Q^T: lane (i, h) = (lane % 32, lane / 32) holds key i's operand and
//     query i's, step s of unit pair j taking dims 8 j + 4 h + s; so one 16-byte read
//     serves four MFMAs. K blocks come by DMA into LDS, their 16-byte units
//     permuted per key (unit u at u ^ key) so that the reads of 16 keys
//     cover all banks;
//   * D holds keys 8 (r / 4) + 4 h + r % 4 of query i, which is the operand
//     layout of O^T = V^T P^T with the keys taken in that order: the
//     probabilities never leave their lane. V rows come straight from global
//     memory, 16 bytes (dims 4 i .. + 3) per lane: dim-block b's MFMA takes
//     dims 4 i + b.
// The rows of a tile may belong to several requests (slots): one pass over the
// keys per distinct slot, rows of other slots masked. Where that costs more
// than walking the rows one by one (tile_pays), the tile is left to row
// workers, extra workgroups at the grid's end.
// Its parts: the f32 MFMAs (154 TFLOP/s on a large product: 35 us of the call
// below; busy for 31% of the time by the counters), the masked half of the blocks on the
// diagonal, the start of a workgroup (9k cycles to its first scores) and the grid's end.
// Measured (rocprofv3) at 4 requests of 358..1000 rows, 10 heads of 128: 711 us
// row by row, 123 us tiled; error against 64 bits 1.41e-7 both ways (one
// chain per score and per output is 7% faster and 3.2e-7 off). Not kept: 8
// waves per workgroup, one per CU (the start is then exposed: 160 us); all 16
// V rows in flight with Q in registers (spills).
// ---------------------------------------------------------------------------
constexpr int kTileQ = 32;        // query rows per tile
constexpr int kTileWaves = 4;
constexpr int tile_resident(int head_dim) { return head_dim == 64 ? 3 : 2; }  // workgroups per CU (40 / 80 KiB of LDS each)
constexpr int kTileSort = kTileWaves * 64;  // tiles that a call orders by their keys (one per thread)
static_assert(kTileSort <= 256, "a tile's index has 8 bits of its sort key");
constexpr int kTileCost = 4;      // row-blocks that a tile's key block costs

// slot and key limit (rows attended, 0 past the end) of query row t
__device__ __forceinline__ void row_limit(const RswaArgs& a, int rows, int t, int& slot, int& limit) {
    slot = -1;
    limit = 0;
    if (t >= rows) return;
    if (a.mode == 3) {
        slot = a.d_slots[t];
        limit = a.d_pos[t] + 1;
    } else {
        const int kv_len = a.mode == 1 ? *a.d_len : a.kv_len;
        slot = 0;
        limit = a.causal ? min(kv_len, a.q_start + t + 1) : kv_len;
    }
    limit = max(limit, 0);
}

// over the 32 lanes of a half wave: DPP within 16 lanes, one LDS exchange between them
// (the row workers ask about every tile, five exchanges per value kept them 6 us)
template <class Op>
__device__ __forceinline__ int half_reduce(int v, Op op) {
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true));   // quad_perm 1, 0, 3, 2
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true));   // quad_perm 2, 3, 0, 1
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true));  // row_half_mirror
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true));  // row_mirror
    return op(v, __shfl_xor(v, 16, 64));
}
__device__ __forceinline__ int half_max(int v) {
    return half_reduce(v, [](int x, int y) { return max(x, y); });
}
__device__ __forceinline__ int half_sum(int v) {
    return half_reduce(v, [](int x, int y) { return x + y; });
}

// Whether a tile runs as a tile; every lane holds row l % 32's slot and limit, the
// answer is that of its half wave's rows (a wave can ask about two tiles). Runs of rows
// of one slot count as passes. (Its buffer loads address up to 2 GiB of a request's
// cache.) Two lines:
//   * throughput: a key block of a pass costs about four row-blocks of the row walk (9
//     against 2.2 ns on the whole chip). Passes are taken at the tile's most keys; where the
//     tiles fill more than 9/16 of the chip, the first request's at its own: a tile where a
//     long request ends then stays a tile, but a call with idle CUs is done earlier by the
//     workers (us, one / own, 8 heads over 2 of 64: 8 requests of 150..500 rows 39 / 33, 4
//     of 90..300 15 / 17.5)
//   * time (rswa_tile_ns, rswa_rows_ns): the passes follow each other while the call's rows
//     are walked side by side. us, always tiled / by this rule / the row kernel, 10 heads
//     of 128: 30 requests of 4 rows 51 / 10.6 / 12.6, 16 of 10 28.1 / 12.9 / 16.6, 100 of 10
//     29.9 / 29.1 / 93, 6 of 20 at position 400 71 / 42 / 45, 2 of 60 at 300 40 / 25.7 / 34.5. A
//     last tile with few rows of one request runs beside its other tiles, at the same time
//     (359 rows, 16 heads of 64: 15.3, by the workers 17.9), unless the call is as short as
//     the tile (20 requests of 5 rows 11.8 / 9.7 / 10.5).
template <int HD>
__device__ __forceinline__ bool tile_pays(const RswaArgs& a, int slot, int limit) {
    const int lane = threadIdx.x & 63;
    const int slot0 = lane & 32 ? __builtin_amdgcn_readlane(slot, 32) : __builtin_amdgcn_readlane(slot, 0);
    const int most0 = half_max(slot == slot0 ? limit : 0), most1 = half_max(slot == slot0 ? 0 : limit);
    const int most = max(most0, most1), blocks = half_sum((limit + 31) / 32);
    const int prev = __builtin_amdgcn_update_dpp(0, slot, 0x138, 0xf, 0xf, true);  // the lane before (wave_shr:1)
    const bool first = slot >= 0 && ((lane & 31) == 0 || slot != prev);
    const int runs = __popc((uint32_t)(__ballot(first) >> (lane & 32)));
    const int live = __popc((uint32_t)(__ballot(slot >= 0) >> (lane & 32)));
    const int passes = a.full ? (most0 + 31) / 32 + (runs - 1) * ((most1 + 31) / 32) : runs * ((most + 31) / 32);
    return (long long)most * a.kv_heads * HD * 4 <= 0x7fffffffll && passes * kTileCost <= blocks &&
           ((runs == 1 && live == kTileQ) ||
            rswa_tile_ns(HD, most, runs) * (runs == 1 ? 1.25f * live : (float)kTileQ) <=
                rswa_rows_ns(HD, a.pairs, live, 32 * blocks - 16 * live, min(runs - 1, 5) * a.kv_share));
}

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int HD>
struct TileLds {
    __attribute__((aligned(16))) float k[kTileWaves][32 * HD];  // K blocks, then the waves' outputs
    union {
        __attribute__((aligned(16))) float q[32 * HD];
        struct {  // once the last scores are done
            float m[kTileWaves][32], l[kTileWaves][32];
            uint32_t redo;  // rows with a non-finite result
        };
    };
};

template <int HD>
__global__ __launch_bounds__(kTileWaves * 64, tile_resident(HD)) void rswa_tile_kernel(RswaArgs a, int rows, int n_tiles, bool sort) {
    constexpr int U = HD / 4;    // 16-byte units per row
    constexpr int NB = HD / 32;  // dims per lane of V, dim-blocks of O
    union Lds {
        TileLds<HD> t;
        RowLds<HD, kTileWaves> r;
        struct {
            RowLds<HD, kTileWaves> r;
            uint8_t pays[kTileSort];
        } w;
        struct {
            __attribute__((aligned(16))) int pos[kTileSort];
            int tile;
        };
    };
    __shared__ Lds s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (scalar: the loads' offsets and buffers are)
    const int i = lane & 31, h = lane >> 5;
    int slot, limit;
    if ((int)blockIdx.x >= n_tiles * a.heads) {  // row worker: the rows of the tiles that don't pay
        // The rows of all such tiles, in order, go to the workers in turn: none is
        // without a row while another has two more. us, restarting with worker 0 at
        // every tile (320 of 512 had all the rows) / this / the row kernel: 10 heads of
        // 128, requests of one row with 1000 keys: 128 289 / 220 / 219, 256 550 / 433 /
        // 431; 100 requests of 3 rows 456 / 370 / 369.
        int next = blockIdx.x - n_tiles * a.heads;  // this worker's next row, counted from tile t0 on
        const int n_workers = gridDim.x - n_tiles * a.heads;
        auto& c = s.w;
        for (int t0 = 0; t0 < n_tiles; t0 += kTileSort) {
            const int n = min(kTileSort, n_tiles - t0);
            for (int k0 = 0; k0 < n; k0 += 4 * 2 * kTileWaves) {  // one tile per half wave, four in flight
                int sl[4], li[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) row_limit(a, rows, (t0 + k0 + j * 2 * kTileWaves + 2 * wave + h) * kTileQ + i, sl[j], li[j]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = k0 + j * 2 * kTileWaves + 2 * wave + h;
                    const bool pays = tile_pays<HD>(a, sl[j], li[j]);
                    if (i == 0 && k < n) c.pays[k] = pays;
                }
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kTileSort / 64; ++q) {
                uint64_t left = __ballot(q * 64 + lane < n && !c.pays[q * 64 + lane]);
                for (; left; left &= left - 1) {
                    const int tile = t0 + q * 64 + __builtin_ctzll(left);
                    // Grouped heads: 8 rows side by side, so that the heads of a row meet
                    // in one XCD's L2 (200 requests of one row, 1000 keys, 8 / 2 heads of
                    // 64: 133 -> 63 us). One head per KV head: the heads of a row side by
                    // side, a whole row of the cache (128 requests, 10 heads of 128: 226 -> 220)
                    const int m = min(kTileQ, rows - tile * kTileQ);
                    const int near = a.heads > a.kv_heads && m % kXcds == 0 ? kXcds : 1;
                    for (; next < m * a.heads; next += n_workers) {
                        const int g = next / near;
                        row_attention<HD, kTileWaves>(a, tile * kTileQ + g / a.heads * near + next % near, g % a.heads, 0, c.r);
                        __syncthreads();
                    }
                    next -= m * a.heads;
                }
            }
            __syncthreads();  // (pays is read)
        }
        return;
    }
    // The tiles with the most keys first, so that the grid's end is made of
    // short ones (sort: more workgroups than the chip holds at once): the tile
    // whose last row's position has rank blockIdx.x / heads (ties by index). Beyond kTileSort tiles: in reverse order.
    const int rank = blockIdx.x / a.heads, head = blockIdx.x % a.heads;
    int tile = n_tiles - 1 - rank;
    if (a.mode == 3 && n_tiles <= kTileSort && sort) {
        // (position, index) in one word: distinct whatever the positions
        const int mine = tid < n_tiles
                             ? (int)((uint32_t)a.d_pos[min(tid * kTileQ + kTileQ, rows) - 1] << 8 | (255 - tid))
                             : INT_MIN;
        s.pos[tid] = mine;
        __syncthreads();
        if (tid < n_tiles) {
            int before = 0;
#pragma unroll 4
            for (int j = 0; j < n_tiles; j += 4) {
                const int4 p = *reinterpret_cast<const int4*>(&s.pos[j]);
                before += (p.x > mine) + (p.y > mine) + (p.z > mine) + (p.w > mine);
            }
            if (before == rank) s.tile = tid;
        }
        __syncthreads();
        tile = __builtin_amdgcn_readfirstlane(s.tile);
        __syncthreads();
    }
    row_limit(a, rows, tile * kTileQ + i, slot, limit);
    if (!__builtin_amdgcn_readfirstlane(tile_pays<HD>(a, slot, limit))) return;
    const int stride = a.kv_heads * HD;
    const int kvh = head / (a.heads / a.kv_heads);
    constexpr float kLog2e = 1.4426950408889634f;

    // the query rows in LDS (registers are for O and V), units permuted as K's
    for (int u = tid; u < 32 * U; u += kTileWaves * 64) {
        const int r = u / U, c = u % U;
        const float* qr = a.q + ((size_t)min(tile * kTileQ + r, rows - 1) * a.heads + head) * HD;
        *reinterpret_cast<f32x4*>(&s.t.q[r * HD + (c ^ (r % U)) * 4]) = *reinterpret_cast<const f32x4*>(qr + 4 * c);
    }
    __syncthreads();
    float m = -INFINITY, l = 0.0f;  // of query i, over this lane's keys (l) / the wave's (m)
    f32x16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) o[b] = f32x16{};

    float* kbuf = s.t.k[wave];
    uint32_t left = (uint32_t)__ballot(limit > 0);
    while (left) {  // one pass per distinct slot
        const int ps = __builtin_amdgcn_readfirstlane(__shfl(slot, __builtin_ctz(left), 64));
        const bool in = slot == ps && limit > 0;
        left &= ~(uint32_t)__ballot(in);
        const int mylim = in ? limit : 0;
        const int kend = __builtin_amdgcn_readfirstlane(half_max(mylim));
        const size_t base = (a.mode == 3 ? (size_t)ps * a.batch_cap * stride : 0) + (size_t)kvh * HD;
        // buffer loads: keys past kend are out of range and read as zeros (base
        // + kvh * HD: the last key's row ends before the next key's). The key's
        // offset is in the vector offset, which alone is certain to be checked against the size.
        const int bytes = ((kend - 1) * stride + HD) * 4, rowb = stride * 4;
        const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.kc + base), 0, bytes, 0x00020000);
        const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.vc + base), 0, bytes, 0x00020000);
        const int nblk = (kend + 31) / 32;
        // DMA n covers 64 / U keys, unit u of key k at u ^ (k % U)
        // (the asm statements keep the 16 offsets from being hoisted out of the
        // key loop, where they would spill)
        const int kvo = (lane / U) * rowb;
        int ku = ((lane % U) ^ (lane / U)) << 4;
        auto load_k = [&](int blk) {
            asm volatile("" : "+v"(ku));
#pragma unroll
            for (int n = 0; n < U / 2; ++n)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    kr, (__attribute__((address_space(3))) void*)(kbuf + n * 256), 16,
                    kvo + (ku ^ ((n * (64 / U)) % U << 4)) + (blk * 32 + n * (64 / U)) * rowb, 0, 0, 0);
        };
        const int vvo = 4 * h * rowb + NB * i * 4;
        if (wave < nblk) load_k(wave);
        for (int blk = wave; blk < nblk; blk += kTileWaves) {
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the K block has landed
            __builtin_amdgcn_sched_barrier(0);
            // V of this block: rows r < 8 in flight during the scores, the
            // others during the softmax (all 16 at once would spill)
            float v[2][8][NB];
            auto load_v = [&](int half) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int so = (blk * 32 + 16 * half + 8 * (r >> 2) + (r & 3)) * rowb;
                    if constexpr (NB == 4) {
                        const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, vvo + so, 0, 0));
#pragma unroll
                        for (int b = 0; b < 4; ++b) v[half][r][b] = t[b];
                    } else {
                        const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, vvo + so, 0, 0));
#pragma unroll
                        for (int b = 0; b < 2; ++b) v[half][r][b] = __uint_as_float(t[b]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            load_v(0);
            // K reads two unit pairs (8 MFMAs) ahead; the barriers keep the
            // scheduler from hoisting all of them (64 registers)
            // (short chains round less: two at a time, over quarters of the dims)
            f32x16 st[2], sum16;
            f32x4 kv[3], qv[3];
            int ko = i * HD + ((h ^ (i % U)) << 2);
            asm volatile("" : "+v"(ko));
            auto read_k = [&](int j) {
                kv[j % 3] = *reinterpret_cast<const f32x4*>(kbuf + (ko ^ (j << 3)));
                qv[j % 3] = *reinterpret_cast<const f32x4*>(s.t.q + (ko ^ (j << 3)));
            };
            read_k(0);
            read_k(1);
#pragma unroll
            for (int j = 0; j < U / 2; ++j) {
                if (j + 2 < U / 2) read_k(j + 2);
                if (j % (U / 8) == 0) st[0] = st[1] = f32x16{};
#pragma unroll
                for (int c = 0; c < 4; ++c) st[c & 1] = mfma_f32(kv[j % 3][c], qv[j % 3][c], st[c & 1]);
                if (j % (U / 8) == U / 8 - 1) {
                    if (j < U / 8) sum16 = st[0] + st[1];
                    else sum16 += st[0] + st[1];
                    asm volatile("" : "+v"(sum16));  // added here (later, the chains would keep their registers)
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): K is in registers, the buffer is free
            __builtin_amdgcn_sched_barrier(0);
            load_v(1);
            if (blk + kTileWaves < nblk) load_k(blk + kTileWaves);
            __builtin_amdgcn_sched_barrier(0);
            // online softmax of query i over this lane's 16 keys and its partner's
            float p[16], mx = -INFINITY;
            const int lim = mylim - blk * 32 - 4 * h;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                p[r] = 8 * (r >> 2) + (r & 3) < lim ? sum16[r] * a.scale : -INFINITY;
                mx = fmaxf(mx, p[r]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m, mx);
            const float mref = mn == -INFINITY ? 0.0f : mn;
            const float alpha = __builtin_amdgcn_exp2f((m - mref) * kLog2e);
            float sum[4] = {};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                p[r] = __builtin_amdgcn_exp2f((p[r] - mref) * kLog2e);
                sum[r & 3] += p[r];
            }
            l = fmaf(l, alpha, (sum[0] + sum[1]) + (sum[2] + sum[3]));
            m = mn;
            // a block's keys are summed from zero in four chains of 8, then
            // added (rounds less than one chain over all keys)
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    f32x16 ob[2] = {};
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int c = 0; c < 2; ++c)
                            ob[c] = mfma_f32(v[half][4 * c + r][b], p[8 * half + 4 * c + r], ob[c]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        o[b][r] = half ? o[b][r] + (ob[0][r] + ob[1][r]) : fmaf(o[b][r], alpha, ob[0][r] + ob[1][r]);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    }
    // combine the waves: each leaves its unnormalised rows [query][dim] in its
    // own K buffer (unit permuted by the query), then every thread sums
    l += __shfl_xor(l, 32, 64);
    __syncthreads();  // the query rows' place takes m and l
    if (tid == 0) s.t.redo = 0;
    if (h == 0) {
        s.t.m[wave][i] = m;
        s.t.l[wave][i] = l;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int rho = 8 * (r >> 2) + 4 * h + (r & 3);  // dims NB * rho .. + NB - 1
        if constexpr (NB == 4) {
            *reinterpret_cast<f32x4*>(kbuf + i * HD + (rho ^ i) * 4) = f32x4{o[0][r], o[1][r], o[2][r], o[3][r]};
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) kbuf[i * HD + (rho ^ i) * NB + b] = o[b][r];
        }
    }
    __syncthreads();
    for (int u = tid; u < 32 * 32; u += kTileWaves * 64) {
        const int qi = u / 32, rho = u % 32, row = tile * kTileQ + qi;
        const int row_keys = __shfl(limit, qi, 64);
        if (row >= rows) continue;
        float M = -INFINITY, L = 0.0f, acc[NB] = {};
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) M = fmaxf(M, s.t.m[w][qi]);
        if (M != -INFINITY) {
#pragma unroll
            for (int w = 0; w < kTileWaves; ++w) {
                const float f = __builtin_amdgcn_exp2f((s.t.m[w][qi] - M) * kLog2e);
                L = fmaf(s.t.l[w][qi], f, L);
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b] = fmaf(s.t.k[w][qi * HD + (rho ^ qi) * NB + b], f, acc[b]);
            }
        }
        float* op = a.out + ((size_t)row * a.heads + head) * HD + NB * rho;
        bool bad = !(L > 0.0f && L < INFINITY);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            acc[b] = L > 0.0f ? acc[b] / L : 0.0f;
            bad |= !(fabsf(acc[b]) < INFINITY);
        }
        // (a row's threads are one half of a wave)
        if ((uint32_t)(__ballot(bad && row_keys > 0) >> (lane & 32))) {
            if ((lane & 31) == 0) atomicOr(&s.t.redo, 1u << qi);
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) op[b] = acc[b];
        }
    }
    // An infinite or NaN value meets a weight of 0 in the rows of the tile that
    // do not see its key (another request's, a later position's): such rows are
    // done again one by one, where every row reads its own keys only. Nothing
    // of them is written before (out may be q).
    __syncthreads();
    uint32_t redo = __builtin_amdgcn_readfirstlane(s.t.redo);
    __syncthreads();  // (the rows' results take its place)
    for (; redo; redo &= redo - 1) {
        row_attention<HD, kTileWaves>(a, tile * kTileQ + __builtin_ctz(redo), head, 0, s.r);
        __syncthreads();
    }
}

// Merge of the n_chunks partial records of each (row, head): the
// flash-decoding combine, chunks in key order.
__global__ __launch_bounds__(256) void rswa_merge_kernel(const float* part, float* out, int heads, int head_dim,
                                                         int n_chunks) {
    constexpr float kLog2e = 1.4426950408889634f;
    const int row = blockIdx.x, head = blockIdx.y;
    const float* rec = part + ((size_t)row * heads + head) * n_chunks * kRswaRec;
    float M = -INFINITY;
    for (int c = 0; c < n_chunks; ++c) M = fmaxf(M, rec[(size_t)c * kRswaRec]);
    for (int d = threadIdx.x; d < head_dim; d += blockDim.x) {
        float L = 0.0f, o = 0.0f;
        if (M != -INFINITY) {
            for (int c = 0; c < n_chunks; ++c) {
                const float m = rec[(size_t)c * kRswaRec];
                const float f = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - M) * kLog2e);
                L = fmaf(rec[(size_t)c * kRswaRec + 1], f, L);
                o = fmaf(rec[(size_t)c * kRswaRec + 4 + d], f, o);
            }
        }
        out[((size_t)row * heads + head) * head_dim + d] = L > 0.0f ? o / L : 0.0f;
    }
}

// Row copy of one token's K and V (stride floats each) into a cache row.
__device__ __forceinline__ void copy_row(const float* k, const float* v, float* kd, float* vd, int stride) {
    for (int i = threadIdx.x * 4; i < stride; i += blockDim.x * 4) {
        *reinterpret_cast<f32x4*>(kd + i) = *reinterpret_cast<const f32x4*>(k + i);
        *reinterpret_cast<f32x4*>(vd + i) = *reinterpret_cast<const f32x4*>(v + i);
    }
}

// The cache row an append writes, with the ring state advanced: grow until
// prefill_len + window, then overwrite prefill_len + ring_pos circularly
// (kv_cache.cpp:54-82; rswa_attention.cu:409-420). One thread updates the
// state; the row reaches the others through LDS.
__device__ __forceinline__ int append_row(int* d_len, int* d_ring_pos, int prefill_len, int window) {
    __shared__ int row_s;
    if (threadIdx.x == 0) {
        const int len = *d_len;
        int row;
        if (len < prefill_len + window) {
            row = len;
            *d_len = len + 1;
            if (len + 1 >= prefill_len + window) *d_ring_pos = 0;
        } else {
            const int rp = *d_ring_pos;
            row = prefill_len + rp;
            *d_ring_pos = (rp + 1) % window;
        }
        row_s = row;
    }
    __syncthreads();
    return row_s;
}

__global__ __launch_bounds__(256) void rswa_append_kernel(const float* k, const float* v, float* kc, float* vc,
                                                          int* d_len, int* d_ring_pos, int prefill_len, int window,
                                                          int stride) {
    const int row = append_row(d_len, d_ring_pos, prefill_len, window);
    copy_row(k, v, kc + (size_t)row * stride, vc + (size_t)row * stride, stride);
}

__global__ __launch_bounds__(256) void rswa_append_batch_kernel(const float* k, const float* v, float* kc, float* vc,
                                                                int* d_len, int* d_ring_pos, const int* d_prefill_len,
                                                                const int* d_slots, int batch_cap, int window,
                                                                int stride) {
    const int b = blockIdx.x, slot = d_slots[b];
    const int row = append_row(d_len + slot, d_ring_pos + slot, d_prefill_len[slot], window);
    const size_t dst = ((size_t)slot * batch_cap + row) * stride;
    copy_row(k + (size_t)b * stride, v + (size_t)b * stride, kc + dst, vc + dst, stride);
}

__global__ __launch_bounds__(256) void rswa_write_ragged_kernel(const float* k, const float* v, float* kc, float* vc,
                                                                const int* d_slots, const int* d_pos, int batch_cap,
                                                                int stride) {
    const int t = blockIdx.x;
    const size_t dst = ((size_t)d_slots[t] * batch_cap + d_pos[t]) * stride;
    copy_row(k + (size_t)t * stride, v + (size_t)t * stride, kc + dst, vc + dst, stride);
}

int check_shape(int heads, int kv_heads, int head_dim) {
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads)
        return set_error(UOCR_HIP_EINVAL, "heads must be a positive multiple of kv_heads");
    if (head_dim <= 0 || head_dim > 256 || head_dim % 4)
        return set_error(UOCR_HIP_EUNSUPPORTED, "head_dim must be a multiple of 4 in [4, 256]");
    return UOCR_HIP_OK;
}

int check_ptrs(std::initializer_list<const void*> ps) {
    for (const void* p : ps) {
        if (!p) return set_error(UOCR_HIP_EINVAL, "null pointer");
        if ((uintptr_t)p % 16) return set_error(UOCR_HIP_EINVAL, "q, k/v caches and out must be 16-byte aligned");
    }
    return UOCR_HIP_OK;
}

// Partial records of the key-split attention: a library-owned device buffer
// (the reference's attention signatures carry no workspace). Calls that split
// on one device share it, so split calls on different streams of one device
// must not overlap; a call whose records would not fit runs unsplit.
constexpr int kRswaPartRecs = 4096;
__device__ float g_rswa_part[(size_t)kRswaPartRecs * kRswaRec];
std::mutex g_rswa_mu;
float* g_rswa_part_ptr[64] = {};
int g_rswa_cus[64] = {};

int device_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        (void)hipGetLastError();
    return n > 0 ? n : 256;
}

// device address of g_rswa_part and the CU count of the current device
int rswa_device(float** part, int* cus) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= 64) return -1;
    std::lock_guard<std::mutex> lock(g_rswa_mu);
    if (!g_rswa_part_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_rswa_part)) != hipSuccess) return -1;
        if (hipDeviceGetAttribute(&g_rswa_cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
        g_rswa_part_ptr[dev] = static_cast<float*>(p);
    }
    *part = g_rswa_part_ptr[dev];
    *cus = g_rswa_cus[dev];
    return 0;
}

// max_len: an upper bound of any row's key count (0: unknown). When rows x
// heads workgroups cannot fill the chip (decode), the keys of each (row, head)
// are split into chunks of at least 128 keys over up to 8 workgroups, then
// merged by a second kernel.
int launch_attention(RswaArgs a, int rows, hipStream_t st, int max_len) {
    if (rows <= 0) return UOCR_HIP_OK;
    a.scale = 1.0f / sqrtf((float)a.head_dim);
    a.n_chunks = 1;
    float* part = nullptr;
    int cus = 0;
    const long long wgs = (long long)rows * a.heads;
    if (wgs < 512 && rswa_device(&part, &cus) == 0) {
        int n = (int)((2LL * cus + wgs - 1) / wgs);
        if (max_len > 0) n = std::min(n, max_len / 128);
        n = std::min(n, 8);
        while (n > 1 && wgs * n > kRswaPartRecs) --n;
        if (n > 1) {
            a.n_chunks = n;
            a.part = part;
        }
    }
    // One cache or ragged rows may run query-tiled (fewer than 512 pairs keep the
    // key split above)
    const bool tiled = a.mode == 0 ? rswa_one_cache_tiled(rows, a.heads, a.head_dim, a.kv_len, a.q_start, a.causal)
                                   : a.mode != 2 && rswa_call_tiled(rows, a.heads, a.head_dim, max_len);
    if (tiled) {
        const int n_tiles = (rows + kTileQ - 1) / kTileQ;
        const int resident = tile_resident(a.head_dim) * device_cus();  // workgroups that the chip holds at once
        const dim3 tgrid(n_tiles * a.heads + (int)std::min<long long>(wgs, resident));
        const bool sort = n_tiles * a.heads > resident;
        a.pairs = (float)wgs;
        a.full = (long long)n_tiles * a.heads * 16 > 9ll * resident;
        a.kv_share = (float)a.kv_heads / a.heads;
        if (a.head_dim == 64) launch_k(rswa_tile_kernel<64>, tgrid, dim3(kTileWaves * 64), 0, st, a, rows, n_tiles, sort);
        else launch_k(rswa_tile_kernel<128>, tgrid, dim3(kTileWaves * 64), 0, st, a, rows, n_tiles, sort);
        const hipError_t te = hipGetLastError();
        return te == hipSuccess ? UOCR_HIP_OK : set_error(UOCR_HIP_EHIP, std::string("rswa launch: ") + hipGetErrorString(te));
    }
    const dim3 grid(rows, a.heads, a.n_chunks), block(kRswaWaves * 64);
    if (a.head_dim <= 64) launch_k(rswa_kernel<64>, grid, block, 0, st, a);
    else if (a.head_dim <= 128) launch_k(rswa_kernel<128>, grid, block, 0, st, a);
    else launch_k(rswa_kernel<256>, grid, block, 0, st, a);
    if (a.n_chunks > 1)
        launch_k(rswa_merge_kernel, dim3(rows, a.heads), dim3(std::min(256, (a.head_dim + 63) / 64 * 64)), 0, st,
                 (const float*)a.part, a.out, a.heads, a.head_dim, a.n_chunks);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? UOCR_HIP_OK : set_error(UOCR_HIP_EHIP, std::string("rswa launch: ") + hipGetErrorString(e));
}

int launch_done(const char* what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? UOCR_HIP_OK : set_error(UOCR_HIP_EHIP, std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace
}  // namespace uocr_hip

using namespace uocr_hip;

extern "C" {

int uocr_hip_rswa_attention_decode(const float* q, const float* kcache, const float* vcache, int kv_len, int heads,
                                   int kv_heads, int head_dim, float* out, void* stream) {
    if (int rc = check_shape(heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({q, kcache, vcache, out})) return rc;
    if (kv_len < 0) return set_error(UOCR_HIP_EINVAL, "kv_len must be >= 0");
    RswaArgs a{q, kcache, vcache, out, heads, kv_heads, head_dim, 0.f, 0, kv_len, 0, 0, nullptr, nullptr, nullptr, 0};
    return launch_attention(a, 1, (hipStream_t)stream, kv_len);
}

int uocr_hip_rswa_attention(const float* q, const float* kcache, const float* vcache, int kv_len, int seq,
                            int q_start, int heads, int kv_heads, int head_dim, int causal, float* out,
                            void* stream) {
    if (int rc = check_shape(heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({q, kcache, vcache, out})) return rc;
    if (kv_len < 0 || seq < 0) return set_error(UOCR_HIP_EINVAL, "kv_len and seq must be >= 0");
    RswaArgs a{q, kcache, vcache, out, heads, kv_heads, head_dim, 0.f, 0, kv_len, q_start, causal != 0,
               nullptr, nullptr, nullptr, 0};
    return launch_attention(a, seq, (hipStream_t)stream, kv_len);
}

int uocr_hip_rswa_attention_devlen(const float* q, const float* kcache, const float* vcache, const int* d_len,
                                   int seq, int q_start, int heads, int kv_heads, int head_dim, int causal,
                                   float* out, void* stream) {
    if (int rc = check_shape(heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({q, kcache, vcache, out})) return rc;
    if (!d_len || seq < 0) return set_error(UOCR_HIP_EINVAL, "null d_len or negative seq");
    RswaArgs a{q, kcache, vcache, out, heads, kv_heads, head_dim, 0.f, 1, 0, q_start, causal != 0,
               d_len, nullptr, nullptr, 0};
    return launch_attention(a, seq, (hipStream_t)stream, 0);
}

int uocr_hip_rswa_attention_batch(const float* q, const float* kcache_base, const float* vcache_base,
                                  const int* d_len, const int* d_slots, int batch, int batch_cap, int heads,
                                  int kv_heads, int head_dim, float* out, void* stream) {
    if (batch <= 0) return UOCR_HIP_OK;  // as the reference: nothing to do
    if (int rc = check_shape(heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({q, kcache_base, vcache_base, out})) return rc;
    if (!d_len || !d_slots || batch_cap <= 0) return set_error(UOCR_HIP_EINVAL, "null d_len/d_slots or batch_cap <= 0");
    RswaArgs a{q, kcache_base, vcache_base, out, heads, kv_heads, head_dim, 0.f, 2, 0, 0, 0,
               d_len, d_slots, nullptr, batch_cap};
    return launch_attention(a, batch, (hipStream_t)stream, batch_cap);
}

int uocr_hip_rswa_attention_ragged(const float* q, const float* kcache_base, const float* vcache_base,
                                   const int* d_slots, const int* d_pos, int total, int batch_cap, int heads,
                                   int kv_heads, int head_dim, float* out, void* stream) {
    if (total <= 0) return UOCR_HIP_OK;
    if (int rc = check_shape(heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({q, kcache_base, vcache_base, out})) return rc;
    if (!d_slots || !d_pos || batch_cap <= 0) return set_error(UOCR_HIP_EINVAL, "null d_slots/d_pos or batch_cap <= 0");
    RswaArgs a{q, kcache_base, vcache_base, out, heads, kv_heads, head_dim, 0.f, 3, 0, 0, 0,
               nullptr, d_slots, d_pos, batch_cap};
    return launch_attention(a, total, (hipStream_t)stream, batch_cap);
}

int uocr_hip_rswa_append_decode(const float* k, const float* v, float* kcache, float* vcache, int* d_len,
                                int* d_ring_pos, int prefill_len, int window, int kv_heads, int head_dim,
                                void* stream) {
    if (int rc = check_shape(kv_heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({k, v, kcache, vcache})) return rc;
    if (!d_len || !d_ring_pos || window <= 0 || prefill_len < 0)
        return set_error(UOCR_HIP_EINVAL, "null state or window <= 0");
    launch_k(rswa_append_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, k, v, kcache, vcache, d_len, d_ring_pos,
             prefill_len, window, kv_heads * head_dim);
    return launch_done("rswa append");
}

int uocr_hip_rswa_append_decode_batch(const float* k, const float* v, float* kcache_base, float* vcache_base,
                                      int* d_len, int* d_ring_pos, const int* d_prefill_len, const int* d_slots,
                                      int batch, int batch_cap, int window, int kv_heads, int head_dim,
                                      void* stream) {
    if (batch <= 0) return UOCR_HIP_OK;
    if (int rc = check_shape(kv_heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({k, v, kcache_base, vcache_base})) return rc;
    if (!d_len || !d_ring_pos || !d_prefill_len || !d_slots || window <= 0 || batch_cap <= 0)
        return set_error(UOCR_HIP_EINVAL, "null state arrays, window <= 0 or batch_cap <= 0");
    launch_k(rswa_append_batch_kernel, dim3(batch), dim3(256), 0, (hipStream_t)stream, k, v, kcache_base, vcache_base,
             d_len, d_ring_pos, d_prefill_len, d_slots, batch_cap, window, kv_heads * head_dim);
    return launch_done("rswa batch append");
}

int uocr_hip_rswa_write_prefill_ragged(const float* k, const float* v, float* kcache_base, float* vcache_base,
                                       const int* d_slots, const int* d_pos, int total, int batch_cap, int kv_heads,
                                       int head_dim, void* stream) {
    if (total <= 0) return UOCR_HIP_OK;
    if (int rc = check_shape(kv_heads, kv_heads, head_dim)) return rc;
    if (int rc = check_ptrs({k, v, kcache_base, vcache_base})) return rc;
    if (!d_slots || !d_pos || batch_cap <= 0) return set_error(UOCR_HIP_EINVAL, "null d_slots/d_pos or batch_cap <= 0");
    launch_k(rswa_write_ragged_kernel, dim3(total), dim3(256), 0, (hipStream_t)stream, k, v, kcache_base, vcache_base,
             d_slots, d_pos, batch_cap, kv_heads * head_dim);
    return launch_done("rswa ragged write");
}

}  // extern "C"
