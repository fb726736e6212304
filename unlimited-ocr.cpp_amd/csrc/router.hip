// Device router: optional RMSNorm prologue, router logits, softmax / sigmoid
// scoring, greedy top-k, and the stable token->expert grouping.
//
// Bit-exactness contract with the reference CPU path:
//   logits   src/kernels/cpu_ops.cpp:26-39 -- one sequential fmaf chain per
//            (token, expert), k ascending (the -march=native build contracts
//            `acc += x * w`); a chain of f32 MFMAs gives exactly those bits.
//   rmsnorm  src/kernels/cpu_ops.cpp:58-67 -- as the reference's -O3
//            -march=native build runs it: each x*x rounded, summed in column
//            order (only a scalar tail of H % 4 terms would be fused),
//            correctly rounded divide and sqrt, (x * inv) * w.
//   softmax  src/kernels/cpu_ops.cpp:93-106 -- exp(l - max) with glibc's expf
//            bits (correctly rounded exp + the generated fix-up table), sum in
//            expert order, p = e * (1 / sum).
//   top-k    src/engine/moe_decoder.cpp:264-287 -- strict '>' greedy selection,
//            ties to the lowest expert index, optional renormalisation.
//   grouping src/engine/gpu_decoder.cu:602-609 -- per expert, tokens in
//            ascending (token, j) order: a stable counting sort, built here from
//            wave ballots (equal-expert masks) and per-wave LDS prefix counts.
#include <mutex>

#include "launch.hpp"
#include "routing.hpp"

namespace uocr_hip {

// Sticky flag of the moe_router_topk mirror: set when an expert received more
// entries than the [n_experts, cap] tables hold (the reference drops them
// silently, src/kernels/cuda/moe_device.cu:90-95). Written with vector atomics,
// read and cleared by router_overflow_read.
__device__ int g_router_overflow;

// Grouping scratch of the moe_router_topk mirror, whose reference signature
// has no workspace: the multi-workgroup grouping's per-entry ranks and
// per-(chunk, expert) counts / bases for up to kMirrorGroupEntries routed
// entries (larger calls run the single-workgroup rounds). One copy per device;
// host code reaches it through hipGetSymbolAddress only.
constexpr int kMirrorGroupEntries = 1 << 17;
constexpr int kMirrorGroupChunks = kMirrorGroupEntries / 1024;
__device__ int g_mirror_lrank[kMirrorGroupEntries];
__device__ int g_mirror_chunk_count[kMirrorGroupChunks * kMaxExperts];
__device__ int g_mirror_chunk_base[kMirrorGroupChunks * kMaxExperts];

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

// Argmax over the wave with the reference's tie rule (first maximum wins).
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const float ov = __shfl_xor(v, o, kWave);
        const int oi = __shfl_xor(i, o, kWave);
        if (ov > v || (ov == v && oi < i)) {
            v = ov;
            i = oi;
        }
    }
}

template <typename XT>
__device__ __forceinline__ void load8_f32(const XT* p, float* out);

template <>
__device__ __forceinline__ void load8_f32<uint16_t>(const uint16_t* p, float* out) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[2 * i] = __uint_as_float(v[i] << 16);
        out[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
    }
}

template <>
__device__ __forceinline__ void load8_f32<float>(const float* p, float* out) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p);
    const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[i] = a[i];
        out[4 + i] = b[i];
    }
}

// ---------------------------------------------------------------------------
// Stable grouping body (one workgroup of 1024 threads), shared by the
// stand-alone group kernel and the router kernel's fused tail.
// ---------------------------------------------------------------------------
constexpr int kGroupThreads = 1024;
constexpr int kGroupWaves = kGroupThreads / 64;

struct GroupLds {
    int hist[kMaxExperts];
    int offs[kMaxExperts + 1];
    int tile0[kMaxExperts + 1];
    int short0[kMaxExperts + 1];
    int nshort[kMaxExperts];
    int run[kMaxExperts];
    int wcnt[kGroupWaves][kMaxExperts];   // per-wave counts of the round
    int wbase[kGroupWaves][kMaxExperts];  // exclusive per-wave prefix of the round
};

// Exclusive prefix sum of v[0..n) (n <= 128) by wave 0; out[n] = total.
__device__ __forceinline__ void wave0_exclusive_scan(const int* v, int* out, int n) {
    const int lane = threadIdx.x & 63;
    const int a = (2 * lane < n) ? v[2 * lane] : 0;
    const int b = (2 * lane + 1 < n) ? v[2 * lane + 1] : 0;
    int inc = a + b;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(inc, o, kWave);
        if (lane >= o) inc += u;
    }
    const int ex = inc - a - b;
    if (2 * lane < n) out[2 * lane] = ex;
    if (2 * lane + 1 < n) out[2 * lane + 1] = ex + a;
    if (lane == 63) out[n] = inc;
}

// Tile list order: every expert's tiles of more than bm/2 rows first, then
// each expert's short last tile (1 .. bm/2 rows), so the short tiles (which
// the large-tile prefill kernel runs in half mode) fill the grid's last round.
// Long / short tile counts of a group of c rows:
__device__ __forceinline__ int short_tiles(int c, int bm) {
    const int rem = c % bm;
    return (rem != 0 && rem <= bm / 2) ? 1 : 0;
}
__device__ __forceinline__ int long_tiles(int c, int bm) { return (c + bm - 1) / bm - short_tiles(c, bm); }
// Write the list from the exclusive scans of the long (tile0) and short
// (short0) counts over Ev groups of hist[] rows. Called by all threads.
__device__ __forceinline__ void write_tile_list(const GroupArgs& g, const int* hist, const int* offs,
                                                const int* tile0, const int* short0, int Ev) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nlong = tile0[Ev];
    if (tid == 0) *g.n_tiles = nlong + short0[Ev];
    for (int e = wave; e < Ev; e += kGroupWaves) {
        const int nt = tile0[e + 1] - tile0[e];
        auto put = [&](int idx, int m0) {
            *reinterpret_cast<int4*>(g.tile_info + 4 * idx) = make_int4(e, m0, min(g.bm, hist[e] - m0), offs[e] + m0);
        };
        for (int m = lane; m < nt; m += 64) put(tile0[e] + m, m * g.bm);
        if (lane == 0 && short0[e + 1] > short0[e]) put(nlong + short0[e], nt * g.bm);
    }
}

// `ids` / `wts` may live in global memory or LDS. Must be called by all 1024 threads.
__device__ void group_body(const int* ids, const float* wts, const GroupArgs& g, GroupLds& s) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int E = g.n_experts, N = g.seq * g.top_k;
    const int Ev = E + g.n_virtual;

    for (int e = tid; e < kMaxExperts; e += kGroupThreads) {
        s.hist[e] = 0;
        s.run[e] = 0;
    }
    __syncthreads();
    for (int i = tid; i < N; i += kGroupThreads) {
        const int e = ids[i];
        if (e >= 0 && e < E) atomicAdd(&s.hist[e], 1);
    }
    __syncthreads();
    if (wave == 0) {
        for (int e = lane; e < g.n_virtual; e += 64) s.hist[E + e] = g.seq;  // virtual groups: all tokens
    }
    __syncthreads();
    if (wave == 0) wave0_exclusive_scan(s.hist, s.offs, Ev);
    if (wave == 1 && g.tile_info) {
        // tiles per expert into run[] (reset below), then scan into tile0[]
        for (int e = lane; e < Ev; e += 64) {
            s.run[e] = long_tiles(s.hist[e], g.bm);
            s.nshort[e] = short_tiles(s.hist[e], g.bm);
        }
    }
    __syncthreads();
    if (g.tile_info && wave == 1) wave0_exclusive_scan(s.run, s.tile0, Ev);
    if (g.tile_info && wave == 2) wave0_exclusive_scan(s.nshort, s.short0, Ev);
    __syncthreads();
    if (g.offsets) {
        for (int e = tid; e < Ev; e += kGroupThreads) g.offsets[e] = s.offs[e];
        if (tid == 0) g.offsets[Ev] = s.offs[Ev];
    }
    if (g.tile_info) write_tile_list(g, s.hist, s.offs, s.tile0, s.short0, Ev);
    for (int e = tid; e < kMaxExperts; e += kGroupThreads) s.run[e] = 0;
    __syncthreads();
    // stable placement of the routed entries, kGroupThreads entries per round
    // (entry i = base + tid, so lane order, then wave order, is (t, j) order)
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int nid = (tid < N) ? ids[tid] : -1;
    float nw = (tid < N) ? wts[tid] : 0.0f;
    for (int base = 0; base < N; base += kGroupThreads) {
        const int i = base + tid;
        const int e = nid;
        const float w = nw;
        if (base + kGroupThreads + tid < N) {  // next round's entry, in flight during this round
            nid = ids[base + kGroupThreads + tid];
            nw = wts[base + kGroupThreads + tid];
        }
        for (int k = tid; k < kGroupWaves * kMaxExperts; k += kGroupThreads) (&s.wcnt[0][0])[k] = 0;
        __syncthreads();
        // i < N: past the last round's end, nid still holds an earlier round's id
        const bool valid = i < N && e >= 0 && e < E;
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 7; ++b) {
            const bool bit = valid && ((e >> b) & 1);
            const uint64_t bal = __ballot(bit);
            m &= bit ? bal : ~bal;
        }
        const int rank = __popcll(m & below);
        if (valid && rank == 0) s.wcnt[wave][e] = __popcll(m);
        __syncthreads();
        // exclusive prefix over waves, one thread per (wave, expert)
        for (int ee = lane; ee < E; ee += 64) {
            int acc = s.run[ee];
            for (int w2 = 0; w2 < wave; ++w2) acc += s.wcnt[w2][ee];
            s.wbase[wave][ee] = acc;
        }
        __syncthreads();
        if (wave == kGroupWaves - 1)
            for (int ee = lane; ee < E; ee += 64) s.run[ee] = s.wbase[wave][ee] + s.wcnt[wave][ee];
        if (valid) {
            const int r = s.wbase[wave][e] + rank;  // position within expert e
            if (g.slot_tok) {
                const int sl = s.offs[e] + r;
                g.slot_tok[sl] = i / g.top_k;
                g.slot_w[sl] = w;
                if (g.pos) g.pos[i] = sl;
            }
            if (g.assign_token && r < g.cap) {
                g.assign_token[(size_t)e * g.cap + r] = i / g.top_k;
                g.assign_w[(size_t)e * g.cap + r] = w;
            }
        }
        __syncthreads();
    }
    if (g.assign_count)
        for (int e = tid; e < E; e += kGroupThreads) {
            g.assign_count[e] = min(s.hist[e], g.cap);
            if (s.hist[e] > g.cap) atomicOr(&g_router_overflow, 1);
        }
    if (g.slot_tok) {
        for (int v = 0; v < g.n_virtual; ++v)
            for (int t = tid; t < g.seq; t += kGroupThreads) {
                g.slot_tok[s.offs[E + v] + t] = t;
                g.slot_w[s.offs[E + v] + t] = 1.0f;
            }
    }
}

__global__ __launch_bounds__(kGroupThreads) void group_kernel(GroupArgs g) {
    __shared__ GroupLds s;
    group_body(g.ids, g.weights, g, s);
}

// ---------------------------------------------------------------------------
// Multi-workgroup stable grouping for large batches: three launches, each of
// which finishes all of its loads before its first store (on gfx9 the vmcnt
// wait for a load also waits for every earlier store).
//   rank:  per 1024-entry chunk, stable rank of each entry among the chunk's
//          entries of the same expert + the chunk's per-expert counts;
//   scan:  expert totals, offsets, tile list and per-(chunk, expert) bases;
//   place: slot = base[chunk][expert] + rank.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kGroupThreads) void group_rank_kernel(GroupArgs g) {
    __shared__ int wcnt[kGroupWaves][kMaxExperts];
    __shared__ int wbase[kGroupWaves][kMaxExperts];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int E = g.n_experts, N = g.seq * g.top_k;
    const int i = blockIdx.x * kGroupThreads + tid;
    const int e = (i < N) ? g.ids[i] : -1;
    for (int k = tid; k < kGroupWaves * kMaxExperts; k += kGroupThreads) (&wcnt[0][0])[k] = 0;
    __syncthreads();
    const bool valid = e >= 0 && e < E;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 7; ++b) {
        const bool bit = valid && ((e >> b) & 1);
        const uint64_t bal = __ballot(bit);
        m &= bit ? bal : ~bal;
    }
    const int rank = __popcll(m & below);
    if (valid && rank == 0) wcnt[wave][e] = __popcll(m);
    __syncthreads();
    for (int ee = lane; ee < E; ee += 64) {
        int acc = 0;
        for (int w2 = 0; w2 < wave; ++w2) acc += wcnt[w2][ee];
        wbase[wave][ee] = acc;
    }
    __syncthreads();
    if (i < N) g.lrank[i] = valid ? wbase[wave][e] + rank : 0;
    if (wave == kGroupWaves - 1)
        for (int ee = lane; ee < E; ee += 64)
            g.chunk_count[(size_t)blockIdx.x * E + ee] = wbase[wave][ee] + wcnt[wave][ee];
}

__global__ __launch_bounds__(kGroupThreads) void group_scan_kernel(GroupArgs g, int n_chunks) {
    extern __shared__ int cc[];  // [n_chunks][E] counts, then bases
    __shared__ int hist[kMaxExperts], offs[kMaxExperts + 1], ntl[kMaxExperts], tile0[kMaxExperts + 1];
    __shared__ int nsh[kMaxExperts], short0[kMaxExperts + 1];
    const int tid = threadIdx.x, wave = tid >> 6;
    const int E = g.n_experts, Ev = E + g.n_virtual;
    for (int k = tid; k < n_chunks * E; k += kGroupThreads) cc[k] = g.chunk_count[k];
    __syncthreads();
    for (int e = tid; e < Ev; e += kGroupThreads) {
        int acc = 0;
        if (e < E)
            for (int c = 0; c < n_chunks; ++c) {
                const int v = cc[c * E + e];
                cc[c * E + e] = acc;  // exclusive base within expert e
                acc += v;
            }
        else
            acc = g.seq;
        hist[e] = acc;
        ntl[e] = long_tiles(acc, g.bm);
        nsh[e] = short_tiles(acc, g.bm);
    }
    __syncthreads();
    if (wave == 0) wave0_exclusive_scan(hist, offs, Ev);
    if (wave == 1) wave0_exclusive_scan(ntl, tile0, Ev);
    if (wave == 2) wave0_exclusive_scan(nsh, short0, Ev);
    __syncthreads();
    for (int k = tid; k < n_chunks * E; k += kGroupThreads) g.chunk_base[k] = cc[k] + (g.slot_tok ? offs[k % E] : 0);
    for (int e = tid; e < Ev; e += kGroupThreads) {
        if (g.offsets) g.offsets[e] = offs[e];
        if (g.assign_count && e < E) {
            g.assign_count[e] = min(hist[e], g.cap);
            if (hist[e] > g.cap) atomicOr(&g_router_overflow, 1);
        }
    }
    if (tid == 0 && g.offsets) g.offsets[Ev] = offs[Ev];
    if (g.tile_info) write_tile_list(g, hist, offs, tile0, short0, Ev);
    // virtual (shared-expert) groups: every token, weight 1
    if (g.slot_tok)
        for (int v = 0; v < g.n_virtual; ++v)
            for (int t = tid; t < g.seq; t += kGroupThreads) {
                g.slot_tok[offs[E + v] + t] = t;
                g.slot_w[offs[E + v] + t] = 1.0f;
            }
}

// Scan and place in one launch, for up to kGroupFusedMaxChunks chunks: every
// workgroup (one per 1024-entry chunk) reduces the per-(chunk, expert) counts
// itself (n_chunks x E ints from L2), so its bases need no other workgroup;
// workgroup 0 also writes the expert totals, offsets and tile list, and the
// virtual groups' slots are spread over all of them. All loads come before
// the first store.
constexpr int kGroupFusedMaxChunks = 64;

__global__ __launch_bounds__(kGroupThreads) void group_scan_place_kernel(GroupArgs g, int n_chunks) {
    extern __shared__ int cc[];  // [n_chunks][E] counts
    __shared__ int hist[kMaxExperts], offs[kMaxExperts + 1], base[kMaxExperts];
    __shared__ int ntl[kMaxExperts], tile0[kMaxExperts + 1], nsh[kMaxExperts], short0[kMaxExperts + 1];
    const int tid = threadIdx.x, wave = tid >> 6;
    const int E = g.n_experts, Ev = E + g.n_virtual, N = g.seq * g.top_k;
    const int b = blockIdx.x;
    const int i = b * kGroupThreads + tid;
    const int e_i = i < N ? g.ids[i] : -1;
    const bool valid = e_i >= 0 && e_i < E;
    const int lr = valid ? g.lrank[i] : 0;
    const float w_i = valid ? g.weights[i] : 0.0f;
    for (int k = tid; k < n_chunks * E; k += kGroupThreads) cc[k] = g.chunk_count[k];
    __syncthreads();
    for (int e = tid; e < Ev; e += kGroupThreads) {
        int acc = 0;
        if (e < E) {
            int mine = 0;
            for (int c = 0; c < n_chunks; ++c) {
                if (c == b) mine = acc;
                acc += cc[c * E + e];
            }
            base[e] = mine;  // entries of expert e in the chunks before this one
        } else {
            acc = g.seq;
        }
        hist[e] = acc;
        ntl[e] = long_tiles(acc, g.bm);
        nsh[e] = short_tiles(acc, g.bm);
    }
    __syncthreads();
    if (wave == 0) wave0_exclusive_scan(hist, offs, Ev);
    if (b == 0 && g.tile_info && wave == 1) wave0_exclusive_scan(ntl, tile0, Ev);
    if (b == 0 && g.tile_info && wave == 2) wave0_exclusive_scan(nsh, short0, Ev);
    __syncthreads();
    if (valid) {
        if (g.slot_tok) {  // the slot
            const int r = offs[e_i] + base[e_i] + lr;
            g.slot_tok[r] = i / g.top_k;
            g.slot_w[r] = w_i;
            if (g.pos) g.pos[i] = r;
        } else if (g.assign_token) {  // the position within expert e_i
            const int r = base[e_i] + lr;
            if (r < g.cap) {
                g.assign_token[(size_t)e_i * g.cap + r] = i / g.top_k;
                g.assign_w[(size_t)e_i * g.cap + r] = w_i;
            }
        }
    }
    if (b == 0) {
        for (int e = tid; e < Ev; e += kGroupThreads) {
            if (g.offsets) g.offsets[e] = offs[e];
            if (g.assign_count && e < E) {
                g.assign_count[e] = min(hist[e], g.cap);
                if (hist[e] > g.cap) atomicOr(&g_router_overflow, 1);
            }
        }
        if (tid == 0 && g.offsets) g.offsets[Ev] = offs[Ev];
        if (g.tile_info) write_tile_list(g, hist, offs, tile0, short0, Ev);
    }
    // virtual (shared-expert) groups: every token, weight 1
    if (g.slot_tok)
        for (int v = 0; v < g.n_virtual; ++v)
            for (int t = i; t < g.seq; t += n_chunks * kGroupThreads) {
                g.slot_tok[offs[E + v] + t] = t;
                g.slot_w[offs[E + v] + t] = 1.0f;
            }
}

__global__ __launch_bounds__(256) void group_place_kernel(GroupArgs g) {
    const int E = g.n_experts, N = g.seq * g.top_k;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int e = g.ids[i];
    if (e < 0 || e >= E) return;
    const int r = g.chunk_base[(size_t)(i / kGroupThreads) * E + e] + g.lrank[i];
    const float w = g.weights[i];
    if (g.slot_tok) {  // r is the slot (bases include the expert offset)
        g.slot_tok[r] = i / g.top_k;
        g.slot_w[r] = w;
        if (g.pos) g.pos[i] = r;
    }
    if (g.assign_token && r < g.cap) {  // r is the position within expert e
        g.assign_token[(size_t)e * g.cap + r] = i / g.top_k;
        g.assign_w[(size_t)e * g.cap + r] = w;
    }
}

// ---------------------------------------------------------------------------
// Router for a bf16 router matrix (E <= 64): 16 tokens per workgroup of 16
// waves, the logits on v_mfma_f32_16x16x4_f32.
//
// The f32 MFMA accumulates its k-slices in ascending order with one rounding
// per term and keeps denormals, so a chain of them gives the bits of the
// reference's sequential fmaf chain. Waves 0..3 own 16 experts each and run one chain for
// all 16 tokens: 32.3 cycles per 4 columns, against
// 4 x (17..23) cycles per column and token for one lane per expert. The
// RMSNorm's sum of squares (each product rounded, then added in column order)
// is the same chain with ones as the other operand: fma(x * x, 1, sum).
//   * x rows in LDS as f32, every 16 columns transposed 4 x 4 so that one
//     16-byte read holds a lane's operand of four consecutive MFMAs; rows are
//     padded by 16 bytes (16 tokens then cover all 64 banks);
//   * router_m holds the weights in the order of the other operand (8 MFMAs
//     per 16-byte load), read from L2 ten loads ahead;
//   * 16 waves, because scoring and top-k take one wave per token.
// Bound by the chain's latency (1280 columns: 320 MFMAs, 10.4k cycles alone,
// 14k measured; with the RMSNorm a second chain), the token rows' arrival and
// the top-k (7k cycles). Measured against one lane per expert and token
// (rocprofv3): 1024 tokens 16.4 -> 13.0 us, 4096 tokens 34 -> 17.8, 1111 tokens
// 30.8 -> 15.7, 283 tokens with the RMSNorm 39 -> 21.7.
// ---------------------------------------------------------------------------
constexpr int kRouterTokens = 16;
constexpr int kMaxRouterHidden = 1792;
constexpr int kLogitStride = 68;  // floats per token of the logits in LDS

// LDS byte offset of column c (a multiple of 16) in a token row: 16 bytes of
// padding per 64 columns, so that the staging writes (64 bytes apart per
// lane) cover all banks too; rows are an odd number of 16-byte units
__host__ __device__ constexpr int router_col_bytes(int c) { return c * 4 + c / 64 * 16; }
__host__ __device__ constexpr int router_row_bytes(int H) { return router_col_bytes(H) + 16; }
__host__ __device__ constexpr size_t router_lds_bytes(int H) {
    return (size_t)kRouterTokens * router_row_bytes(H) + (size_t)kRouterTokens * kLogitStride * 4 +
           (size_t)kRouterTokens * 64 * 4;
}

// HC: hidden as a compile-time constant (the k-loops are then unrolled and the
// weights stay four 32-column steps ahead in registers); 0: a.hidden, one step
template <typename XT, bool RMS, int HC>
__global__ __launch_bounds__(kRouterTokens * 64) void router_kernel(RouterArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int H = HC ? HC : a.hidden, E = a.n_experts, K = a.top_k;
    const int rowb = router_row_bytes(H), n_steps = H / 32;
    float* logits = reinterpret_cast<float*>(smem + (size_t)kRouterTokens * rowb);
    float* scr = logits + kRouterTokens * kLogitStride + wave * 64;
    __shared__ uint64_t etab[32];
    __shared__ float inv_s[kRouterTokens];
    if (threadIdx.x < 32) etab[threadIdx.x] = uocr_exp2_tab[threadIdx.x];
    const int t = blockIdx.x * kRouterTokens + wave;
    const bool live = t < a.seq;
    const XT* x = static_cast<const XT*>(a.x) + (size_t)min(t, a.seq - 1) * H;
    const int m16 = lane & 15, g = lane >> 4;

    // waves 0..3: the weights of 16 experts. 32-column step i: 8 bf16 of
    // expert 16 * wave + m16, MFMA s of the step taking column 4 s + g
    constexpr int RING = HC ? 10 : 1;
    u32x4 wreg[RING];
    const u32x4* wsrc = reinterpret_cast<const u32x4*>(a.router_m) + g * 64 + wave * 16 + m16;
    if (wave < 4) {
#pragma unroll
        for (int i = 0; i < RING; ++i) wreg[i] = wsrc[i * 256];
    }

    // this wave's token row: 16 columns per lane and step. store_x16 writes
    // the experts' f16 input
    auto store_x16 = [&](int c, const float* v) {
        f16x8 h[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) h[i >> 3][i & 7] = (f16)v[i];
        f16* d = a.x16 + (size_t)t * H + c;
        reinterpret_cast<f16x8*>(d)[0] = h[0];
        reinterpret_cast<f16x8*>(d)[1] = h[1];
    };
    // (RMS: the row stays in registers and LDS first holds the rounded squares)
    unsigned char* xrow = smem + (size_t)wave * rowb;
    auto put = [&](int c, const float* v) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(xrow + router_col_bytes(c) + q * 16) = f32x4{v[q], v[4 + q], v[8 + q], v[12 + q]};
    };
    constexpr int NV = (kMaxRouterHidden + 1023) / 1024;
    float v[NV][16];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = lane * 16 + j * 1024;
        if (c < H) {
            load8_f32<XT>(x + c, v[j]);
            load8_f32<XT>(x + c + 8, v[j] + 8);
        }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = lane * 16 + j * 1024;
        if (c < H) {
            float sq[16];
            if constexpr (RMS) {
#pragma unroll
                for (int i = 0; i < 16; ++i) sq[i] = __fmul_rn(v[j][i], v[j][i]);
            }
            put(c, RMS ? sq : v[j]);
            if (!RMS && live) store_x16(c, v[j]);
        }
    }
    __syncthreads();

    // operand reads: token m16, k-slice g, the 8 MFMAs of 32-column step i
    const unsigned char* xop = smem + (size_t)m16 * rowb + g * 16;
    auto read_x = [&](int i, f32x4* v) {
        const int c = (i < n_steps ? i : n_steps - 1) * 32;  // (past the end: the last step again)
        v[0] = *reinterpret_cast<const f32x4*>(xop + router_col_bytes(c));
        v[1] = *reinterpret_cast<const f32x4*>(xop + router_col_bytes(c) + 64);
    };
    // One chain step per MFMA, accumulating in place (asm: the compiler would
    // rotate the accumulator through other registers, which costs the chain
    // wait states). A VALU op between two MFMAs of a chain costs it 13 cycles,
    // eight of them after eight MFMAs 5.7 per MFMA, a ds_read 3 (measured on
    // one wave: 32.3 cycles per MFMA alone), so a step's other work comes in
    // one piece. s_nop 1 covers a VALU write of an operand, which the hazard
    // recognizer does not see in asm, and chain_end() the wait states before
    // the result is read.
    auto mac = [](f32x4& acc, float p, float q) {
        asm volatile("s_nop 1\n\tv_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(acc) : "v"(p), "v"(q));
    };
    auto chain_begin = [](f32x4& acc) {
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("s_nop 7" : "+v"(acc));
    };
    auto chain_end = [](f32x4& acc) { asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc)); };
    if constexpr (RMS) {
        if (wave == 0) {
            f32x4 ss, cur[2], nx[2];
            read_x(0, cur);
            const float one = 1.0f;
            chain_begin(ss);
            auto step = [&](int i, f32x4* u, f32x4* next) {
                read_x(i + 1, next);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < 8; ++s) mac(ss, u[s >> 2][s & 3], one);
                __builtin_amdgcn_sched_barrier(0);
            };
            for (int i = 0; i < n_steps; i += 2) {  // (H % 128 == 0)
                step(i, cur, nx);
                step(i + 1, nx, cur);
            }
            chain_end(ss);
            // lane holds the sums of tokens 4 g + r (the same in every column m16)
            float s = ss[0];
#pragma unroll
            for (int r = 1; r < 4; ++r) s = (m16 & 3) == r ? ss[r] : s;
            if (m16 < 4)
                inv_s[4 * g + m16] = __fdiv_rn(1.0f, sqrt_rn(__fadd_rn(__fdiv_rn(s, (float)H), a.rms_eps)));
        }
        __syncthreads();
        const float inv = inv_s[wave];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = lane * 16 + j * 1024;
            if (c < H) {
                float w[16];
                load8_f32<float>(a.rms_weight + c, w);
                load8_f32<float>(a.rms_weight + c + 8, w + 8);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[j][i] = __fmul_rn(__fmul_rn(v[j][i], inv), w[i]);
                put(c, v[j]);
                if (live) store_x16(c, v[j]);
            }
        }
        __syncthreads();
    }

    if (wave < 4) {
        f32x4 acc, xa[2], xb[2];
        float wa[8], wb[8];
        auto widen = [](const u32x4& w, float* o) {
#pragma unroll
            for (int s = 0; s < 8; ++s) o[s] = __uint_as_float(s & 1 ? w[s >> 1] & 0xffff0000u : w[s >> 1] << 16);
        };
        // rows: experts, columns: tokens. Step i: x of step i + 1 is requested,
        // the MFMAs run, then the weights of step i + 1 are widened and those
        // of step i + RING requested
        read_x(0, xa);
        widen(wreg[0], wa);
        chain_begin(acc);
        auto step = [&](int i, const float* wc, const f32x4* xc, float* wn, f32x4* xn, const u32x4& w, u32x4& refill) {
            read_x(i + 1, xn);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 8; ++s) mac(acc, wc[s], xc[s >> 2][s & 3]);
            __builtin_amdgcn_sched_barrier(0);
            widen(w, wn);
            if (i + RING < n_steps) refill = wsrc[(size_t)(i + RING) * 256];
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr (HC > 0) {
#pragma unroll
            for (int i = 0; i < HC / 32; i += 2) {
                step(i, wa, xa, wb, xb, wreg[(i + 1) % RING], wreg[i % RING]);
                step(i + 1, wb, xb, wa, xa, wreg[(i + 2) % RING], wreg[(i + 1) % RING]);
            }
        } else {
            u32x4 none;
            for (int i = 0; i < n_steps; i += 2) {
                const u32x4 w1 = wsrc[(size_t)(i + 1) * 256];
                step(i, wa, xa, wb, xb, w1, none);
                const u32x4 w2 = wsrc[(size_t)min(i + 2, n_steps - 1) * 256];
                step(i + 1, wb, xb, wa, xa, w2, none);
            }
        }
        chain_end(acc);
        // lane holds experts 16 * wave + 4 g + r of token m16
        *reinterpret_cast<f32x4*>(logits + m16 * kLogitStride + wave * 16 + 4 * g) = acc;
    }
    __syncthreads();

    // scoring and greedy top-k of one token per wave
    const WaveTopk pick = wave_topk(logits[wave * kLogitStride + lane], E, K, a.scoring_sigmoid, a.norm_topk_prob,
                                    a.scaling, scr, etab);
    if (live && lane < K) a.weights[(size_t)t * K + lane] = pick.w;
    if (live && pick.rank < K) a.ids[(size_t)t * K + pick.rank] = lane;
}

// Router from precomputed logits [seq, E] (mirror of moe_router_topk,
// src/kernels/cuda/moe_device.cu:24-98), any E: one wave per token, experts
// strided over lanes; reduction orders match the CPU reference.
__global__ __launch_bounds__(256) void router_from_logits_kernel(RouterArgs a, const float* logits) {
    extern __shared__ float lds[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int E = a.n_experts, K = a.top_k;
    float* row = lds + (size_t)wave * E;
    __shared__ uint64_t etab[32];
    if (threadIdx.x < 32) etab[threadIdx.x] = uocr_exp2_tab[threadIdx.x];
    __syncthreads();
    const int t = blockIdx.x * (blockDim.x >> 6) + wave;
    const bool live = t < a.seq;
    const float* src = logits + (size_t)(live ? t : 0) * E;
    if (a.scoring_sigmoid) {
        for (int e = lane; e < E; e += 64)
            row[e] = __fdiv_rn(1.0f, 1.0f + ref_expf(-src[e], etab));
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) mx = fmaxf(mx, src[e]);
        mx = wave_max(mx);
        for (int e = lane; e < E; e += 64) row[e] = ref_expf(src[e] - mx, etab);
        __syncthreads();
        float sum = 0.0f;
        for (int e = 0; e < E; ++e) sum += row[e];
        const float inv = __fdiv_rn(1.0f, sum);
        __syncthreads();
        for (int e = lane; e < E; e += 64) row[e] *= inv;
    }
    __syncthreads();
    float wj = 0.0f;
    int idj = 0;
    for (int j = 0; j < K; ++j) {
        float v = -INFINITY;
        int i = 0x7fffffff;
        for (int e = lane; e < E; e += 64)
            if (row[e] > v) {
                v = row[e];
                i = e;
            }
        wave_argmax(v, i);
        if (!(v > -1e30f)) i = -1;
        if (lane == j) {
            idj = i;
            wj = v;
        }
        __syncthreads();
        if (i >= 0 && lane == (i & 63)) row[i] = -1e30f;
        __syncthreads();
    }
    if (K > 1 && a.norm_topk_prob) {
        float s = 0.0f;
        for (int j = 0; j < K; ++j) s += __shfl(wj, j, kWave);
        wj = __fdiv_rn(wj, s + 1e-20f) * a.scaling;
    } else {
        wj *= a.scaling;
    }
    if (live && lane < K) {
        a.ids[(size_t)t * K + lane] = idj;
        a.weights[(size_t)t * K + lane] = wj;
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
template <typename XT, bool RMS, int HC>
static hipError_t launch_router_h(const RouterArgs& a, hipStream_t st) {
    // > 64 KiB of dynamic LDS: raise the limit once per kernel
    static hipError_t attr = hipFuncSetAttribute((const void*)router_kernel<XT, RMS, HC>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
    if (attr != hipSuccess) return attr;
    launch_k((router_kernel<XT, RMS, HC>), dim3((a.seq + kRouterTokens - 1) / kRouterTokens),
             dim3(kRouterTokens * 64), router_lds_bytes(a.hidden), st, a);
    return hipGetLastError();
}

template <typename XT, bool RMS>
static hipError_t launch_router_t(const RouterArgs& a, hipStream_t st) {
    return a.hidden == 1280 ? launch_router_h<XT, RMS, 1280>(a, st) : launch_router_h<XT, RMS, 0>(a, st);
}

hipError_t launch_router(const RouterArgs& a, bool x_is_bf16, hipStream_t st) {
    if (a.n_experts > 64 || a.hidden > kMaxRouterHidden || a.hidden % 128 || a.seq <= 0 || !a.router_m)
        return hipErrorInvalidValue;
    const bool rms = a.rms_weight != nullptr;
    if (x_is_bf16) return rms ? launch_router_t<uint16_t, true>(a, st) : launch_router_t<uint16_t, false>(a, st);
    return rms ? launch_router_t<float, true>(a, st) : launch_router_t<float, false>(a, st);
}

hipError_t launch_router_from_logits(const RouterArgs& a, const float* logits, hipStream_t st) {
    const int waves = 4;
    const dim3 grid((a.seq + waves - 1) / waves);
    const size_t lds = (size_t)waves * a.n_experts * sizeof(float);
    launch_k(router_from_logits_kernel, grid, dim3(64 * waves), lds, st, a, logits);
    return hipGetLastError();
}

int group_chunks(int seq, int top_k) { return (seq * top_k + kGroupThreads - 1) / kGroupThreads; }

bool group_fits(int seq, int top_k, int n_experts) {
    return (size_t)group_chunks(seq, top_k) * n_experts * sizeof(int) <= kGroupScanLds;
}

hipError_t router_overflow_read(int clear, int* flag) {
    hipError_t e = hipMemcpyFromSymbol(flag, HIP_SYMBOL(g_router_overflow), sizeof(int), 0, hipMemcpyDeviceToHost);
    if (e != hipSuccess || !clear) return e;
    const int zero = 0;
    return hipMemcpyToSymbol(HIP_SYMBOL(g_router_overflow), &zero, sizeof(int), 0, hipMemcpyHostToDevice);
}

hipError_t launch_group_mirror(GroupArgs g, hipStream_t st) {
    if (group_chunks(g.seq, g.top_k) > 1 && (long long)g.seq * g.top_k <= kMirrorGroupEntries) {
        static std::mutex mu;
        static void* addr[3][64] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (!addr[0][dev]) {
                if ((e = hipGetSymbolAddress(&addr[0][dev], HIP_SYMBOL(g_mirror_lrank))) != hipSuccess ||
                    (e = hipGetSymbolAddress(&addr[1][dev], HIP_SYMBOL(g_mirror_chunk_count))) != hipSuccess ||
                    (e = hipGetSymbolAddress(&addr[2][dev], HIP_SYMBOL(g_mirror_chunk_base))) != hipSuccess) {
                    addr[0][dev] = nullptr;
                    return e;
                }
            }
        }
        g.lrank = static_cast<int*>(addr[0][dev]);
        g.chunk_count = static_cast<int*>(addr[1][dev]);
        g.chunk_base = static_cast<int*>(addr[2][dev]);
    }
    return launch_group(g, st);
}

hipError_t launch_group(const GroupArgs& g, hipStream_t st) {
    const int n_chunks = group_chunks(g.seq, g.top_k);
    // one workgroup for a single 1024-entry round (or without the multi-kernel
    // scratch); measured slower than rank / scan / place from 6 rounds on
    if (n_chunks <= 1 || !g.lrank) {
        launch_k(group_kernel, dim3(1), dim3(kGroupThreads), 0, st, g);
        return hipGetLastError();
    }
    if (g.slot_tok && g.assign_token) return hipErrorInvalidValue;  // bases are slots or positions, not both
    // checked before the first launch, so an oversized call enqueues nothing
    const size_t lds = (size_t)n_chunks * g.n_experts * sizeof(int);
    if (lds > kGroupScanLds) return hipErrorInvalidValue;
    launch_k(group_rank_kernel, dim3(n_chunks), dim3(kGroupThreads), 0, st, g);
    if (n_chunks <= kGroupFusedMaxChunks) {
        launch_k(group_scan_place_kernel, dim3(n_chunks), dim3(kGroupThreads), lds, st, g, n_chunks);
        return hipGetLastError();
    }
    static hipError_t attr = hipFuncSetAttribute((const void*)group_scan_kernel,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, kGroupScanLds);
    if (attr != hipSuccess) return attr;
    launch_k(group_scan_kernel, dim3(1), dim3(kGroupThreads), lds, st, g, n_chunks);
    const int n = g.seq * g.top_k;
    launch_k(group_place_kernel, dim3((n + 255) / 256), dim3(256), 0, st, g);
    return hipGetLastError();
}

}  // namespace uocr_hip
