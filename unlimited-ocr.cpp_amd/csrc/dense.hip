// Unquantised expert weights: the reference's BF16 (and, after the AWQ fold,
// F32) matrices on f16 MFMA.
//
// The reference keeps the shared expert unquantised (src/runtime/weights.cpp:
// 289-292; F32 after scale_columns, weights.cpp:185-207) and runs it as three
// bf16 linear_forward calls (src/engine/gpu_decoder.cu:647-652); its default
// routed-expert format is BF16 too (include/uocr/config.h:111), grouped by
// moe_grouped_gate_up_bf16 / _down_bf16 (src/kernels/cuda/moe_gemm_bf16.cu:
// 122-353). Here those matrices are uploaded once as f16, row-major
// [rows][cols] (exact for every bf16 value in f16's normal range; finer than
// bf16 for f32 values), and multiplied with f16 activations on
// v_mfma_f32_*_f16 with f32 accumulation. Two kernels share one argument
// block and one work description (the grouping's tile list, or consecutive
// slot tiles for the shared MLP, which sees every token):
//   * dense_skinny_kernel -- up to 16 slots per tile (decode). A workgroup owns
//     16 output columns of one tile and splits K across its waves; every wave
//     issues all of its weight and activation loads at once (16-byte
//     fragments straight from global memory into MFMA operand order), so the
//     weight stream is limited by HBM, not by latency; the waves' partial sums
//     meet in LDS.
//   * dense_tile_kernel -- 64 or 128 slots per tile (prefill): both operands by
//     DMA through LDS, several k-tiles ahead.
// Gate/up (GU) pairs a gate block with the same up rows and writes
// silu(g) * u as f16 act; down writes y (f16 per slot for the combine of the
// grouped path, f32 per token for the shared MLP).
#include "experts_prefill.hpp"
#include "xcd_order.hpp"

namespace uocr_hip {

namespace {

// 8 consecutive activations as f16: f16 rows (AK 0) or bf16 rows (AK 1,
// converted exactly within f16's range)
template <int AK>
__device__ __forceinline__ f16x8 load_a8(const void* base, size_t idx) {
    if constexpr (AK == 0) {
        return *reinterpret_cast<const f16x8*>(static_cast<const f16*>(base) + idx);
    } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + idx);
        f16x8 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            r[2 * i] = (f16)__uint_as_float(v[i] << 16);
            r[2 * i + 1] = (f16)__uint_as_float(v[i] & 0xffff0000u);
        }
        return r;
    }
}

__device__ __forceinline__ f16x8 load_w8(const f16* p) { return *reinterpret_cast<const f16x8*>(p); }

struct TileDesc {
    int e, m0, rows, slot0;
};

// tile `tile` of the work list; false past its end
__device__ __forceinline__ bool tile_desc(const DenseArgs& a, int tile, int bm, TileDesc& t) {
    if (a.tile_info) {
        if (tile >= *a.n_tiles) return false;
        const int4 ti = *reinterpret_cast<const int4*>(a.tile_info + 4 * tile);
        t = TileDesc{ti.x, ti.y, ti.z, ti.w};
        return true;
    }
    const int m0 = tile * bm;
    if (m0 >= a.seq) return false;
    t = TileDesc{0, m0, min(bm, a.seq - m0), m0};
    return true;
}

// four values staged as f16 (a value beyond f16's range is reported)
__device__ __forceinline__ void store_f16x4(f16* p, float v0, float v1, float v2, float v3, int* status) {
    f16x4 h = {(f16)v0, (f16)v1, (f16)v2, (f16)v3};
    *reinterpret_cast<f16x4*>(p) = h;
    report_f16_overflow(status, f16_overflow(v0) || f16_overflow(v1) || f16_overflow(v2) || f16_overflow(v3));
}

}  // namespace

// ---------------------------------------------------------------------------
// Decode-sized tiles (<= 16 slots). Workgroup = (tile, 16 output columns),
// NW waves; wave w covers k-steps [w * KSW, (w + 1) * KSW) of 32 columns.
// KSW == 0: runtime k-step count, in chunks of 8.
// ---------------------------------------------------------------------------
template <int NW, int KSW, bool GU, int AK>
__global__ __launch_bounds__(64 * NW) void dense_skinny_kernel(DenseArgs a) {
    constexpr int CH = KSW > 0 ? KSW : 8;
    __shared__ f32x4 red[NW > 1 ? NW - 1 : 1][GU ? 2 : 1][64];
    const int n_nb = a.n_out / 16;
    const int tile = blockIdx.x / n_nb, nb = blockIdx.x % n_nb;
    TileDesc t;
    if (!tile_desc(a, tile, 16, t)) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int K = a.k;
    const int ksw = KSW > 0 ? KSW : (K / 32) / NW;
    const int kc0 = wave * ksw * 32 + 8 * (lane >> 4);  // this lane's first column
    const int m = lane & 15;
    const int slot = t.slot0 + min(m, t.rows - 1);
    const int arow = a.slot_tok ? a.slot_tok[slot] : slot;
    const size_t abase = (size_t)arow * K + kc0;
    const size_t wbase = (size_t)t.e * a.w_stride + (size_t)(nb * 16 + m) * K + kc0;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < ksw; c += CH) {
        f16x8 b0[CH], b1[CH], af[CH];
        // the weight stream first (HBM), then the activations (L2)
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (KSW > 0 || c + i < ksw) {
                b0[i] = load_w8(a.w0 + wbase + (c + i) * 32);
                if constexpr (GU) b1[i] = load_w8(a.w1 + wbase + (c + i) * 32);
            }
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (KSW > 0 || c + i < ksw) af[i] = load_a8<AK>(a.a, abase + (c + i) * 32);
        // every load of the chunk is in flight before the first use (left to
        // itself the scheduler sinks loads to their uses, one round trip each)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (KSW > 0 || c + i < ksw) {
                acc0 = mfma16(b0[i], af[i], acc0);
                if constexpr (GU) acc1 = mfma16(b1[i], af[i], acc1);
            }
    }
    if constexpr (NW > 1) {
        if (wave > 0) {
            red[wave - 1][0][lane] = acc0;
            if constexpr (GU) red[wave - 1][1][lane] = acc1;
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 0; w < NW - 1; ++w) {
            acc0 += red[w][0][lane];
            if constexpr (GU) acc1 += red[w][1][lane];
        }
    }
    // lane holds D[weight row 4 * (lane / 16) + r][slot lane % 16]
    if (m >= t.rows) return;
    const size_t o = (size_t)(t.slot0 + m) * a.n_out + nb * 16 + 4 * (lane >> 4);
    if constexpr (GU) {
        store_f16x4(a.out16 + o, silu_mul_f(acc0[0], acc1[0]), silu_mul_f(acc0[1], acc1[1]),
                    silu_mul_f(acc0[2], acc1[2]), silu_mul_f(acc0[3], acc1[3]), a.status);
    } else if (a.out32) {
        *reinterpret_cast<f32x4*>(a.out32 + o) = acc0;
    } else {
        store_f16x4(a.out16 + o, acc0[0], acc0[1], acc0[2], acc0[3], a.status);
    }
}

// ---------------------------------------------------------------------------
// Prefill-sized tiles: BM (64 or 128) slots x NJ 64-row blocks of weights (GU:
// the gate and the up rows of 64 act columns; down: 64 or 128 output columns) per
// workgroup of 2 x 2 waves, v_mfma_f32_32x32x16_f16 with the weights as the A operand (a lane
// ends with 4 consecutive output columns of one slot).
//   * A (gathered) and B rows come by 16-byte DMA in k-tiles of 64 columns,
//     kStages - 1 k-tiles ahead, one barrier per k-tile; 8 lanes read a row's 128
//     contiguous bytes (the operand-order DMA of the older kernel touched 32
//     lines per instruction and had one k-tile in flight);
//   * unit u (16 bytes) of row r sits at u ^ (r / 2 % 8): the operand reads of 16
//     rows then cover all 64 banks;
//   * the LDS reads are asm with counted waits (the compiler would wait for
//     every DMA in flight before each of them).
// Small batches are bound by latency (few workgroups, K / 64 dependent steps). 64
// experts at 1111 tokens: HBM, gate/up 374 MB in 96 us (303 of weights), down 312 MB in 57
// (5.4 TB/s; 151 of weights, every XCD reads all act rows); MFMA 21 and 17% of the time, LDS
// 10 and 8%. Measured against the older kernel (128 slots, one
// k-tile of operand-order DMA ahead, 42 and 15 workgroups at 283 tokens), both
// launches of the shared MLP, weights from HBM: 283 tokens 102 -> 22 us, 1024 108 -> 37, 4096
// 137 -> 93.
// ---------------------------------------------------------------------------
template <int BM, int NJ>
struct DenseTile {
    static constexpr int BN = 64 * NJ;  // weight rows
    static constexpr int stage = (BM + BN) * 128;
    static constexpr int fit = 81920 / stage;  // two workgroups per CU
    static constexpr int stages = fit > 4 ? 4 : fit;
    static constexpr int dmas = (BM + BN) / 32;  // per wave and k-tile
};

template <int BM, bool GU, int NJ>
__global__ __launch_bounds__(256, 2) void dense_tile_kernel(DenseArgs a, int n_tiles) {
    static_assert(!GU || NJ == 2, "one gate and one up block");
    using T = DenseTile<BM, NJ>;
    constexpr int JM = BM / 64, JN = NJ;      // 32-slot and 32-weight-row blocks per wave
    constexpr int NC = GU ? 64 : 64 * NJ;     // output columns
    constexpr int kStages = T::stages, ND = T::dmas;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kStages * T::stage];
    const int n_nt = a.n_out / NC;
    // an XCD takes an even run of the live (n-tile, tile) items, tiles fastest: those of
    // one n-tile share its weights in that XCD's L2. (n-tiles fastest: 2048 tokens
    // 262 -> 242 us, but 283 with Zipf routing 73 -> 84. Runs over the list's capacity
    // gave some XCDs mostly dead entries: 256 tokens 132 us against 120.)
    const int n_live = a.tile_info ? *a.n_tiles : n_tiles, xcd = blockIdx.x % kXcds;
    const int item = xcd_first_item(xcd, n_live * n_nt) + blockIdx.x / kXcds;
    if (item >= xcd_first_item(xcd + 1, n_live * n_nt)) return;
    const int nt = item / n_live;
    TileDesc t;
    if (!tile_desc(a, item % n_live, BM, t)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int K = a.k, KT = K / 64;
    const int l32 = lane & 31, lh = lane >> 5;

    // this wave's DMAs: 8 rows each (A rows, then weight rows)
    const f16* src[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int r = (wave + 4 * d) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
        const f16* row;
        if (r < BM) {
            const int slot = t.slot0 + min(r, t.rows - 1);
            row = static_cast<const f16*>(a.a) + (size_t)(a.slot_tok ? a.slot_tok[slot] : slot) * K;
        } else {
            const int n = r - BM;
            row = (GU && n >= 64 ? a.w1 : a.w0) + (size_t)t.e * a.w_stride + (size_t)(nt * NC + (GU ? n & 63 : n)) * K;
        }
        src[d] = row + u * 8;
    }
    auto issue = [&](int kt) {
        uint8_t* dst = smem + (kt % kStages) * T::stage;
#pragma unroll
        for (int d = 0; d < ND; ++d) load_lds16(src[d] + kt * 64, dst + (wave + 4 * d) * 1024);
    };
    // operand reads of k-step s: row l32 of a 32-row block, unit 2 s + lh
    uint32_t off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = l32 * 128 + (((2 * s + lh) ^ ((l32 >> 1) & 7)) << 4);

    f32x16 acc[JN][JM];
#pragma unroll
    for (int n = 0; n < JN; ++n)
#pragma unroll
        for (int m = 0; m < JM; ++m) acc[n][m] = f32x16{};
    const uint32_t base = lds_addr(smem);
    for (int kt = 0; kt < kStages - 1 && kt < KT; ++kt) issue(kt);
    for (int kt = 0; kt < KT; ++kt) {
        // this wave's part of k-tile kt has landed; after the barrier every
        // wave's has, and k-tile kt - 1 is read
        if (kt + kStages - 2 < KT) vm_wait<ND * (kStages - 2)>();
        else vm_wait<0>();
        asm volatile("s_barrier" ::: "memory");
        if (kt + kStages - 1 < KT) issue(kt + kStages - 1);
        const uint32_t st = base + (kt % kStages) * T::stage;
        const uint32_t sa = st + wm * (32 * JM) * 128, sb = st + (BM + wn * 32) * 128;
        f16x8 af[2][JM], bf[2][JN];
        auto read = [&](auto sc) {
            constexpr int s = decltype(sc)::value;
            static_for<JM>([&](auto m) { lds_read16<decltype(m)::value * 4096>(af[s & 1][decltype(m)::value], sa + off[s]); });
            static_for<JN>([&](auto n) { lds_read16<decltype(n)::value * 8192>(bf[s & 1][decltype(n)::value], sb + off[s]); });
        };
        read(std::integral_constant<int, 0>{});
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if constexpr (s < 3) read(std::integral_constant<int, s + 1>{});
            lgkm_wait<(s < 3 ? JM + JN : 0)>();
#pragma unroll
            for (int m = 0; m < JM; ++m) tie(af[s & 1][m]);
#pragma unroll
            for (int n = 0; n < JN; ++n) tie(bf[s & 1][n]);
#pragma unroll
            for (int n = 0; n < JN; ++n)
#pragma unroll
                for (int m = 0; m < JM; ++m) acc[n][m] = mfma32(bf[s & 1][n], af[s & 1][m], acc[n][m]);
        });
    }
    // D lane l: weight row 8 * (r / 4) + 4 * (l / 32) + r % 4 of the block, slot l % 32
#pragma unroll
    for (int m = 0; m < JM; ++m) {
        const int mm = (wm * JM + m) * 32 + l32;
        if (mm >= t.rows) continue;
        const size_t orow = (size_t)(t.slot0 + mm) * a.n_out + nt * NC + wn * 32;
#pragma unroll
        for (int n = 0; n < (GU ? 1 : JN); ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const size_t o = orow + n * 64 + 8 * q + 4 * lh;
                const f32x16& v = acc[n][m];
                if constexpr (GU) {
                    const f32x16& u = acc[JN - 1][m];
                    store_f16x4(a.out16 + o, silu_mul_f(v[4 * q], u[4 * q]), silu_mul_f(v[4 * q + 1], u[4 * q + 1]),
                                silu_mul_f(v[4 * q + 2], u[4 * q + 2]), silu_mul_f(v[4 * q + 3], u[4 * q + 3]), a.status);
                } else if (a.out32) {
                    *reinterpret_cast<f32x4*>(a.out32 + o) = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                } else {
                    store_f16x4(a.out16 + o, v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], a.status);
                }
            }
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
bool dense_shapes_ok(int k, int n_out, bool gate_up, int bm) {
    if (k <= 0 || n_out <= 0 || k % kTileK) return false;
    if (bm == kDenseSkinnyBM) return n_out % 16 == 0 && (k / 32) % 4 == 0;
    if (bm == kDenseTiledBM || bm == kDenseTiledSmallBM) return n_out % 64 == 0;
    return false;
}

template <bool GU, int AK>
static hipError_t launch_skinny(const DenseArgs& a, int n_tiles, hipStream_t st) {
    const int ks = a.k / 32;
    const dim3 grid(n_tiles * (a.n_out / 16));
    if (ks == 40)
        launch_k(dense_skinny_kernel<4, 10, GU, AK>, grid, dim3(256), 0, st, a);
    else if (ks == 28)
        launch_k(dense_skinny_kernel<4, 7, GU, AK>, grid, dim3(256), 0, st, a);
    else if (ks == 56)
        launch_k(dense_skinny_kernel<8, 7, GU, AK>, grid, dim3(512), 0, st, a);
    else
        launch_k(dense_skinny_kernel<4, 0, GU, AK>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The f16 input rows of an unquantised shared MLP that runs ahead of the
// single-kernel decode, for f32 hidden states or the RMSNorm prologue
// (src/kernels/cpu_ops.cpp:58-67: (x * inv) * w with inv = 1 / sqrt(mean(x^2)
// + eps)). One workgroup per token; the sum of squares is added in parallel,
// which moves inv by a few units of f32 roundoff, far below the f16 rounding
// of the result.
// ---------------------------------------------------------------------------
constexpr int kPrepThreads = 256;
constexpr int kPrepCols = 8;  // columns per thread (hidden <= 2048)

__global__ __launch_bounds__(kPrepThreads) void x16_prep_kernel(const void* x, int x_bf16, const float* rms_w,
                                                                float eps, int H, f16* x16) {
    __shared__ float wsum[kPrepThreads / 64];
    const int t = blockIdx.x, tid = threadIdx.x;
    float v[kPrepCols];
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kPrepCols; ++i) {
        const int c = tid + kPrepThreads * i;
        v[i] = 0.0f;
        if (c < H)
            v[i] = x_bf16 ? __uint_as_float((uint32_t)static_cast<const uint16_t*>(x)[(size_t)t * H + c] << 16)
                          : static_cast<const float*>(x)[(size_t)t * H + c];
        ss += v[i] * v[i];
    }
    float inv = 1.0f;
    if (rms_w) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        if ((tid & 63) == 0) wsum[tid >> 6] = ss;
        __syncthreads();
        float tot = 0.0f;
#pragma unroll
        for (int w = 0; w < kPrepThreads / 64; ++w) tot += wsum[w];
        inv = 1.0f / sqrtf(tot / (float)H + eps);
    }
#pragma unroll
    for (int i = 0; i < kPrepCols; ++i) {
        const int c = tid + kPrepThreads * i;
        if (c < H) x16[(size_t)t * H + c] = (f16)(rms_w ? (v[i] * inv) * rms_w[c] : v[i]);
    }
}

hipError_t launch_x16_prep(const void* x, bool x_bf16, const float* rms_w, float eps, int seq, int H, f16* x16,
                           hipStream_t st) {
    if (seq <= 0) return hipSuccess;
    if (H > kPrepThreads * kPrepCols || !x || !x16) return hipErrorInvalidValue;
    launch_k(x16_prep_kernel, dim3(seq), dim3(kPrepThreads), 0, st, x, x_bf16 ? 1 : 0, rms_w, eps, H, x16);
    return hipGetLastError();
}

hipError_t launch_dense(const DenseArgs& a, bool gate_up, int bm, int max_tiles, hipStream_t st) {
    if (!dense_shapes_ok(a.k, a.n_out, gate_up, bm)) return hipErrorInvalidValue;
    if (gate_up ? !(a.out16 && a.w1) : !(a.out16 || a.out32)) return hipErrorInvalidValue;
    const int n_tiles = a.tile_info ? max_tiles : (a.seq + bm - 1) / bm;
    if (n_tiles <= 0) return hipSuccess;
    if (bm == kDenseSkinnyBM) {
        if (a.a_kind == 1) return gate_up ? launch_skinny<true, 1>(a, n_tiles, st) : launch_skinny<false, 1>(a, n_tiles, st);
        return gate_up ? launch_skinny<true, 0>(a, n_tiles, st) : launch_skinny<false, 0>(a, n_tiles, st);
    }
    if (a.a_kind != 0) return hipErrorInvalidValue;
    auto launch = [&](auto kernel, int cols) {
        launch_k(kernel, dim3((n_tiles * (a.n_out / cols) + 7) / 8 * 8), dim3(256), 0, st, a, n_tiles);
        return hipGetLastError();
    };
    // down: 128 output columns per workgroup (twice the MFMAs per LDS read) once
    // that leaves a workgroup per CU (grouped experts at 1111 tokens 73.8 -> 56.9
    // us; the shared MLP at 1536 tokens would lose 7 us)
    const bool wide = a.n_out % 128 == 0 && n_tiles * (a.n_out / 128) >= 256;
    if (gate_up) return bm == 64 ? launch(dense_tile_kernel<64, true, 2>, 64) : launch(dense_tile_kernel<128, true, 2>, 64);
    if (wide) return bm == 64 ? launch(dense_tile_kernel<64, false, 2>, 128) : launch(dense_tile_kernel<128, false, 2>, 128);
    return bm == 64 ? launch(dense_tile_kernel<64, false, 1>, 64) : launch(dense_tile_kernel<128, false, 1>, 64);
}

}  // namespace uocr_hip
