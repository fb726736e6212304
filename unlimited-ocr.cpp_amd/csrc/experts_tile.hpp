// Grouped INT4 expert GEMM (prefill): 64 or 128 slots x 128 weight rows per
// workgroup of 2 x 2 waves, two workgroups per CU, v_mfma_f32_32x32x16_f16 with
// the weights as the A operand (a lane ends with 4 consecutive output columns
// of one slot).
//
// Counterpart of the reference's grouped pair moe_grouped_gate_up_int4 /
// moe_grouped_down_int4 (src/kernels/cuda/moe_gemm_int4.cu:535-732), which
// stages bf16 panels for mma.sync m16n8k16. Here:
//   * activation rows (gathered through the slot -> token list) come by 16-byte
//     DMA in k-tiles of 64 columns, 2 (128 slots) or 3 k-tiles ahead; 8 lanes read a row's 128
//     contiguous bytes;
//   * weights: each thread loads 2 units (16 bytes of nibbles and the row's
//     scales) per 128 columns into registers, 1 .. 2 of those ahead, and
//     dequantises them exactly to f16 into a double-buffered k-tile in LDS, one
//     k-tile ahead, between the MFMAs of the current one;
//   * in LDS unit u (16 bytes) of row r sits at u ^ (r / 2 % 8): the reads and writes of
//     16 rows then cover all 64 banks;
//   * every load, LDS access and wait is asm in a fixed order with counted
//     waits (the build fails if a kernel spills); one barrier per k-tile.
// A workgroup's load and store phases run under the other workgroup's MFMAs
// (the 256-slot kernel of experts_prefill.hpp has one workgroup per CU). Bound by
// the k-tile's chain (barrier, LDS latency, 8 or 16 MFMAs, staging): about 2400
// cycles per 64 columns for two workgroups (counters, gate/up at 283 tokens: MFMA 17% of
// the time, LDS 31%, 2.1 TB/s from HBM). Measured at 283 tokens, 64 experts, top-6, group
// 32: gate/up 50.4 -> 42 us, down 37.5 -> 25.5 against the 256-slot kernel.
#pragma once
#include "experts_prefill.hpp"
#include "xcd_order.hpp"

namespace uocr_hip {

// 16-byte DMA per lane to lds + 16 * lane, in program order with the other asm
__device__ __forceinline__ void tile_dma16(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}

template <int BM>
struct Int4Tile {
    static constexpr int a_stage = BM * 128, b_stage = 128 * 128;
    static constexpr int a_stages = BM == 128 ? 3 : 4;
    static constexpr int lds = a_stages * a_stage + 2 * b_stage;  // 80 / 64 KiB
};

template <int BM, bool GU, int GPT, bool ZP>
__global__ __launch_bounds__(256, 2) void int4_tile_kernel(ExpertArgs a) {
    using T = Int4Tile<BM>;
    constexpr int JM = BM / 64, SA = T::a_stages;
    constexpr int DA = BM / 32;                    // activation DMAs per wave and k-tile
    constexpr int NBL = 2 * (ZP ? 3 : 2);          // weight loads per thread and 128 columns
    constexpr int NC = GU ? 64 : 128;              // output columns
    __shared__ __attribute__((aligned(16))) uint8_t smem[T::lds];
    const int n_nt = a.n_rows / NC;
    // an XCD takes an even run of the live (tile, n-tile) items, n-tiles fastest: those of
    // one tile share its activation rows in that XCD's L2. (Runs over the list's
    // capacity gave some XCDs mostly dead entries: the whole call, us, 1024 tokens at hidden
    // 1792, inter 256 110 -> 94; tiles fastest: 597 tokens of the decoder 107.7 against 105.4)
    const int n_live = *a.n_tiles, xcd = blockIdx.x % kXcds;
    const int item = xcd_first_item(xcd, n_live * n_nt) + blockIdx.x / kXcds;
    if (item >= xcd_first_item(xcd + 1, n_live * n_nt)) return;
    const int tile = item / n_nt, nt = item % n_nt;
    const int4 ti = *reinterpret_cast<const int4*>(a.tile_info + 4 * tile);  // expert, first row, live rows, first slot
    const int e = ti.x, rows = ti.z, slot0 = ti.w;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int K = a.k, KT2 = K / 128;
    const int l32 = lane & 31, lh = lane >> 5;
    const int NG = scale_row_stride(K, kTileK / GPT);

    // activations: DMA d of this wave covers rows (wave + 4 d) * 8 .. + 7
    const f16* asrc[DA];
#pragma unroll
    for (int d = 0; d < DA; ++d) {
        const int r = (wave + 4 * d) * 8 + (lane >> 3), u = (lane & 7) ^ ((r >> 1) & 7);
        const int slot = slot0 + min(r, rows - 1);
        asrc[d] = a.a + (size_t)(a.gather ? a.slot_tok[slot] : slot) * K + u * 8;
    }
    // weights: unit i is row block wave of half i (GU: gate, up; down: columns
    // 0 .. 63, 64 .. 127), row lane % 16, columns 8 (lane / 16) .. of every 32
    const uint8_t* wsrc[2];
    const f16* ssrc[2];
    const f16* zsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int rb = GU ? nt * 4 + wave : nt * 8 + i * 4 + wave;
        const size_t so = (size_t)e * a.s_stride + (size_t)(rb * 16 + (lane & 15)) * NG;
        wsrc[i] = (GU && i ? a.w1 : a.w0) + (size_t)e * a.w_stride + (size_t)rb * KT2 * kTileBytes + lane * 16;
        ssrc[i] = reinterpret_cast<const f16*>(GU && i ? a.s1 : a.s0) + so;
        zsrc[i] = ZP ? reinterpret_cast<const f16*>(GU && i ? a.z1 : a.z0) + so : nullptr;
    }
    const uint32_t base = lds_addr(smem), bbase = base + SA * T::a_stage;
    // LDS destination of unit i's run s: row i * 64 + wave * 16 + lane % 16, unit
    // (s % 2) * 4 + lane / 16 of k-tile s / 2
    uint32_t bdst;
    {
        const int r = wave * 16 + (lane & 15);
        bdst = bbase + r * 128 + (((lane >> 4) ^ ((r >> 1) & 7)) << 4);
    }
    // operand reads of k-step s: row l32 of a 32-row block, unit 2 s + lh
    uint32_t off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = l32 * 128 + (((2 * s + lh) ^ ((l32 >> 1) & 7)) << 4);

    u32x4 braw[3][2];
    typename std::conditional<GPT == 4, u32x2, uint32_t>::type bsc[3][2], bz[3][2];
    auto issue_b = [&](int t2, auto setc) {  // weights of columns t2 * 128 ..
        constexpr int set = decltype(setc)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            gload<0>(braw[set][i], wsrc[i] + (size_t)t2 * kTileBytes);
            if constexpr (GPT == 1) gload_u16<0>(bsc[set][i], ssrc[i] + t2);
            else gload<0>(bsc[set][i], ssrc[i] + t2 * GPT);
            if constexpr (ZP) {
                if constexpr (GPT == 1) gload_u16<0>(bz[set][i], zsrc[i] + t2);
                else gload<0>(bz[set][i], zsrc[i] + t2 * GPT);
            }
        }
    };
    auto tie_b = [&](auto setc) {
        constexpr int set = decltype(setc)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            tie(braw[set][i]);
            tie(bsc[set][i]);
            if constexpr (ZP) tie(bz[set][i]);
        }
    };
    auto issue_a = [&](int kt) {
        const uint32_t dst = base + (kt % SA) * T::a_stage;
        kt = min(kt, 2 * KT2 - 1);
#pragma unroll
        for (int d = 0; d < DA; ++d) tile_dma16(asrc[d] + kt * 64, dst + (wave + 4 * d) * 1024);
    };
    auto half_of = [](const auto& w, int g) -> f16 {
        uint32_t v;
        if constexpr (GPT == 4) v = w[g >> 1];
        else v = w;
        return __builtin_bit_cast(f16, (uint16_t)(g & 1 ? v >> 16 : v & 0xffffu));
    };
    // run s (0 .. 3) of unit i, dequantised, for the k-tile buffer of parity s / 2
    auto dequant = [&](auto setc, auto ic, auto sc) {
        constexpr int set = decltype(setc)::value, i = decltype(ic)::value, s = decltype(sc)::value;
        constexpr int g = s * GPT >> 2;
        const f16x2 scl = scale2(half_of(bsc[set][i], g));
        if constexpr (ZP) return dequant8z(braw[set][i][s], scl, half_of(bz[set][i], g));
        else return dequant8(braw[set][i][s], scl);
    };
    auto stage = [&](auto ic, auto sc, const f16x8& v) {
        constexpr int i = decltype(ic)::value, s = decltype(sc)::value;
        lds_write16<(s >> 1) * T::b_stage + i * 8192>(bdst ^ ((s & 1) << 6), v);
    };

    f32x16 acc[2][JM];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < JM; ++m) acc[n][m] = f32x16{};

    using std::integral_constant;
    typedef integral_constant<int, 0> C0;
    typedef integral_constant<int, 1> C1;
    typedef integral_constant<int, 2> C2;
    // prologue: weights of the first two 128-column tiles, activations of the
    // first SA - 1 k-tiles; stage the first k-tile's weights. Loads past the
    // last column repeat the last tile's (never used), so every count below holds to the end.
    issue_b(0, C0{});
    issue_b(min(1, KT2 - 1), C1{});
#pragma unroll
    for (int kt = 0; kt < SA - 1; ++kt) issue_a(kt);
    vm_wait<NBL + (SA - 1) * DA>();
    tie_b(C0{});
    static_for<2>([&](auto ic) {
        stage(ic, C0{}, dequant(C0{}, ic, C0{}));
        stage(ic, C1{}, dequant(C0{}, ic, C1{}));
    });

    // k-tile kt = 2 t2 + PAR, set = t2 % 3. Order of the loads: [weights of t2 + 2
    // (PAR 0)], activations of kt + SA - 1.
    auto step = [&](int t2, auto parc, auto setc) {
        constexpr int PAR = decltype(parc)::value, set = decltype(setc)::value;
        const int kt = 2 * t2 + PAR;
        // activations of k-tile kt: later loads are the activations of kt + 1 ..
        // kt + SA - 2 and, from the third k-tile before on (SA 4) or the last
        // (SA 3), one tile's weights; at kt 0 the prologue's activations only
        if (SA == 3 ? PAR == 0 : kt == 0) vm_wait<(SA - 2) * DA>();
        else vm_wait<(SA - 2) * DA + NBL>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // staged weights; k-tile kt - 1 is read
        if constexpr (PAR == 0) issue_b(min(t2 + 2, KT2 - 1), integral_constant<int, (set + 2) % 3>{});
        issue_a(kt + SA - 1);
        const uint32_t sa = base + (kt % SA) * T::a_stage + wm * (32 * JM) * 128;
        const uint32_t sb = bbase + PAR * T::b_stage + wn * 32 * 128;
        // every operand of the k-tile is requested at once (one LDS latency per k-tile)
        f16x8 af[4][JM], bf[4][2];
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            static_for<JM>([&](auto m) { lds_read16<decltype(m)::value * 4096>(af[s][decltype(m)::value], sa + off[s]); });
            static_for<2>([&](auto n) { lds_read16<decltype(n)::value * 8192>(bf[s][decltype(n)::value], sb + off[s]); });
        });
        // the next k-tile's weights: PAR 0, runs 2 and 3 of this tile; PAR 1, runs
        // 0 and 1 of the next, whose loads are older than the activations of
        // the last 4 k-tiles and one tile's weights
        constexpr int nset = PAR ? (set + 1) % 3 : set;
        typedef integral_constant<int, nset> NS;
        f16x8 wv[4];
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            lgkm_wait<(3 - s) * (JM + 2)>();
#pragma unroll
            for (int m = 0; m < JM; ++m) tie(af[s][m]);
#pragma unroll
            for (int n = 0; n < 2; ++n) tie(bf[s][n]);
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int m = 0; m < JM; ++m) acc[n][m] = mfma32(bf[s][n], af[s][m], acc[n][m]);
            if constexpr (PAR == 1 && s == 0) {
                vm_wait<4 * DA + NBL>();
                tie_b(NS{});
            }
            wv[s] = dequant(NS{}, integral_constant<int, s & 1>{}, integral_constant<int, (PAR ? 0 : 2) + (s >> 1)>{});
            tie(wv[s]);  // (here, under this step's MFMAs)
        });
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            stage(integral_constant<int, s & 1>{}, integral_constant<int, (PAR ? 0 : 2) + (s >> 1)>{}, wv[s]);
        });
    };
    for (int t2 = 0;;) {
        step(t2, C0{}, C0{});
        step(t2, C1{}, C0{});
        if (++t2 == KT2) break;
        step(t2, C0{}, C1{});
        step(t2, C1{}, C1{});
        if (++t2 == KT2) break;
        step(t2, C0{}, C2{});
        step(t2, C1{}, C2{});
        if (++t2 == KT2) break;
    }
    // The last step's weight loads (repeats of the last tile) have no use: they are
    // waited for while their registers are still theirs, or one that lands later
    // would overwrite what the epilogue holds in them. No DMA may outlive the
    // workgroup's LDS either.
    vm_wait<0>();
    tie_b(C0{});
    tie_b(C1{});
    tie_b(C2{});

    // D lane l: weight row 8 * (r / 4) + 4 * (l / 32) + r % 4 of the block, slot l % 32
    bool ovf = false;
#pragma unroll
    for (int m = 0; m < JM; ++m) {
        const int mm = (wm * JM + m) * 32 + l32;
        if (mm >= rows) continue;
        f16* orow = (GU ? a.act_out : a.y_out) + (size_t)(slot0 + mm) * a.n_rows + nt * NC + wn * 32;
#pragma unroll
        for (int n = 0; n < (GU ? 1 : 2); ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = GU ? silu_mul_f(acc[0][m][4 * q + r], acc[1][m][4 * q + r]) : acc[n][m][4 * q + r];
                    ovf |= f16_overflow(v[r]);
                }
                *reinterpret_cast<f16x4*>(orow + n * 64 + 8 * q + 4 * lh) =
                    f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
            }
    }
    report_f16_overflow(a.status, ovf);
}

template <bool GU, bool ZP>
static hipError_t launch_int4_tile(const ExpertArgs& a, int max_tiles, hipStream_t st) {
    const int cols = GU ? 64 : 128;
    if (a.n_rows % cols || a.k % kTileK) return hipErrorInvalidValue;
    const dim3 grid((max_tiles * (a.n_rows / cols) + 7) / 8 * 8);
    auto go = [&](auto bm) {
        constexpr int BM = decltype(bm)::value;
        switch (a.group) {
            case 32: launch_k((int4_tile_kernel<BM, GU, 4, ZP>), grid, dim3(256), 0, st, a); break;
            case 64: launch_k((int4_tile_kernel<BM, GU, 2, ZP>), grid, dim3(256), 0, st, a); break;
            case 128: launch_k((int4_tile_kernel<BM, GU, 1, ZP>), grid, dim3(256), 0, st, a); break;
            default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    };
    if (a.bm == kPrefillSmallTileRows) return go(std::integral_constant<int, 64>{});
    if (a.bm == kPrefillTileRows) return go(std::integral_constant<int, 128>{});
    return hipErrorInvalidValue;
}

}  // namespace uocr_hip
