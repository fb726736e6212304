// Body of the row walk: one (query row `row`, head `head`) by a workgroup of WAVES waves, keys
// split over n_chunks calls (`chunk` is this one's), results of the waves in
// `s`. Included into the row kernel and into the row workers' function rather than
// called from both: inlined from a function, the loop's V loads are scheduled behind
// the next branch, and batched decode (16 requests x 1128 rows) takes 37.0 us instead of 36.5.
    constexpr int D = HDP / 8;  // dims per lane
    constexpr int NV = D / 4;   // float4 per lane per row
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int j = lane >> 3, p = lane & 7;
    const int hd = a.head_dim, stride = a.kv_heads * hd;
    const int kvh = head / (a.heads / a.kv_heads);
    const float* kc = a.kc;
    const float* vc = a.vc;
    int limit;
    if (a.mode <= 1) {
        const int kv_len = a.mode == 1 ? *a.d_len : a.kv_len;
        limit = a.causal ? min(kv_len, a.q_start + row + 1) : kv_len;
    } else {
        const int slot = a.d_slots[row];
        limit = a.mode == 2 ? a.d_len[slot] : a.d_pos[row] + 1;
        kc += (size_t)slot * a.batch_cap * stride;
        vc += (size_t)slot * a.batch_cap * stride;
    }
    const size_t qoff = ((size_t)row * a.heads + head) * hd;
    kc += (size_t)kvh * hd;
    vc += (size_t)kvh * hd;
    // lane p's dims: 4 at 4p + 32i (i < NV), so the 8 lanes of a key read one
    // contiguous 128-byte run per load
    auto dim_of = [&](int i) { return 4 * p + 32 * i; };

    f32x4 qv[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i)
        qv[i] = dim_of(i) < hd ? *reinterpret_cast<const f32x4*>(a.q + qoff + dim_of(i)) : f32x4{0.f, 0.f, 0.f, 0.f};

    float m = -INFINITY, l = 0.0f;
    f32x4 acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // this workgroup's keys [kbeg, kend): chunk blockIdx.z of n_chunks (chunks
    // of whole 8-key groups; a chunk past the limit has no keys)
    int kbeg = 0, kend = limit;
    if (a.n_chunks > 1) {
        const int cs = ((limit + a.n_chunks - 1) / a.n_chunks + 7) & ~7;
        kbeg = min(limit, chunk * cs);
        kend = min(limit, kbeg + cs);
    }
    const int n_groups = (kend - kbeg + 7) / 8;
    // Unpredicated loads (a lane-predicated load makes the compiler wait for
    // every outstanding load before the first use, defeating the prefetch):
    // keys past the limit re-read the last valid row (their weight is 0),
    // dims past head_dim re-read the last 4 (their q is 0 and they are never
    // stored). Called only with limit >= 1.
    auto load = [&](int g, f32x4 (&kv)[NV], f32x4 (&vv)[NV]) {
        const int t = min(kbeg + g * 8 + j, kend - 1);
        const float* kr = kc + (size_t)t * stride;
        const float* vr = vc + (size_t)t * stride;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int d = min(dim_of(i), hd - 4);
            kv[i] = *reinterpret_cast<const f32x4*>(kr + d);
            vv[i] = *reinterpret_cast<const f32x4*>(vr + d);
        }
    };
    f32x4 k0[NV], v0[NV], k1[NV], v1[NV], k2[NV], v2[NV];
    constexpr float kLog2e = 1.4426950408889634f;
    auto step = [&](int g, const f32x4 (&kv)[NV], const f32x4 (&vv)[NV]) {
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) part = fmaf(qv[i][c], kv[i][c], part);
        part += __shfl_xor(part, 1, 64);
        part += __shfl_xor(part, 2, 64);
        part += __shfl_xor(part, 4, 64);
        const bool valid = kbeg + g * 8 + j < kend;
        const float sc = valid ? part * a.scale : -INFINITY;
        float mg = fmaxf(sc, __shfl_xor(sc, 8, 64));
        mg = fmaxf(mg, __shfl_xor(mg, 16, 64));
        mg = fmaxf(mg, __shfl_xor(mg, 32, 64));
        const float m_new = fmaxf(m, mg);  // finite: key 0 of the group is valid
        const float alpha = __builtin_amdgcn_exp2f((m - m_new) * kLog2e);
        const float beta = valid ? __builtin_amdgcn_exp2f((sc - m_new) * kLog2e) : 0.0f;
        float bs = beta + __shfl_xor(beta, 8, 64);
        bs += __shfl_xor(bs, 16, 64);
        bs += __shfl_xor(bs, 32, 64);
        l = fmaf(l, alpha, bs);
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[i][c] = fmaf(acc[i][c], alpha, beta * vv[i][c]);
        m = m_new;
    };
    // groups wave, wave + 8, ...; two groups' loads in flight beyond the one in
    // use (three register buffers in rotation), one for head_dim > 128
    constexpr int GS = WAVES;
    int g = wave;
    if constexpr (HDP <= 128) {
        if (g < n_groups) {
            load(g, k0, v0);
            load(g + GS, k1, v1);
        }
        while (g < n_groups) {
            load(g + 2 * GS, k2, v2);
            step(g, k0, v0);
            g += GS;
            if (g >= n_groups) break;
            load(g + 2 * GS, k0, v0);
            step(g, k1, v1);
            g += GS;
            if (g >= n_groups) break;
            load(g + 2 * GS, k1, v1);
            step(g, k2, v2);
            g += GS;
        }
    } else {
        if (g < n_groups) load(g, k0, v0);
        while (g < n_groups) {
            load(g + GS, k1, v1);
            step(g, k0, v0);
            g += GS;
            if (g >= n_groups) break;
            load(g + GS, k0, v0);
            step(g, k1, v1);
            g += GS;
        }
    }
    // sum the 8 key slots of the wave (same m within the wave)
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float x = acc[i][c];
            x += __shfl_xor(x, 8, 64);
            x += __shfl_xor(x, 16, 64);
            x += __shfl_xor(x, 32, 64);
            acc[i][c] = x;
        }
    auto& wm = s.m;
    auto& wl = s.l;
    auto& wacc = s.acc;
    if (lane < 8) {
#pragma unroll
        for (int i = 0; i < NV; ++i) *reinterpret_cast<f32x4*>(&wacc[wave][dim_of(i)]) = acc[i];
    }
    if (lane == 0) {
        wm[wave] = m;
        wl[wave] = l;
    }
    __syncthreads();
    // combine the waves (a wave without keys has m = -inf and weight 0)
    float* rec = a.n_chunks > 1 ? a.part + (((size_t)row * a.heads + head) * a.n_chunks + chunk) * kRswaRec
                                : nullptr;
    if (rec && tid == 0) {
        float M = -INFINITY, L = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) M = fmaxf(M, wm[w]);
        if (M != -INFINITY) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
                L = fmaf(wl[w], wm[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((wm[w] - M) * kLog2e), L);
        }
        rec[0] = M;
        rec[1] = L;
    }
    for (int d = tid; d < hd; d += WAVES * 64) {
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) M = fmaxf(M, wm[w]);
        float L = 0.0f, o = 0.0f;
        if (M != -INFINITY) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const float f = wm[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((wm[w] - M) * kLog2e);
                L = fmaf(wl[w], f, L);
                o = fmaf(wacc[w][d], f, o);
            }
        }
        if (rec)
            rec[4 + d] = o;  // unnormalised, relative to this chunk's max
        else
            a.out[qoff + d] = L > 0.0f ? o / L : 0.0f;
    }
