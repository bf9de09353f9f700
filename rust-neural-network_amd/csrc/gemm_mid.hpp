// gemm_mid.hpp -- the int8 and ternary GEMM for outputs of few tiles, included
// by gemm.hip (Epilogue, dma16_buf, ternary_perm_decode).
//
//   acc[m,n] = sum_k A[m,k] * B[n,k]   A [M,K] int8, B [N,K] int8 or 2-bit codes
//                                      in the MFMA layout; K % 16 == 0
//
// The prefill kernels of gemm.hip give each workgroup 256 x 224 (or 128 x 128)
// outputs, so a layer of a few hundred rows keeps a fraction of the CUs busy.
// What bounds such a product is the stream of weights from HBM and, per CU,
// the rate at which it takes in operand bytes (about 136 GB/s), so this kernel
// takes a small tile and splits K over the waves of the workgroup:
//  * 8 waves: WN x WM waves of 16 TN weight rows x 16 TM rows of x, times WK K
//    groups. Stage s holds WK blocks of KB bytes of K; group g works on block g.
//  * Both operands go to LDS by DMA in whole 128- or 256-byte row pieces (a
//    weight fragment loaded straight into registers takes 64 bytes of each of
//    16 rows per instruction and came in at about 40 GB/s per CU). A ring of R
//    stages; one barrier per stage. The 16-byte chunk c of row r is at
//    c ^ swizzle(r), so the 16 rows of a fragment fall on different banks.
//  * K % (WK KB) != 0: in the last stage the lanes whose chunk lies past K use
//    an offset past the buffer's range, which lands as zeros in LDS.
//  * Ternary codes are a quarter of the bytes and belong to one wave alone:
//    they go to registers, one load of KB/64 consecutive words per lane and
//    block, so a lane's k order is q KB/4 + 16 j where the int8 order is
//    64 j + 16 q; the fragments of x are read in the same order.
//  * The K groups' partial tiles are added through LDS (wrapping int32: exact,
//    so the result does not depend on the split), each group finishing the
//    16 x 16 blocks f with f % WK == group.
#pragma once

namespace rnn {

typedef int v2i_mid __attribute__((ext_vector_type(2)));

template <int WN_, int WM_, int TN_, int TM_, int KB_, bool TER_>
struct MidCfg {
    static constexpr int WN = WN_, WM = WM_, WK = 8 / (WN * WM), TN = TN_, TM = TM_, KB = KB_;
    static constexpr bool TER = TER_;
    static constexpr int NT = 512, BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int CH = KB / 16;                  // 16-byte chunks of a row per block
    static constexpr int NJ = KB / 64;                  // MFMA K steps per block
    static constexpr int X_BYTES = WK * BM * KB, W_BYTES = TER ? 0 : WK * BN * KB;
    static constexpr int STAGE = X_BYTES + W_BYTES;     // bytes of LDS per stage
    static constexpr int XL = X_BYTES / 8192, WL = W_BYTES / 8192;  // 1 KiB loads per wave
    static constexpr int R = 160 * 1024 / STAGE < 4 ? 160 * 1024 / STAGE : 4;
    static constexpr int OPS = XL + (TER ? TN : WL);    // memory operations per wave and stage
    static constexpr int F = TN * TM;                   // 16 x 16 blocks per wave
    // partial tiles: with two groups only the blocks the other one finishes
    static constexpr int RED = WK == 1 ? 0 : WK == 2 ? 8 * ((F + 1) / 2) * 1024 : 8 * F * 1024;
    static constexpr int LDS = R * STAGE > RED ? R * STAGE : RED;
    static_assert(WN * WM * WK == 8, "8 waves");
    static_assert((KB == 128 || KB == 256) && X_BYTES % 8192 == 0 && W_BYTES % 8192 == 0, "loads");
    static_assert(R >= 2 && LDS <= 160 * 1024, "gfx950 has 160 KiB of LDS per CU");
    static_assert((R - 2) * OPS < 64, "vmcnt range");
};

// stage(0, s), stage(1, s + 1), ... while they return true
template <class Fn, int... Is>
__device__ __forceinline__ bool mid_stages(Fn &f, int s, std::integer_sequence<int, Is...>) {
    return (f(std::integral_constant<int, Is>{}, s + Is) && ...);
}

template <class C>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_mid_kernel(const int8_t *__restrict__ A, const int8_t *__restrict__ B, int64_t M,
                     int64_t N, int64_t K, int tiles_m, int tiles_n, bool vec, Epilogue epi) {
    constexpr int TN = C::TN, TM = C::TM, WK = C::WK, NJ = C::NJ, CH = C::CH, R = C::R;
    __shared__ __attribute__((aligned(1024))) int8_t smem[C::LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (C::WN * C::WM), wm = wave / C::WN % C::WM, wn = wave % C::WN;
    const int fr = lane & 15, fq = lane >> 4;
    int tm, tn;
    xcd_tile((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * C::BM, n0 = (int64_t)tn * C::BN;
    const int ns = (int)((K + (int64_t)WK * C::KB - 1) / (WK * C::KB));

    // DMA instruction j of a stage covers 64 / CH rows of block j / (rows * CH
    // / 64): lane l fills chunk l % CH of row l / CH with the row's logical
    // chunk (l % CH) ^ swizzle(row). `o`: byte offset from the tile's first
    // row in the whole stages, `t`: in the last one. Rows past M or N repeat
    // the last row (their outputs are not stored).
    constexpr uint32_t kPast = 0xfffffff0u;  // past every descriptor's range: zeros
    const int ktail = (int)(K - (int64_t)(ns - 1) * WK * C::KB);
    auto offsets = [&](int j, int rows, int64_t left, uint32_t &o, uint32_t &t) {
        const int f = 64 * j + lane, r = f / CH % rows, b = f / CH / rows;
        const int c = (f % CH) ^ (CH == 8 ? (r >> 1) & 7 : r & 15);
        o = (uint32_t)(std::min<int64_t>(r, left - 1) * K + b * C::KB + 16 * c);
        t = b * C::KB + 16 * c < ktail ? o : kPast;
    };
    uint32_t xo[C::XL], xt[C::XL], wo[C::TER ? TN : C::WL], wt[C::TER ? TN : C::WL];
#pragma unroll
    for (int i = 0; i < C::XL; ++i) offsets(wave + 8 * i, C::BM, M - m0, xo[i], xt[i]);
    constexpr int WDIV = C::TER ? 4 : 1;  // k per byte
    const int64_t nw = n0 + 16 * TN * wn;
    if constexpr (C::TER) {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int kk = kg * C::KB + 16 * NJ * fq;  // the lane's first k in the stage
            wo[t] = (uint32_t)(std::min<int64_t>(16 * (TN * wn + t) + fr, N - 1 - n0) * (K / 4) + kk / 4);
            // codes past K meet zeros of x; past the last row: out of range
            wt[t] = kk < ktail ? wo[t] : kPast;
        }
    } else {
#pragma unroll
        for (int i = 0; i < C::WL; ++i) offsets(wave + 8 * i, C::BN, N - n0, wo[i], wt[i]);
    }
    // (ranges past 2 GiB are cut there: a tile's rows span less, host-checked)
    const uint32_t xr = (uint32_t)std::min<int64_t>((M - m0) * K, 0x7fffffff);
    const uint32_t wr = (uint32_t)std::min<int64_t>((N - n0) * (K / WDIV), 0x7fffffff);
    const int8_t *const xa = A + m0 * K, *const wb = B + n0 * (K / WDIV);

    struct Raw {
        uint32_t w[C::TER ? TN : 1][C::TER ? NJ : 1];
    };
    Raw raw[C::TER ? R : 1];
    // the loads of stage s (past the last: every lane out of range, so that
    // the number in flight stays the same)
    auto load = [&](auto ic, int s) {
        constexpr int slot = decltype(ic)::value;
        int8_t *const buf = smem + slot * C::STAGE;
        auto go = [&](const uint32_t (&x)[C::XL], const uint32_t (&w)[C::TER ? TN : C::WL]) {
#pragma unroll
            for (int i = 0; i < C::XL; ++i)
                dma16_buf(xa, xr, x[i], (uint32_t)s * (WK * C::KB), buf + 1024 * (wave + 8 * i));
            if constexpr (!C::TER) {
#pragma unroll
                for (int i = 0; i < C::WL; ++i)
                    dma16_buf(wb, wr, w[i], (uint32_t)s * (WK * C::KB),
                              buf + C::X_BYTES + 1024 * (wave + 8 * i));
            } else {
                const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<int8_t *>(wb), 0, (int)wr, 0x00020000);
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    const uint32_t so = (uint32_t)s * (WK * C::KB / 4);
                    if constexpr (NJ == 4) {
                        const v4i v = __builtin_bit_cast(
                            v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, w[t], so, 0));
#pragma unroll
                        for (int j = 0; j < 4; ++j) raw[slot].w[t][j] = (uint32_t)v[j];
                    } else {
                        const v2i_mid v = __builtin_bit_cast(
                            v2i_mid, __builtin_amdgcn_raw_buffer_load_b64(rb, w[t], so, 0));
                        raw[slot].w[t][0] = (uint32_t)v.x;
                        raw[slot].w[t][1] = (uint32_t)v.y;
                    }
                }
            }
        };
        if (s + 1 < ns)
            go(xo, wo);
        else if (s + 1 == ns)
            go(xt, wt);
        else {
            uint32_t xp[C::XL], wp[C::TER ? TN : C::WL];
#pragma unroll
            for (auto &v : xp) v = kPast;
#pragma unroll
            for (auto &v : wp) v = kPast;
            go(xp, wp);
        }
    };

    v4i acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int u = 0; u < TM; ++u) acc[t][u] = v4i{0, 0, 0, 0};
    const int sw = CH == 8 ? (fr >> 1) & 7 : fr;
    auto compute = [&](auto ic) {
        constexpr int slot = decltype(ic)::value;
        const int8_t *xb = smem + slot * C::STAGE + (kg * C::BM + 16 * TM * wm + fr) * C::KB;
        const int8_t *ww = smem + slot * C::STAGE + C::X_BYTES + (kg * C::BN + 16 * TN * wn + fr) * C::KB;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int c = 16 * ((C::TER ? NJ * fq + j : 4 * j + fq) ^ sw);
            v4i x[TM], w[TN];
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if constexpr (C::TER)
                    w[t] = ternary_perm_decode(raw[slot].w[t][j]);
                else
                    w[t] = *reinterpret_cast<const v4i *>(ww + 16 * t * C::KB + c);
            }
#pragma unroll
            for (int u = 0; u < TM; ++u)
                x[u] = *reinterpret_cast<const v4i *>(xb + 16 * u * C::KB + c);
#pragma unroll
            for (int u = 0; u < TM; ++u)
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    acc[t][u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[t], x[u], acc[t][u], 0, 0, 0);
        }
    };
    auto barrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    static_for<R - 1>([&](auto ic) { load(ic, decltype(ic)::value); });
    // Stage s: its loads have landed when at most those of the R - 2 stages
    // after it are in flight; behind the barrier every wave has read stage
    // s - 1, whose slot takes stage s + R - 1.
    auto stage = [&](auto ic, int s) {
        constexpr int i = decltype(ic)::value;
        wait_vmcnt<(R - 2) * C::OPS>();
        barrier();
        load(std::integral_constant<int, (i + R - 1) % R>{}, s + R - 1);
        compute(ic);
        return s + 1 < ns;
    };
    for (int s = 0; mid_stages(stage, s, std::make_integer_sequence<int, R>{}); s += R) {
    }
    wait_vmcnt<0>();  // the loads past the last stage land before LDS is reused
    barrier();

    // lane: columns nw + 16 t + 4 fq + e, row mw + 16 u + fr
    const int64_t mw = m0 + 16 * TM * wm;
    float sam[TM];
    float4 swv[TN], bv[TN];
    v4i csv[TN];
    const bool has_bias = epi.bias != nullptr, relu = epi.relu != 0;
#pragma unroll
    for (int u = 0; u < TM; ++u)
        sam[u] = epi.y ? epi.sa[std::min<int64_t>(mw + 16 * u + fr, M - 1)] : 0.0f;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int64_t n = nw + 16 * t + 4 * fq;
        swv[t] = bv[t] = float4{0.f, 0.f, 0.f, 0.f};
        csv[t] = v4i{0, 0, 0, 0};
        if (!C::TER && epi.colsum) {
#pragma unroll
            for (int e = 0; e < 4; ++e) csv[t][e] = epi.colsum[std::min(n + e, N - 1)];
        }
        if (vec) {  // N % 4 == 0 and 16-byte aligned vectors
            const int64_t nc = std::min(n, N - 4);
            if (epi.y) swv[t] = *reinterpret_cast<const float4 *>(epi.sw + nc);
            if (has_bias) bv[t] = *reinterpret_cast<const float4 *>(epi.bias + nc);
        } else if (epi.y) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t nc = std::min(n + e, N - 1);
                reinterpret_cast<float *>(&swv[t])[e] = epi.sw[nc];
                if (has_bias) reinterpret_cast<float *>(&bv[t])[e] = epi.bias[nc];
            }
        }
    }
    if constexpr (WK > 1) {
        v4i *red = reinterpret_cast<v4i *>(smem);
        // block f of group g: with two groups only the blocks that the other
        // group finishes have a place
        auto place = [&](int g, int f) {
            constexpr int P = WK == 2 ? (C::F + 1) / 2 : C::F;
            return (((g * C::WM + wm) * C::WN + wn) * P + (WK == 2 ? f / 2 : f)) * 64 + lane;
        };
#pragma unroll
        for (int f = 0; f < C::F; ++f)
            if (f % WK != kg) red[place(kg, f)] = acc[f / TM][f % TM];
        barrier();
#pragma unroll
        for (int f = 0; f < C::F; ++f)
            if (f % WK == kg) {
                v4i &a = acc[f / TM][f % TM];
#pragma unroll
                for (int g = 0; g < WK; ++g)
                    if (g != kg) {
                        const v4i p = red[place(g, f)];
                        a.x = (int)((uint32_t)a.x + (uint32_t)p.x);
                        a.y = (int)((uint32_t)a.y + (uint32_t)p.y);
                        a.z = (int)((uint32_t)a.z + (uint32_t)p.z);
                        a.w = (int)((uint32_t)a.w + (uint32_t)p.w);
                    }
            }
    }
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int u = 0; u < TM; ++u) {
            if (WK > 1 && (t * TM + u) % WK != kg) continue;
            const int64_t m = mw + 16 * u + fr, n = nw + 16 * t + 4 * fq;
            if (m >= M || n >= N) continue;
            const v4i a = acc[t][u];
            v4i ao;  // the raw output, with igemm's zero-point correction
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ao[e] = (int)((uint32_t)a[e] + 128u * (uint32_t)csv[t][e]);
                // src/int8.rs:159-162's order
                v[e] = (float)a[e] * sam[u] * reinterpret_cast<const float *>(&swv[t])[e];
                if (has_bias) v[e] = v[e] + reinterpret_cast<const float *>(&bv[t])[e];
                if (relu) v[e] = fmaxf(v[e], 0.0f);
            }
            if (vec) {
                if (epi.y) *reinterpret_cast<float4 *>(epi.y + m * N + n) = float4{v[0], v[1], v[2], v[3]};
                if (epi.acc_out) *reinterpret_cast<v4i *>(epi.acc_out + m * N + n) = ao;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) {
                        if (epi.y) epi.y[m * N + n + e] = v[e];
                        if (epi.acc_out) epi.acc_out[m * N + n + e] = ao[e];
                    }
            }
        }
}

template <class C>
static int launch_mid(const int8_t *A, const int8_t *B, int64_t M, int64_t N, int64_t K,
                      const Epilogue &epi, hipStream_t st, const char *name) {
    const int64_t tm = ceil_div(M, C::BM), tn = ceil_div(N, C::BN);
    RNN_REQUIRE(tm * tn <= 0x7fffffffLL, "%s: too many tiles", name);
    auto al = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    const bool vec = N % 4 == 0 && al(epi.y) && al(epi.acc_out) && al(epi.sw) && al(epi.bias);
    gemm_mid_kernel<C><<<(unsigned)(tm * tn), C::NT, 0, st>>>(A, B, M, N, K, (int)tm, (int)tn, vec,
                                                             epi);
    return check_launch(name);
}

// The kernel addresses a tile's rows (at most 256) with 32-bit byte offsets.
static bool mid_fits(int64_t K) { return K > 0 && K % 16 == 0 && K <= (1 << 22); }

// Estimated time (us) of M x N outputs on BM x BN tiles: a launch, and per
// round of one tile per CU a start-up plus K times what the tile's operand
// bytes (its edges) and its products (its area) cost. Fitted to graph-replay
// times at K = 4096 and 768, one tile per CU (K = 4096, measured / estimate):
// 64 x 32 9.0 / 9.0, 64 x 64 11.3 / 11.5, 64 x 128 16.6 / 16.4, 128 x 128
// 24.6 / 24.1, 128 x 256 39.7 / 39.6. `edge_w`: weight bytes per x byte (1,
// or 1/4 for ternary codes); `area`: cost per product, higher where the codes
// are decoded next to the products (ternary, K = 4096: 16 x 16 5.1, 48 x 32
// 8.7, 32 x 64 8.5, 64 x 64 13.0).
static double mid_cost(int64_t M, int64_t N, int64_t K, int bm, int bn, double edge_w, double area,
                       int cus) {
    const double rounds = (double)ceil_div(ceil_div(M, bm) * ceil_div(N, bn), cus);
    return 3.0 + rounds * (1.5 + (double)K / 4096.0 * (0.032 * (bm + edge_w * bn) + area * bm * bn));
}
constexpr double kMidArea = 0.000696, kMidAreaTer = 0.0019;
// the 256 x 224 prefill tiles (K = 4096: 39.7 us at one round, 102.5 at two)
static double pp_cost(int64_t M, int64_t N, int64_t K) {
    const double rounds = (double)ceil_div(ceil_div(M, 256) * ceil_div(N, 224), device_cu_count());
    return 3.0 + rounds * (1.5 + (double)K / 4096.0 * 44.0);
}
// the 64 x 128 ternary tiles (K = 4096: 10.3-12.6 us at one round, 32 at three)
static double l128_ter_cost(int64_t M, int64_t N, int64_t K) {
    const double rounds = (double)ceil_div(ceil_div(M, 64) * ceil_div(N, 128), device_cu_count());
    return 3.0 + rounds * (1.5 + (double)K / 4096.0 * 7.5);
}

// The tile shape with the smallest estimate; *cost receives it.
struct MidShape {
    int bm, bn;
    int (*run)(const int8_t *, const int8_t *, int64_t, int64_t, int64_t, const Epilogue &,
               hipStream_t, const char *);
};
template <bool TER>
static const MidShape *mid_choose(int64_t M, int64_t N, int64_t K, double *cost) {
#define RNN_MID(WN, WM, TN, TM, KB) \
    {16 * (TM) * (WM), 16 * (TN) * (WN), launch_mid<MidCfg<WN, (WM), TN, (TM), (KB), TER>>}
    static const MidShape shapes[] = {
        RNN_MID(1, 1, 1, 1, 128), RNN_MID(1, 1, 1, 2, 128), RNN_MID(2, 1, 1, 2, 128),
        RNN_MID(2, 1, 1, 3, 128), RNN_MID(2, 1, 1, 4, 128), RNN_MID(2, 1, 2, 2, TER ? 256 : 128),
        RNN_MID(2, TER ? 1 : 2, 2, TER ? 4 : 2, 128), RNN_MID(4, 1, 2, 4, TER ? 256 : 128),
        RNN_MID(4, 2, 2, 4, 128), RNN_MID(4, 2, 4, 4, 128),
    };
#undef RNN_MID
    const MidShape *best = nullptr;
    const int cus = device_cu_count();
    for (const MidShape &s : shapes) {
        const double c = mid_cost(M, N, K, s.bm, s.bn, TER ? 0.25 : 1.0, TER ? kMidAreaTer : kMidArea,
                                  cus);
        if (!best || c < *cost) best = &s, *cost = c;
    }
    return best;
}

}  // namespace rnn
