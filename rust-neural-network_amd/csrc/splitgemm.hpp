// splitgemm.hpp -- f32 x . W^T on the bf16 matrix cores, at f32 precision.
//
//   C[m,n] = alpha * sum_k x[m,k] W[n,k] (+ bias[n], ReLU) + beta * C[m,n]
//
// x (and f32 weights) are split into three bf16 parts, v = h + m + l: h and m
// round v and v - h to nearest, which leaves an l of at most 8 significant
// bits, so the split is exact. Weights that bf16 holds exactly (integer codes,
// E2M1, bf16) have one part and take 3 bf16 products per product; f32 weights
// take the 6 largest of the 9 (the dropped ones are below 2^-25 of the
// product). v_mfma_f32_16x16x32_bf16 runs at 16 times the rate of
// v_mfma_f32_16x16x4f32, so 6 products leave 2.7 times its rate and 3 leave
// 5.3 times. A group's codes are summed first and enter the total in one
// fused multiply-add by the group's scale.
//
//  * split_x_kernel writes the parts of x once per call in MFMA fragment
//    order (K step of 32, 16-row tile, part: 1 KiB), so that a tile's parts
//    are contiguous, go to LDS by DMA as they are and are read without bank
//    conflicts. Rows past M and k past K are zeros.
//  * Weights go to LDS by DMA as they are stored (16-byte chunk c of row r at
//    c ^ swizzle(r)) and each wave splits or decodes its rows in registers.
//  * 8 waves: WN x WM of 16 TN columns x 16 TM rows, times WK K groups whose
//    partial tiles are added through LDS in a fixed order. A ring of R stages,
//    one barrier per stage.
//  * Values the split does not hold: infinities and NaN become NaN in the
//    parts, x below 2^-108 (whose l would fall under bf16's range) gets a NaN
//    l, and f32 weights below it are noticed as they are split. A workgroup
//    whose tile holds a NaN or infinity, or that saw such a weight, computes
//    the tile again on v_mfma_f32_16x16x4f32 from the stored operands.
#pragma once

#include <algorithm>
#include <utility>

#include "common.hpp"

namespace rnn {

typedef float sg_f4 __attribute__((ext_vector_type(4)));
typedef float sg_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 sg_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 sg_b8 __attribute__((ext_vector_type(8)));
typedef unsigned int sg_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int sg_u2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kTinyBits = 19u << 23;  // 2^-108: below it a bf16 l loses bits

__device__ __forceinline__ uint32_t sg_pk(float a, float b) {  // two bf16, round to nearest even
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(sg_f2{a, b}, sg_b2));
}
// The parts of a pair of floats, packed; part[0] = h, [1] = m, [2] = l.
__device__ __forceinline__ void sg_split2(float a, float b, uint32_t (&part)[3]) {
    part[0] = sg_pk(a, b);
    a -= __uint_as_float(part[0] << 16), b -= __uint_as_float(part[0] & 0xFFFF0000u);
    part[1] = sg_pk(a, b);
    a -= __uint_as_float(part[1] << 16), b -= __uint_as_float(part[1] & 0xFFFF0000u);
    part[2] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

__device__ __forceinline__ uint32_t sg_hi2(float lo, float hi) {  // two floats that bf16 holds
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// x [M, K] (row stride ldx) -> parts in fragment order: lane (r = l % 16, q =
// l / 16) of fragment (K step s, tile t, part p) holds x[16 t + r][32 s + 8 q
// .. + 7]. A wave per (s, t). VEC: 16-byte loads (ldx % 4 == 0, aligned x).
template <bool VEC>
__global__ __launch_bounds__(256) void split_x_kernel(const float *__restrict__ x, int64_t ldx,
                                                      int64_t M, int64_t K, int mt, int64_t frags,
                                                      uint32_t *__restrict__ xp) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    for (int64_t f = blockIdx.x * 4 + (threadIdx.x >> 6); f < frags; f += 4 * (int64_t)gridDim.x) {
        const int64_t m = 16 * (f % mt) + r, k = 32 * (f / mt) + 8 * q;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const float *src = x + m * ldx + k;
        if (m < M) {
            if (VEC && k + 8 <= K) {
                *reinterpret_cast<sg_f4 *>(v) = *reinterpret_cast<const sg_f4 *>(src);
                *reinterpret_cast<sg_f4 *>(v + 4) = *reinterpret_cast<const sg_f4 *>(src + 4);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (k + e < K) v[e] = src[e];
            }
        }
        sg_u4 o[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t p[3];
            sg_split2(v[2 * e], v[2 * e + 1], p);
            // 0 < |v| < 2^-108: a NaN in l
            if ((__float_as_uint(v[2 * e]) << 1) - 1u < 2u * kTinyBits - 1u) p[2] |= 0x7FFFu;
            if ((__float_as_uint(v[2 * e + 1]) << 1) - 1u < 2u * kTinyBits - 1u) p[2] |= 0x7FFF0000u;
#pragma unroll
            for (int j = 0; j < 3; ++j) o[j][e] = p[j];
        }
        sg_u4 *dst = reinterpret_cast<sg_u4 *>(xp) + f * 192 + lane;
#pragma unroll
        for (int j = 0; j < 3; ++j) dst[64 * j] = o[j];
    }
}

struct SplitArgs {
    const uint32_t *xp;      // parts of x (split_x_kernel), mt tiles per K step
    const float *x;          // x itself, for the tiles computed again
    const void *w;
    const float *scales;     // of a scaled format: scale of (n, k) at n * sc_n / sc_d + k / 32 / sc_k
    const float *bias;       // null: none
    float *c;
    int64_t ldx, ldw, ldc;   // ldw in bytes
    int64_t M, N, K;
    int64_t sc_n, sc_d;
    uint32_t sc_k;           // K steps per group (0: a group spans whole rows)
    float alpha, beta;
    int relu;                // 0, or 1: v > 0 ? v : 0
    int mt, tiles_m, tiles;  // 16-row tiles of xp; block tiles (m fastest)
    int kps;                 // K steps per split range
    int64_t cstride;         // C of range s at c + s * cstride
};

// 16-byte (or 4-byte) buffer -> LDS DMA: lane l's bytes land at lds + size * l.
template <int SIZE>
__device__ __forceinline__ void sg_dma(const void *base, uint32_t bytes, uint32_t voff, uint32_t soff,
                                       void *lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
    auto *const to = (__attribute__((address_space(3))) void *)lds;
    if constexpr (SIZE == 16)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 16, voff, soff, 0, 0);
    else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, voff, soff, 0, 0);
#endif
}

// Weight formats. B32: bytes of 32 elements; PW: bf16 parts; frag(): the
// parts of elements 8 q .. 8 q + 7 of a step, from the row's LDS piece.
// chunk(c) gives the address of the row's 16-byte chunk c.
template <bool ALIGNED>
struct SplitWF32 {
    static constexpr int B32 = 128, PW = 3, DMA = ALIGNED ? 16 : 4;
    static constexpr bool SCALED = false;
    static constexpr float SMUL = 1.0f;
    template <class Fn>
    static __device__ __forceinline__ void frag(Fn chunk, int step, int q, sg_u4 (&part)[PW],
                                                uint32_t &tiny) {
        const sg_f4 a = *reinterpret_cast<const sg_f4 *>(chunk(8 * step + 2 * q));
        const sg_f4 b = *reinterpret_cast<const sg_f4 *>(chunk(8 * step + 2 * q + 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float u = e < 2 ? a[2 * e] : b[2 * e - 4], v = e < 2 ? a[2 * e + 1] : b[2 * e - 3];
            uint32_t p[3];
            sg_split2(u, v, p);
            part[0][e] = p[0], part[1][e] = p[1], part[2][e] = p[2];
            tiny = std::min(tiny, std::min((__float_as_uint(u) << 1) - 1u, (__float_as_uint(v) << 1) - 1u));
        }
    }
    static __device__ __forceinline__ float at(const void *w, int64_t ldw, int64_t n, int64_t k, float) {
        return *reinterpret_cast<const float *>(static_cast<const uint8_t *>(w) + n * ldw + 4 * k);
    }
    static __device__ __forceinline__ sg_f4 at4(const void *w, int64_t ldw, int64_t n, int64_t k, float) {
        const float *p = reinterpret_cast<const float *>(static_cast<const uint8_t *>(w) + n * ldw) + k;
        if constexpr (ALIGNED) return *reinterpret_cast<const sg_f4 *>(p);
        return sg_f4{p[0], p[1], p[2], p[3]};
    }
};

enum { SPLIT_I4, SPLIT_I8, SPLIT_BF16, SPLIT_E2M1 };

template <int FMT>
struct SplitWQ {
    static constexpr bool NIB = FMT == SPLIT_I4 || FMT == SPLIT_E2M1;
    static constexpr int B32 = NIB ? 16 : FMT == SPLIT_I8 ? 32 : 64, PW = 1, DMA = 16;
    static constexpr bool SCALED = FMT != SPLIT_BF16;
    static constexpr float SMUL = FMT == SPLIT_I4 ? 16.0f : 1.0f;  // INT4 codes decode to q / 16
    template <class Fn>
    static __device__ __forceinline__ void frag(Fn chunk, int step, int q, sg_u4 (&part)[PW],
                                                uint32_t &) {
        if constexpr (FMT == SPLIT_BF16) {
            part[0] = *reinterpret_cast<const sg_u4 *>(chunk(4 * step + q));
        } else if constexpr (FMT == SPLIT_I8) {
            const sg_u2 w = *reinterpret_cast<const sg_u2 *>(chunk(2 * step + q / 2) + 8 * (q & 1));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t d = w[e / 2] >> (16 * (e & 1));
                part[0][e] = sg_hi2((float)(int8_t)d, (float)(int8_t)(d >> 8));
            }
        } else {
            const uint32_t w = *reinterpret_cast<const uint32_t *>(chunk(step) + 4 * q);
            if constexpr (FMT == SPLIT_I4) {
                // the low nibble of byte e is element 2e, the high one 2e + 1
                uint32_t h = w >> 4;
                asm("" : "+v"(h));  // a register of its own: each conversion selects a byte
#pragma unroll
                for (int e = 0; e < 4; ++e)  // v_cvt_off_f32_i4: the low 4 bits q as q / 16
                    part[0][e] = sg_hi2(__builtin_amdgcn_cvt_off_f32_i4((int)((w >> (8 * e)) & 0xFFu)),
                                        __builtin_amdgcn_cvt_off_f32_i4((int)((h >> (8 * e)) & 0xFFu)));
            } else {
                // E2M1 magnitudes 0 .5 1 1.5 2 3 4 6 as bf16: the bytes of both
                // halves by permutes, the sign moved to the high byte's top bit
                const uint32_t il = w & 0x07070707u, ih = (w >> 4) & 0x07070707u;
                const uint32_t hl = __builtin_amdgcn_perm(0x40404040u, 0x3F3F3F00u, il) | (w & 0x08080808u) << 4;
                const uint32_t hh = __builtin_amdgcn_perm(0x40404040u, 0x3F3F3F00u, ih) | (w & 0x80808080u);
                const uint32_t ll = __builtin_amdgcn_perm(0xC0804000u, 0xC0800000u, il);
                const uint32_t lh = __builtin_amdgcn_perm(0xC0804000u, 0xC0800000u, ih);
                // pair e: bytes {ll[e], hl[e], lh[e], hh[e]}
                const uint32_t a0 = __builtin_amdgcn_perm(hl, ll, 0x05010400u);  // ll0 hl0 ll1 hl1
                const uint32_t a1 = __builtin_amdgcn_perm(hl, ll, 0x07030602u);
                const uint32_t b0 = __builtin_amdgcn_perm(hh, lh, 0x05010400u);
                const uint32_t b1 = __builtin_amdgcn_perm(hh, lh, 0x07030602u);
                part[0][0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
                part[0][1] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
                part[0][2] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
                part[0][3] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
            }
        }
    }
    // the stored weight's f32 value (src/quantize.rs:252-269)
    static __device__ __forceinline__ float at(const void *w, int64_t ldw, int64_t n, int64_t k, float s) {
        const uint8_t *row = static_cast<const uint8_t *>(w) + n * ldw;
        if constexpr (FMT == SPLIT_BF16)
            return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t *>(row)[k] << 16);
        else if constexpr (FMT == SPLIT_I8)
            return (float)(int8_t)row[k] * s;
        return nibble(row[k / 2] >> (4 * (k & 1))) * s;
    }
    // elements k .. k + 3 (k % 4 == 0)
    static __device__ __forceinline__ sg_f4 at4(const void *w, int64_t ldw, int64_t n, int64_t k, float s) {
        const uint8_t *row = static_cast<const uint8_t *>(w) + n * ldw;
        sg_f4 v;
        if constexpr (FMT == SPLIT_BF16) {
            uint32_t d[2];
            __builtin_memcpy(d, row + 2 * k, 8);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = __uint_as_float(e & 1 ? d[e / 2] & 0xFFFF0000u : d[e / 2] << 16);
        } else if constexpr (FMT == SPLIT_I8) {
            uint32_t d;
            __builtin_memcpy(&d, row + k, 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (float)(int8_t)(d >> (8 * e)) * s;
        } else {
            uint16_t d;
            __builtin_memcpy(&d, row + k / 2, 2);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = nibble((uint32_t)d >> (4 * e)) * s;
        }
        return v;
    }
    static __device__ __forceinline__ float nibble(uint32_t nib) {  // of the low 4 bits
        if constexpr (FMT == SPLIT_I4) return (float)((int)(nib << 28) >> 28);
        const float mag = nib & 4 ? (nib & 2 ? (nib & 1 ? 6.0f : 4.0f) : (nib & 1 ? 3.0f : 2.0f))
                                  : 0.5f * (float)(nib & 3);
        return nib & 8 ? -mag : mag;
    }
};

template <class W_, int WN_, int WM_, int TN_, int TM_, int KS_>
struct SplitCfg {
    using W = W_;
    static constexpr int WN = WN_, WM = WM_, WK = 8 / (WN * WM), TN = TN_, TM = TM_, KS = KS_;
    static constexpr int NT = 512, BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int ST = KS / 32;              // K steps per block of a stage
    static constexpr int SK = WK * ST;              // K steps per stage
    static constexpr int P = ST * W::B32;           // bytes of a weight row per block
    static constexpr int CPR = P / 16;              // 16-byte chunks of them
    static constexpr int X_BYTES = SK * (BM / 16) * 3072;
    static constexpr int W_BYTES = (WK * BN * P + 8191) / 8192 * 8192;  // whole loads of 8 waves
    static constexpr int STAGE = X_BYTES + W_BYTES;
    static constexpr int XL = X_BYTES / 8192, WL = W_BYTES / (8 * 64 * W::DMA);  // per wave
    static constexpr int R = 160 * 1024 / STAGE < 3 ? 160 * 1024 / STAGE : 3;
    static constexpr int OPS = XL + WL + (W::SCALED ? TN * ST : 0);
    static constexpr int F = TN * TM;
    static constexpr int RED = WK == 1 ? 0 : WK == 2 ? 8 * ((F + 1) / 2) * 1024 : 8 * F * 1024;
    static constexpr int LDS = R * STAGE > RED ? R * STAGE : RED;
    static_assert(WN * WM * WK == 8 && (P == 16 || P == 32 || P == 64 || P == 128), "shape");
    static_assert(X_BYTES % 8192 == 0, "loads");
    static_assert(R >= 2 && LDS <= 160 * 1024 && (R - 2) * OPS < 64, "ring");
};

template <class Fn, int... Is>
__device__ __forceinline__ bool split_stages(Fn &f, int s, std::integer_sequence<int, Is...>) {
    return (f(std::integral_constant<int, Is>{}, s + Is) && ...);
}
template <class Fn, int... Is>
__device__ __forceinline__ void split_each(Fn &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}

template <class C>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(2)))
void split_gemm_kernel(SplitArgs a) {
    using W = typename C::W;
    constexpr int TN = C::TN, TM = C::TM, WK = C::WK, R = C::R, ST = C::ST, PW = W::PW;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (C::WN * C::WM), wm = wave / C::WN % C::WM, wn = wave % C::WN;
    const int fr = lane & 15, fq = lane >> 4;
    const int tile = (int)(blockIdx.x % (unsigned)a.tiles), split = (int)(blockIdx.x / (unsigned)a.tiles);
    const int tm = tile % a.tiles_m, tn = tile / a.tiles_m;
    const int64_t m0 = (int64_t)tm * C::BM, n0 = (int64_t)tn * C::BN;
    // this range's K steps [s0, s0 + steps)
    const int total = (int)((a.K + 31) / 32);
    const int s0 = split * a.kps, steps = std::min(a.kps, total - s0);
    const int ns = (steps + C::SK - 1) / C::SK;

    // x parts: load j of a stage is 1 KiB j % (3 BM / 16) of step j / (3 BM / 16)
    constexpr int XF = 3 * (C::BM / 16);
    const uint32_t *const xt = a.xp + ((int64_t)s0 * a.mt + m0 / 16) * 768;
    const int64_t xleft = ((int64_t)(total - s0) * a.mt - m0 / 16) * 3072;  // bytes to the end
    const uint32_t xrange = (uint32_t)std::min<int64_t>(xleft, 0x7fffffff);
    const uint32_t xstage = (uint32_t)(C::SK * a.mt) * 3072u;
    constexpr uint32_t kPast = 0xfffffff0u;
    uint32_t xo[C::XL], xe[C::XL];
    const int tail = steps - (ns - 1) * C::SK;  // K steps of the last stage
#pragma unroll
    for (int i = 0; i < C::XL; ++i) {
        const int j = wave + 8 * i, st = j / XF;
        xo[i] = (uint32_t)(st * a.mt) * 3072u + (j % XF) * 1024 + 16 * lane;
        xe[i] = st < tail ? xo[i] : kPast;  // steps past the range: zeros
    }
    // weights: load j covers 64 * DMA / P rows of block j / (BN P / (64 DMA))
    const uint8_t *const wb = static_cast<const uint8_t *>(a.w) + n0 * a.ldw + (int64_t)s0 * W::B32;
    const int64_t kbytes = a.K * W::B32 / 32 - (int64_t)s0 * W::B32;  // a row's bytes from s0
    const uint32_t wrange =
        (uint32_t)std::min<int64_t>((a.N - n0 - 1) * a.ldw + kbytes, 0x7fffffff);
    const int wtail = (int)std::min<int64_t>(kbytes - (int64_t)(ns - 1) * WK * C::P,
                                             (int64_t)tail * W::B32);
    uint32_t wo[C::WL], we[C::WL];
#pragma unroll
    for (int i = 0; i < C::WL; ++i) {
        const int b = (wave + 8 * i) * 64 * W::DMA + lane * W::DMA;  // byte of the stage's weights
        const int r = b / C::P % C::BN, g = b / C::P / C::BN, o = b % C::P;
        const int c = (o / 16) ^ (C::P == 128 ? (r >> 1) & 7 : C::P == 64 ? (r >> 2) & 3 : C::P == 32 ? (r >> 3) & 1 : 0);
        const int kb = g * C::P + 16 * c + o % 16;  // byte of the row within the stage
        wo[i] = g < WK && n0 + r < a.N ? (uint32_t)(r * a.ldw + kb) : kPast;
        we[i] = kb < wtail ? wo[i] : kPast;
    }
    const int64_t nw = n0 + 16 * TN * wn;
    float sc[W::SCALED ? R : 1][W::SCALED ? ST : 1][TN];
    int64_t sb[W::SCALED ? TN : 1];  // a column's first scale
    if constexpr (W::SCALED)
#pragma unroll
        for (int t = 0; t < TN; ++t) sb[t] = std::min(nw + 16 * t + fr, a.N - 1) * a.sc_n / a.sc_d;
    auto load = [&](auto ic, int s) {
        constexpr int slot = decltype(ic)::value;
        uint8_t *const buf = smem + slot * C::STAGE;
        auto go = [&](const uint32_t (&xv)[C::XL], const uint32_t (&wv)[C::WL]) {
#pragma unroll
            for (int i = 0; i < C::XL; ++i)
                sg_dma<16>(xt, xrange, xv[i], (uint32_t)s * xstage, buf + 1024 * (wave + 8 * i));
#pragma unroll
            for (int i = 0; i < C::WL; ++i)
                sg_dma<W::DMA>(wb, wrange, wv[i], (uint32_t)s * (WK * C::P),
                               buf + C::X_BYTES + 64 * W::DMA * (wave + 8 * i));
        };
        if (s + 1 < ns)
            go(xo, wo);
        else if (s + 1 == ns)
            go(xe, we);
        else {  // past the range: nothing lands, the number in flight stays the same
            uint32_t xp[C::XL], wp[C::WL];
#pragma unroll
            for (auto &v : xp) v = kPast;
#pragma unroll
            for (auto &v : wp) v = kPast;
            go(xp, wp);
        }
        if constexpr (W::SCALED) {
#pragma unroll
            for (int st = 0; st < ST; ++st) {
                const int step = std::min(s0 + std::min(s, ns - 1) * C::SK + kg * ST + st, total - 1);
                const int64_t col = a.sc_k ? (uint32_t)step / a.sc_k : 0;
#pragma unroll
                for (int t = 0; t < TN; ++t) sc[slot][st][t] = a.scales[sb[t] + col];
            }
        }
    };

    sg_f4 acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int u = 0; u < TM; ++u) acc[t][u] = sg_f4{0.f, 0.f, 0.f, 0.f};
    // One-part weights: the sums of 8 stages are added to a second level, so
    // that fewer additions round at the total's magnitude (error against the
    // 64-bit product at K = 4096, INT4 groups of 128: 1.7e-7 -> 1.2e-7; the
    // 16-row GEMVs 1.4e-7). f32 weights have no registers left for it, and
    // their one level (2.2e-7) is below the f32 MFMA GEMM's 3.0e-7 (split K)
    // to 1.15e-6.
    constexpr bool TWO = PW == 1;
    sg_f4 top[TWO ? TN : 1][TWO ? TM : 1];
#pragma unroll
    for (auto &row : top)
#pragma unroll
        for (auto &v : row) v = sg_f4{0.f, 0.f, 0.f, 0.f};
    auto lift = [&]() {
        if constexpr (TWO) {
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int u = 0; u < TM; ++u) {
                    top[t][u] += acc[t][u];
                    acc[t][u] = sg_f4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    uint32_t tiny = 0xffffffffu;  // smallest 2|w| - 1 (as bits) of this lane's f32 weights
    const int swz = C::P == 128 ? (fr >> 1) & 7 : C::P == 64 ? (fr >> 2) & 3 : C::P == 32 ? (fr >> 3) & 1 : 0;
    auto mm = [](const sg_u4 &xv, const sg_u4 &wv, const sg_f4 &c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sg_b8, xv),
                                                       __builtin_bit_cast(sg_b8, wv), c, 0, 0, 0);
    };
    auto compute = [&](auto ic) {
        constexpr int slot = decltype(ic)::value;
        const uint8_t *const xb = smem + slot * C::STAGE + 16 * lane;
        const uint8_t *const wp = smem + slot * C::STAGE + C::X_BYTES + (kg * C::BN + 16 * TN * wn + fr) * C::P;
#pragma unroll
        for (int st = 0; st < ST; ++st) {
            sg_u4 w[TN][PW];
#pragma unroll
            for (int t = 0; t < TN; ++t)
                W::frag([&](int c) { return wp + 16 * t * C::P + 16 * (c ^ swz); }, st, fq, w[t], tiny);
#pragma unroll
            for (int u = 0; u < TM; ++u) {
                sg_u4 xv[3];
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    xv[p] = *reinterpret_cast<const sg_u4 *>(
                        xb + (((kg * ST + st) * (C::BM / 16) + TM * wm + u) * 3 + p) * 1024);
                // smallest products first
                sg_f4 v[TN];
                auto each = [&](auto pc, auto wc) {
                    constexpr int p = decltype(pc)::value, j = decltype(wc)::value;
#pragma unroll
                    for (int t = 0; t < TN; ++t) v[t] = mm(xv[p], w[t][j], v[t]);
                };
                using I0 = std::integral_constant<int, 0>;
                using I1 = std::integral_constant<int, 1>;
                using I2 = std::integral_constant<int, 2>;
#pragma unroll
                for (int t = 0; t < TN; ++t) v[t] = sg_f4{0.f, 0.f, 0.f, 0.f};
                if constexpr (PW == 3) {
                    each(I2{}, I0{}), each(I0{}, I2{}), each(I1{}, I1{});
                    each(I1{}, I0{}), each(I0{}, I1{}), each(I0{}, I0{});
                } else {
                    each(I2{}, I0{}), each(I1{}, I0{}), each(I0{}, I0{});
                }
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    if constexpr (W::SCALED) {
                        const float s = sc[slot][st][t] * W::SMUL;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[t][u][e] = __builtin_fmaf(v[t][e], s, acc[t][u][e]);
                    } else {
                        acc[t][u] += v[t];
                    }
                }
            }
        }
    };
    auto barrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    split_each([&](auto ic) { load(ic, decltype(ic)::value); }, std::make_integer_sequence<int, R - 1>{});
    auto stage = [&](auto ic, int s) {
        constexpr int i = decltype(ic)::value;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 2) * C::OPS) : "memory");
        barrier();
        load(std::integral_constant<int, (i + R - 1) % R>{}, s + R - 1);
        compute(ic);
        if (TWO && (s & 7) == 7) lift();
        return s + 1 < ns;
    };
    for (int s = 0; split_stages(stage, s, std::make_integer_sequence<int, R>{}); s += R) {
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier();
    if constexpr (TWO) {
        lift();
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int u = 0; u < TM; ++u) acc[t][u] = top[t][u];
    }

    if constexpr (WK > 1) {
        sg_f4 *red = reinterpret_cast<sg_f4 *>(smem);
        auto place = [&](int g, int f) {
            constexpr int PL = WK == 2 ? (C::F + 1) / 2 : C::F;
            return (((g * C::WM + wm) * C::WN + wn) * PL + (WK == 2 ? f / 2 : f)) * 64 + lane;
        };
#pragma unroll
        for (int f = 0; f < C::F; ++f)
            if (f % WK != kg) red[place(kg, f)] = acc[f / TM][f % TM];
        barrier();
#pragma unroll
        for (int f = 0; f < C::F; ++f)
            if (f % WK == kg) {
                sg_f4 &o = acc[f / TM][f % TM];
#pragma unroll
                for (int g = 0; g < WK; ++g)
                    if (g != kg) o += red[place(g, f)];
            }
    }
    // A tile that the parts do not hold is computed again in f32.
    bool again = tiny < 2u * kTinyBits - 1u;
#pragma unroll
    for (int f = 0; f < C::F; ++f)
        if (WK == 1 || f % WK == kg) {
            const sg_f4 v = acc[f / TM][f % TM];
            // (v - v is 0 for finite v, NaN otherwise)
            again |= !((v[0] - v[0]) + (v[1] - v[1]) + (v[2] - v[2]) + (v[3] - v[3]) == 0.0f);
        }
    const int64_t mw = m0 + 16 * TM * wm;
    barrier();  // the partial tiles are read
    uint32_t *const flags = reinterpret_cast<uint32_t *>(smem);
    if (lane == 0) flags[wave] = 0u;
    if (again) flags[wave] = 1u;  // (after lane 0's store: one wave's LDS operations are in order)
    barrier();
    uint32_t any = 0u;
#pragma unroll
    for (int v = 0; v < 8; ++v) any |= flags[v];
    if (any) {
        // Each wave its own fragments, TM + TN operand loads for TN TM of them.
        // Per 16 k, lane group fq takes k + 4 fq .. + 3 of both operands (one
        // 16-byte load where x is aligned); a pass is 32 k. Bound by the loads'
        // latency and lines. With every tile computed again, 2000 x 4096 x 4096
        // f32 takes 1.1 ms and Q8_0 300 x 4096 x 11008 1.08 (one fragment at a
        // time in steps of 4 k: 7.4 and 5.4 ms; without such values 0.38, 0.14).
        const int64_t k0 = 32 * (int64_t)s0, k1 = std::min<int64_t>(a.K, 32 * (int64_t)(s0 + steps));
        const bool vec = (a.ldx & 3) == 0 && ((uintptr_t)a.x & 15) == 0;
#pragma unroll
        for (auto &row : acc)
#pragma unroll
            for (auto &v : row) v = sg_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int64_t kb = k0; kb < k1; kb += 32) {
            const bool whole = kb + 32 <= k1;
            sg_f4 xv[2][TM], wv[2][TN];
#pragma unroll
            for (int u = 0; u < TM; ++u) {
                const float *const xr = a.x + std::min(mw + 16 * u + fr, a.M - 1) * a.ldx;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int64_t k = kb + 16 * h + 4 * fq;
                    if (whole && vec) {
                        xv[h][u] = *reinterpret_cast<const sg_f4 *>(xr + k);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) xv[h][u][e] = k + e < k1 ? xr[k + e] : 0.0f;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const int64_t n = std::min(nw + 16 * t + fr, a.N - 1);
                float s = 1.0f;
                if constexpr (W::SCALED)
                    s = a.scales[n * a.sc_n / a.sc_d + (a.sc_k ? (uint32_t)(kb / 32) / a.sc_k : 0)];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int64_t k = kb + 16 * h + 4 * fq;
                    if (whole) {
                        wv[h][t] = W::at4(a.w, a.ldw, n, k, s);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            wv[h][t][e] = k + e < k1 ? W::at(a.w, a.ldw, n, k + e, s) : 0.0f;
                    }
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int t = 0; t < TN; ++t)
#pragma unroll
                        for (int u = 0; u < TM; ++u)
                            if (WK == 1 || (t * TM + u) % WK == kg)
                                acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                    xv[h][u][e], wv[h][t][e], acc[t][u], 0, 0, 0);
        }
    }
    // lane: rows mw + 16 u + 4 fq + e, column nw + 16 t + fr
    float *const cp = a.c + split * a.cstride;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int64_t n = nw + 16 * t + fr;
        if (n >= a.N) continue;
        const float bn = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
        for (int u = 0; u < TM; ++u) {
            if (WK > 1 && (t * TM + u) % WK != kg) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t m = mw + 16 * u + 4 * fq + e;
                if (m >= a.M) continue;
                float v = a.alpha * acc[t][u][e];
                if (a.beta != 0.0f) v = v + a.beta * cp[m * a.ldc + n];
                if (a.bias) v = v + bn;
                if (a.relu) v = v > 0.0f ? v : 0.0f;
                cp[m * a.ldc + n] = v;
            }
        }
    }
}

// C = alpha * (P_0 + ... + P_{S-1}) + beta * C (+ bias, ReLU): the ranges'
// partial products (M x N each, cstride apart) added in order.
static __global__ __launch_bounds__(256) void split_sum_kernel(const float *__restrict__ P, int S,
                                                        SplitArgs a) {
    for (int64_t m = blockIdx.y; m < a.M; m += gridDim.y)
        for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < a.N;
             n += (int64_t)gridDim.x * blockDim.x) {
            const float *p = P + m * a.N + n;
            float v = p[0];
            for (int s = 1; s < S; ++s) v += p[s * a.M * a.N];
            v = a.alpha * v;
            float *cp = a.c + m * a.ldc + n;
            if (a.beta != 0.0f) v = v + a.beta * *cp;
            if (a.bias) v = v + a.bias[n];
            if (a.relu) v = v > 0.0f ? v : 0.0f;
            *cp = v;
        }
}

// A tile shape: `step` is the time (us) of one K step of a round of tiles (one
// per CU), measured by graph replay at K = 4096.
struct SplitShape {
    int bm, bn, sk;
    double step;
    void (*run)(const SplitArgs &, unsigned, hipStream_t);
};
template <class C>
static void split_run(const SplitArgs &a, unsigned grid, hipStream_t st) {
    split_gemm_kernel<C><<<grid, C::NT, 0, st>>>(a);
}
template <class C>
constexpr SplitShape split_shape(double step) {
    return SplitShape{C::BM, C::BN, C::SK, step, split_run<C>};
}

struct SplitPlan {
    const SplitShape *s = nullptr;
    int S = 1, kps = 0, mt = 0;
    size_t planes = 0, bytes = 0;  // scratch: the parts of x, then the partial products
    double cost = 0.0;
};

// The shape and number of K ranges with the smallest estimate: the two
// launches, the rounds of tiles times their K steps, and for several ranges
// the sum's launch and traffic.
static inline SplitPlan split_plan(const SplitShape *shapes, int count, int64_t M, int64_t N, int64_t K) {
    SplitPlan best;
    const int64_t total = ceil_div(K, 32), cus = device_cu_count();
    for (int i = 0; i < count; ++i) {
        const SplitShape &s = shapes[i];
        const int64_t tiles = ceil_div(M, s.bm) * ceil_div(N, s.bn);
        for (int64_t S = 1; S <= 8; S *= 2) {
            const int64_t kps = ceil_div(ceil_div(total, S), s.sk) * s.sk;
            const int64_t ranges = ceil_div(total, kps);
            if (S > 1 && (ranges != S || tiles * S > 4 * cus)) break;
            const double rounds = (double)ceil_div(tiles * ranges, cus);
            double c = 6.0 + rounds * (1.0 + (double)kps * s.step);
            if (S > 1) c += 3.0 + (double)(S * M * N) * 2e-6;
            if (!best.s || c < best.cost) {
                best.s = &s, best.cost = c, best.S = (int)ranges, best.kps = (int)kps;
                best.mt = (int)(ceil_div(M, s.bm) * s.bm / 16);
            }
        }
    }
    best.planes = (size_t)(total * best.mt) * 3072;
    best.bytes = best.planes + (best.S > 1 ? (size_t)(best.S * M * N) * 4 : 0);
    return best;
}
// 32-bit offsets: a tile's weight rows, and the parts of x.
static inline bool split_fits(int64_t M, int64_t K, int64_t ldw_bytes) {
    return 256 * ldw_bytes < (int64_t(1) << 31) && ceil_div(K, 32) * (M + 128) * 192 < (int64_t(1) << 31);
}

// `a` as the caller has filled it (operands, sizes, alpha, beta, bias, relu).
static inline int split_launch(const SplitPlan &pl, SplitArgs a, void *scratch, hipStream_t st,
                               const char *name) {
    const int64_t total = ceil_div(a.K, 32), frags = total * pl.mt;
    uint32_t *xp = static_cast<uint32_t *>(scratch);
    const unsigned g = (unsigned)std::min<int64_t>(ceil_div(frags, 4), 8 * device_cu_count());
    if (a.ldx % 4 == 0 && ((uintptr_t)a.x & 15) == 0)
        split_x_kernel<true><<<g, 256, 0, st>>>(a.x, a.ldx, a.M, a.K, pl.mt, frags, xp);
    else
        split_x_kernel<false><<<g, 256, 0, st>>>(a.x, a.ldx, a.M, a.K, pl.mt, frags, xp);
    RNN_TRY(check_launch(name));
    SplitArgs k = a;
    k.xp = xp;
    k.mt = pl.mt;
    k.tiles_m = (int)ceil_div(a.M, pl.s->bm);
    const int64_t tiles = k.tiles_m * ceil_div(a.N, pl.s->bn);
    RNN_REQUIRE(tiles * pl.S <= 0x7fffffffLL, "%s: too many tiles", name);
    k.tiles = (int)tiles;
    k.kps = pl.kps;
    if (pl.S > 1) {
        k.c = reinterpret_cast<float *>(static_cast<uint8_t *>(scratch) + pl.planes);
        k.ldc = a.N, k.cstride = a.M * a.N;
        k.alpha = 1.0f, k.beta = 0.0f, k.bias = nullptr, k.relu = 0;
    }
    pl.s->run(k, (unsigned)(tiles * pl.S), st);
    RNN_TRY(check_launch(name));
    if (pl.S > 1) {
        const dim3 sg((unsigned)ceil_div(a.N, 256), (unsigned)std::min<int64_t>(a.M, 65535));
        split_sum_kernel<<<sg, 256, 0, st>>>(k.c, pl.S, a);
        return check_launch(name);
    }
    return RNN_OK;
}

}  // namespace rnn
