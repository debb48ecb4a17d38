// Wave GEMV for Q4_K / Q5_K / Q6_K with f32 activations on gfx950 (CDNA4,
// wave64): the default decode projection, the arithmetic of the reference's
// warp kernels (crates/nvidia/src/kernels/quantized/q4_k.cu:103-159,
// q5_k.cu:37-98, q6_k.cu:45-109): f32 activations against weights dequantised
// in registers, f32 accumulation. Optional fused RMSNorm or SwiGLU prologue,
// grouped weights sharing one input (q/k/v, gate/up) and gate/up pairs with a
// SwiGLU epilogue, as in gemv_wave.hip.
//
// Mapping: the wave / lane layout of wave_rows.hpp (a lane owns 64 weights of
// one super-block per unit of row x slice).
//
// Activations
//  - Each workgroup stages x (times gamma, or silu(x) * x2) once, in f32, into
//    LDS "lane records": the 64 activations a lane multiplies, in the order it
//    uses them, then the f32 sum X_g of each of its scale groups. A record is
//    68 dwords (17 x 16 bytes, odd), so 16 lanes' 128-bit reads hit distinct
//    banks. One member's slice is 17 KB.
//  - One or two members: a lane keeps its record in VGPRs (64 floats a member)
//    for every row it reduces. Three to eight: gemv_f32_many_kernel below.
//
// Arithmetic of one lane and one unit, per scale group g (32 elements for
// Q4_K / Q5_K, 16 for Q6_K; crates/gguf/src/lib.rs:596-661):
//      S_g  = sum_i q_i * x_i          (f32 FMAs, element order)
//      Q4_K / Q5_K:  part += (d*sc_g) * S_g - (dmin*m_g) * X_g
//      Q6_K:         part += (d*sc_g) * (S_g - 32 X_g)
//  which is sum_i ((d*sc_g)*q_i - dmin*m_g) * x_i (respectively (q_i - 32)) with
//  the same products: the dequantised weight times x, regrouped per scale
//  group. Every quantity is f32; nothing is rounded to a narrower format.
//
// Canonical order of a row (every launch shape and member count follows it,
// so a member's output bits never depend on the batch it runs in):
//   P_s = DPP/readlane wave sum of the lanes' parts of slice s (fixed tree),
//   T   = ((P_0 + P_1) + P_2) ... in slice order,
//   y   = T * inv with inv = 1/sqrt(sum(x^2)/K + eps) for RMSNorm (else y = T),
//   sum(x^2) = per 256-element block, a fixed lane tree; blocks added in order.
#include "per_device.hpp"
#include "wave_rows.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace ribn_amd {

namespace {

template <int T> struct F32Rec {
    static constexpr int group = (T == kQ6K) ? 16 : 32;  // elements per scale group
    static constexpr int groups = 64 / group;            // scale groups per lane
    static constexpr int stride = 68;                    // dwords per lane record
};

constexpr int kF32Blocks = kWaveMaxK / 256;  // super-blocks of the largest K staged

// Lane record and position of element e (a multiple of 4, within one slice).
template <int T>
__device__ __forceinline__ void f32_slot(int e, int& rec, int& pos) {
    if constexpr (T == kQ6K) {
        const int bs = e >> 8, c = (e >> 7) & 1, v = (e >> 5) & 3, s = (e >> 4) & 1;
        rec = 4 * bs + 2 * c + s;
        pos = 16 * v + (e & 15);
    } else {
        rec = e >> 6;
        pos = e & 63;
    }
}

// Sum over the consecutive lanes holding one scale group (8 or 4 lanes of 4
// elements); every lane of the group receives the same value.
template <int T>
__device__ __forceinline__ float group_sum_f(float v) {
    v = dpp_step<0xb1>(v);  // quad_perm [1,0,3,2]
    v = dpp_step<0x4e>(v);  // quad_perm [2,3,0,1]
    if constexpr (F32Rec<T>::group == 32) v = dpp_step<0x141>(v);  // row_half_mirror
    return v;
}

__device__ __forceinline__ float byte_f(uint32_t w, int t) { return (float)((w >> (8 * t)) & 0xffu); }

// The value passes through an empty asm statement, so the compiler no longer
// knows its bits: byte_f of a masked word then stays one v_cvt_f32_ubyte{t}
// instead of a bit-field extract plus a convert.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}
// ------------------------------------------------- scales and quants of a unit
//
// Q4_K / Q5_K: (d*sc, dmin*m) of the lane's groups 2p (a0, b0) and 2p+1 (a1, b1).
template <int T>
__device__ __forceinline__ void group_scales(const uint4 h, int p, float& a0, float& a1, float& b0, float& b1) {
    const float dd = half_bits_to_float(h.x & 0xffffu);
    const float dmin = half_bits_to_float(h.x >> 16);
    // six-bit scales / minima of all 8 groups, four per word (lib.rs:573-587)
    const uint32_t lo_sc = h.y & 0x3f3f3f3fu;
    const uint32_t lo_mn = h.z & 0x3f3f3f3fu;
    const uint32_t hi_sc = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
    const uint32_t hi_mn = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    const uint32_t scw = (p < 2) ? lo_sc : hi_sc;
    const uint32_t mnw = (p < 2) ? lo_mn : hi_mn;
    const int sh = (p & 1) * 16;
    // Q4_K quants enter as q * 2^-9 (quant_quads): scales carry the 2^9, exactly
    constexpr float kQScale = (T == kQ4K) ? 512.0f : 1.0f;
    a0 = (dd * (float)((scw >> sh) & 0xffu)) * kQScale;
    a1 = (dd * (float)((scw >> (sh + 8)) & 0xffu)) * kQScale;
    b0 = dmin * (float)((mnw >> sh) & 0xffu);
    b1 = dmin * (float)((mnw >> (sh + 8)) & 0xffu);
}

// Q4_K / Q5_K: quants 4j .. 4j+3 of group A = 2p (low nibbles) and B = 2p+1
// (high nibbles), with Q5_K's fifth bit, as f32.
template <int T>
__device__ __forceinline__ void quant_quads(const RowData<T>& d, int j, int p, float (&fa)[4], float (&fb)[4]) {
    const uint32_t qw[8] = {d.qa.x, d.qa.y, d.qa.z, d.qa.w, d.qb.x, d.qb.y, d.qb.z, d.qb.w};
    uint32_t qa = qw[j] & 0x0f0f0f0fu;
    uint32_t qb = (qw[j] >> 4) & 0x0f0f0f0fu;
    if constexpr (T == kQ4K) {
        // Bytes 0..15 read as OCP E4M3 are exactly q * 2^-9: two quants per
        // convert (the 2^9 is folded into the scales).
        const auto a01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qa, false);
        const auto a23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qa, true);
        const auto b01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qb, false);
        const auto b23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qb, true);
        fa[0] = a01[0];
        fa[1] = a01[1];
        fa[2] = a23[0];
        fa[3] = a23[1];
        fb[0] = b01[0];
        fb[1] = b01[1];
        fb[2] = b23[0];
        fb[3] = b23[1];
    } else {
        const uint32_t hw[8] = {d.ha.x, d.ha.y, d.ha.z, d.ha.w, d.hb.x, d.hb.y, d.hb.z, d.hb.w};
        qa = opaque(qa | (((hw[j] >> (2 * p)) & 0x01010101u) << 4));
        qb = opaque(qb | (((hw[j] >> (2 * p + 1)) & 0x01010101u) << 4));
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            fa[t] = byte_f(qa, t);
            fb[t] = byte_f(qb, t);
        }
    }
}

// Q6_K: the lane's four d*scale factors and its quant words, windows joined.
__device__ __forceinline__ void q6_fields(const RowData<kQ6K>& d, int p, float (&a)[4], uint32_t (&law)[4],
                                          uint32_t (&lbw)[4], uint32_t (&qhw)[4]) {
    const int c = p >> 1, s = p & 1;
    const uint4 la = funnel(d.la, d.la_t, d.shift);
    const uint4 lb = funnel(d.lb, d.lb_t, d.shift);
    const uint4 qh = funnel(d.qh, d.qh_t, d.shift);
    const uint4 sc = funnel(d.sc, d.sc_t, d.shift);  // int8 scales
    const float dd = half_bits_to_float(d.d16);
    const uint32_t w0 = c ? sc.z : sc.x;  // scales 8c+0..8c+3
    const uint32_t w1 = c ? sc.w : sc.y;  // scales 8c+4..8c+7
    a[0] = dd * (float)(int8_t)((w0 >> (8 * s)) & 0xffu);
    a[1] = dd * (float)(int8_t)((w0 >> (8 * (2 + s))) & 0xffu);
    a[2] = dd * (float)(int8_t)((w1 >> (8 * s)) & 0xffu);
    a[3] = dd * (float)(int8_t)((w1 >> (8 * (2 + s))) & 0xffu);
    law[0] = la.x; law[1] = la.y; law[2] = la.z; law[3] = la.w;
    lbw[0] = lb.x; lbw[1] = lb.y; lbw[2] = lb.z; lbw[3] = lb.w;
    qhw[0] = qh.x; qhw[1] = qh.y; qhw[2] = qh.z; qhw[3] = qh.w;
}

// Q6_K: four quants (0..63) of 16-element group v from its low-nibble word
// (la for even v, lb for odd) and high-bit word; the -32 enters through X_v.
__device__ __forceinline__ void q6_quad(uint32_t lw, uint32_t qh, int v, float (&f)[4]) {
    uint32_t q;
    if (v == 0) q = (lw & 0x0f0f0f0fu) | ((qh << 4) & 0x30303030u);
    else if (v == 1) q = (lw & 0x0f0f0f0fu) | ((qh << 2) & 0x30303030u);
    else if (v == 2) q = ((lw >> 4) & 0x0f0f0f0fu) | (qh & 0x30303030u);
    else q = ((lw >> 4) & 0x0f0f0f0fu) | ((qh >> 2) & 0x30303030u);
    q = opaque(q);
#pragma unroll
    for (int t = 0; t < 4; ++t) f[t] = byte_f(q, t);
}

// --------------------------------------------------------- lane dot product
//
// part[m] = this lane's share of the unit's row . x_m. xf(m, i) returns the
// i-th float4 of member m's lane record, sf(m, g) its group sum X_g. Each
// member sees the same operation sequence whatever MT is.
template <int T, int MT, class XF, class SF>
__device__ __forceinline__ void row_dot(const RowData<T>& d, int p, XF xf, SF sf, float (&part)[MT]) {
    auto mac4 = [](const float (&f)[4], const float4 x, float s) {
        s = __builtin_fmaf(f[0], x.x, s);
        s = __builtin_fmaf(f[1], x.y, s);
        s = __builtin_fmaf(f[2], x.z, s);
        return __builtin_fmaf(f[3], x.w, s);
    };
    if constexpr (T == kQ4K || T == kQ5K) {
        float a0, a1, b0, b1;
        group_scales<T>(d.h, p, a0, a1, b0, b1);
        float sA[MT], sB[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) sA[m] = sB[m] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float fa[4], fb[4];
            quant_quads<T>(d, j, p, fa, fb);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                sA[m] = mac4(fa, xf(m, j), sA[m]);
                sB[m] = mac4(fb, xf(m, 8 + j), sB[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float tA = __builtin_fmaf(a0, sA[m], -(b0 * sf(m, 0)));
            const float tB = __builtin_fmaf(a1, sB[m], -(b1 * sf(m, 1)));
            part[m] = tA + tB;
        }
    } else {
        float a[4];
        uint32_t law[4], lbw[4], qhw[4];
        q6_fields(d, p, a, law, lbw, qhw);
        // one 16-element group v at a time: element 16v + 4j + t of the lane's record
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float sv[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) sv[m] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float f[4];
                q6_quad((v & 1) ? lbw[j] : law[j], qhw[j], v, f);
#pragma unroll
                for (int m = 0; m < MT; ++m) sv[m] = mac4(f, xf(m, 4 * v + j), sv[m]);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float t = a[v] * (sv[m] - 32.0f * sf(m, v));  // 32 X exact
                part[m] = (v == 0) ? t : part[m] + t;
            }
        }
    }
}

// row_dot for gemv_f32_kernel's ring, the same operations in the same order. It
// spells out what the helpers above compute, and Q6_K keeps two loops of one
// trip, because the compiler's order of loads and conversions depends on both,
// and the ring's rate on that order: through row_dot one member of Q6_K
// 12288 -> 4096 took 11.8 us, without the two loops 11.3, as it stands 10.6; Q5_K
// 12288 -> 4096 10.2 against 10.0. (Two members of Q6_K in one slice are faster
// through row_dot, gate/up of 2048 -> 2 x 3072 8.7 against 9.1 us.)
template <int T, int MT, class XF, class SF>
__device__ __forceinline__ void ring_row_dot(const RowData<T>& row, int p, XF xf, SF sf, float (&part)[MT]) {
    const RowData<T> d = row;
    if constexpr (T == kQ4K || T == kQ5K) {
        const uint4 h = d.h;
        const float dd = half_bits_to_float(h.x & 0xffffu);
        const float dmin = half_bits_to_float(h.x >> 16);
        // six-bit scales / minima of all 8 groups, four per word (lib.rs:573-587)
        const uint32_t lo_sc = h.y & 0x3f3f3f3fu;
        const uint32_t lo_mn = h.z & 0x3f3f3f3fu;
        const uint32_t hi_sc = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
        const uint32_t hi_mn = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
        const uint32_t scw = (p < 2) ? lo_sc : hi_sc;
        const uint32_t mnw = (p < 2) ? lo_mn : hi_mn;
        const int sh = (p & 1) * 16;
        // Q4_K quants enter as q * 2^-9 (see below): scales carry the 2^9, exactly
        constexpr float kQScale = (T == kQ4K) ? 512.0f : 1.0f;
        const float a0 = (dd * (float)((scw >> sh) & 0xffu)) * kQScale;
        const float a1 = (dd * (float)((scw >> (sh + 8)) & 0xffu)) * kQScale;
        const float b0 = dmin * (float)((mnw >> sh) & 0xffu);
        const float b1 = dmin * (float)((mnw >> (sh + 8)) & 0xffu);
        float sA[MT], sB[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) sA[m] = sB[m] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // group A = 2p (low nibbles), group B = 2p+1 (high nibbles), 5th bit for Q5_K
            float fa[4], fb[4];
            const uint32_t qw[8] = {d.qa.x, d.qa.y, d.qa.z, d.qa.w, d.qb.x, d.qb.y, d.qb.z, d.qb.w};
            uint32_t qa = qw[j] & 0x0f0f0f0fu;
            uint32_t qb = (qw[j] >> 4) & 0x0f0f0f0fu;
            if constexpr (T == kQ5K) {
                const uint32_t hw[8] = {d.ha.x, d.ha.y, d.ha.z, d.ha.w, d.hb.x, d.hb.y, d.hb.z, d.hb.w};
                qa |= ((hw[j] >> (2 * p)) & 0x01010101u) << 4;
                qb |= ((hw[j] >> (2 * p + 1)) & 0x01010101u) << 4;
            }
            if constexpr (T == kQ4K) {
                // Bytes 0..15 read as OCP E4M3 are exactly q * 2^-9: two
                // quants per convert (the 2^9 is folded into the scales).
                const auto a01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qa, false);
                const auto a23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qa, true);
                const auto b01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qb, false);
                const auto b23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)qb, true);
                fa[0] = a01[0];
                fa[1] = a01[1];
                fa[2] = a23[0];
                fa[3] = a23[1];
                fb[0] = b01[0];
                fb[1] = b01[1];
                fb[2] = b23[0];
                fb[3] = b23[1];
            } else {
                qa = opaque(qa);
                qb = opaque(qb);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    fa[t] = byte_f(qa, t);
                    fb[t] = byte_f(qb, t);
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float4 xa = xf(m, j);
                const float4 xb = xf(m, 8 + j);
                sA[m] = __builtin_fmaf(fa[0], xa.x, sA[m]);
                sA[m] = __builtin_fmaf(fa[1], xa.y, sA[m]);
                sA[m] = __builtin_fmaf(fa[2], xa.z, sA[m]);
                sA[m] = __builtin_fmaf(fa[3], xa.w, sA[m]);
                sB[m] = __builtin_fmaf(fb[0], xb.x, sB[m]);
                sB[m] = __builtin_fmaf(fb[1], xb.y, sB[m]);
                sB[m] = __builtin_fmaf(fb[2], xb.z, sB[m]);
                sB[m] = __builtin_fmaf(fb[3], xb.w, sB[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float xA = sf(m, 0), xB = sf(m, 1);
            const float tA = __builtin_fmaf(a0, sA[m], -(b0 * xA));
            const float tB = __builtin_fmaf(a1, sB[m], -(b1 * xB));
            part[m] = tA + tB;
        }
    } else {
        const int c = p >> 1, s = p & 1;
        float a[4];
        uint32_t law[4], lbw[4], qhw[4];
#pragma unroll
        for (int once = 0; once < 1; ++once) {
            const uint32_t sh = d.shift;
            const uint4 la = funnel(d.la, d.la_t, sh);
            const uint4 lb = funnel(d.lb, d.lb_t, sh);
            const uint4 qh = funnel(d.qh, d.qh_t, sh);
            const uint4 sc = funnel(d.sc, d.sc_t, sh);  // int8 scales
            const float dd = half_bits_to_float(d.d16);
            const uint32_t w0 = c ? sc.z : sc.x;  // scales 8c+0..8c+3
            const uint32_t w1 = c ? sc.w : sc.y;  // scales 8c+4..8c+7
            a[0] = dd * (float)(int8_t)((w0 >> (8 * s)) & 0xffu);
            a[1] = dd * (float)(int8_t)((w0 >> (8 * (2 + s))) & 0xffu);
            a[2] = dd * (float)(int8_t)((w1 >> (8 * s)) & 0xffu);
            a[3] = dd * (float)(int8_t)((w1 >> (8 * (2 + s))) & 0xffu);
            law[0] = la.x; law[1] = la.y; law[2] = la.z; law[3] = la.w;
            lbw[0] = lb.x; lbw[1] = lb.y; lbw[2] = lb.z; lbw[3] = lb.w;
            qhw[0] = qh.x; qhw[1] = qh.y; qhw[2] = qh.z; qhw[3] = qh.w;
        }
        // One 16-element group v at a time: quants 0..63 of group v are
        // element 16v + 4j + t of the lane's record (the -32 offset enters
        // through X_v).
        float acc[MT];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float sv[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) sv[m] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float f[4];
                uint32_t q;
                const uint32_t lw = (v & 1) ? lbw[j] : law[j];
                if (v == 0) q = (lw & 0x0f0f0f0fu) | ((qhw[j] << 4) & 0x30303030u);
                else if (v == 1) q = (lw & 0x0f0f0f0fu) | ((qhw[j] << 2) & 0x30303030u);
                else if (v == 2) q = ((lw >> 4) & 0x0f0f0f0fu) | (qhw[j] & 0x30303030u);
                else q = ((lw >> 4) & 0x0f0f0f0fu) | ((qhw[j] >> 2) & 0x30303030u);
                q = opaque(q);
#pragma unroll
                for (int t = 0; t < 4; ++t) f[t] = byte_f(q, t);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const float4 xv = xf(m, 4 * v + j);
                    sv[m] = __builtin_fmaf(f[0], xv.x, sv[m]);
                    sv[m] = __builtin_fmaf(f[1], xv.y, sv[m]);
                    sv[m] = __builtin_fmaf(f[2], xv.z, sv[m]);
                    sv[m] = __builtin_fmaf(f[3], xv.w, sv[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float x32 = 32.0f * sf(m, v);  // exact
#pragma unroll
                for (int once = 0; once < 1; ++once) {
                    const float t = a[v] * (sv[m] - x32);
                    acc[m] = (v == 0) ? t : acc[m] + t;
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) part[m] = acc[m];
    }
}

}  // namespace

// ------------------------------------------------------------------ kernel

// SPLIT: K spans several slices and each workgroup takes one of them
// (blockIdx.y); it stores each row's slice total P_s (before any RMSNorm
// factor) to args.partial[s][members][rows], and f32_split_reduce_kernel adds
// the slices in order. The result equals the one-launch form bit for bit.
template <int T, int MT, int PRO, bool ONE_SLICE, int NBUF, int WAVES, int GROUP, bool PAIR, bool SPLIT = false>
__global__ __launch_bounds__(WAVES * 64) void gemv_f32_kernel(WaveGemvArgs args) {
    static_assert(NBUF % GROUP == 0, "the ring holds whole row groups");
    static_assert(!SPLIT || (ONE_SLICE && !PAIR && PRO == kProPlain), "slice splits are plain one-slice passes");
    static_assert(!PAIR || (ONE_SLICE && NBUF % 2 == 0), "pairs are whole ring slots of one-slice rows");
    static_assert(MT <= 2, "lane records are held in VGPRs");
    constexpr bool NORM = PRO == kProNorm;
    constexpr bool SWIGLU = PRO == kProSwiglu;
    constexpr int G = F32Rec<T>::groups;
    constexpr int STRIDE = F32Rec<T>::stride;
    constexpr int BB = BlockTraits<T>::bytes;
    constexpr int NBMAX = ONE_SLICE ? 16 : kF32Blocks;
    constexpr int NBW = (NBMAX + WAVES - 1) / WAVES;  // staging blocks per wave
    extern __shared__ __attribute__((aligned(16))) float xs[];  // [MT][slices][64 records][STRIDE]
    __shared__ float ssq_s[NORM ? MT : 1][NORM ? NBMAX : 1];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = args.K;
    const int nb = K >> 8;
    const int slices = ONE_SLICE ? 1 : (nb + 15) >> 4;
    const int slice0 = SPLIT ? (int)blockIdx.y : 0;  // the slice this workgroup covers (SPLIT)
    const int members = args.members;
    const int p = lane & 3;
    const int bs = lane >> 2;
    const int nwaves = gridDim.x * WAVES;
    const int wg = blockIdx.x * WAVES + wave;
    const int split = PAIR ? args.total_rows >> 1 : args.total_rows;
    const int r_begin = (PAIR ? 2 : 1) * (int)((long long)split * wg / nwaves);
    const int r_end = (PAIR ? 2 : 1) * (int)((long long)split * (wg + 1) / nwaves);
    const uint32_t row_bytes = (uint32_t)nb * BB;

    auto locate = [&](int row, int& mat, int& local) {
        if constexpr (PAIR) {
            mat = row & 1;
            local = row >> 1;
            return;
        }
        mat = 0;
        int start = 0;
#pragma unroll
        for (int i = 0; i < kMaxGroup - 1; ++i) {
            if (i + 1 < args.count && row >= args.rows_end[i]) {
                mat = i + 1;
                start = args.rows_end[i];
            }
        }
        local = row - start;
    };
    auto pick_w = [&](int mat) {
        const uint8_t* w = args.w[0];
        uint32_t bytes = args.wbytes[0];
#pragma unroll
        for (int i = 1; i < kMaxGroup; ++i) {
            if (mat == i) {
                w = args.w[i];
                bytes = args.wbytes[i];
            }
        }
        return make_rsrc(w, bytes);
    };
    auto pick_y = [&](int mat, int& rows_mat) {
        float* y = args.y[0];
        int begin = 0, end = args.rows_end[0];
#pragma unroll
        for (int i = 1; i < kMaxGroup; ++i) {
            if (mat == i) {
                y = args.y[i];
                begin = args.rows_end[i - 1];
                end = args.rows_end[i];
            }
        }
        rows_mat = end - begin;
        return make_rsrc(y, (uint32_t)members * (uint32_t)rows_mat * 4u);
    };

    // Rows only move forward in one-slice launches, so the matrix of the
    // current row (and its weight / output resources) is tracked by cursors
    // that change only at matrix boundaries instead of being selected per unit.
    struct Cursor {
        int mat, start, end;
        __amdgpu_buffer_rsrc_t rs;
        int rows_mat;
    };
    auto cursor_at = [&](int row, bool out) {
        Cursor c;
        int local;
        locate(row, c.mat, local);
        c.start = row - local;
        const __amdgpu_buffer_rsrc_t yr = pick_y(c.mat, c.rows_mat);
        c.end = c.start + c.rows_mat;
        c.rs = out ? yr : pick_w(c.mat);
        return c;
    };
    auto seek = [&](Cursor& c, int row, bool out) {
        if (row >= c.end && c.mat + 1 < args.count) c = cursor_at(row, out);
    };

    // ---- activation loads first (vector memory returns in order, so the
    // staging waits for these, not for the weight loads issued after them).
    // Wave w stages super-blocks w, w + WAVES, ... of every member.
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(args.x, (uint32_t)members * (uint32_t)K * 4u);
    const __amdgpu_buffer_rsrc_t gr = make_rsrc(args.gamma, NORM ? (uint32_t)K * 4u : 0u);
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(args.x2, SWIGLU ? (uint32_t)members * (uint32_t)K * 4u : 0u);
    float4 xv[NBW][MT];
    float4 gv[NORM ? NBW : 1];
    float4 uv[SWIGLU ? NBW : 1][SWIGLU ? MT : 1];
#pragma unroll
    for (int k = 0; k < NBW; ++k) {
        const int b = 16 * slice0 + wave + WAVES * k;
        const int e = 256 * b + 4 * lane;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint32_t off = (b < nb && m < members) ? (uint32_t)(m * K + e) * 4u : kOutOfRange;
            xv[k][m] = load_f4(xr, off);
            if constexpr (SWIGLU) uv[k][m] = load_f4(ur, off);
        }
        if constexpr (NORM) gv[k] = load_f4(gr, b < nb ? (uint32_t)e * 4u : kOutOfRange);
    }
    asm volatile("" ::: "memory");

    // ---- weight ring, primed now; loads are unconditional (dead units read
    // from an out-of-range offset and return zeros), so each wait covers
    // exactly the unit reduced next.
    RowData<T> ring[NBUF];
    int lrow = r_begin, lslice = 0;
    constexpr bool kCursor = ONE_SLICE && !PAIR;
    Cursor lcur = cursor_at(r_begin, false);
    Cursor ccur = cursor_at(r_begin, true);
    // gate/up pairs: the two weights alternate row by row into one output
    const __amdgpu_buffer_rsrc_t pair_w0 = make_rsrc(args.w[0], PAIR ? args.wbytes[0] : 0u);
    const __amdgpu_buffer_rsrc_t pair_w1 = make_rsrc(args.w[1], PAIR ? args.wbytes[1] : 0u);
    const int pair_rows = args.rows_end[0];
    const __amdgpu_buffer_rsrc_t pair_y =
        make_rsrc(args.y[0], PAIR ? (uint32_t)members * (uint32_t)pair_rows * 4u : 0u);
    auto load_next = [&](RowData<T>& dst, int r) {
        const int row = ONE_SLICE ? lrow : lrow + r % GROUP;
        const bool live_row = row < r_end;
        int mat, local;
        __amdgpu_buffer_rsrc_t rs;
        if constexpr (kCursor) {
            if (live_row) seek(lcur, row, false);
            rs = lcur.rs;
            local = row - lcur.start;
        } else if constexpr (PAIR) {
            rs = (row & 1) ? pair_w1 : pair_w0;
            local = row >> 1;
        } else {
            locate(live_row ? row : r_begin, mat, local);
            rs = pick_w(mat);
        }
        const int b = (SPLIT ? slice0 : lslice) * 16 + bs;
        const bool live = live_row && b < nb;
        load_row<T>(dst, rs, live ? (uint32_t)local * row_bytes + (uint32_t)b * BB : kOutOfRange, p);
        if constexpr (ONE_SLICE) {
            ++lrow;
        } else if (r % GROUP == GROUP - 1 && ++lslice == slices) {
            lslice = 0;
            lrow += GROUP;
        }
    };
#pragma unroll
    for (int r = 0; r < NBUF; ++r) load_next(ring[r], r);

    // ---- staging: f32 activations into the lane records, group sums, and
    // per-block sums of squares for RMSNorm.
#pragma unroll
    for (int k = 0; k < NBW; ++k) {
        const int b = 16 * slice0 + wave + WAVES * k;
        const int e = 256 * b + 4 * lane;
        const int slice = (b >> 4) - slice0;  // staged slice (LDS index)
        int rec, pos;
        f32_slot<T>(e - (b >> 4) * kSliceElems, rec, pos);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float4 v = xv[k][m];
            if constexpr (SWIGLU) {
                // silu(gate) * up, in the reference's operation order (model_ops.rs:316-328)
                v.x = (v.x / (1.0f + expf(-v.x))) * uv[k][m].x;
                v.y = (v.y / (1.0f + expf(-v.y))) * uv[k][m].y;
                v.z = (v.z / (1.0f + expf(-v.z))) * uv[k][m].z;
                v.w = (v.w / (1.0f + expf(-v.w))) * uv[k][m].w;
            }
            if constexpr (NORM) {
                const float sq = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                const float blk = wave_sum_uniform(sq);
                if (lane == 0 && b < nb && m < members) ssq_s[m][b] = blk;
                v.x *= gv[k].x;
                v.y *= gv[k].y;
                v.z *= gv[k].z;
                v.w *= gv[k].w;
            }
            const float gsum = group_sum_f<T>(((v.x + v.y) + v.z) + v.w);
            // Blocks past K inside the last slice are staged as zeros: their
            // lanes multiply zero weights, and 0 * (stale LDS) could be NaN.
            if (b < 16 * (slice0 + slices) && m < members) {
                float* dst = xs + ((m * slices + slice) * 64 + rec) * STRIDE;
                *reinterpret_cast<float4*>(dst + pos) = v;
                if ((lane & (F32Rec<T>::group / 4 - 1)) == 0) dst[64 + pos / F32Rec<T>::group] = gsum;
            }
        }
    }
    __syncthreads();

    float inv[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        inv[m] = 1.f;
        if constexpr (NORM) {
            float total = 0.f;
            for (int b = 0; b < nb; ++b) total += ssq_s[m][b];
            // RMSNorm (qwen_reference.rs:550-556): x * (1/sqrt(sum(x^2)/K + eps)) * gamma
            inv[m] = 1.0f / sqrtf(total / (float)K + args.eps);
        }
    }

    const bool accumulate = args.accumulate != 0;
    auto put = [&](float value, __amdgpu_buffer_rsrc_t yr, uint32_t off) {
        if (accumulate) {
            __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(value, yr, (int)off, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, value), yr, (int)off, 0, 0);
        }
    };
    // silu(gate) * up of one output row (model_ops.rs:316-328)
    auto swiglu = [](float g, float u) { return (g / (1.0f + expf(-g))) * u; };
    const __amdgpu_buffer_rsrc_t partial_r =
        make_rsrc(args.partial, SPLIT ? (uint32_t)gridDim.y * (uint32_t)members * (uint32_t)args.total_rows * 4u : 0u);

    // ---- one or two members: records in VGPRs; the ring is reduced one
    // unit at a time and each slot refilled with the unit NBUF ahead.
    float4 xq[MT][16];
    float xg[MT][G];
    auto read_rec = [&](int slice) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float* src = xs + ((m * slices + slice) * 64 + lane) * STRIDE;
#pragma unroll
            for (int i = 0; i < 16; ++i) xq[m][i] = *reinterpret_cast<const float4*>(src + 4 * i);
            const float4 sums = *reinterpret_cast<const float4*>(src + 64);
            const float sv[4] = {sums.x, sums.y, sums.z, sums.w};
#pragma unroll
            for (int g = 0; g < G; ++g) xg[m][g] = sv[g];
        }
    };
    auto xf = [&](int m, int i) { return xq[m][i]; };
    auto sf = [&](int m, int g) { return xg[m][g]; };
    if constexpr (ONE_SLICE) read_rec(0);

    int crow = r_begin, cslice = 0;
    constexpr int kAcc = ONE_SLICE ? 1 : GROUP;
    float acc[kAcc][MT];
    float gk[MT];
#pragma unroll
    for (int r = 0; r < kAcc; ++r)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[r][m] = 0.f;
    auto consume = [&](const RowData<T>& d, int r) {
        if constexpr (!ONE_SLICE) {
            if (r % GROUP == 0) read_rec(cslice);
        }
        float part[MT];
        if constexpr (T == kQ6K && MT == 2 && ONE_SLICE) {
            row_dot<T, MT>(d, p, xf, sf, part);
        } else {
            ring_row_dot<T, MT>(d, p, xf, sf, part);
        }
        const int ai = ONE_SLICE ? 0 : r % GROUP;
        const int row = ONE_SLICE ? crow : crow + r % GROUP;
        const bool last = ONE_SLICE || cslice == slices - 1;
        int mat, local, rows_mat;
        __amdgpu_buffer_rsrc_t yr;
        if constexpr (kCursor) {
            if (row < r_end) seek(ccur, row, true);
            yr = ccur.rs;
            local = row - ccur.start;
            rows_mat = ccur.rows_mat;
        } else if constexpr (PAIR) {
            yr = pair_y;
            local = row >> 1;
            rows_mat = pair_rows;
        } else {
            locate(row < r_end ? row : r_begin, mat, local);
            yr = pick_y(mat, rows_mat);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float ps = wave_sum_uniform(part[m]);
            acc[ai][m] = (ONE_SLICE || cslice == 0) ? ps : acc[ai][m] + ps;
            const float total = acc[ai][m] * inv[m];
            const uint32_t off = (last && row < r_end && lane == 0 && m < members)
                                     ? (uint32_t)(m * rows_mat + local) * 4u
                                     : kOutOfRange;
            if constexpr (SPLIT) {
                // this workgroup's slice total P_s, as the several-member pass stores it
                const uint32_t poff = (row < r_end && lane == 0 && m < members)
                                          ? (uint32_t)((slice0 * members + m) * args.total_rows + row) * 4u
                                          : kOutOfRange;
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, ps), partial_r, (int)poff, 0, 0);
            } else if constexpr (PAIR) {
                if (r % 2 == 0) {
                    gk[m] = total;
                } else {
                    put(swiglu(gk[m], total), yr, off);
                }
            } else {
                put(total, yr, off);
            }
        }
        if constexpr (ONE_SLICE) {
            ++crow;
        } else if (r % GROUP == GROUP - 1 && ++cslice == slices) {
            cslice = 0;
            crow += GROUP;
        }
    };

    const int rows_w = r_end - r_begin;
    const int units = ONE_SLICE ? rows_w : (rows_w + GROUP - 1) / GROUP * GROUP * slices;
    const int passes = (units + NBUF - 1) / NBUF;
    for (int ps = 0; ps + 1 < passes; ++ps) {
#pragma unroll
        for (int r = 0; r < NBUF; ++r) {
            consume(ring[r], r);
            load_next(ring[r], r);
        }
    }
    if (passes > 0) {
        const int left = units - (passes - 1) * NBUF;
#pragma unroll
        for (int r = 0; r < NBUF; ++r) {
            if (r < left) consume(ring[r], r);
        }
    }
}

namespace {

// ---------------------------------------- one or two members, any super-blocks
//
// gemv_f32_slices_kernel: rows whose super-blocks are not one whole slice (K
// above 4096, or at most 2048). A slice of 8 or fewer blocks leaves lanes idle
// when a unit is one row, so a unit is RP = 1, 2 or 4 rows of a slice of up to
// 16, 8 or 4 blocks (each row in 64 / RP lanes), and a wave keeps one slice's
// records in VGPRs while it walks that slice's units: the workgroup's rows give
// one sequence of units, slice by slice, cut evenly over its waves, so a wave
// rereads records from LDS only where its share crosses a slice (before, at
// every second row). Slice totals P_s meet in LDS; after one barrier a thread
// per value adds them in slice order and applies the epilogue. The DPP row sums
// of a unit's rows and the zeros an absent block would add make every row's
// bits those of the one-slice form.
//
// Measured, one member, us (before: one row a unit, or pairs of rows over all
// slices): Q4_K 5120 -> 17408 23.6 -> 16.3, Q6_K 29.7 -> 22.0; Q4_K 12288 ->
// 17408 38.0 -> 32.0; 1024 -> 17408 8.9 -> 6.3; two members 5120 -> 17408 30.4 ->
// 20.9. What bounds it: 3.1-4.0 TB/s of weights after a 4-6 us ramp. Where it
// serves is chosen by launch_few (pairs_form) and launch_split (one_launch_long_k).
constexpr int kSliceWaves = 8;

// Rows of one slice a unit takes.
__device__ __host__ constexpr int unit_rows(int blocks) { return blocks > 8 ? 1 : blocks > 4 ? 2 : 4; }

template <int T, int MT, int PRO, bool MULTI, int NBUF, bool PAIR>
__global__ __launch_bounds__(kSliceWaves * 64) void gemv_f32_slices_kernel(WaveGemvArgs args) {
    static_assert(!PAIR || !MULTI, "pairs are one slice");
    constexpr bool NORM = PRO == kProNorm;
    constexpr bool SWIGLU = PRO == kProSwiglu;
    constexpr int G = F32Rec<T>::groups;
    constexpr int STRIDE = F32Rec<T>::stride;
    constexpr int BB = BlockTraits<T>::bytes;
    constexpr int WAVES = kSliceWaves;
    constexpr int NBMAX = MULTI ? (MT == 1 ? 2 : 1) * kF32Blocks : 8;
    constexpr int NBW = MULTI ? 6 : 1;                // blocks a wave stages at a time
    extern __shared__ __attribute__((aligned(16))) float xs[];  // [MT][slices][64 records][STRIDE], then the slice totals
    __shared__ float ssq_s[NORM ? MT : 1][NORM ? NBMAX : 1];
    __shared__ float inv_s[MT];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = args.K;
    const int nb = K >> 8;
    const int slices = MULTI ? (nb + 15) >> 4 : 1;
    const int members = args.members;
    const uint32_t row_bytes = (uint32_t)nb * BB;

    // Rows in quads, numbered through the matrices (a matrix's last quad may be
    // short); pairs: each quad of gate rows, then the up rows beside it.
    int quad_end[kMaxGroup];
#pragma unroll
    for (int i = 0; i < kMaxGroup; ++i) {
        const int rows = args.rows_end[i] - (i > 0 ? args.rows_end[i - 1] : 0);
        quad_end[i] = (i > 0 ? quad_end[i - 1] : 0) + (i < args.count ? (rows + 3) >> 2 : 0);
    }
    const int quads_all = PAIR ? quad_end[0] : quad_end[kMaxGroup - 1];
    const int q_begin = (int)((long long)quads_all * blockIdx.x / gridDim.x);
    const int q_end = (int)((long long)quads_all * (blockIdx.x + 1) / gridDim.x);
    const int quads = (PAIR ? 2 : 1) * (q_end - q_begin);  // of this workgroup
    auto locate = [&](int quad, int& mat, int& row0) {
        const int q = q_begin + (PAIR ? quad >> 1 : quad);
        mat = 0;
        int start = 0;
        if constexpr (PAIR) {
            mat = quad & 1;
        } else {
#pragma unroll
            for (int i = 0; i < kMaxGroup - 1; ++i) {
                if (i + 1 < args.count && q >= quad_end[i]) {
                    mat = i + 1;
                    start = quad_end[i];
                }
            }
        }
        row0 = 4 * (q - start);
    };
    // units of the last slice per quad, and the wave's share of the sequence
    const int last_blocks = nb - 16 * (slices - 1);
    const int last_rp = unit_rows(last_blocks);
    const int full_units = 4 * quads * (slices - 1);
    const int units = full_units + (4 / last_rp) * quads;
    const int u_begin = (int)((long long)units * wave / WAVES);
    const int u_end = (int)((long long)units * (wave + 1) / WAVES);

    const __amdgpu_buffer_rsrc_t xr = make_rsrc(args.x, (uint32_t)members * (uint32_t)K * 4u);
    const __amdgpu_buffer_rsrc_t gr = make_rsrc(args.gamma, NORM ? (uint32_t)K * 4u : 0u);
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(args.x2, SWIGLU ? (uint32_t)members * (uint32_t)K * 4u : 0u);

    // A position in the unit sequence: the slice, the unit in it, and what that
    // makes of this lane (its row of the unit, its record of the slice).
    struct Place {
        int slice, idx, end;  // unit of the slice, units the slice has
        int rp;
        uint32_t lane_off;    // of the lane's row and block from the unit's first row
        bool live;            // the lane's block exists
        int rec;
    };
    auto enter = [&](Place& c, int slice, int idx) {
        c.slice = slice;
        c.idx = idx;
        c.rp = slice + 1 < slices ? 1 : last_rp;
        c.end = (4 / c.rp) * quads;
        const int lanes = 64 / c.rp;  // a power of two
        c.rec = lane & (lanes - 1);
        const int block = 16 * slice + (c.rec >> 2);
        c.live = block < nb;
        c.lane_off = (uint32_t)(lane / lanes) * row_bytes + (uint32_t)block * BB;
    };
    auto place = [&](int unit) {
        Place c;
        const int s = min(unit / (4 * quads > 0 ? 4 * quads : 1), slices - 1);
        enter(c, s, unit - 4 * quads * s);
        return c;
    };
    auto step = [&](Place& c) {
        if (++c.idx == c.end) enter(c, min(c.slice + 1, slices - 1), 0);
    };
    const int p = lane & 3;
    Place lp = place(u_begin);
    RowData<T> ring[NBUF];
    int lunit = u_begin;
    auto load_next = [&](RowData<T>& dst) {
        const int shift = lp.rp == 1 ? 2 : lp.rp == 2 ? 1 : 0;  // log2 units per quad
        int mat, row0;
        locate(lp.idx >> shift, mat, row0);
        row0 += (lp.idx & ((1 << shift) - 1)) * lp.rp;
        const uint8_t* w = args.w[0];
        uint32_t bytes = args.wbytes[0];
#pragma unroll
        for (int i = 1; i < kMaxGroup; ++i) {
            if (mat == i) {
                w = args.w[i];
                bytes = args.wbytes[i];
            }
        }
        // dead units read through an empty resource; rows past the matrix lie
        // past its bytes: zeros
        load_row<T>(dst, make_rsrc(w, lunit < u_end ? bytes : 0u),
                    lp.live ? lp.lane_off + (uint32_t)row0 * row_bytes : kOutOfRange, p);
        ++lunit;
        step(lp);
    };

    // ---- staging, as the one-slice form's, NBW blocks a wave at a time (all of
    // K up to 12288; a longer unrolled run costs more in cold code): activation
    // loads first, then, the first time, the first units of weights
#pragma unroll 1
    for (int b0 = wave; b0 < 16 * slices; b0 += WAVES * NBW) {
        float4 xv[NBW][MT];
        float4 gv[NORM ? NBW : 1];
        float4 uv[SWIGLU ? NBW : 1][SWIGLU ? MT : 1];
#pragma unroll
        for (int k = 0; k < NBW; ++k) {
            const int b = b0 + WAVES * k;
            const int e = 256 * b + 4 * lane;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                xv[k][m] = float4{0.f, 0.f, 0.f, 0.f};
                if constexpr (SWIGLU) uv[k][m] = float4{0.f, 0.f, 0.f, 0.f};
            }
            if constexpr (NORM) gv[k] = float4{0.f, 0.f, 0.f, 0.f};
            if (b < nb) {  // uniform: a wave issues only the loads its K has
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const uint32_t off = m < members ? (uint32_t)(m * K + e) * 4u : kOutOfRange;
                    xv[k][m] = load_f4(xr, off);
                    if constexpr (SWIGLU) uv[k][m] = load_f4(ur, off);
                }
                if constexpr (NORM) gv[k] = load_f4(gr, (uint32_t)e * 4u);
            }
        }
        asm volatile("" ::: "memory");
        if (b0 == wave) {
#pragma unroll
            for (int r = 0; r < NBUF; ++r) load_next(ring[r]);
        }
#pragma unroll
        for (int k = 0; k < NBW; ++k) {
            const int b = b0 + WAVES * k;
            // blocks past K inside the last slice are staged as zeros
            if (b >= 16 * slices) break;
            const int slice = b >> 4;
            int rec, pos;
            f32_slot<T>(256 * (b & 15) + 4 * lane, rec, pos);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                float4 v = xv[k][m];
                if constexpr (SWIGLU) {
                    // silu(gate) * up, in the reference's operation order (model_ops.rs:316-328)
                    v.x = (v.x / (1.0f + expf(-v.x))) * uv[k][m].x;
                    v.y = (v.y / (1.0f + expf(-v.y))) * uv[k][m].y;
                    v.z = (v.z / (1.0f + expf(-v.z))) * uv[k][m].z;
                    v.w = (v.w / (1.0f + expf(-v.w))) * uv[k][m].w;
                }
                if constexpr (NORM) {
                    const float sq = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                    const float blk = wave_sum_uniform(sq);
                    if (lane == 0 && b < nb && m < members) ssq_s[m][b] = blk;
                    v.x *= gv[k].x;
                    v.y *= gv[k].y;
                    v.z *= gv[k].z;
                    v.w *= gv[k].w;
                }
                const float gsum = group_sum_f<T>(((v.x + v.y) + v.z) + v.w);
                float* dst = xs + ((m * slices + slice) * 64 + rec) * STRIDE;
                *reinterpret_cast<float4*>(dst + pos) = v;
                if ((lane & (F32Rec<T>::group / 4 - 1)) == 0) dst[64 + pos / F32Rec<T>::group] = gsum;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < MT) {
        float inv = 1.f;
        if constexpr (NORM) {
            if ((int)threadIdx.x < members) {
                float total = 0.f;
                for (int b = 0; b < nb; ++b) total += ssq_s[threadIdx.x][b];
                // RMSNorm (qwen_reference.rs:550-556): x * (1/sqrt(sum(x^2)/K + eps)) * gamma
                inv = 1.0f / sqrtf(total / (float)K + args.eps);
            }
        }
        inv_s[threadIdx.x] = inv;
    }

    // slice totals: [row of the workgroup][slice][member]
    float* const sums = xs + (size_t)MT * slices * 64 * STRIDE;
    float4 xq[MT][16];
    float xg[MT][G];
    auto read_rec = [&](int slice, int rec) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float* src = xs + ((m * slices + slice) * 64 + rec) * STRIDE;
#pragma unroll
            for (int i = 0; i < 16; ++i) xq[m][i] = *reinterpret_cast<const float4*>(src + 4 * i);
            const float4 s4 = *reinterpret_cast<const float4*>(src + 64);
            const float sv[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
            for (int g = 0; g < G; ++g) xg[m][g] = sv[g];
        }
    };
    auto xf = [&](int m, int i) { return xq[m][i]; };
    auto sf = [&](int m, int g) { return xg[m][g]; };
    Place cp = place(u_begin);
    if (u_begin < u_end) read_rec(cp.slice, cp.rec);
    auto consume = [&](const RowData<T>& d) {
        float part[MT];
        row_dot<T, MT>(d, p, xf, sf, part);
        float* dst = sums + ((size_t)cp.idx * cp.rp * slices + cp.slice) * MT;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float v = part[m];
            v = dpp_step<0xb1>(v);   // quad_perm [1,0,3,2]
            v = dpp_step<0x4e>(v);   // quad_perm [2,3,0,1]
            v = dpp_step<0x141>(v);  // row_half_mirror
            v = dpp_step<0x140>(v);  // row_mirror
            const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
            const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
            const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
            const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
            // (+ 0: the sum an absent half or quarter of the slice would add)
            if (cp.rp == 1) {
                const float t = (r0 + r1) + (r2 + r3);
                if (lane == 0) dst[m] = t;
            } else if (cp.rp == 2) {
                const float t = (lane == 0 ? r0 + r1 : r2 + r3) + 0.0f;
                if (lane < 2) dst[lane * slices * MT + m] = t;
            } else {
                const float t = (lane == 0 ? r0 : lane == 1 ? r1 : lane == 2 ? r2 : r3) + 0.0f;
                if (lane < 4) dst[lane * slices * MT + m] = t;
            }
        }
        const int slice = cp.slice;
        step(cp);
        if (MULTI && cp.slice != slice) read_rec(cp.slice, cp.rec);
    };
    int left = u_end - u_begin;
    for (; left > NBUF; left -= NBUF) {
#pragma unroll
        for (int r = 0; r < NBUF; ++r) {
            consume(ring[r]);
            load_next(ring[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < NBUF; ++r) {
        if (r < left) consume(ring[r]);
    }

    // ---- rows: a value per thread, its address found before the barrier
    const int rows_wg = 4 * (PAIR ? quads >> 1 : quads);
    struct Out {
        float* y;  // null: no value
        int at, m;
    };
    auto out_of = [&](int v) {
        Out o{nullptr, 0, MT == 1 ? 0 : v & 1};
        const int r = MT == 1 ? v : v >> 1;
        const int quad = PAIR ? 2 * (r >> 2) : r >> 2;
        o.at = (4 * quad + (r & 3)) * slices * MT + o.m;
        int mat, row0;
        locate(quad, mat, row0);
        const int rows = args.rows_end[mat] - (mat > 0 ? args.rows_end[mat - 1] : 0);
        const int row = row0 + (r & 3);
        if (r < rows_wg && row < rows && o.m < members) {
            float* y = args.y[0];
#pragma unroll
            for (int i = 1; i < kMaxGroup; ++i)
                if (!PAIR && mat == i) y = args.y[i];
            o.y = y + (size_t)o.m * rows + row;
        }
        return o;
    };
    Out out = out_of(threadIdx.x);
    __syncthreads();
#pragma unroll 1
    for (int v = threadIdx.x; v < rows_wg * MT; v += WAVES * 64) {
        if (v >= WAVES * 64) out = out_of(v);
        if (out.y == nullptr) continue;
        auto total_at = [&](int at) {
            float t = sums[at];
            for (int s = 1; s < slices; ++s) t = t + sums[at + s * MT];
            return t * inv_s[out.m];
        };
        float value = total_at(out.at);
        if constexpr (PAIR) {
            // silu(gate) * up (model_ops.rs:316-328); the up quad follows
            const float up = total_at(out.at + 4 * slices * MT);
            value = (value / (1.0f + expf(-value))) * up;
        }
        if (args.accumulate) {
            unsafeAtomicAdd(out.y, value);
        } else {
            *out.y = value;
        }
    }
}

// ------------------------------------------- three to eight members, MFMA
//
// gemv_f32_many_kernel: the same rows for 3..8 members, one slice per
// workgroup. The products run on v_mfma_f32_4x4x1_16b_f32: 16 independent
// 4 x 4 outer products, D[i][j] += x_i * q_j, each element one fused f32
// multiply-add (checked bit for bit against fmaf over normal, denormal,
// overflowing, infinite and NaN operands), so a chain of them over a scale
// group's elements is the S_g of the single-member kernel, in its order. (The
// minimum terms m * X are formed onto +0, so one of -0 becomes +0: a row of zero
// weights may give the other zero.)
//
// Mapping. A wave owns one quarter of the slice (4 super-blocks, 16 lane
// records) and walks units of 4 rows x that quarter: lane l holds record
// l >> 2 of row l & 3 as the B operand, and in VGPRs, for the whole launch,
// the activations of member (l & 3) (and 4 + (l & 3)) at that record as the A
// operand. The accumulator of lane l then holds its own row and record for
// members 0..3, so scales and minima apply where they were loaded, and the
// activations reach four rows and four members per instruction without an LDS
// read. (The f32 matrix rate equals the VALU's here, 117 against 110 TFLOP/s
// measured, and they share time; what goes is the LDS traffic, 1 KB per 4 rows
// and record piece at the 90 B/clk it is read at, and the issue slots.)
//
// A unit's 16 records per row reduce in canonical order: 4 lanes of a block by
// two DPP steps, then blocks (b0 + b1) + (b2 + b3) and quarters
// (r0 + r1) + (r2 + r3) through LDS, where the records were; one barrier per
// kManyItems units.
//
// Measured (us a call over distinct weights, against rows through VALU FMAs with
// the records in LDS), 8 members, K 4096 at 256 / 4096 / 12288 rows: Q4_K 9.5 / 9.9 /
// 20.4 -> 7.2 / 9.4 / 16.1; Q5_K 10.0 / 10.7 / 21.3 -> 7.6 / 10.4 / 17.9; Q6_K 12.5 /
// 13.2 / 26.0 -> 8.3 / 11.5 / 19.9; 4 members, Q4_K 6.3 / 6.6 / 13.5 -> 5.1 / 6.5 / 10.7.
// (Slower in one place: Q5_K, 3 or 4 members, two units a wave, 4096 rows 7.1 -> 7.6:
// the second unit runs the loop's code cold.) What bounds it: with the weights in
// cache 26.9 us of Q4_K 4096 -> 24576's 30.7, so the f32 multiply-adds and the
// conversions; an MFMA takes 4.5 ns of a SIMD. A ring of four units, two
// workgroups per CU (4 members), and weights loaded as whole rows through an LDS
// slab were level or slower.
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kManyWaves = 8;
constexpr int kManyItems = 32;                     // units a wave reduces between barriers
constexpr int kManyStride = 64 * 68 + 8;           // dwords per member's records: quads of lanes (members) in distinct banks
constexpr int kManyLds = 4 * kManyStride * 4;      // bytes per four members

template <int CTRL>
__device__ __forceinline__ float dpp_shift_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// part[m] = this lane's share of its row . x_m (m = 0 .. 4 MG - 1): row_dot's
// operation sequence per (row, member), the FMAs on the matrix cores.
template <int T, int MG>
__device__ __forceinline__ void unit_dot(const RowData<T>& d, int p, const float4 (&x)[MG][16], const float (&xg)[MG][4],
                                         float (&part)[4 * MG]) {
    constexpr int CH = T == kQ5K && MG == 2 ? 4 : 8;  // dwords of quants per run (of two groups)
    auto mac = [](float xv, float q, f32x4 s) { return __builtin_amdgcn_mfma_f32_4x4x1f32(xv, q, s, 0, 0, 0); };
    // Quants are converted in runs, then multiplied in runs: 64 (CH dwords of two
    // groups) for Q4_K and Q5_K, 32 for Q5_K at 5 to 8 members and Q6_K at 3 and 4, 16
    // for Q6_K at 5 to 8. Q5_K, 8 members, 4096 -> 12288, 64 / 32: 18.5 / 17.6 us, 12288
    // -> 4096 24.3 / 22.3; Q4_K level, runs of 8 too. The minimum terms m * X run
    // as one more MFMA each.
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    if constexpr (T == kQ4K || T == kQ5K) {
        float a0, a1, b0, b1;
        group_scales<T>(d.h, p, a0, a1, b0, b1);
        f32x4 sA[MG], sB[MG], mA[MG], mB[MG];
#pragma unroll
        for (int h = 0; h < 8; h += CH) {
            float fa[CH][4], fb[CH][4];
#pragma unroll
            for (int j = 0; j < CH; ++j) quant_quads<T>(d, h + j, p, fa[j], fb[j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int g = 0; g < MG; ++g) {
                        const float4 xa = x[g][h + j], xb = x[g][8 + h + j];
                        const float va[4] = {xa.x, xa.y, xa.z, xa.w}, vb[4] = {xb.x, xb.y, xb.z, xb.w};
                        sA[g] = mac(va[t], fa[j][t], h + j + t == 0 ? zero : sA[g]);
                        sB[g] = mac(vb[t], fb[j][t], h + j + t == 0 ? zero : sB[g]);
                    }
            if (h + CH == 8) {
#pragma unroll
                for (int g = 0; g < MG; ++g) {
                    mA[g] = mac(xg[g][0], b0, zero);
                    mB[g] = mac(xg[g][1], b1, zero);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < MG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float tA = __builtin_fmaf(a0, sA[g][i], -mA[g][i]);
                const float tB = __builtin_fmaf(a1, sB[g][i], -mB[g][i]);
                part[4 * g + i] = tA + tB;
            }
    } else {
        float a[4];
        uint32_t law[4], lbw[4], qhw[4];
        q6_fields(d, p, a, law, lbw, qhw);
        float acc[4 * MG];
        // two 16-element groups at a time: their chains are independent
#pragma unroll
        for (int v = 0; v < 4; v += 2) {
            f32x4 s0[MG], s1[MG], m0[MG], m1[MG];
            constexpr int CH6 = MG == 1 ? 4 : 2;  // two groups of members leave registers for half a run
#pragma unroll
            for (int h = 0; h < 4; h += CH6) {
                float f0[CH6][4], f1[CH6][4];
#pragma unroll
                for (int j = 0; j < CH6; ++j) {
                    q6_quad(law[h + j], qhw[h + j], v, f0[j]);
                    q6_quad(lbw[h + j], qhw[h + j], v + 1, f1[j]);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < CH6; ++j)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int g = 0; g < MG; ++g) {
                            const float4 x0 = x[g][4 * v + h + j], x1 = x[g][4 * v + 4 + h + j];
                            const float w0[4] = {x0.x, x0.y, x0.z, x0.w}, w1[4] = {x1.x, x1.y, x1.z, x1.w};
                            s0[g] = mac(w0[t], f0[j][t], h + j + t == 0 ? zero : s0[g]);
                            s1[g] = mac(w1[t], f1[j][t], h + j + t == 0 ? zero : s1[g]);
                        }
                if (h + CH6 == 4) {
#pragma unroll
                    for (int g = 0; g < MG; ++g) {  // 32 X, exact
                        m0[g] = mac(xg[g][v], 32.0f, zero);
                        m1[g] = mac(xg[g][v + 1], 32.0f, zero);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int g = 0; g < MG; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float t0 = a[v] * (s0[g][i] - m0[g][i]);
                    const float t1 = a[v + 1] * (s1[g][i] - m1[g][i]);
                    acc[4 * g + i] = ((v == 0) ? t0 : acc[4 * g + i] + t0) + t1;
                }
        }
#pragma unroll
        for (int m = 0; m < 4 * MG; ++m) part[m] = acc[m];
    }
}

}  // namespace

// MG: groups of four members (1: 3..4 members, 2: 5..8). SPLIT: K spans
// several slices; the first `wgs` workgroups take slice 0, the next slice 1,
// ..., the rest the last one (which may be short), and each row's slice total
// P_s goes to args.partial[s][members][rows] for f32_split_reduce_kernel, and
// with an RMSNorm the blocks' sums of squares to [members][super-blocks] after
// the partials.
template <int T, int MG, int PRO, int NBUF, bool PAIR, bool SPLIT>
__global__ __launch_bounds__(kManyWaves * 64) void gemv_f32_many_kernel(WaveGemvArgs args, int wgs) {
    static_assert(kManyItems % NBUF == 0, "whole ring passes between barriers");
    static_assert(!PAIR || NBUF == 2, "pairs are whole rings");
    static_assert(!SPLIT || !PAIR, "slice splits store slice totals");
    constexpr bool NORM = PRO == kProNorm;
    constexpr int MT = 4 * MG;
    constexpr int BB = BlockTraits<T>::bytes;
    constexpr int NBW = 16 / kManyWaves;  // staging blocks per wave
    extern __shared__ __attribute__((aligned(16))) float xs[];  // [MT][64 records][68] (member stride kManyStride), then the units' block sums
    __shared__ float ssq_s[NORM && !SPLIT ? MT : 1][NORM && !SPLIT ? 16 : 1];
    __shared__ float inv_s[MT];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = args.K;
    const int nb = K >> 8;
    const int members = args.members;
    const int last_slice = (nb - 1) >> 4;
    const int slice0 = SPLIT ? min((int)blockIdx.x / wgs, last_slice) : 0;
    const int wg = SPLIT ? (int)blockIdx.x - slice0 * wgs : (int)blockIdx.x;
    const int wg_count = !SPLIT ? (int)gridDim.x : slice0 < last_slice ? wgs : (int)gridDim.x - last_slice * wgs;
    // quarters with blocks in this slice, and the sets of waves that share them out
    const int quarters = (min(nb - 16 * slice0, 16) + 3) >> 2;
    const int sets = quarters == 1 ? 8 : quarters == 2 ? 4 : 2;
    const int quarter = wave % quarters;
    const int set = wave / quarters;  // sets..: idle (three quarters use six waves)
    const uint32_t row_bytes = (uint32_t)nb * BB;

    // units of four rows, numbered through the matrices; a matrix's last one may be short
    int unit_end[kMaxGroup];
#pragma unroll
    for (int i = 0; i < kMaxGroup; ++i) {
        const int rows = args.rows_end[i] - (i > 0 ? args.rows_end[i - 1] : 0);
        unit_end[i] = (i > 0 ? unit_end[i - 1] : 0) + (i < args.count ? (rows + 3) >> 2 : 0);
    }
    const int units = PAIR ? unit_end[0] : unit_end[kMaxGroup - 1];
    const int u_begin = (int)((long long)units * wg / wg_count);
    const int u_end = (int)((long long)units * (wg + 1) / wg_count);
    // this wave's item k: unit u_begin + set + sets * k (pairs: gate rows for even k, up rows of the same unit for odd k)
    const int items = (PAIR ? 2 : 1) * ((u_end - u_begin + sets - 1) / sets);
    auto unit_of = [&](int s, int k) { return u_begin + s + sets * (PAIR ? k >> 1 : k); };
    auto locate = [&](int unit, int k, int& mat, int& row0) {
        mat = 0;
        int start = 0;
        if constexpr (PAIR) {
            mat = k & 1;
        } else {
#pragma unroll
            for (int i = 0; i < kMaxGroup - 1; ++i) {
                if (i + 1 < args.count && unit >= unit_end[i]) {
                    mat = i + 1;
                    start = unit_end[i];
                }
            }
        }
        row0 = 4 * (unit - start);
    };

    // ---- activation loads first, then the first units of weights, then the
    // staging (vector memory returns in order)
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(args.x, (uint32_t)members * (uint32_t)K * 4u);
    const __amdgpu_buffer_rsrc_t gr = make_rsrc(args.gamma, NORM ? (uint32_t)K * 4u : 0u);
    float4 xv[NBW][MT];
    float4 gv[NORM ? NBW : 1];
#pragma unroll
    for (int k = 0; k < NBW; ++k) {
        const int b = 16 * slice0 + wave + kManyWaves * k;
        const int e = 256 * b + 4 * lane;
#pragma unroll
        for (int m = 0; m < MT; ++m)
            xv[k][m] = load_f4(xr, (b < nb && m < members) ? (uint32_t)(m * K + e) * 4u : kOutOfRange);
        if constexpr (NORM) gv[k] = load_f4(gr, b < nb ? (uint32_t)e * 4u : kOutOfRange);
    }
    asm volatile("" ::: "memory");

    const int slot = lane >> 2;      // record of the quarter
    const int p = slot & 3;          // quarter of its super-block
    const int block = 16 * slice0 + 4 * quarter + (slot >> 2);
    const uint32_t lane_off = (uint32_t)(lane & 3) * row_bytes + (uint32_t)block * BB;
    RowData<T> ring[NBUF];
    auto load_item = [&](RowData<T>& dst, int k) {
        const int unit = unit_of(set, k);
        int mat, row0;
        locate(unit, k, mat, row0);
        const uint8_t* w = args.w[0];
        uint32_t bytes = args.wbytes[0];
#pragma unroll
        for (int i = 1; i < kMaxGroup; ++i) {
            if (mat == i) {
                w = args.w[i];
                bytes = args.wbytes[i];
            }
        }
        // dead items read through an empty resource; rows past the matrix lie
        // past its bytes: zeros
        const bool live = set < sets && unit < u_end;
        load_row<T>(dst, make_rsrc(w, live ? bytes : 0u), block < nb ? lane_off + (uint32_t)row0 * row_bytes : kOutOfRange, p);
    };
#pragma unroll
    for (int r = 0; r < NBUF; ++r) load_item(ring[r], r);

#pragma unroll
    for (int k = 0; k < NBW; ++k) {
        const int b = 16 * slice0 + wave + kManyWaves * k;
        int rec, pos;
        f32_slot<T>(256 * (b - 16 * slice0) + 4 * lane, rec, pos);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float4 v = xv[k][m];
            if constexpr (NORM) {
                const float sq = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                const float blk = wave_sum_uniform(sq);
                if (lane == 0 && b < nb && m < members) {
                    if constexpr (SPLIT) {
                        if (wg == 0)
                            args.partial[(size_t)(last_slice + 1) * members * args.total_rows + (size_t)m * nb + b] = blk;
                    } else {
                        ssq_s[m][b] = blk;
                    }
                }
                v.x *= gv[k].x;
                v.y *= gv[k].y;
                v.z *= gv[k].z;
                v.w *= gv[k].w;
            }
            const float gsum = group_sum_f<T>(((v.x + v.y) + v.z) + v.w);
            // blocks past K are staged as zeros, absent members' too
            float* dst = xs + m * kManyStride + rec * F32Rec<T>::stride;
            *reinterpret_cast<float4*>(dst + pos) = v;
            if ((lane & (F32Rec<T>::group / 4 - 1)) == 0) dst[64 + pos / F32Rec<T>::group] = gsum;
        }
    }
    __syncthreads();
    if (threadIdx.x < MT) {
        float inv = 1.f;
        if constexpr (NORM && !SPLIT) {
            if ((int)threadIdx.x < members) {
                float total = 0.f;
                for (int b = 0; b < nb; ++b) total += ssq_s[threadIdx.x][b];
                // RMSNorm (qwen_reference.rs:550-556): x * (1/sqrt(sum(x^2)/K + eps)) * gamma
                inv = 1.0f / sqrtf(total / (float)K + args.eps);
            }
        }
        inv_s[threadIdx.x] = inv;
    }
    float4 x[MG][16];
    float xg[MG][4];
#pragma unroll
    for (int g = 0; g < MG; ++g) {
        const float* src = xs + (4 * g + (lane & 3)) * kManyStride + (16 * quarter + slot) * F32Rec<T>::stride;
#pragma unroll
        for (int i = 0; i < 16; ++i) x[g][i] = *reinterpret_cast<const float4*>(src + 4 * i);
        const float4 sums = *reinterpret_cast<const float4*>(src + 64);
        xg[g][0] = sums.x;
        xg[g][1] = sums.y;
        xg[g][2] = sums.z;
        xg[g][3] = sums.w;
    }
    __syncthreads();

    // block sums: [item][wave][block of the quarter][row of the unit][member]
    constexpr int kWaveSums = 16 * MT;
    constexpr int kItemSums = kManyWaves * kWaveSums;
    static_assert((size_t)kManyItems * kItemSums * 4 <= (size_t)MG * kManyLds, "block sums fit the records' room");
    const __amdgpu_buffer_rsrc_t partial_r =
        make_rsrc(args.partial, SPLIT ? (uint32_t)(last_slice + 1) * (uint32_t)members * (uint32_t)args.total_rows * 4u : 0u);

    // The rows of items [first, first + count): value v = (item, set, row of
    // the unit, member), the members fastest.
    auto finish = [&](int first, int count) {
        const int values = (PAIR ? count >> 1 : count) * sets * (4 * MT);
        for (int v = threadIdx.x; v < values; v += kManyWaves * 64) {
            const int m = v % MT, j = (v / MT) & 3;
            const int s = (v / (4 * MT)) & (sets - 1);
            const int item = (v / (4 * MT) / sets) * (PAIR ? 2 : 1);
            auto total_of = [&](int it) {
                float r[4] = {0.f, 0.f, 0.f, 0.f};
                const float* src = xs + it * kItemSums + s * quarters * kWaveSums + j * MT + m;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (q < quarters)
                        r[q] = (src[q * kWaveSums] + src[q * kWaveSums + 4 * MT]) +
                               (src[q * kWaveSums + 8 * MT] + src[q * kWaveSums + 12 * MT]);
                return (r[0] + r[1]) + (r[2] + r[3]);
            };
            const int unit = unit_of(s, first + item);
            int mat, row0;
            locate(unit, PAIR ? 0 : first + item, mat, row0);
            const int begin = mat > 0 ? args.rows_end[mat - 1] : 0;
            const int rows = args.rows_end[mat] - begin;
            const int row = row0 + j;
            if (unit >= u_end || row >= rows || m >= members) continue;
            const float total = total_of(item);
            if constexpr (SPLIT) {
                const uint32_t off = (uint32_t)((slice0 * members + m) * args.total_rows + begin + row) * 4u;
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, total), partial_r, (int)off, 0, 0);
            } else {
                float* y = args.y[0];
#pragma unroll
                for (int i = 1; i < kMaxGroup; ++i)
                    if (mat == i) y = args.y[i];
                float value = total * inv_s[m];
                if constexpr (PAIR) {
                    // silu(gate) * up (model_ops.rs:316-328)
                    const float up = total_of(item + 1) * inv_s[m];
                    value = (value / (1.0f + expf(-value))) * up;
                }
                float* dst = y + (size_t)m * rows + row;
                if (args.accumulate) {
                    unsafeAtomicAdd(dst, value);
                } else {
                    *dst = value;
                }
            }
        }
    };

    // Item c0 + k from its ring slot, which then takes the item NBUF ahead (a
    // wave's last item takes none: a load there would make every ring pass wait
    // for both slots).
    auto reduce_item = [&](RowData<T>& d, int c0, int k, auto refill) {
        float part[MT];
        unit_dot<T, MG>(d, p, x, xg, part);
        if constexpr (decltype(refill)::value) load_item(d, c0 + k + NBUF);
        // a block's four records: ((0 + 1) + (2 + 3)), in the block's first quad
#pragma unroll
        for (int m = 0; m < MT; ++m) part[m] = dpp_shift_add<0x108>(dpp_shift_add<0x104>(part[m]));  // row_shl 4, 8
        if ((lane & 12) == 0 && set < sets) {
            float* dst = xs + k * kItemSums + wave * kWaveSums + (4 * (lane >> 4) + (lane & 3)) * MT;
#pragma unroll
            for (int g = 0; g < MG; ++g)
                *reinterpret_cast<float4*>(dst + 4 * g) =
                    float4{part[4 * g], part[4 * g + 1], part[4 * g + 2], part[4 * g + 3]};
        }
    };
    for (int c0 = 0; c0 < items; c0 += kManyItems) {
        const int count = min(kManyItems, items - c0);
        int k0 = 0;
        for (; k0 + NBUF <= count; k0 += NBUF) {
#pragma unroll
            for (int r = 0; r < NBUF; ++r) reduce_item(ring[r], c0, k0 + r, std::true_type{});
        }
        // a wave's last items, where they are no whole ring (pairs are)
        if constexpr (!PAIR) {
#pragma unroll
            for (int r = 0; r + 1 < NBUF; ++r)
                if (k0 + r < count) reduce_item(ring[r], c0, k0 + r, std::false_type{});
        }
        __syncthreads();
        finish(c0, count);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- launcher

namespace {

template <int T>
size_t f32_lds_bytes(int members, int K) {
    const int slices = ((K >> 8) + 15) >> 4;
    return (size_t)members * slices * 64 * F32Rec<T>::stride * sizeof(float);
}

template <int T, int MT, int PRO, bool ONE_SLICE, int NBUF, int WAVES, int GROUP = 1, bool PAIR = false,
          bool SPLIT = false>
struct F32Instance {
    static std::atomic<int> occupancy;  // resident workgroups per CU at the largest LDS size (0: not queried)
    static hipError_t launch(const WaveGemvArgs& a, int cu_count, int per_cu, hipStream_t stream) {
        auto kern = gemv_f32_kernel<T, MT, PRO, ONE_SLICE, NBUF, WAVES, GROUP, PAIR, SPLIT>;
        const size_t lds = f32_lds_bytes<T>(MT, ONE_SLICE ? std::min(a.K, (int)kSliceElems) : a.K);
        const int max_lds = (int)f32_lds_bytes<T>(MT, ONE_SLICE ? kSliceElems : kWaveMaxK);
        static PerDevice sized;
        (void)sized.once(a.device, [&] {
            return hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
        });
        int occ = occupancy.load(std::memory_order_relaxed);
        if (occ == 0) {
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void*)kern, WAVES * 64, max_lds) !=
                    hipSuccess ||
                occ < 1) {
                occ = 1;
            }
            occupancy.store(occ, std::memory_order_relaxed);
        }
        const int slices = ONE_SLICE ? 1 : ((a.K >> 8) + 15) >> 4;
        const long long units = (long long)a.total_rows * slices;
        const long long want = (units + 2 * WAVES - 1) / (2 * WAVES);
        long long grid = want;
        if (want >= cu_count) {
            grid = (long long)cu_count * std::min<long long>({(want + cu_count - 1) / cu_count, (long long)occ,
                                                               (long long)per_cu});
        }
        if (grid < 1) grid = 1;
        unsigned gy = 1;
        if constexpr (SPLIT) {
            // one slice per grid row; about one workgroup per CU in all
            gy = (unsigned)(((a.K >> 8) + 15) >> 4);
            grid = std::max<long long>(1, std::min<long long>(want, cu_count / (long long)gy));
        }
        hipLaunchKernelGGL(kern, dim3((unsigned)grid, gy), dim3(WAVES * 64), lds, stream, a);
        return hipGetLastError();
    }
};
template <int T, int MT, int PRO, bool ONE_SLICE, int NBUF, int WAVES, int GROUP, bool PAIR, bool SPLIT>
std::atomic<int> F32Instance<T, MT, PRO, ONE_SLICE, NBUF, WAVES, GROUP, PAIR, SPLIT>::occupancy{0};

// y[m][row] (+)= ((P_0 + P_1) + P_2) ... over the slices of a SPLIT launch,
// in slice order, times the RMSNorm factor: the slice totals of the one-launch
// form, added the same way.
// (NORM is a template argument: with a branch on args.gamma the plain reduction
// was longer, one member of Q6_K 24576 -> 256 8.8 instead of 8.1 us.)
template <bool NORM>
__global__ __launch_bounds__(256) void f32_split_reduce_kernel(WaveGemvArgs a, int slices) {
    const int total = a.members * a.total_rows;
    __shared__ float inv_s[NORM ? kWaveMaxMembers : 1];
    if constexpr (NORM) {
        const int nb = a.K >> 8;
        if ((int)threadIdx.x < a.members) {
            const float* ssq = a.partial + (size_t)slices * total + (size_t)threadIdx.x * nb;
            float sum = 0.f;
            for (int b = 0; b < nb; ++b) sum += ssq[b];
            inv_s[threadIdx.x] = 1.0f / sqrtf(sum / (float)a.K + a.eps);
        }
        __syncthreads();
    }
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int m = i / a.total_rows;
        const int row = i - m * a.total_rows;
        float t = a.partial[(size_t)m * a.total_rows + row];
        for (int s = 1; s < slices; ++s) t = t + a.partial[((size_t)s * a.members + m) * a.total_rows + row];
        if constexpr (NORM) t = t * inv_s[m];
        int mat = 0, start = 0;
        for (int g = 0; g + 1 < a.count; ++g) {
            if (row >= a.rows_end[g]) {
                mat = g + 1;
                start = a.rows_end[g];
            }
        }
        float* y = a.y[0];
        for (int g = 1; g < kMaxGroup; ++g) {
            if (mat == g) y = a.y[g];
        }
        const int rows_mat = a.rows_end[mat] - start;
        float* dst = y + (size_t)m * rows_mat + (row - start);
        *dst = a.accumulate ? *dst + t : t;
    }
}

// One or two members whose K is not one slice of more than 8 blocks.
template <int T, int MT, int PRO, bool MULTI, bool PAIR = false>
hipError_t launch_slices(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    constexpr int kRing = 2;
    constexpr int kMaxLds = 158 * 1024;  // beside the kernel's own few hundred bytes
    auto kern = gemv_f32_slices_kernel<T, MT, PRO, MULTI, kRing, PAIR>;
    static PerDevice sized;
    const hipError_t e = sized.once(a.device, [&] {
        return hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    });
    if (e != hipSuccess) return e;
    const int nb = a.K >> 8, slices = (nb + 15) >> 4;
    long long quads = 0;
    for (int i = 0; i < (PAIR ? 1 : a.count); ++i)
        quads += (a.rows_end[i] - (i > 0 ? a.rows_end[i - 1] : 0) + 3) / 4;
    // one workgroup per CU, fewer where a wave would have less than a unit or
    // two, more where a workgroup's slice totals would not fit beside its records
    const long long records = (long long)MT * slices * 64 * F32Rec<T>::stride * 4;
    const long long quad_bytes = (PAIR ? 2LL : 1LL) * 4 * slices * MT * 4;
    const long long quad_units = (PAIR ? 2 : 1) * (4LL * (slices - 1) + 4 / unit_rows(nb - 16 * (slices - 1)));
    long long grid = std::min<long long>(cu_count, (quads * quad_units + kSliceWaves - 1) / kSliceWaves);
    const long long most = (kMaxLds - records) / quad_bytes;  // quads a workgroup holds
    if (most < 1) return hipErrorInvalidValue;
    grid = std::max<long long>({grid, 1, (quads + most - 1) / most});
    grid = std::min(grid, quads);
    const long long held = (quads + grid - 1) / grid;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kSliceWaves * 64), (size_t)(records + held * quad_bytes), stream, a);
    return hipGetLastError();
}

// K above 4096, one or two members: whether pairs of rows over all slices (a wave
// rereads the slices' records for every pair) beat the units of
// gemv_f32_slices_kernel. A wave takes ceil(rows / 16 per CU) pairs, `pair_units`
// units. Plain products: the slices form costs about as much more a launch as two
// units take, so it has to save two, or one where two members make the rereads
// dearer (Q4_K, and a short last slice after one whole slice); longer launches
// hide it. With a SwiGLU pairs are faster only where nothing is saved over four
// slices (three for one member of Q5_K and Q6_K), with an RMSNorm nowhere. Pairs time / slices time over K 4608 .. 16384 and 2 .. 68 rows a CU,
// Q4_K / Q5_K / Q6_K:
//   plain, one member, two or more units saved 1.04-1.7 / 1.02-1.8 / 1.03-1.7, one
//   saved 0.86-0.99 / 0.94-1.03 / 0.88-1.04, none 0.84-1.13 (0.91-0.99 up to 32 rows
//   a CU; two whole slices 0.95-0.99 at 48); e.g. us, Q4_K: 5120 at 3072 and 4096 rows
//   6.9 / 6.1 and 7.0 / 7.6; 8192 at 2560 rows 6.3 / 7.0; 12288 at 2048, 2560 and 5120
//   rows 8.1 / 7.4, 8.2 / 9.0 and 13.8 / 11.3
//   SwiGLU, K up to 9728 1.03-1.7, 12288 0.96-1.5, 16384 at 13 to 16 rows a CU 0.92-0.97
//   RMSNorm 0.98-1.7
template <int T, int MT, int PRO>
bool pairs_form(const WaveGemvArgs& a, int cu_count) {
    const long long per_cu = ((long long)a.total_rows + cu_count - 1) / cu_count;
    const int nb = a.K >> 8, slices = (nb + 15) >> 4;
    const long long quad_units = 4 * (slices - 1) + 4 / unit_rows(nb - 16 * (slices - 1));
    const long long slice_units = ((per_cu + 3) / 4 * quad_units + kSliceWaves - 1) / kSliceWaves;
    const long long pair_units = 2 * slices * ((per_cu + 15) / 16);
    if (PRO == kProSwiglu) {
        return per_cu <= 16 && pair_units <= slice_units && (slices > 3 || (slices == 3 && MT == 1 && T != kQ4K));
    }
    if (per_cu > (slices == 2 ? 48 : 32)) return false;
    const int save = MT == 2 && (T == kQ4K || (slices == 2 && unit_rows(nb - 16) > 1)) ? 1 : 2;
    return pair_units - slice_units < save;
}

// One or two members.
template <int T, int MT, int PRO, bool ONE_SLICE, bool PAIR = false>
hipError_t launch_few(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    if constexpr (!ONE_SLICE) {
        if constexpr (PRO != kProNorm) {
            if (pairs_form<T, MT, PRO>(a, cu_count)) return F32Instance<T, MT, PRO, false, 2, 8, 2>::launch(a, cu_count, 1, stream);
        }
        return launch_slices<T, MT, PRO, true>(a, cu_count, stream);
    } else {
        // Short rows: several to a unit, where the launch is long enough for it
        // (us, one member, one row / several: Q4_K 1024 at 4096, 5120, 12288
        // rows 4.2 / 4.6, 5.0 / 4.7, 7.0 / 5.7; 1536 at 10240, 10496, 16384 rows
        // 6.2 / 6.2, 6.4 / 6.3, 8.1 / 7.2; 2048 at 10496, 12288, 14336 rows 6.4 / 6.8,
        // 6.7 / 6.9, 7.7 / 7.5, with an RMSNorm 7.0 / 7.0, 7.2 / 7.1, 8.0 / 7.7; two
        // members of K 1536 and 2048 at 10496 rows 1.10-1.15 times as fast).
        const bool late = T == kQ4K && MT == 1 && PRO != kProNorm && a.K > 1536;
        if (a.total_rows > (a.K <= 1024 ? 16LL : late ? 48LL : 40LL) * cu_count && a.K <= 2048) {
            return launch_slices<T, MT, PRO, false, PAIR>(a, cu_count, stream);
        }
        const long long per_cu = ((long long)a.total_rows + cu_count - 1) / cu_count;
        if constexpr (MT == 1) {
            // Streams of more than 48 units per CU (gate/up, the lm_head): a
            // three-unit ring (four for gate/up pairs) over 8-wave workgroups,
            // one per CU. MI355X sweep over ring {2,3,4,6,8} x waves {4,8,16} x
            // workgroups per CU {1,2,4}: 13.3 us for the gate+up group
            // (Q4_K 4096 -> 2 x 12288) against 14.3 us for ring 2 x 2 per CU,
            // and 97 us for the Q6_K 4096 -> 151936 head against 124 us for
            // ring 8 x 4 waves.
            if (per_cu > 48) {
                return F32Instance<T, 1, PRO, true, (PAIR ? 4 : 3), 8, 1, PAIR>::launch(a, cu_count, 1, stream);
            }
        }
        return F32Instance<T, MT, PRO, true, 2, 8, 1, PAIR>::launch(a, cu_count, per_cu > 48 ? 2 : 1, stream);
    }
}

// Three to eight members (one form for all; four members of 4096 rows 7.5 us on
// the VALU rows, 6.6 here; three use the four-member form): one workgroup per CU
// over the slice (or, SPLIT, over the slices in proportion to their super-blocks).
template <int T, int MG, int PRO, bool PAIR, bool SPLIT = false>
hipError_t launch_many_instance(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    constexpr int kRing = 2;
    auto kern = gemv_f32_many_kernel<T, MG, PRO, kRing, PAIR, SPLIT>;
    static PerDevice sized;
    const hipError_t e = sized.once(a.device, [&] {
        return hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, MG * kManyLds);
    });
    if (e != hipSuccess) return e;
    const int nb = a.K >> 8;
    const int slices = SPLIT ? (nb + 15) >> 4 : 1;
    long long units = 0;
    for (int i = 0; i < (PAIR ? 1 : a.count); ++i)
        units += (a.rows_end[i] - (i > 0 ? a.rows_end[i - 1] : 0) + 3) / 4;
    // workgroups of a whole slice, and of the last one (its share of the quarters)
    const int quarters = (nb + 3) >> 2, last = quarters - 4 * (slices - 1);
    const int sets = last == 1 ? 8 : last == 2 ? 4 : 2;
    const int wgs = (int)std::max<long long>(1, std::min<long long>((units + 1) / 2, (long long)cu_count * (slices == 1 ? last : 4) / quarters));
    const int tail = (int)std::max<long long>(1, std::min<long long>((units + sets - 1) / sets, cu_count - (long long)wgs * (slices - 1)));
    const int grid = slices == 1 ? tail : wgs * (slices - 1) + tail;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kManyWaves * 64), MG * kManyLds, stream, a, wgs);
    return hipGetLastError();
}

template <int T, int PRO, bool PAIR, bool SPLIT = false>
hipError_t launch_many(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    return a.members <= 4 ? launch_many_instance<T, 1, PRO, PAIR, SPLIT>(a, cu_count, stream)
                          : launch_many_instance<T, 2, PRO, PAIR, SPLIT>(a, cu_count, stream);
}

template <int T, int PRO>
hipError_t launch_plain(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    const bool one = a.K <= kSliceElems;
    if (a.members <= 1) {
        return one ? launch_few<T, 1, PRO, true>(a, cu_count, stream) : launch_few<T, 1, PRO, false>(a, cu_count, stream);
    }
    if (a.members <= 2 || !one) {
        if (a.members > 2) return hipErrorInvalidValue;
        return one ? launch_few<T, 2, PRO, true>(a, cu_count, stream) : launch_few<T, 2, PRO, false>(a, cu_count, stream);
    }
    if constexpr (PRO == kProSwiglu) {
        return hipErrorInvalidValue;  // the host splits SwiGLU-prologue launches into pairs of members
    } else {
        return launch_many<T, PRO, false>(a, cu_count, stream);
    }
}

template <int T, int PRO>
hipError_t launch_pair(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    if (a.members <= 1) return launch_few<T, 1, PRO, true, true>(a, cu_count, stream);
    if (a.members <= 2) return launch_few<T, 2, PRO, true, true>(a, cu_count, stream);
    return launch_many<T, PRO, true>(a, cu_count, stream);
}

template <int T>
hipError_t launch_type(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    if (a.members < 1 || a.members > f32_max_members(a.K)) return hipErrorInvalidValue;
    if (a.pair_swiglu) {
        if (a.x2 != nullptr || a.count != 2 || a.rows_end[1] != 2 * a.rows_end[0] || a.K > kSliceElems) {
            return hipErrorInvalidValue;
        }
        return a.gamma != nullptr ? launch_pair<T, kProNorm>(a, cu_count, stream)
                                  : launch_pair<T, kProPlain>(a, cu_count, stream);
    }
    if (a.x2 != nullptr) {
        if (a.gamma != nullptr || a.members > kSwigluMaxMembers) return hipErrorInvalidValue;
        return launch_plain<T, kProSwiglu>(a, cu_count, stream);
    }
    if (a.gamma != nullptr) return launch_plain<T, kProNorm>(a, cu_count, stream);
    return launch_plain<T, kProPlain>(a, cu_count, stream);
}

// One member, K above kWaveMaxK: whether one launch of the slices form, whose
// workgroups stage all of K, beats a workgroup per slice and the reduction. Past
// five slices staging costs more than the second launch where a workgroup has
// one short run of units, or (Q4_K, and Q5_K of seven slices on) more than a few.
// Split time / one launch, Q4_K / Q5_K / Q6_K: K 16640 .. 17408 at 1 and 2 rows a CU
// 1.06-1.11 / 0.95-1.02 / 0.97-1.01, more 1.00-1.09 / 1.01-1.07 / 1.00-1.10 (Q6_K at 14
// and 16 rows a CU 0.90-1.02; at K 17408 itself also 0.90 at 32 and 0.96 at 40); K 18432
// .. 24576 at 1 and 2 rows a CU 1.01-1.09 / 0.94-0.98 / 0.94-0.97, 4 to 16 rows
// 0.99-1.13, more 0.94-1.03 / 0.96-1.10 / 1.00-1.07; K 28672 and 32768 at 1 and 2 rows
// 0.85-0.92, 4 and 8 rows 0.98-1.07, 12 and more 0.92-0.98 / 0.94-1.05 / 0.99-1.05.
template <int T>
bool one_launch_long_k(const WaveGemvArgs& a, int cu_count) {
    if (a.K > 2 * kWaveMaxK) return false;
    const long long per_cu = ((long long)a.total_rows + cu_count - 1) / cu_count;
    if (a.K <= 17408) return T == kQ4K || (per_cu > 2 && (T == kQ5K || per_cu <= 12 || per_cu > 16));
    const bool any_longer = T == kQ6K || (T == kQ5K && a.K <= 24576);
    return per_cu > 2 && (any_longer || per_cu <= (a.K <= 24576 ? 16 : 8));
}

// Members over a K of several slices: one workgroup per (row range, slice),
// then the ordered slice reduction. One member (a K beyond kWaveMaxK) keeps
// its records in VGPRs, as the one-launch form does.
template <int T>
hipError_t launch_split(const WaveGemvArgs& a, int cu_count, hipStream_t stream) {
    if (a.members == 1 && one_launch_long_k<T>(a, cu_count)) return launch_slices<T, 1, kProPlain, true>(a, cu_count, stream);
    hipError_t e = (a.members == 1)
                       ? F32Instance<T, 1, kProPlain, true, 3, 8, 1, false, true>::launch(a, cu_count, 1, stream)
                   : a.gamma != nullptr ? launch_many<T, kProNorm, false, true>(a, cu_count, stream)
                                        : launch_many<T, kProPlain, false, true>(a, cu_count, stream);
    if (e != hipSuccess) return e;
    const int slices = ((a.K >> 8) + 15) >> 4;
    const long long total = (long long)a.members * a.total_rows;
    const unsigned grid = (unsigned)std::min<long long>((total + 255) / 256, (long long)cu_count * 4);
    if (a.gamma != nullptr) {
        hipLaunchKernelGGL(f32_split_reduce_kernel<true>, dim3(grid), dim3(256), 0, stream, a, slices);
    } else {
        hipLaunchKernelGGL(f32_split_reduce_kernel<false>, dim3(grid), dim3(256), 0, stream, a, slices);
    }
    return hipGetLastError();
}

}  // namespace

size_t f32_split_partial_bytes(int members, int K, int total_rows) {
    const int slices = ((K >> 8) + 15) >> 4;
    return (size_t)slices * members * total_rows * sizeof(float);
}

hipError_t launch_gemv_f32_split(int value_type, const WaveGemvArgs& args, int cu_count, hipStream_t stream) {
    const int min_members = args.K > kWaveMaxK ? 1 : 3;
    if (args.members < min_members || args.members > kWaveMaxMembers || args.K <= kSliceElems ||
        args.K > kF32SplitMaxK || args.K % 256 != 0 || (args.gamma != nullptr && args.members < 3) || args.x2 != nullptr ||
        args.pair_swiglu || args.partial == nullptr ||
        f32_split_partial_bytes(args.members, args.K, args.total_rows) > (args.K > kWaveMaxK ? kF32SplitScratchBytes : kF32MmaPartialBytes)) {
        return hipErrorInvalidValue;
    }
    switch (value_type) {
    case kQ4K: return launch_split<kQ4K>(args, cu_count, stream);
    case kQ5K: return launch_split<kQ5K>(args, cu_count, stream);
    case kQ6K: return launch_split<kQ6K>(args, cu_count, stream);
    default: return hipErrorInvalidValue;
    }
}

int f32_long_k_members(int K, int total_rows) {
    if (K <= kWaveMaxK || K > kF32SplitMaxK || K % 256 != 0 || total_rows < 1) return 0;
    int m = kWaveMaxMembers;
    while (m > 0 && f32_split_partial_bytes(m, K, total_rows) > kF32SplitScratchBytes) --m;
    return m;
}

int f32_max_members(int K) {
    if (K < 256 || K > kWaveMaxK) return 0;
    return K <= kSliceElems ? kWaveMaxMembers : 2;
}

hipError_t launch_gemv_f32(int value_type, const WaveGemvArgs& args, int cu_count, hipStream_t stream) {
    switch (value_type) {
    case kQ4K: return launch_type<kQ4K>(args, cu_count, stream);
    case kQ5K: return launch_type<kQ5K>(args, cu_count, stream);
    case kQ6K: return launch_type<kQ6K>(args, cu_count, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace ribn_amd
