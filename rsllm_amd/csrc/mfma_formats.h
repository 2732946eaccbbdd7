// The quantized formats as operands of v_mfma_f32_16x16x32_f16 (exact f16
// integers with fp32 scales) and the hi + lo f16 activations they meet, shared
// by the batched GEMV (gemv_mfma.hip) and the many-token GEMM
// (gemm_exact.hip).
#pragma once

#include <type_traits>

#include "gemv_formats.h"

namespace rsllm_hip {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMfStep = 128;  // K elements per step

// Max over a wavefront (every lane gets it): DPP row reductions plus lane reads.
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false)));
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 15));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 31));
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 47));
    const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

__device__ __forceinline__ uint32_t bload4(__amdgpu_buffer_rsrc_t r, uint32_t voff) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, 0, 0);
}

// The weights are the B operand of v_mfma_f32_16x16x32_f16 (K x 16 weight
// rows) and the activations the A operand (16 tokens x K), so lane
// (r16, q) = (lane % 16, lane / 16) supplies weights of row r16 and receives
// D[4q + i][r16], i = 0..3: four tokens of its own row. Every B value is an
// exact integer in f16 — Q4_K sc * q (at most 63 * 15), Q6_K sc * (q - 32)
// (an f16 part and a -1/0/1 remainder where |.| > 2048), Q8_0 q — and the
// per-row scales the reference multiplies in f32 (d, dmin * m) are applied
// to each step's MFMA result in fp32 by the lane that holds that row.
// Products of two f16 values are exact in fp32, so the weights are exact;
// the activations enter as hi + lo f16 planes (about 2^-22 relative).
//
// Each format gives: W (a lane's bytes for one step), elem / piece (the K
// order: element of MFMA j, lane group q, step s), load, and step<NT, PACK>:
// the MFMAs of one step for one 16-row tile against NT token tiles, folded
// into acc[NT] with the scales. With PACK (up to 8 tokens) the A operand x
// holds the hi plane of tokens 0..7 in its rows 0..7 and the lo plane in
// rows 8..15, and xl is not read: one MFMA per sub-step, and D rows t and
// t + 8 add up to token t.

__device__ __forceinline__ f32x4 mfma16x32(const uint4 &x, const f16x8 &w, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x), w, c, 0, 0, 0);
}

// Q4_K (GGUF layout). Step s = half (s & 1) of super-block s >> 1. Lane group
// q reads qs bytes 32q + 16 (s & 1) .. + 15 (sub-block pair q): low nibbles are
// sub-block 2q, positions 16 (s & 1) + 0..15; high nibbles sub-block 2q + 1.
// MFMA j: low (j even) / high (j odd) nibbles of bytes 0..7 (j < 2) or 8..15.
// B = sc_j * q (exact); a second MFMA per j with B = m_j gives sum m_j x, and
// the step adds d * P - dmin * M (dequant_q4_k, q4_k.rs:66-88: w = d sc q -
// dmin m).
struct MQ4K {
    struct W {
        uint4 hdr, qs;
    };
    __device__ static int elem(int s, int j, int q) {
        return 256 * (s >> 1) + 64 * q + 32 * (j & 1) + 16 * (s & 1) + 8 * (j >> 1);
    }
    // inverse of elem for an 8-aligned element offset: (s, j, q)
    __device__ static void piece(int e, int &s, int &j, int &q) {
        const int r = e & 255;
        q = r >> 6;
        s = 2 * (e >> 8) + ((r >> 4) & 1);
        j = ((r >> 5) & 1) + 2 * ((r >> 3) & 1);
    }
    __device__ static void load(W &w, __amdgpu_buffer_rsrc_t r, int row, int s, int q, int in_dim,
                                int) {
        const uint32_t off = ((uint32_t)row * (uint32_t)(in_dim >> 8) + (uint32_t)(s >> 1)) * 144u;
        w.hdr = bload16(r, off, 0);
        w.qs = bload16(r, off + 16u + 32u * (uint32_t)q + 16u * (uint32_t)(s & 1), 0);
    }
    template <int NT, bool PACK = false>
    __device__ static void step(const W &w, int q, const uint4 (&x)[4][NT], const uint4 (&xl)[4][NT],
                                f32x4 (&acc)[NT]) {
        const float d = f16_to_f32(w.hdr.x & 0xFFFFu), dmin = f16_to_f32(w.hdr.x >> 16);
        // (sc, m) of sub-blocks 2q and 2q + 1 (q4_k_scale_min,
        // dequant/mod.rs:48-58), all four bytes of a word at once: sub-block
        // j < 4 has sc = s0[j] & 63, m = s1[j] & 63; j >= 4 has sc =
        // s2[j - 4] & 15 | (s0[j - 4] >> 6) << 4, m = s2[j - 4] >> 4 |
        // (s1[j - 4] >> 6) << 4. Lane group q takes bytes 2 (q & 1) and
        // 2 (q & 1) + 1 of the low (q < 2) or high words, each paired with
        // 0x64 by v_perm_b32 (the f16 1024 + v, exact) less 1024.
        // (masks and selectors as arithmetic: a conditional here became a
        // branch per tile)
        const uint32_t s0 = w.hdr.y, s1 = w.hdr.z, s2 = w.hdr.w;
        const uint32_t hm = 0u - (uint32_t)(q >> 1);  // all ones for q >= 2
        const uint32_t sc4 = (((s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)) & hm) |
                             (s0 & 0x3F3F3F3Fu & ~hm);
        const uint32_t m4 = ((((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) & hm) |
                            (s1 & 0x3F3F3F3Fu & ~hm);
        const uint32_t sel = 0x04010400u + (uint32_t)(q & 1) * 0x00020002u;
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const f16x2 scp = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, sc4, sel)) - k1024;
        const f16x2 mp = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m4, sel)) - k1024;
        const _Float16 sl = scp[0], sh = scp[1];
        const f16x2 zero = {(_Float16)0.0f, (_Float16)0.0f};
        const f16x2 ssl = {sl, sl}, ssh = {sh, sh};
        f16x8 b[4];
        b[0] = dequant_q4x8_f16(w.qs.x, w.qs.y, false, ssl, zero);
        b[1] = dequant_q4x8_f16(w.qs.x, w.qs.y, true, ssh, zero);
        b[2] = dequant_q4x8_f16(w.qs.z, w.qs.w, false, ssl, zero);
        b[3] = dequant_q4x8_f16(w.qs.z, w.qs.w, true, ssh, zero);
        const _Float16 ml = mp[0], mh = mp[1];
        const f16x8 bml = {ml, ml, ml, ml, ml, ml, ml, ml}, bmh = {mh, mh, mh, mh, mh, mh, mh, mh};
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            f32x4 P = {0.f, 0.f, 0.f, 0.f}, M = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                P = mfma16x32(x[j][nt], b[j], P);
                if (!PACK) P = mfma16x32(xl[j][nt], b[j], P);
                M = mfma16x32(x[j][nt], (j & 1) ? bmh : bml, M);
                if (!PACK) M = mfma16x32(xl[j][nt], (j & 1) ? bmh : bml, M);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[nt][i] = fmaf(-dmin, M[i], fmaf(d, P[i], acc[nt][i]));
        }
    }
};

// Four 6-bit codes (bytes 0..63 of q6) -> f16 q - 32 (exact): v_perm_b32
// pairs each byte with 0x64, the f16 pattern of 1024 + q, and subtracting
// 1056 leaves q - 32.
__device__ __forceinline__ void q6x4_f16(uint32_t q6, f16x2 &w01, f16x2 &w23) {
    const uint32_t p01 = __builtin_amdgcn_perm(0x64646464u, q6, 0x04010400u);
    const uint32_t p23 = __builtin_amdgcn_perm(0x64646464u, q6, 0x04030402u);
    const f16x2 bias = {(_Float16)1056.0f, (_Float16)1056.0f};
    w01 = __builtin_bit_cast(f16x2, p01) - bias;
    w23 = __builtin_bit_cast(f16x2, p23) - bias;
}

// Q6_K (super-tile device layout). Step s = half h = s & 1 of block s >> 1.
// Lane group q reads ql bytes 64h + 16q .. + 15 and qh bytes 32h + 16 (q & 1)
// .. + 15: low nibbles are elements 128h + 16q + b (high bits at 2 (q >> 1)),
// high nibbles elements 128h + 64 + 16q + b (high bits at 4 + 2 (q >> 1));
// their scales are sc[8h + q] and sc[8h + q + 4]. B = sc * (q - 32), and the
// step adds d * P (dequant_q6_k, q6_k.rs:86-92: w = d sc (q - 32)).
// |sc (q - 32)| <= 128 * 32 = 4096: exact in f16 up to 2048, and above that
// (|sc| > 64, which GGUF's int8 scales allow) f16 keeps the even integers
// only. So B = f16(sc (q - 32)) and B_lo = sc (q - 32) - B (one fused f16
// multiply-add, exact, in {-1, 0, 1}); a step whose wavefront has any
// |sc| > 64 adds x_hi * B_lo as a third MFMA per sub-step, which leaves out
// only x_lo * B_lo (below 2^-22 of the term). A step without such scales
// builds 2^-15 B instead, with one FMA per two weights on subnormal codes
// (the same products scaled by a power of two, so the same sums).
struct MQ6K {
    struct W {
        uint4 ql, qh;
        uint32_t sl, sh, d;
    };
    __device__ static int elem(int s, int j, int q) {
        return 256 * (s >> 1) + 128 * (s & 1) + 16 * q + 64 * (j & 1) + 8 * (j >> 1);
    }
    __device__ static void piece(int e, int &s, int &j, int &q) {
        const int r = e & 255;
        s = 2 * (e >> 8) + (r >> 7);
        j = ((r >> 6) & 1) + 2 * ((r >> 3) & 1);
        q = (r >> 4) & 3;
    }
    __device__ static void load(W &w, __amdgpu_buffer_rsrc_t r, int row, int s, int q, int in_dim,
                                int out_dim) {
        const uint32_t nb = (uint32_t)(in_dim >> 8);
        const uint32_t nblk = (uint32_t)out_dim * nb;
        const uint32_t bi = (uint32_t)row * nb + (uint32_t)(s >> 1);
        const uint32_t S = bi >> 3, jb = bi & 7u;
        const uint32_t rS = (S < (nblk >> 3)) ? 8u : (nblk & 7u);
        const uint32_t base = S * 1680u, h = (uint32_t)(s & 1);
        w.ql = bload16(r, base + jb * 128u + 64u * h + 16u * (uint32_t)q, 0);
        w.qh = bload16(r, base + rS * 128u + jb * 64u + 32u * h + 16u * (uint32_t)(q & 1), 0);
        w.sl = bload4(r, base + rS * 192u + jb * 16u + 8u * h);
        w.sh = bload4(r, base + rS * 192u + jb * 16u + 8u * h + 4u);
        w.d = bload2(r, base + rS * 208u + jb * 2u, 0);
    }
    // lane holds a scale with |sc| > 64
    __device__ static bool wide_lane(const W &w, int q) {
        const int il = (int)(int8_t)(w.sl >> (8 * q)), ih = (int)(int8_t)(w.sh >> (8 * q));
        return il > 64 || il < -64 || ih > 64 || ih < -64;
    }
    template <int NT, bool PACK = false>
    __device__ static void step(const W &w, int q, const uint4 (&x)[4][NT], const uint4 (&xl)[4][NT],
                                f32x4 (&acc)[NT]) {
        step_m<NT, 2, PACK>(w, q, x, xl, acc);
    }
    // WIDE 0: no scale of the wavefront's step has |sc| > 64 (the caller
    // checked); 1: add the B_lo MFMAs; 2: decide here, per step
    template <int NT, int WIDE, bool PACK>
    __device__ static void step_m(const W &w, int q, const uint4 (&x)[4][NT],
                                  const uint4 (&xl)[4][NT], f32x4 (&acc)[NT]) {
        const float d = f16_to_f32(w.d);
        const int il = (int)(int8_t)(w.sl >> (8 * q)), ih = (int)(int8_t)(w.sh >> (8 * q));
        const bool wide = WIDE == 1 || (WIDE == 2 && __ballot(wide_lane(w, q)) != 0);
        // the high bit pairs sit at bits 2 (q >> 1) (low nibbles) and 4 + 2 (q >> 1)
        // (high nibbles) of each qh byte; one shift puts either pair at bits 4, 5
        const uint32_t shl = 2u * (uint32_t)(q >> 1), sup = 4u - shl;
        const uint32_t l[4] = {w.ql.x, w.ql.y, w.ql.z, w.ql.w};
        const uint32_t hb[4] = {w.qh.x, w.qh.y, w.qh.z, w.qh.w};
        // four 6-bit codes of MFMA j, word u (bytes in K order)
        auto codes = [&](int j, int u) {
            const bool hi = j & 1;
            const int p = 2 * (j >> 1) + u;
            const uint32_t nib = hi ? (l[p] >> 4) & 0x0F0F0F0Fu : l[p] & 0x0F0F0F0Fu;
            const uint32_t top = (hi ? hb[p] >> shl : hb[p] << sup) & 0x30303030u;
            return nib | top;
        };
        f32x4 P[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) P[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto mma = [&](const f16x8 (&b)[4]) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    P[nt] = mfma16x32(x[j][nt], b[j], P[nt]);
                    if (!PACK) P[nt] = mfma16x32(xl[j][nt], b[j], P[nt]);
                }
        };
        float dd = d;
        if (!wide) {
            // |sc| <= 64: B = 2^-15 sc (q - 32), exact, in one FMA per pair:
            // v_perm_b32 zero-extends two codes to f16 bit patterns (the
            // subnormals code * 2^-24), times sc * 2^9, plus -sc * 2^-10; the
            // step's sum is scaled back by 2^15 with d
            const _Float16 ml = (_Float16)((float)il * 512.0f), mh = (_Float16)((float)ih * 512.0f);
            const _Float16 cl = (_Float16)((float)il * -0x1p-10f), ch = (_Float16)((float)ih * -0x1p-10f);
            f16x8 b[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f16x2 m2 = (j & 1) ? f16x2{mh, mh} : f16x2{ml, ml};
                const f16x2 c2 = (j & 1) ? f16x2{ch, ch} : f16x2{cl, cl};
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const uint32_t c = codes(j, u);
                    const f16x2 t01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0u, c, 0x0c010c00u));
                    const f16x2 t23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0u, c, 0x0c030c02u));
                    const f16x2 w01 = __builtin_elementwise_fma(t01, m2, c2);
                    const f16x2 w23 = __builtin_elementwise_fma(t23, m2, c2);
                    b[j][4 * u] = w01[0];
                    b[j][4 * u + 1] = w01[1];
                    b[j][4 * u + 2] = w23[0];
                    b[j][4 * u + 3] = w23[1];
                }
            }
            mma(b);
            dd = d * 32768.0f;
        } else {
            const _Float16 scl = (_Float16)(float)il, sch = (_Float16)(float)ih;
            f16x8 a[4], b[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                f16x2 v[4];
#pragma unroll
                for (int u = 0; u < 2; u++) q6x4_f16(codes(j, u), v[2 * u], v[2 * u + 1]);
                f16x8 r;
                r[0] = v[0][0]; r[1] = v[0][1]; r[2] = v[1][0]; r[3] = v[1][1];
                r[4] = v[2][0]; r[5] = v[2][1]; r[6] = v[3][0]; r[7] = v[3][1];
                const _Float16 sc = (j & 1) ? sch : scl;
                const f16x8 sv = {sc, sc, sc, sc, sc, sc, sc, sc};
                a[j] = r;
                b[j] = r * sv;
            }
            mma(b);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const _Float16 sc = (j & 1) ? sch : scl;
                const f16x8 sv = {sc, sc, sc, sc, sc, sc, sc, sc};
                const f16x8 bl = __builtin_elementwise_fma(a[j], sv, -b[j]);
#pragma unroll
                for (int nt = 0; nt < NT; nt++) P[nt] = mfma16x32(x[j][nt], bl, P[nt]);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[nt][i] = fmaf(dd, P[nt][i], acc[nt][i]);
    }
};

// Q8_0 (super-tile device layout [qs 8x32 | d 8x2]). Step s = blocks 4s ..
// 4s + 3 of the row (in_dim is a multiple of 256, so they share one
// super-tile); MFMA j is block 4s + j, lane group q its elements 8q .. 8q + 7.
// A code q (int8) becomes f16 exactly as the pattern 0x64 with byte q ^ 0x80
// (1024 + q + 128) minus 1152; each block's MFMA result is multiplied by its
// scale d in fp32 (dequant_q8_0, q8_0.rs:25-63: w = d q).
struct MQ8 {
    struct W {
        uint2 q[4];
        uint2 d;  // the four blocks' f16 scales
    };
    __device__ static int elem(int s, int j, int q) { return 128 * s + 32 * j + 8 * q; }
    __device__ static void piece(int e, int &s, int &j, int &q) {
        s = e >> 7;
        j = (e >> 5) & 3;
        q = (e >> 3) & 3;
    }
    __device__ static void load(W &w, __amdgpu_buffer_rsrc_t r, int row, int s, int q, int in_dim,
                                int out_dim) {
        const uint32_t nb = (uint32_t)(in_dim >> 5);
        const uint32_t nblk = (uint32_t)out_dim * nb;
        const uint32_t bi = (uint32_t)row * nb + 4u * (uint32_t)s;  // jb is 0 or 4
        const uint32_t S = bi >> 3, jb = bi & 7u;
        const uint32_t rS = (S < (nblk >> 3)) ? 8u : (nblk & 7u);
        const uint32_t base = S * 272u;
#pragma unroll
        for (int j = 0; j < 4; j++)
            w.q[j] = bload8(r, base + (jb + (uint32_t)j) * 32u + 8u * (uint32_t)q, 0);
        w.d = bload8(r, base + rS * 32u + jb * 2u, 0);
    }
    template <int NT, bool PACK = false>
    __device__ static void step(const W &w, int, const uint4 (&x)[4][NT], const uint4 (&xl)[4][NT],
                                f32x4 (&acc)[NT]) {
        const f16x2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
        f16x8 b[4];
        float d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            d[j] = f16_to_f32(((j & 2) ? w.d.y : w.d.x) >> (16 * (j & 1)));
            f16x8 r;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t bb = (u ? w.q[j].y : w.q[j].x) ^ 0x80808080u;
                const f16x2 w01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, bb, 0x04010400u)) - bias;
                const f16x2 w23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, bb, 0x04030402u)) - bias;
                r[4 * u] = w01[0];
                r[4 * u + 1] = w01[1];
                r[4 * u + 2] = w23[0];
                r[4 * u + 3] = w23[1];
            }
            b[j] = r;
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 P0 = mfma16x32(x[j][nt], b[j], f32x4{0.f, 0.f, 0.f, 0.f});
                const f32x4 P = PACK ? P0 : mfma16x32(xl[j][nt], b[j], P0);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[nt][i] = fmaf(d[j], P[i], acc[nt][i]);
            }
    }
};

// Q2_K (super-tile device layout [qs 8x64 | scales 8x16 | (d, dmin) 8x4],
// 672 bytes per 8 blocks; the matrix's last super-tile holds the blocks
// left). Step s = half n = s & 1 of block s >> 1, its elements in order:
// element 128 n + 32 j + l (l < 32) is bits 2j, 2j + 1 of qs byte 32 n + l
// under scale byte 8 n + 2 j + l / 16 (low nibble sc, high nibble m)
// (dequant_q2_k, q2_k.rs:73-95: w = d sc q - dmin m). MFMA j takes the codes at
// shift 2j; lane group q reads qs bytes 32 n + 8 q .. + 7, all of sub-block
// 8 n + 2 j + q / 2. B = sc * q (exact, at most 45); a second MFMA per j
// with B = m gives sum m x; the step adds d * P - dmin * M.
struct MQ2K {
    struct W {
        uint2 qs, sc;  // the lane's 8 qs bytes; the half's 8 scale bytes
        uint32_t dd;   // f16 d, dmin
    };
    __device__ static int elem(int s, int j, int q) { return 128 * s + 32 * j + 8 * q; }
    __device__ static void piece(int e, int &s, int &j, int &q) {
        s = e >> 7;
        j = (e >> 5) & 3;
        q = (e >> 3) & 3;
    }
    __device__ static void load(W &w, __amdgpu_buffer_rsrc_t r, int row, int s, int q, int in_dim,
                                int out_dim) {
        const uint32_t nb = (uint32_t)(in_dim >> 8);
        const uint32_t nblk = (uint32_t)out_dim * nb;
        const uint32_t bi = (uint32_t)row * nb + (uint32_t)(s >> 1);
        const uint32_t S = bi >> 3, jb = bi & 7u;
        const uint32_t rS = (S < (nblk >> 3)) ? 8u : (nblk & 7u);
        const uint32_t base = S * 672u, n = (uint32_t)(s & 1);
        w.qs = bload8(r, base + jb * 64u + 32u * n + 8u * (uint32_t)q, 0);
        w.sc = bload8(r, base + rS * 64u + jb * 16u + 8u * n, 0);
        w.dd = bload4(r, base + rS * 80u + jb * 4u);
    }
    template <int NT, bool PACK = false>
    __device__ static void step(const W &w, int q, const uint4 (&x)[4][NT], const uint4 (&xl)[4][NT],
                                f32x4 (&acc)[NT]) {
        const float d = f16_to_f32(w.dd & 0xFFFFu), dmin = f16_to_f32(w.dd >> 16);
        // the scale bytes 2 j + q / 2 (j = 0..3) of the half, then sc and m
        // as f16 integers (v_perm_b32 against 0x64: the f16 1024 + v, exact,
        // less 1024)
        const uint32_t b4 = __builtin_amdgcn_perm(w.sc.y, w.sc.x,
                                                  0x06040200u + (uint32_t)(q >> 1) * 0x01010101u);
        const uint32_t sc4 = b4 & 0x0F0F0F0Fu, m4 = (b4 >> 4) & 0x0F0F0F0Fu;
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const f16x2 s01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, sc4, 0x04010400u)) - k1024;
        const f16x2 s23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, sc4, 0x04030402u)) - k1024;
        const f16x2 m01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m4, 0x04010400u)) - k1024;
        const f16x2 m23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m4, 0x04030402u)) - k1024;
        const _Float16 scj[4] = {s01[0], s01[1], s23[0], s23[1]};
        const _Float16 mj[4] = {m01[0], m01[1], m23[0], m23[1]};
        const f16x2 zero = {(_Float16)0.0f, (_Float16)0.0f};
        f16x8 b[4], bm[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t c0 = (w.qs.x >> (2 * j)) & 0x03030303u;
            const uint32_t c1 = (w.qs.y >> (2 * j)) & 0x03030303u;
            const f16x2 sc2 = {scj[j], scj[j]};
            b[j] = dequant_q4x8_f16(c0, c1, false, sc2, zero);
            const _Float16 m = mj[j];
            bm[j] = f16x8{m, m, m, m, m, m, m, m};
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            f32x4 P = {0.f, 0.f, 0.f, 0.f}, M = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                P = mfma16x32(x[j][nt], b[j], P);
                if (!PACK) P = mfma16x32(xl[j][nt], b[j], P);
                M = mfma16x32(x[j][nt], bm[j], M);
                if (!PACK) M = mfma16x32(xl[j][nt], bm[j], M);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[nt][i] = fmaf(-dmin, M[i], fmaf(d, P[i], acc[nt][i]));
        }
    }
};

// IQ2_XXS operands as f16: codebook entry i as 8 f16 magnitudes (8, 25, 43,
// exact), and for each 7-bit sign index the 8 f16 sign bits (its parity as
// the 8th), so a lane's 8 weights are one XOR of two 16-byte table reads.
struct Iq2F16Tables {
    uint32_t grid[256][4];
    uint32_t sign[128][4];
    constexpr Iq2F16Tables() : grid(), sign() {
        constexpr uint32_t f16v[3] = {0x4800u, 0x4E40u, 0x5160u};  // 8, 25, 43
        for (int i = 0; i < 256; i++) {
            uint32_t code = kIq2Codes[i];
            uint32_t h[8] = {};
            for (int j = 0; j < 8; j++) {
                h[j] = f16v[code % 3];
                code /= 3;
            }
            for (int k = 0; k < 4; k++) grid[i][k] = h[2 * k] | h[2 * k + 1] << 16;
        }
        for (uint32_t si = 0; si < 128; si++) {
            uint32_t par = 0;
            for (int b = 0; b < 7; b++) par ^= (si >> b) & 1u;
            const uint32_t s8 = si | par << 7;
            for (int k = 0; k < 4; k++)
                sign[si][k] = ((s8 >> (2 * k)) & 1u) << 15 | ((s8 >> (2 * k + 1)) & 1u) << 31;
        }
    }
};
static __constant__ Iq2F16Tables kIq2F16 = Iq2F16Tables();
// The workgroup's LDS copy (6 KB), staged by MIQ2::stage_tables before the
// first step of a kernel that runs MIQ2::step.
static __shared__ uint4 s_iq2_grid[256];
static __shared__ uint4 s_iq2_sign[128];

// IQ2_XXS (super-tile device layout [qs 8x64 | d 8x2], 528 bytes per 8
// blocks). Step s = sub-groups 4 (s & 1) .. + 3 of block s >> 1, its
// elements in order: MFMA j is sub-group 4 (s & 1) + j (32 elements: 8
// bytes aux0, aux1), lane group q its grid slot q, 8 values from the
// codebook entry aux0 byte q with the sign bits of aux1 bits 7q .. 7q + 6
// (and their parity), each +-{8, 25, 43} (iq2_xxs.rs:66-111), read as f16
// from the tables in LDS; the sub-group's scale db = d (0.5 + (aux1 >> 28)) / 4 is
// exact in fp32 (one FMA: ls d/4 + d/8). B = the value; the step adds
// db_j * P_j.
struct MIQ2 {
    struct W {
        uint4 a[2];  // the step's 4 sub-groups: (aux0, aux1) of 2 per uint4
        uint32_t d;  // f16 d in the low half
    };
    __device__ static int elem(int s, int j, int q) { return 128 * s + 32 * j + 8 * q; }
    __device__ static void piece(int e, int &s, int &j, int &q) {
        s = e >> 7;
        j = (e >> 5) & 3;
        q = (e >> 3) & 3;
    }
    // every thread of the workgroup, before its first step
    __device__ static void stage_tables() {
        for (int i = threadIdx.x; i < 384; i += blockDim.x) {
            if (i < 256)
                s_iq2_grid[i] = *reinterpret_cast<const uint4 *>(kIq2F16.grid[i]);
            else
                s_iq2_sign[i - 256] = *reinterpret_cast<const uint4 *>(kIq2F16.sign[i - 256]);
        }
        __syncthreads();
    }
    __device__ static void load(W &w, __amdgpu_buffer_rsrc_t r, int row, int s, int, int in_dim,
                                int out_dim) {
        const uint32_t nb = (uint32_t)(in_dim >> 8);
        const uint32_t nblk = (uint32_t)out_dim * nb;
        const uint32_t bi = (uint32_t)row * nb + (uint32_t)(s >> 1);
        const uint32_t S = bi >> 3, jb = bi & 7u;
        const uint32_t rS = (S < (nblk >> 3)) ? 8u : (nblk & 7u);
        const uint32_t base = S * 528u, off = base + jb * 64u + 32u * (uint32_t)(s & 1);
        w.a[0] = bload16(r, off, 0);
        w.a[1] = bload16(r, off + 16u, 0);
        w.d = bload2(r, base + rS * 64u + jb * 2u, 0);
    }
    template <int NT, bool PACK = false>
    __device__ static void step(const W &w, int q, const uint4 (&x)[4][NT], const uint4 (&xl)[4][NT],
                                f32x4 (&acc)[NT]) {
        const float d = f16_to_f32(w.d & 0xFFFFu), d4 = d * 0.25f, d8 = d * 0.125f;
        f16x8 b[4];
        float db[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint4 &a = w.a[j >> 1];
            const uint32_t aux0 = (j & 1) ? a.z : a.x, aux1 = (j & 1) ? a.w : a.y;
            db[j] = fmaf((float)(aux1 >> 28), d4, d8);
            const uint4 gv = s_iq2_grid[(aux0 >> (8 * q)) & 0xFFu];
            const uint4 sv = s_iq2_sign[(aux1 >> (7 * q)) & 0x7Fu];
            b[j] = __builtin_bit_cast(f16x8, make_uint4(gv.x ^ sv.x, gv.y ^ sv.y, gv.z ^ sv.z,
                                                        gv.w ^ sv.w));
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 P0 = mfma16x32(x[j][nt], b[j], f32x4{0.f, 0.f, 0.f, 0.f});
                const f32x4 P = PACK ? P0 : mfma16x32(xl[j][nt], b[j], P0);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[nt][i] = fmaf(db[j], P[i], acc[nt][i]);
            }
    }
};

// ---- activation pre-pass ---------------------------------------------------------
// Every activation image has two planes of the same layout: hi = f16(v) and
// lo = f16(v - hi) for v = 2^e x (v - hi is exact in fp32), so hi + lo holds
// v to about 2^-22 relative, and each weight operand meets both planes.
__device__ __forceinline__ void hilo8(const float4 &v0, const float4 &v1, float up, uint4 &hi,
                                      uint4 &lo) {
    const float v[8] = {v0.x * up, v0.y * up, v0.z * up, v0.w * up,
                        v1.x * up, v1.y * up, v1.z * up, v1.w * up};
    f16x8 h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        h[i] = (_Float16)v[i];
        l[i] = (_Float16)(v[i] - (float)h[i]);
    }
    hi = __builtin_bit_cast(uint4, h);
    lo = __builtin_bit_cast(uint4, l);
}

// Scale exponent of a row whose largest magnitude is amax: amax * 2^e in
// [2^14, 2^15) (e clamped to [-126, 126]; 0 for a zero or non-finite amax).
// hilo8 with both roundings toward zero, two values per conversion
// instruction: hi keeps a prefix of v's bits, so v - hi is exact in fp32,
// and hi + lo is within 2^-21 |v| (the one-pass kernel converts its slice of
// the activations in every workgroup, where the conversion's VALU time
// shows).
typedef __fp16 h2rtz __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void hilo8_rtz(const float4 &v0, const float4 &v1, float up, uint4 &hi,
                                          uint4 &lo) {
    const float v[8] = {v0.x * up, v0.y * up, v0.z * up, v0.w * up,
                        v1.x * up, v1.y * up, v1.z * up, v1.w * up};
    uint32_t h[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const h2rtz p = __builtin_amdgcn_cvt_pkrtz(v[2 * k], v[2 * k + 1]);
        h[k] = __builtin_bit_cast(uint32_t, p);
        l[k] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(v[2 * k] - (float)p[0],
                                                                       v[2 * k + 1] - (float)p[1]));
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}
__device__ __forceinline__ int mf_exponent(float amax) {
    int e = 0;
    if (amax > 0.f && amax <= 3.4e38f) {
        int ex;
        frexpf(amax, &ex);  // amax in [2^(ex-1), 2^ex)
        e = min(max(15 - ex, -126), 126);
    }
    return e;
}

__device__ __forceinline__ float max8(const float4 &a, const float4 &b) {
    return fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                 fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w))));
}

// Max over a workgroup of TH threads (every thread gets it); `red`
// holds one float per wavefront.
constexpr int kMfxThreads = 1024;
template <int TH = 1024>
__device__ __forceinline__ float block_max(float m, float *red) {
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int i = 1; i < TH / 64; i++) r = fmaxf(r, red[i]);
    return r;
}

}  // namespace rsllm_hip
