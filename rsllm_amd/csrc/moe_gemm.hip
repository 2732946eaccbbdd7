// Routed experts on the matrix cores, 16 slots of one expert at a time: for a
// batch (up to 16 sorted slots of an expert, moe.hip routing) y[slot, o] =
// sum_i W_e[o, i] x[row(slot), i], with the exact f16 weights and hi + lo
// activations of mfma_formats.h and the per-row activation image of
// gemv_mfma.hip (row r's 8-element pieces in operand order, hi then lo 16
// bytes, from byte 4 r in_dim).
//
// A workgroup of 8 wavefronts covers 512 rows of one expert's matrix and walks
// K in steps of 128 elements; wavefront w owns four row tiles (rows 64 w ..).
// The activations of a step (16 rows x 512 bytes, shared by all wavefronts)
// reach LDS by 16-byte buffer-to-LDS pieces through a ring of three steps. The
// weights are read half a super-tile (1024 elements) at a time into registers,
// four lanes to a row, one half ahead: a row's 256 bytes of codes are
// consecutive loads of one wavefront, so its cache lines are fetched once.
// Block by block (256 elements) they pass through a small LDS buffer of the
// wavefront's own, which hands each lane its row's fields.
//
// (The direct operand loads of mf_rows give neighbouring lanes different rows,
// 64 cache-line lookups an instruction. Copying each block's 64 code bytes,
// scales and d of 512 rows to LDS when it is needed fetched every line up to
// eight times: 4.4 GB from memory for 1.1 GB of weights.)
//
// DS-V4 experts (256 x IQ2_XXS gate/up 2048 x 4096, Q2_K down 4096 x 2048,
// top-6) at 512 tokens: gate/up 688 us, down 358 us, the call 1062 us, against
// 941, 482 and 1480 us on mf_rows (gate/up 803 us before its steps were
// staggered and the loop freed of spilled addresses). Gate/up is bound by the
// vector work of the decode (about 97 instructions per 16 x 128 weights) and
// its table reads. Calls whose workgroups leave CUs idle stay on mf_rows
// (moe_gemm16_fills).
#include <algorithm>
#include <cmath>

#include "mfma_formats.h"
#include "buffer_lds.h"

namespace rsllm_hip {

// IQ2_XXS operand tables in LDS, 16 copies of each entry side by side (lane l
// reads copy l % 16): gathers of random entries without bank conflicts.
constexpr int kXmCopies = 16;
constexpr int kXmTables = (256 + 128) * kXmCopies * 16;
__device__ __forceinline__ void xm_stage_tables(uint4 *tab, int threads) {
#pragma unroll 2
    for (int i = threadIdx.x; i < 384 * kXmCopies; i += threads) {
        const int e = i / kXmCopies;
        tab[i] = e < 256 ? *reinterpret_cast<const uint4 *>(kIq2F16.grid[e])
                         : *reinterpret_cast<const uint4 *>(kIq2F16.sign[e - 256]);
    }
}

// Per format: a lane's share of a row tile's half super-tile. load(): blocks 2 p
// and 2 p + 1 of the half (rp: the row lane / 4's byte offset plus 16 (lane %
// 4); so: the super-tile's offset, half hf); load_aux(): what serves the whole
// half, into the next half's fields (rr: row r16's offset), next(): makes it
// current. put(): block b's bytes into the wavefront's LDS rows (stride 80
// bytes; row lane / 4, piece lane % 4); put_half(): those of the half's scales.
// Then step() adds the MFMAs of step half h of block b (128 elements) and
// fold() closes the block, or step_all() does both for all row tiles.
constexpr int kXmRow = 80;  // LDS bytes per row: 16 rows spread over the banks
template <class F> struct XmFmt;
template <> struct XmFmt<MIQ2> {
    static constexpr bool kSums = false, kTables = true;
    static constexpr int kAux = 1;  // loads of load_aux
    static constexpr int kBuf = 16 * kXmRow;
    __device__ static uint32_t row_bytes(int in_dim) { return (uint32_t)(in_dim >> 11) * 528u; }
    static constexpr uint32_t kTile = 528;
    uint4 qs[4];
    uint2 d, dn;
    __device__ void load(__amdgpu_buffer_rsrc_t r, uint32_t rp, uint32_t so, int hf, int p) {
#pragma unroll
        for (int b = 2 * p; b < 2 * p + 2; b++)
            qs[b] = bload16(r, rp + 64u * (uint32_t)b, so + 256u * (uint32_t)hf);
    }
    __device__ void load_aux(__amdgpu_buffer_rsrc_t r, uint32_t, uint32_t rr, uint32_t so, int hf) {
        dn = bload8(r, rr + 512u, so + 8u * (uint32_t)hf);
    }
    __device__ void next() { d = dn; }
    __device__ void put(uint8_t *buf, int lane, int b) const {
        *reinterpret_cast<uint4 *>(buf + (lane >> 2) * kXmRow + 16 * (lane & 3)) = qs[b];
    }
    // The sub-group scales differ within a step, so each MFMA result is scaled
    // (as MIQ2::step) into P, the block's sum, which joins acc at its end: a
    // chain of 8 and one of in_dim / 256 terms, whose rounding error is that
    // of a K split over four wavefronts. Row tiles go through in units of two
    // MFMA operands, staggered by hand: the records of unit u + 2 and the table
    // entries of u + 1 are read, then u is multiplied and u - 1 scaled. (Left
    // to the compiler every table read and every MFMA was waited for at once.)
    template <int RT>
    __device__ static void step_all(const XmFmt (&w)[RT], const uint8_t *buf, int r16, int q, int b, int h,
                                    const uint4 (&x)[4], const uint4 (&xl)[4], f32x4 (&P)[RT],
                                    f32x4 (&acc)[RT], const uint8_t *tab) {
        constexpr int U = 2 * RT;
        uint4 a[U], gv[U][2], sv[U][2];
        f32x4 S[U][2];
        auto record = [&](int u) {
            a[u] = *reinterpret_cast<const uint4 *>(buf + (u >> 1) * kBuf + r16 * kXmRow + 32 * h + 16 * (u & 1));
        };
        auto gather = [&](int u) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t aux0 = k ? a[u].z : a[u].x, aux1 = k ? a[u].w : a[u].y;
                gv[u][k] = *reinterpret_cast<const uint4 *>(tab + ((aux0 >> (8 * q)) & 0xFFu) * (16 * kXmCopies));
                sv[u][k] = *reinterpret_cast<const uint4 *>(tab + 256 * 16 * kXmCopies +
                                                            ((aux1 >> (7 * q)) & 0x7Fu) * (16 * kXmCopies));
            }
        };
        auto multiply = [&](int u) {
            f16x8 bv[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint4 &g = gv[u][k], &s = sv[u][k];
                bv[k] = __builtin_bit_cast(f16x8, make_uint4(g.x ^ s.x, g.y ^ s.y, g.z ^ s.z, g.w ^ s.w));
            }
#pragma unroll
            for (int k = 0; k < 2; k++) S[u][k] = mfma16x32(x[2 * (u & 1) + k], bv[k], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int k = 0; k < 2; k++) S[u][k] = mfma16x32(xl[2 * (u & 1) + k], bv[k], S[u][k]);
        };
        auto scale = [&](int u) {
            const int rt = u >> 1;
            const float dv = f16_to_f32(((b & 2) ? w[rt].d.y : w[rt].d.x) >> (16 * (b & 1)) & 0xFFFFu);
            const float d4 = dv * 0.25f, d8 = dv * 0.125f;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float db = fmaf((float)((k ? a[u].w : a[u].y) >> 28), d4, d8);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    P[rt][i] = h || (u & 1) || k ? fmaf(db, S[u][k][i], P[rt][i]) : db * S[u][k][i];
            }
            if (h && (u & 1)) acc[rt] += P[rt];
        };
        record(0);
        record(1);
        gather(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u + 2 < U) record(u + 2);
            if (u + 1 < U) gather(u + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(u);
            if (u > 0) scale(u - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        scale(U - 1);
    }
};
// Q2_K: w = d sc q - dmin m per 16-element sub-block. B = 2^-15 sc q: a qs
// byte zero-extended to 16 bits and masked to code j is the f16 subnormal q
// 4^j 2^-24, times sc 2^(9 - 2 j) (exact: sc q <= 45). The mins meet the
// sums of x over each sub-block (f32 sums as hi + lo f16 planes, 2^-4 of
// them, [16 hi | 16 lo] per block after the image): one MFMA per block with
// the 16 m twice along K (as the subnormals 16 m 2^-24), where the m of
// every element would take 16.
template <> struct XmFmt<MQ2K> {
    static constexpr bool kSums = true, kTables = false;
    static constexpr int kAux = 2;
    static constexpr int kBuf = 2 * 16 * kXmRow;  // the block's qs, the half's scales
    __device__ static uint32_t row_bytes(int in_dim) { return (uint32_t)(in_dim >> 11) * 672u; }
    static constexpr uint32_t kTile = 672;
    uint4 qs[4], scp, dd, ddn;
    __device__ void load(__amdgpu_buffer_rsrc_t r, uint32_t rp, uint32_t so, int hf, int p) {
#pragma unroll
        for (int b = 2 * p; b < 2 * p + 2; b++)
            qs[b] = bload16(r, rp + 64u * (uint32_t)b, so + 256u * (uint32_t)hf);
    }
    __device__ void load_aux(__amdgpu_buffer_rsrc_t r, uint32_t rp, uint32_t rr, uint32_t so, int hf) {
        scp = bload16(r, rp + 512u, so + 64u * (uint32_t)hf);
        ddn = bload16(r, rr + 640u, so + 16u * (uint32_t)hf);
    }
    __device__ void next() { dd = ddn; }
    __device__ void put_half(uint8_t *buf, int lane) const {
        *reinterpret_cast<uint4 *>(buf + 16 * kXmRow + (lane >> 2) * kXmRow + 16 * (lane & 3)) = scp;
    }
    __device__ void put(uint8_t *buf, int lane, int b) const {
        *reinterpret_cast<uint4 *>(buf + (lane >> 2) * kXmRow + 16 * (lane & 3)) = qs[b];
    }
    __device__ void step(const uint8_t *buf, int r16, int q, int b, int h, const uint4 (&x)[4],
                         const uint4 (&xl)[4], f32x4 &P) const {
        const uint2 v = *reinterpret_cast<const uint2 *>(buf + r16 * kXmRow + 32 * h + 8 * q);
        const uint2 sc = *reinterpret_cast<const uint2 *>(buf + 16 * kXmRow + r16 * kXmRow + 16 * b + 8 * h);
        // scale bytes 2 j + q / 2, j = 0..3, as f16 sc 2^(9 - 2 j)
        const uint32_t b4 = __builtin_amdgcn_perm(sc.y, sc.x, 0x06040200u + (uint32_t)(q >> 1) * 0x01010101u) &
                            0x0F0F0F0Fu;
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const f16x2 f01 = {(_Float16)512.0f, (_Float16)128.0f}, f23 = {(_Float16)32.0f, (_Float16)8.0f};
        const f16x2 s01 = (__builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, b4, 0x04010400u)) - k1024) * f01;
        const f16x2 s23 = (__builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, b4, 0x04030402u)) - k1024) * f23;
        const uint32_t z[4] = {__builtin_amdgcn_perm(0u, v.x, 0x0c010c00u), __builtin_amdgcn_perm(0u, v.x, 0x0c030c02u),
                               __builtin_amdgcn_perm(0u, v.y, 0x0c010c00u), __builtin_amdgcn_perm(0u, v.y, 0x0c030c02u)};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const f16x2 s2 = j < 2 ? s01 : s23;
            const f16x2 sj = (j & 1) ? s2.yy : s2.xx;
            f16x8 bv;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const f16x2 t = __builtin_bit_cast(f16x2, z[k] & (0x00030003u << (2 * j))) * sj;
                bv[2 * k] = t[0];
                bv[2 * k + 1] = t[1];
            }
            P = mfma16x32(x[j], bv, P);
            P = mfma16x32(xl[j], bv, P);
        }
    }
    __device__ void fold(const uint8_t *buf, int r16, int q, int b, const uint4 &xs, f32x4 &P,
                         f32x4 &acc) const {
        const uint2 mb = *reinterpret_cast<const uint2 *>(buf + 16 * kXmRow + r16 * kXmRow + 16 * b + 8 * (q & 1));
        const uint32_t m0 = mb.x & 0xF0F0F0F0u, m1 = mb.y & 0xF0F0F0F0u;
        const uint4 bm = make_uint4(__builtin_amdgcn_perm(0u, m0, 0x0c010c00u), __builtin_amdgcn_perm(0u, m0, 0x0c030c02u),
                                    __builtin_amdgcn_perm(0u, m1, 0x0c010c00u), __builtin_amdgcn_perm(0u, m1, 0x0c030c02u));
        const f32x4 M = mfma16x32(xs, __builtin_bit_cast(f16x8, bm), f32x4{0.f, 0.f, 0.f, 0.f});
        // P holds 2^-15 of its sum, M 2^-20 2^-4
        const uint32_t dv = sel4(dd, b);
        const float d = f16_to_f32(dv & 0xFFFFu) * 32768.0f, dmin = f16_to_f32(dv >> 16) * 16777216.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] += fmaf(-dmin, M[i], d * P[i]);
        P = f32x4{0.f, 0.f, 0.f, 0.f};
    }
};

constexpr int kXmNW = 8, kXmRT = 4, kXmRows = 16 * kXmRT * kXmNW;
template <class F> struct XmGeo {
    static constexpr int X = 16 * 512;                  // a step's activations: one copy per wavefront
    static constexpr int SN = XmFmt<F>::kSums ? 1 : 0;  // sub-block sums: 16 columns x 256 bytes a half
    static constexpr int S = SN * 4096;
    static constexpr int TAB = XmFmt<F>::kTables ? kXmTables : 0;
    static constexpr int LDS = TAB + 3 * X + 2 * S + kXmNW * kXmRT * XmFmt<F>::kBuf;
};

// Grid (row blocks, batch slots, matrices) as k_gemv_mfgs.
template <class F>
__global__ __launch_bounds__(64 * kXmNW) void k_xm(const uint8_t *__restrict__ w0,
                                                   const uint8_t *__restrict__ w1, size_t w_stride,
                                                   const _Float16 *__restrict__ xh, uint32_t x_bytes,
                                                   const _Float16 *__restrict__ sums, uint32_t s_bytes,
                                                   const float *__restrict__ unscale,
                                                   const int *__restrict__ tok,
                                                   const MfgBatch *__restrict__ bat,
                                                   const int *__restrict__ n_bat,
                                                   float *__restrict__ y0, float *__restrict__ y1,
                                                   int in_dim, int out_dim) {
    extern __shared__ __align__(16) uint8_t smem[];
    using X = XmFmt<F>;
    using G = XmGeo<F>;
    constexpr int RT = kXmRT;
    const int bi = blockIdx.y;
    if (bi >= *n_bat) return;
    const MfgBatch bt = bat[bi];
    const bool m1 = blockIdx.z != 0;
    float *y = (m1 ? y1 : y0) + (size_t)bt.first * out_dim;
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = ((int)blockIdx.x * kXmNW + wv) * (16 * RT);  // this wavefront's rows
    const int nh = in_dim >> 10, ns = 8 * nh;                     // halves, steps
    const __amdgpu_buffer_rsrc_t rw =
        make_rsrc((m1 ? w1 : w0) + (size_t)bt.expert * w_stride, (uint32_t)w_stride);
    const bl_rsrc rx = bl_make_rsrc(xh, x_bytes), rsum = bl_make_rsrc(sums, s_bytes);
    uint8_t *const xbuf = smem + G::TAB;
    uint8_t *const sbuf = xbuf + 3 * G::X;
    uint8_t *const wbuf = sbuf + 2 * G::S + wv * RT * X::kBuf;
    const uint32_t lds_x = bl_lds(xbuf), lds_s = bl_lds(sbuf);

    // Activation copies: wavefront w moves image rows of columns 2 w and 2 w
    // + 1, lane l to slot l % 32 of row l / 32, holding 16-byte piece (l % 32)
    // ^ (row & 15) of the step's 512 bytes (columns past the batch repeat its
    // first; their results are not stored). Sums: wavefront w columns 2 w, 2
    // w + 1 of the half's 256 bytes (lanes 0..31).
    auto image_row = [&](int c) {
        const int slot = bt.first + (c < bt.count ? c : 0);
        return (uint32_t)(tok ? tok[slot] : slot);
    };
    const int xc = 2 * wv + (lane >> 5);
    const uint32_t xrow = image_row(xc);
    const uint32_t xo = xrow * (uint32_t)in_dim * 4u + 16u * (uint32_t)((lane & 31) ^ xc);
    uint32_t so = 0;
    if constexpr (G::SN != 0)
        so = image_row(2 * wv + ((lane >> 4) & 1)) * (uint32_t)(in_dim >> 2) + 16u * (uint32_t)(lane & 15);
    // slot: byte offset of step s's place in the ring, X (s % 3)
    auto dma_x = [&](int s, uint32_t slot) {
        const bl_rsrc r = {rx[0], rx[1], s < ns ? rx[2] : 0u, rx[3]};
        bl_dma16(r, xo, 512u * (uint32_t)s, lds_x + slot + 1024u * (uint32_t)wv);
    };
    auto dma_s = [&](int hb) {
        const bl_rsrc r = {rsum[0], rsum[1], hb < nh ? rsum[2] : 0u, rsum[3]};
        if (lane < 32) bl_dma16(r, so, 256u * (uint32_t)hb, lds_s + (uint32_t)(hb & 1) * 4096u + 512u * (uint32_t)wv);
    };
    // row tile rt's first row (uniform; a tile past the end repeats the last
    // rows, a tile across it starts early), and the lane's place in a tile
    auto tile_row = [&](int rt) { return max(min(row0 + 16 * rt, out_dim - 16), 0); };
    const uint32_t rp = (uint32_t)min(lane >> 2, out_dim - 1) * X::row_bytes(in_dim) + 16u * (uint32_t)(lane & 3);
    const uint32_t rr = (uint32_t)min(r16, out_dim - 1) * X::row_bytes(in_dim);
    X wc[RT];
    // blocks 2 p, 2 p + 1 of half hb, with p = 0 also what serves the half
    auto load_w = [&](int hb, int p) {
        const __amdgpu_buffer_rsrc_t r = hb < nh ? rw : make_rsrc(w0, 0);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const uint32_t so = (uint32_t)tile_row(rt) * X::row_bytes(in_dim) + (uint32_t)(hb >> 1) * X::kTile;
            wc[rt].load(r, rp, so, hb & 1, p);
            if (p == 0) wc[rt].load_aux(r, rp, rr, so, hb & 1);
        }
    };
    dma_x(0, 0);
    dma_x(1, (uint32_t)G::X);
    if constexpr (G::SN != 0) dma_s(0);
    load_w(0, 0);
    load_w(0, 1);
#pragma unroll
    for (int rt = 0; rt < RT; rt++) wc[rt].next();
    if constexpr (X::kTables) xm_stage_tables(reinterpret_cast<uint4 *>(smem), 64 * kXmNW);
    f32x4 acc[RT], P[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) acc[rt] = P[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint8_t *const tab = smem + 16 * (lane & (kXmCopies - 1));
    // slot 2 (4 j + q) + plane of the step, XOR-ed with r16: j / 2 is an
    // offset of 16 slots, j % 2 flips bit 3
    uint32_t xa[2][2];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int l = 0; l < 2; l++) xa[j][l] = 512u * (uint32_t)r16 + 16u * (uint32_t)((8 * j + 2 * q + l) ^ r16);
    // The compiler is kept from seeing through these offsets and the ring's:
    // it would hold every step's sum of them in registers for the whole loop
    // (50 spilled to scratch, reloaded with full waits once a half).
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int l = 0; l < 2; l++) asm("" : "+v"(xa[j][l]));
    uint32_t slot = 0;
    // step i of half hb
    auto step = [&](int hb, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value, b = i >> 1, h = i & 1;
        const int s = 8 * hb + i;
        // landed after this barrier: step s's activations (and the half's
        // sums); the next step's copy and, in the two steps after their
        // issue, the weights of the next half may still be in flight (they
        // are issued after their step's copy: blocks 0, 1 in step 4, 2, 3 in
        // step 7, when their registers are free)
        constexpr int kA = RT * (2 + X::kAux) + G::SN, kB = RT * 2;
        bl_barrier<1 + (i == 5 || i == 6 ? kA : i == 0 || i == 1 ? kB : 0)>();
        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot);
        dma_x(s + 2, slot == 0 ? 2u * (uint32_t)G::X : slot - (uint32_t)G::X);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i == 4) {
            if constexpr (G::SN != 0) dma_s(hb + 1);
            load_w(hb + 1, 0);
        }
        if constexpr (i == 7) load_w(hb + 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (G::SN != 0)
            if constexpr (i == 0)
#pragma unroll
                for (int rt = 0; rt < RT; rt++) wc[rt].put_half(wbuf + rt * X::kBuf, lane);
        if constexpr (h == 0)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) wc[rt].put(wbuf + rt * X::kBuf, lane, b);
        const uint8_t *xs = xbuf + slot;
        slot = slot == 2u * (uint32_t)G::X ? 0u : slot + (uint32_t)G::X;
        uint4 xr[4], xl[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            xr[j] = *reinterpret_cast<const uint4 *>(xs + xa[j & 1][0] + 256 * (j >> 1));
            xl[j] = *reinterpret_cast<const uint4 *>(xs + xa[j & 1][1] + 256 * (j >> 1));
        }
        uint4 sm = make_uint4(0, 0, 0, 0);
        if constexpr (h == 1 && G::SN != 0)
            sm = *reinterpret_cast<const uint4 *>(sbuf + 4096 * (hb & 1) + 256 * r16 + 64 * b + 16 * q);
        if constexpr (X::kTables) {
            X::step_all(wc, wbuf, r16, q, b, h, xr, xl, P, acc, tab);
            if constexpr (i == 7)
#pragma unroll
                for (int rt = 0; rt < RT; rt++) wc[rt].next();
            return;
        } else
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const uint8_t *buf = wbuf + rt * X::kBuf;
            wc[rt].step(buf, r16, q, b, h, xr, xl, P[rt]);
            if constexpr (h == 1) wc[rt].fold(buf, r16, q, b, sm, P[rt], acc[rt]);
            if constexpr (i == 7) wc[rt].next();
            if (rt & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int hb = 0; hb < nh; hb++) {
        step(hb, std::integral_constant<int, 0>{});
        step(hb, std::integral_constant<int, 1>{});
        step(hb, std::integral_constant<int, 2>{});
        step(hb, std::integral_constant<int, 3>{});
        step(hb, std::integral_constant<int, 4>{});
        step(hb, std::integral_constant<int, 5>{});
        step(hb, std::integral_constant<int, 6>{});
        step(hb, std::integral_constant<int, 7>{});
    }
    bl_barrier<0>();
    // D: columns 4 q + 0..3 of row r16
    float us[4];
#pragma unroll
    for (int i = 0; i < 4; i++) us[i] = unscale[image_row(4 * q + i)];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const int o = tile_row(rt) + r16;
        if (row0 + 16 * rt >= out_dim || o >= out_dim) continue;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4 * q + i < bt.count) y[(size_t)(4 * q + i) * out_dim + o] = acc[rt][i] * us[i];
    }
}

template <class F>
static hipError_t xm_go(const uint8_t *w0, const uint8_t *w1, size_t w_stride, const _Float16 *xh,
                        uint32_t x_bytes, const _Float16 *sums, uint32_t s_bytes, const float *us,
                        const int *tok, const MfgBatch *bat, const int *n_bat, int max_b, float *y0,
                        float *y1, int in_dim, int out_dim, hipStream_t s) {
    constexpr int LDS = XmGeo<F>::LDS;
    static_assert(LDS <= 160 * 1024, "one workgroup's LDS");
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void *>(&k_xm<F>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (attr != hipSuccess) return attr;
    const dim3 g((unsigned)((out_dim + kXmRows - 1) / kXmRows), (unsigned)max_b, w1 ? 2u : 1u);
    k_xm<F><<<g, 64 * kXmNW, LDS, s>>>(w0, w1, w_stride, xh, x_bytes, sums, s_bytes, us, tok, bat,
                                       n_bat, y0, y1, in_dim, out_dim);
    return hipGetLastError();
}

// One workgroup fits a CU and takes the same time whether or not the others are
// busy, so this kernel pays once most CUs of every round have one: against
// k_gemv_mfg, by workgroups per round of 256 CUs (kernel times, us; IQ2_XXS
// gate/up of K 4096: 16: 20 -> 60, 64: 44 -> 65, 96: 52 -> 66, 128: 65 -> 68,
// 144: 74 -> 68, 192: 85 -> 73, 234: 98 -> 73; two rounds of 144: 126 -> 140, of
// 192: 169 -> 145, of 256: 209 -> 158; Q2_K down of K 2048: 64: 22 -> 32, 128: 32
// -> 33, 144: 38 -> 34, 192: 45 -> 35; K 8192 the same by the round). The line
// is where all of the traced shapes win or are level: seven tenths of the CUs
// for IQ2_XXS, whose workgroups also stage the tables (three rounds of 172, 64
// experts of 2048 x 2048 at 9 slots: the call 191 -> 207; of 184: 233 -> 197 for
// the gate/up of 8 experts at 130), six tenths for Q2_K. The number of batches
// is known on the device alone; this is what slots dealt evenly at random make:
// with m a mean expert's slots, m / 16 batches and half of one more each, and
// below 18 slots, where few experts have a second batch, about 1 + (m - 8)^2 /
// 150.
bool moe_gemm16_fills(uint32_t dtype, int in_dim, int out_dim, int mats, int n_pairs, int n_expert) {
    if ((dtype != T_IQ2_XXS && dtype != T_Q2_K) || in_dim % 2048 != 0) return false;
    const double m = (double)n_pairs / n_expert;
    const double batches = n_expert * std::min(m / 16 + 0.5, 1 + (m - 8) * (m - 8) / 150);
    const double wgs = batches * ((out_dim + kXmRows - 1) / kXmRows) * mats;
    const double cus = device_cus();
    return wgs >= (dtype == T_IQ2_XXS ? 0.7 : 0.6) * cus * std::ceil(wgs / cus);
}

hipError_t launch_moe_gemm16(uint32_t dtype, const uint8_t *w0, const uint8_t *w1, size_t w_stride,
                             const void *xh, size_t x_bytes, const void *sums, size_t s_bytes,
                             const float *us, const int *tok, const MfgBatch *bat, const int *n_bat,
                             int max_b, float *y0, float *y1, int in_dim, int out_dim,
                             hipStream_t s) {
    if (w_stride > 0xFFFFFF00u || x_bytes > 0xFFFFFFFFu || s_bytes > 0xFFFFFFFFu ||
        in_dim % 2048 != 0 || (moe_gemm_sums(dtype) && !sums) ||
        (((uintptr_t)w0 | (uintptr_t)(w1 ? w1 : w0) | (uintptr_t)w_stride) & 15) != 0)
        return hipErrorNotSupported;
    const _Float16 *x = static_cast<const _Float16 *>(xh), *sm = static_cast<const _Float16 *>(sums);
    switch (dtype) {
    case T_IQ2_XXS:
        return xm_go<MIQ2>(w0, w1, w_stride, x, (uint32_t)x_bytes, sm, (uint32_t)s_bytes, us, tok,
                           bat, n_bat, max_b, y0, y1, in_dim, out_dim, s);
    case T_Q2_K:
        return xm_go<MQ2K>(w0, w1, w_stride, x, (uint32_t)x_bytes, sm, (uint32_t)s_bytes, us, tok,
                           bat, n_bat, max_b, y0, y1, in_dim, out_dim, s);
    default: return hipErrorNotSupported;
    }
}

}  // namespace rsllm_hip
