// Matrix-core GEMM with exact weights for many tokens: y[t, o] = sum_i
// W[o, i] x[t, i] where each 16-row weight tile is decoded once for up to 48
// token columns. The weights are the exact f16 integers of mfma_formats.h
// with their fp32 scales, the activations hi + lo f16 planes (about 2^-22
// relative), as in the batched GEMV (gemv_mfma.hip), whose 16- and 32-token
// passes decode every weight and stream every row again per pass.
//
// 1. k_xg_rows: a per-row activation image. Row r's 8-element pieces in MFMA
//    operand order, scaled by 2^e_r: piece p's hi 16 bytes at byte 4 r in_dim
//    + 32 p, its lo 16 bytes after them, unscale[r] = 2^-e_r.
// 2. k_xg: a workgroup of 16 wavefronts covers 256 rows x 16 NT columns in
//    steps of 64 elements. Wavefront w holds two row tiles (rows 32 (w & 7)
//    ..) for all columns and 32 elements of each step (K group w >> 3): four
//    wavefronts per SIMD, since one alone issues vector work at about half
//    rate and the decode and the block scales need as much as the MFMAs.
//    Weights (raw bytes) and activations reach LDS by 16-byte buffer-to-LDS
//    pieces: the activations through a ring of four steps, the
//    weights one 256-element tile at a time (a row's tile is one contiguous
//    run: few cache lines per instruction), which every wavefront reads into
//    registers a step before it needs it, so the buffer takes the next tile
//    while this one is computed. A step's operands are decoded during the
//    step before. The K groups' sums are added through LDS at the end.
//
// 8 x [1024 x 4096] Q8_0 at 300 tokens, kernel trace over three sets of
// operands in turn: 78 us (72 at best; 40 GFLOP counting both planes, 0.51
// PFLOP/s) after 17 us for the image (39 MB read and 79 MB written, part of it
// in the last-level cache), against 197 + 38 us for the 16-token passes. Calls
// one after the other overlap at their ends: 82 us each (74 on one set of
// operands). What bounds it: per 32 x 16 x 16 products two MFMAs (32 cycles),
// 4 FMAs for the block scales and a share of the decode, with the copies and
// the LDS reads of the activations beside them.
//
// (Tried on that shape, before the tile sums, when the kernel's trace read 74
// us: the weights straight to the operand registers, each
// lane its own row, 107 us: neighbouring lanes hit 64 different lines per
// instruction. Both through two buffers of 128 elements, 76 us; both through
// a ring of four 64-element steps, 89 us: a row's 64 bytes and its scales per
// step touch three times the lines of a whole tile. 8 wavefronts of four row
// tiles, 77 us.)
#include "buffer_lds.h"
#include "mfma_formats.h"

namespace rsllm_hip {

// Per format: a row's tile of 256 elements is PR 16-byte pieces (PR odd, so
// 16 rows at a stride of PR pieces start on distinct LDS bank groups). The
// lane (row r16, lane group q) of K group kg reads its raw bytes of a tile
// (elements 64 u + 32 kg + 8 q .. + 7 of steps u = 0..3) with load(); op(u)
// is step u's MFMA operand (exact f16 integers), scale(u) its fp32 factor.
template <class F> struct XgFmt;
template <> struct XgFmt<MQ8> {
    static constexpr int PR = 17;  // super-tile [qs 8x32 | d 8x2]
    uint2 v[4];
    uint4 d;
    __device__ void load(const uint8_t *row, int kg, int q) {
#pragma unroll
        for (int u = 0; u < 4; u++)
            v[u] = *reinterpret_cast<const uint2 *>(row + 64 * u + 32 * kg + 8 * q);
        d = *reinterpret_cast<const uint4 *>(row + 256);
    }
    __device__ f16x8 op(int u) const {
        const f16x2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
        f16x8 r;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t bb = (i ? v[u].y : v[u].x) ^ 0x80808080u;
            const f16x2 w01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, bb, 0x04010400u)) - bias;
            const f16x2 w23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, bb, 0x04030402u)) - bias;
            r[4 * i] = w01[0];
            r[4 * i + 1] = w01[1];
            r[4 * i + 2] = w23[0];
            r[4 * i + 3] = w23[1];
        }
        return r;
    }
    __device__ float scale(int u, int kg) const {
        return f16_to_f32((sel4(d, u) >> (16 * kg)) & 0xFFFFu);
    }
};

struct XgShape {
    int in_dim;
    int n_cols;      // columns (tokens)
    int groups;      // row groups: group g's rows read image rows c * groups + g
    int group_rows;
    int y_stride;
    uint32_t x_bytes;  // of the image
    uint32_t w_bytes;
};

// Bytes between image rows: a row's hi and lo planes and 256 bytes, so the
// rows of a token tile start in different L2 channels (in_dim is often a
// power of two; without the pad a step's token rows all come from one channel).
__host__ __device__ inline uint32_t xg_row_bytes(int in_dim) { return (uint32_t)in_dim * 4u + 256u; }

constexpr int kXgRows = 256;
constexpr int kXgRing = 4;  // (step s uses slot s % 4: its place within the tile)
constexpr int kXgRT = 2;                              // row tiles per wavefront
constexpr int kXgWR = kXgRows / (16 * kXgRT);         // wavefronts over the rows
constexpr int kXgWaves = 2 * kXgWR;
template <class F, int NT> struct XgGeo {
    static constexpr int PR = XgFmt<F>::PR;
    static constexpr int WN = kXgRows * PR / 64, WI = (WN + kXgWaves - 1) / kXgWaves;  // weight copies per tile, per wavefront
    static constexpr int XN = 4 * NT, XI = (XN + kXgWaves - 1) / kXgWaves;  // activation copies per step
    static constexpr int W = kXgRows * PR * 16;
    static constexpr int X = 16 * NT * 256;
    static constexpr int H0 = (kXgRT * NT + 1) / 2;  // exchanged tiles per wavefront
    static constexpr int XCH = kXgWaves * H0 * 1024;
    static constexpr int LDS = W + kXgRing * X > XCH ? W + kXgRing * X : XCH;
};

template <class F, int NT>
__global__ __launch_bounds__(64 * kXgWaves) void k_xg(const uint8_t *__restrict__ w,
                                               const _Float16 *__restrict__ xh,
                                               const float *__restrict__ unscale,
                                               float *__restrict__ y, XgShape sh, int n_tiles) {
    extern __shared__ __align__(16) uint8_t smem[];
    using X = XgFmt<F>;
    using G = XgGeo<F, NT>;
    constexpr int RT = kXgRT;
    // tile order: row blocks of a group's token tile side by side, and an
    // eighth of the tiles per XCD (workgroups are dealt to the XCDs in turn)
    const int per = (int)gridDim.x >> 3;
    const int tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (tile >= n_tiles) return;
    const int rbs = (sh.group_rows + kXgRows - 1) / kXgRows;
    const int tts = (sh.n_cols + 16 * NT - 1) / (16 * NT);
    const int rb = tile % rbs, tg = tile / rbs, tt = tg % tts, g = tg / tts;
    const int row0 = g * sh.group_rows + rb * kXgRows, row_end = (g + 1) * sh.group_rows;
    const int col0 = tt * 16 * NT;

    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wv & (kXgWR - 1), kg = wv / kXgWR;
    const int nt256 = sh.in_dim / 256, ns = 4 * nt256;  // tiles, steps
    const bl_rsrc rw = bl_make_rsrc(w, sh.w_bytes), rx = bl_make_rsrc(xh, sh.x_bytes);
    const uint32_t lds0 = bl_lds(smem);
    const uint8_t *const wbuf = smem + kXgRing * G::X;  // after the activations' ring

    // Copies, the same number from every wavefront (those past the last
    // repeat it). Weights: instruction i moves pieces 64 i + lane of the tile
    // (piece j: row j / PR, piece j % PR; rows past the group's end repeat
    // its last). Activations: instruction i moves token rows 4 i .. + 3, lane
    // l to slot l % 16 of row l / 16, which holds 16-byte piece (l % 16) ^
    // (row & 15), so the operand reads of 16 tokens spread over all banks.
    // Steps and tiles past the end copy nothing (an empty
    // resource) but count as issued, so the waits below stay the same.
    uint32_t wo[G::WI], xo[G::XI];
#pragma unroll
    for (int p = 0; p < G::WI; p++) {
        const int j = 64 * min(wv + kXgWaves * p, G::WN - 1) + lane, row = j / G::PR, k = j - row * G::PR;
        wo[p] = (uint32_t)min(row0 + row, row_end - 1) * (uint32_t)nt256 * (16u * G::PR) + 16u * (uint32_t)k;
    }
#pragma unroll
    for (int p = 0; p < G::XI; p++) {
        const int tr = 4 * min(wv + kXgWaves * p, G::XN - 1) + (lane >> 4);
        const int c = min(col0 + tr, sh.n_cols - 1);
        xo[p] = (uint32_t)(c * sh.groups + g) * xg_row_bytes(sh.in_dim) +
                16u * (uint32_t)((lane & 15) ^ (tr & 15));
    }
    auto dma_w = [&](int t) {
        const bl_rsrc r = {rw[0], rw[1], t < nt256 ? rw[2] : 0u, rw[3]};
#pragma unroll
        for (int p = 0; p < G::WI; p++)
            bl_dma16(r, wo[p], (uint32_t)t * (16u * G::PR),
                     lds0 + (uint32_t)(kXgRing * G::X) + 1024u * (uint32_t)min(wv + kXgWaves * p, G::WN - 1));
    };
    auto dma_x = [&](int s) {
        const uint32_t dst = lds0 + (uint32_t)((s & (kXgRing - 1)) * G::X);
        const bl_rsrc r = {rx[0], rx[1], s < ns ? rx[2] : 0u, rx[3]};
#pragma unroll
        for (int p = 0; p < G::XI; p++)
            bl_dma16(r, xo[p], 256u * (uint32_t)s,
                     dst + 1024u * (uint32_t)min(wv + kXgWaves * p, G::XN - 1));
    };
    f32x4 acc[RT][NT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[rt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int slot = 8 * kg + 2 * q;
    const uint8_t *const xhi = smem + 256 * r16 + 16 * (slot ^ r16);
    const uint8_t *const xlo = smem + 256 * r16 + 16 * ((slot + 1) ^ r16);
    auto read_x = [&](int u, int nt, uint4 &hi, uint4 &lo) {
        hi = *reinterpret_cast<const uint4 *>(xhi + u * G::X + 4096 * nt);
        lo = *reinterpret_cast<const uint4 *>(xlo + u * G::X + 4096 * nt);
    };
    // A step has two phases: the MFMAs (their results kept in P), and the
    // vector work (P times the block scales into acc, the next operands'
    // decode). A vector instruction does not issue beside an MFMA of its own
    // wavefront, so the K groups run them in opposite order: on every SIMD
    // one wavefront feeds the matrix core while the other does vector work.
    // Group 0: MFMAs of step s, fold s, decode s + 1. Group 1: fold s - 1,
    // decode s, MFMAs of step s.
    auto run = [&](auto kg_c) __attribute__((always_inline)) {
        constexpr int KG = decltype(kg_c)::value;
        X raw[RT];
        f16x8 b[RT];
        float d[RT];
        f32x4 P[NT][RT];
        uint4 hi0, lo0;  // the next token tile to multiply
        auto load_raw = [&]() {
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
                raw[rt].load(wbuf + (16 * RT * wr + 16 * rt + r16) * (16 * G::PR), KG, q);
        };
        auto decode = [&](int u) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                b[rt] = raw[rt].op(u);
                d[rt] = raw[rt].scale(u, KG);
            }
        };
        // A tile's sum, added to acc at its end: chains of 4 and of in_dim /
        // 256 terms round like a K split over four wavefronts (in_dim 4096:
        // error against 64 bits 1.2e-7, one chain 1.6e-7, the
        // 16-token passes 1.3e-7).
        f32x4 part[RT][NT];
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) part[rt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto fold = [&](int u) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float v = u == 0 ? d[rt] * P[nt][rt][i]
                                               : fmaf(d[rt], P[nt][rt][i], part[rt][nt][i]);
                        if (u == 3) acc[rt][nt][i] += v;
                        else part[rt][nt][i] = v;
                    }
        };
        auto mfmas = [&](int u) {
            uint4 hi = hi0, lo = lo0;
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint4 h = hi, l = lo;
                if (nt + 1 < NT) read_x(u, nt + 1, hi, lo);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    P[nt][rt] = mfma16x32(h, b[rt], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int rt = 0; rt < RT; rt++) P[nt][rt] = mfma16x32(l, b[rt], P[nt][rt]);
            }
        };
        auto step = [&](int s, auto u_c) __attribute__((always_inline)) {
            constexpr int u = decltype(u_c)::value;
            // landed after this barrier: step s + 1's activations, and before
            // the tile's last step the next tile's weights; newer copies may
            // still be in flight. (Order of issue: steps' activations, a
            // tile's weights after those issued in its first step.)
            bl_barrier<(u == 1 || u == 2) ? G::XI + G::WI : G::XI>();
            dma_x(s + 3);
            if constexpr (u == 0) dma_w((s >> 2) + 1);
            if constexpr (KG == 0) {
                if constexpr (u == 3) load_raw();
                mfmas(u);
                __builtin_amdgcn_sched_barrier(0);
                read_x((u + 1) & 3, 0, hi0, lo0);
                fold(u);
                decode((u + 1) & 3);
            } else {
                read_x(u, 0, hi0, lo0);
                fold((u + 3) & 3);
                decode(u);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (u == 3) load_raw();
                mfmas(u);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        load_raw();
        if constexpr (KG == 0) {
            read_x(0, 0, hi0, lo0);
            decode(0);
        } else {
#pragma unroll
            for (int rt = 0; rt < RT; rt++) d[rt] = 0.f;
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int rt = 0; rt < RT; rt++) P[nt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int t = 0; t < nt256; t++) {
            step(4 * t, std::integral_constant<int, 0>{});
            step(4 * t + 1, std::integral_constant<int, 1>{});
            step(4 * t + 2, std::integral_constant<int, 2>{});
            step(4 * t + 3, std::integral_constant<int, 3>{});
        }
        if constexpr (KG == 1) fold(3);
    };

    dma_w(0);
    dma_x(0);
    dma_x(1);
    dma_x(2);
    bl_barrier<2 * G::XI>();
    if (kg == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    bl_barrier<0>();
    // the K groups' sums: group 0 keeps the lower half of each wavefront's
    // (row tile, column tile) pairs, group 1 the upper
    constexpr int PAIRS = RT * NT, H0 = G::H0;
    f32x4 *xch = reinterpret_cast<f32x4 *>(smem);
    auto slot_of = [&](int grp, int i) { return ((grp * kXgWR + wr) * H0 + i) * 64 + lane; };
#pragma unroll
    for (int i = 0; i < PAIRS; i++) {
        if (i < H0 && kg == 1) xch[slot_of(0, i)] = acc[i / NT][i % NT];
        if (i >= H0 && kg == 0) xch[slot_of(1, i - H0)] = acc[i / NT][i % NT];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PAIRS; i++) {
        if ((i < H0) != (kg == 0)) continue;
        const f32x4 v = acc[i / NT][i % NT] + xch[i < H0 ? slot_of(0, i) : slot_of(1, i - H0)];
        const int o = row0 + 16 * RT * wr + 16 * (i / NT) + r16;
        if (o >= row_end) continue;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = col0 + 16 * (i % NT) + 4 * q + k;
            if (c < sh.n_cols)
                y[(size_t)c * sh.y_stride + o] = v[k] * unscale[c * sh.groups + g];
        }
    }
}

// One workgroup of 256 threads per image row (in_dim a multiple of 256): the
// row is read once (up to 4 pieces of 8 elements a thread; longer rows
// twice), in whole cache lines both ways.
template <class F>
__global__ __launch_bounds__(256) void k_xg_rows(const float *__restrict__ x,
                                                 _Float16 *__restrict__ xh,
                                                 float *__restrict__ unscale, int in_dim) {
    __shared__ float red[4];
    constexpr int C = 4;
    const size_t r = blockIdx.x;
    const int tid = threadIdx.x, n8 = in_dim >> 3;
    const float4 *xt = reinterpret_cast<const float4 *>(x + r * in_dim);
    uint4 *ht = reinterpret_cast<uint4 *>(xh + r * (xg_row_bytes(in_dim) / 2));
    const bool cached = n8 <= 256 * C;
    float4 c[C][2];
    float m = 0.f;
    if (cached) {
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int i = tid + 256 * k;
            if (i < n8) {
                c[k][0] = xt[2 * i];
                c[k][1] = xt[2 * i + 1];
                m = fmaxf(m, max8(c[k][0], c[k][1]));
            }
        }
    } else {
        for (int i = tid; i < n8; i += 256) m = fmaxf(m, max8(xt[2 * i], xt[2 * i + 1]));
    }
    const int e = mf_exponent(block_max<256>(m, red));
    const float up = ldexpf(1.0f, e);
    if (tid == 0) unscale[r] = ldexpf(1.0f, -e);
    auto store = [&](int i, const float4 &a, const float4 &b) {
        int s, j, q;
        F::piece(8 * i, s, j, q);
        uint4 hi, lo;
        hilo8(a, b, up, hi, lo);
        uint4 *p = ht + 2 * ((s * 4 + j) * 4 + q);
        p[0] = hi;
        p[1] = lo;
    };
    if (cached) {
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int i = tid + 256 * k;
            if (i < n8) store(i, c[k][0], c[k][1]);
        }
    } else {
        for (int i = tid; i < n8; i += 256) store(i, xt[2 * i], xt[2 * i + 1]);
    }
}

template <class F, int NT>
static hipError_t xg_go(const uint8_t *w, const _Float16 *xh, const float *us, float *y,
                        const XgShape &sh, hipStream_t s) {
    constexpr int LDS = XgGeo<F, NT>::LDS;
    static_assert(LDS <= 160 * 1024, "one workgroup's LDS");
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void *>(&k_xg<F, NT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (attr != hipSuccess) return attr;
    const long tiles = (long)sh.groups * ((sh.group_rows + kXgRows - 1) / kXgRows) *
                       ((sh.n_cols + 16 * NT - 1) / (16 * NT));
    if (tiles > (1 << 28)) return hipErrorInvalidValue;
    k_xg<F, NT><<<(unsigned)((tiles + 7) / 8 * 8), 64 * kXgWaves, LDS, s>>>(w, xh, us, y, sh, (int)tiles);
    return hipGetLastError();
}

// Column tiles per workgroup: the fewest (rounds of one workgroup per CU) x
// (work of one), counting one column tile's time for what a workgroup does
// whatever its width. That picked the faster of the two in all of 158 measured
// calls (3 to 16 groups, K of 512 to 4096, 256 to 1000 tokens): 8 x [1024 x
// 4096] at 256 / 300 / 400 / 640 tokens two tiles 63 / 109 / 115 / 174 us, three
// 69 / 73 / 132 / 148. Four do not fit the registers beside the tile sums (65
// spilled); with one chain of sums instead they served 16 x [512 x 1024] at
// 400 tokens in 34 us (three: 42 us, the 16-token passes 76 us) at an error
// above the passes' own (1.1e-7 against 9.9e-8; now 9.6e-8).
template <class F>
static hipError_t xg_launch(const uint8_t *w, const float *x, uint8_t *scratch, float *y,
                            const XgShape &sh, hipStream_t s) {
    const size_t rows = (size_t)sh.n_cols * sh.groups;
    _Float16 *xh = reinterpret_cast<_Float16 *>(scratch);
    float *us = reinterpret_cast<float *>(scratch + rows * xg_row_bytes(sh.in_dim));
    k_xg_rows<F><<<(unsigned)rows, 256, 0, s>>>(x, xh, us, sh.in_dim);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const long cus = device_cus();
    int best = 3;
    long cost = -1;
    for (int nt = 3; nt >= 2; nt--) {
        const long tiles = (long)sh.groups * ((sh.group_rows + 255) / 256) *
                           ((sh.n_cols + 16 * nt - 1) / (16 * nt));
        const long c = (tiles + cus - 1) / cus * (nt + 1);
        if (cost < 0 || c < cost) {
            cost = c;
            best = nt;
        }
    }
    switch (best) {
    case 2: return xg_go<F, 2>(w, xh, us, y, sh, s);
    default: return xg_go<F, 3>(w, xh, us, y, sh, s);
    }
}

size_t gemm_exact_scratch_bytes(int n_tok, int in_dim, int groups) {
    const size_t rows = (size_t)n_tok * groups;
    return rows * xg_row_bytes(in_dim) + rows * 4;
}

bool gemm_exact_supported(uint32_t dtype, const uint8_t *w, size_t w_bytes, const float *x,
                          int n_tok, int in_dim, int groups, int group_rows) {
    return dtype == T_Q8_0 && n_tok > 0 && in_dim > 0 && in_dim % 256 == 0 && group_rows > 0 &&
           (size_t)n_tok * groups * xg_row_bytes(in_dim) <= 0x7FFFFFFFu && w_bytes <= 0xFFFFFF00u &&
           (((uintptr_t)w | (uintptr_t)x) & 15) == 0;
}

hipError_t launch_gemm_exact(uint32_t dtype, const uint8_t *w, size_t w_bytes, const float *x,
                             uint8_t *scratch, float *y, int n_tok, int in_dim, int groups,
                             int group_rows, int y_stride, hipStream_t s) {
    if (!gemm_exact_supported(dtype, w, w_bytes, x, n_tok, in_dim, groups, group_rows))
        return hipErrorNotSupported;
    const XgShape sh{in_dim, n_tok, groups, group_rows, y_stride,
                     (uint32_t)((size_t)n_tok * groups * xg_row_bytes(in_dim)), (uint32_t)w_bytes};
    return xg_launch<MQ8>(w, x, scratch, y, sh, s);
}

}  // namespace rsllm_hip
