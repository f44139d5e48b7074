// gemm_rows.hip -- fp32-activation quant matmul for M > 1, bit-identical to TR's CPU order.
//
// tensor/cpu_quant.go:103-147 (quantGemmPanels) and the tile path (:59-82, gemmPart in
// cpu_matmul.go:330-380) both compute, for every output (m, n): for each 256-deep K chunk a fresh
// fused chain from +0 in ascending k (sgemm6x16, cpu_micro_amd64.s:14-64), the chunk results added
// in chunk order into a cleared `part`, then c[m, n] += part.
//
// Mapping: a wave is 64 weight rows (lane = row) on one 256-deep chunk. It decodes its rows' weights 32 elements at
// a time, exactly as tensor/quant.go does, and advances the chains of up to 16 activation rows with K = 1 matrix
// instructions, each of whose outputs is one fused multiply-add. A wave's 64 row images of a chunk are loaded with
// whole cache lines per instruction and staged in LDS, where each lane reads its own row back; the activations of a
// group are staged the same way. A workgroup is kStageWaves (or, for grids of few row blocks, 4) such waves on
// consecutive chunks of the same 64 rows. Their chain results are added to `part` in chunk order in LDS, or, when
// the chunks of a row block are split over several workgroups, written out per chunk and added in chunk order by
// a second kernel.
#include "trhip_internal.hpp"

#include <type_traits>

namespace trhip {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
// Plain vector types for registers carried across loop iterations (the HIP uint4 / float4 structs are copied with
// memcpy, which keeps them in private memory there).
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kStageWaves = 8;  // chunk-waves per workgroup when one workgroup covers a row block's chunks
constexpr int kSplitWaves = 4;  // chunk-waves per workgroup when a row block's chunks are split over workgroups
constexpr int kXPitch = 36;     // floats per activation row of a staged 32-wide group: rows land on distinct banks
constexpr int kRPitch = 68;     // floats per row of a wave's 16 x 64 chain results

// f(integral_constant<int, I>) for I = B .. E - 1, so that loop indices are constants in the body.
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// 32 consecutive elements (group G of a 32-element grid along the row) of one block, decoded exactly as
// tensor/quant.go:139-205.
template <int DT>
struct Group;

template <>
struct Group<kQ8> {
    uint4 a, b;
    uint32_t d;
    __device__ __forceinline__ void decode(int, float y[32]) const {
        const float dv = f16_to_f32((uint16_t)d), nd = -128.0f * dv;  // q*d = d*(u - 128), u = q + 128: exact
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t u = opaque(w[i] ^ 0x80808080u);
#pragma unroll
            for (int k = 0; k < 4; k++) y[4 * i + k] = fmaf(dv, ubyte_f(u, k), nd);
        }
    }
};

template <>
struct Group<kQ4> {
    uint4 a;
    uint32_t d;
    __device__ __forceinline__ void decode(int, float y[32]) const {
        const float dv = f16_to_f32((uint16_t)d), n8 = -8.0f * dv;  // (q - 8)*d, exact
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = opaque(w[i] & 0x0F0F0F0Fu), hi = opaque((w[i] >> 4) & 0x0F0F0F0Fu);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                y[4 * i + k] = fmaf(dv, ubyte_f(lo, k), n8);
                y[16 + 4 * i + k] = fmaf(dv, ubyte_f(hi, k), n8);
            }
        }
    }
};

template <>
struct Group<kQ4K> {
    uint4 h, a, b;
    __device__ __forceinline__ void decode(int j, float y[32]) const {
        uint32_t sc_lo, sc_hi, m_lo, m_hi;
        q4k_scales(h.y, h.z, h.w, sc_lo, sc_hi, m_lo, m_hi);
        const int sh = 8 * (j & 3);
        const float d = f16_to_f32((uint16_t)(h.x & 0xFFFF)), dmin = f16_to_f32((uint16_t)(h.x >> 16));
        const float d1 = d * (float)(((j < 4 ? sc_lo : sc_hi) >> sh) & 0xFF);
        const float m1 = dmin * (float)(((j < 4 ? m_lo : m_hi) >> sh) & 0xFF);
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t nib = opaque((j & 1) ? (w[i] >> 4) & 0x0F0F0F0Fu : w[i] & 0x0F0F0F0Fu);
#pragma unroll
            for (int k = 0; k < 4; k++) y[4 * i + k] = fmaf(d1, ubyte_f(nib, k), -m1);  // d1*q exact: one rounding
        }
    }
};

template <>
struct Group<kQ6K> {
    uint2 ql[4], qh[4];
    uint32_t d, sc;  // sc: the two int8 scales of the group's halves
    __device__ __forceinline__ void decode(int G, float y[32]) const {
        const int k4 = G & 3;
        const float dv = f16_to_f32((uint16_t)d);
        const float s0 = dv * (float)(int8_t)(sc & 0xFF), s1 = dv * (float)(int8_t)(sc >> 8);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t lw[2] = {ql[t].x, ql[t].y}, hw[2] = {qh[t].x, qh[t].y};
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                const uint32_t nib = (k4 < 2) ? (lw[hh] & 0x0F0F0F0Fu) : ((lw[hh] >> 4) & 0x0F0F0F0Fu);
                const uint32_t code = opaque(nib | (((hw[hh] >> (2 * k4)) & 0x03030303u) << 4));
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int e = 8 * t + 4 * hh + k;
                    y[e] = (e < 16 ? s0 : s1) * (ubyte_f(code, k) - 32.0f);  // fl(fl(d*sc) * (q - 32))
                }
            }
        }
    }
};

// A weight row's bytes for one 256-wide chunk, as the 16-byte pieces of an LDS image. A wave loads the 64 rows'
// images with consecutive lanes on consecutive pieces of a row (whole cache lines per instruction) and then reads
// its own row back, a lane per row. kPitch (bytes per row image) keeps 16 consecutive rows on distinct LDS banks.
template <int DT>
struct Image;

template <>
struct Image<kQ8> {  // 8 blocks x 32 codes, then the 8 fp16 scales
    static constexpr int kPieces = 16, kPitch = 272, kScaleOff = 256, kBlocks = 8;
    __device__ static const uint8_t *piece(const Planes &p, int64_t b0, int q) { return p.qs + b0 * 32 + 16 * q; }
    __device__ static int piece_block(int q) { return q >> 1; }
};

template <>
struct Image<kQ4> {  // 8 blocks x 16 code bytes, then the 8 fp16 scales
    static constexpr int kPieces = 8, kPitch = 144, kScaleOff = 128, kBlocks = 8;
    __device__ static const uint8_t *piece(const Planes &p, int64_t b0, int q) { return p.qs + b0 * 16 + 16 * q; }
    __device__ static int piece_block(int q) { return q; }
};

template <>
struct Image<kQ4K> {  // the lane-sliced qs block (128), then the header d, dmin, scales (16)
    static constexpr int kPieces = 9, kPitch = 144, kScaleOff = -1, kBlocks = 1;
    __device__ static const uint8_t *piece(const Planes &p, int64_t b0, int q) {
        return q < 8 ? p.qs + b0 * 128 + 16 * q : p.aux + b0 * 16;
    }
    __device__ static int piece_block(int) { return 0; }
};

template <>
struct Image<kQ6K> {  // ql (128), qh (64), the 16 int8 scales (16); d stays in a register
    static constexpr int kPieces = 13, kPitch = 208, kScaleOff = -1, kBlocks = 1;
    __device__ static const uint8_t *piece(const Planes &p, int64_t b0, int q) {
        return q < 8 ? p.qs + b0 * 128 + 16 * q : q < 12 ? p.aux + b0 * 64 + 16 * (q - 8) : p.sc + b0 * 16;
    }
    __device__ static int piece_block(int) { return 0; }
};

// One wave's staging registers for the images of 64 rows: piece P = 64 i + lane is piece P % kPieces of row
// P / kPieces. Blocks past the end of a row (a short last chunk of q8_0 / q4_0) are neither loaded nor read.
template <int DT>
struct Stage {
    using I = Image<DT>;
    static constexpr int kScales = I::kScaleOff >= 0 ? 8 : 0;
    u32x4 w[I::kPieces];
    uint32_t s[kScales > 0 ? kScales : 1];
    uint32_t d6;  // q6_k: the fp16 scale of the lane's own row
    __device__ __forceinline__ void load(const Planes &p, int64_t row0, int64_t rbase, int64_t N, int64_t chunk,
                                         int lane) {
        const int64_t nblk = p.nb - chunk * I::kBlocks;  // blocks of the row from this chunk on
#pragma unroll
        for (int i = 0; i < I::kPieces; i++) {
            const int P = 64 * i + lane, rr = P / I::kPieces, q = P % I::kPieces;
            const int64_t row = row0 + (rbase + rr < N ? rbase + rr : N - 1);
            if (I::kBlocks == 1 || I::piece_block(q) < nblk)  // a k-quant chunk is one whole block
                w[i] = *reinterpret_cast<const u32x4 *>(I::piece(p, row * p.nb + chunk * I::kBlocks, q));
        }
#pragma unroll
        for (int i = 0; i < kScales; i++) {
            const int S = 64 * i + lane, rr = S >> 3, blk = S & 7;
            const int64_t row = row0 + (rbase + rr < N ? rbase + rr : N - 1);
            if (blk < nblk) s[i] = p.d[row * p.nb + chunk * 8 + blk];
        }
        if (DT == kQ6K) {
            const int64_t row = row0 + (rbase + lane < N ? rbase + lane : N - 1);
            d6 = p.d[row * p.nb + chunk];
        }
    }
    __device__ __forceinline__ void store(uint8_t *ws, int lane) const {
#pragma unroll
        for (int i = 0; i < I::kPieces; i++) {
            const int P = 64 * i + lane, rr = P / I::kPieces, q = P % I::kPieces;
            *reinterpret_cast<u32x4 *>(ws + rr * I::kPitch + 16 * q) = w[i];
        }
#pragma unroll
        for (int i = 0; i < kScales; i++) {
            const int S = 64 * i + lane, rr = S >> 3, blk = S & 7;
            *reinterpret_cast<uint16_t *>(ws + rr * I::kPitch + I::kScaleOff + 2 * blk) = (uint16_t)s[i];
        }
    }
};

// Group G of a row's chunk from its LDS image (the same bytes Group<DT>::load fetches from the planes).
template <int DT>
__device__ __forceinline__ void group_from_image(Group<DT> &g, const uint8_t *img, int G, uint32_t d6);

template <>
__device__ __forceinline__ void group_from_image<kQ8>(Group<kQ8> &g, const uint8_t *img, int G, uint32_t) {
    g.a = *reinterpret_cast<const uint4 *>(img + 32 * G);
    g.b = *reinterpret_cast<const uint4 *>(img + 32 * G + 16);
    g.d = *reinterpret_cast<const uint16_t *>(img + 256 + 2 * G);
}

template <>
__device__ __forceinline__ void group_from_image<kQ4>(Group<kQ4> &g, const uint8_t *img, int G, uint32_t) {
    g.a = *reinterpret_cast<const uint4 *>(img + 16 * G);
    g.d = *reinterpret_cast<const uint16_t *>(img + 128 + 2 * G);
}

template <>
__device__ __forceinline__ void group_from_image<kQ4K>(Group<kQ4K> &g, const uint8_t *img, int j, uint32_t) {
    g.h = *reinterpret_cast<const uint4 *>(img + 128);
    g.a = *reinterpret_cast<const uint4 *>(img + 16 * (j >> 1));
    g.b = *reinterpret_cast<const uint4 *>(img + 64 + 16 * (j >> 1));
}

template <>
__device__ __forceinline__ void group_from_image<kQ6K>(Group<kQ6K> &g, const uint8_t *img, int G, uint32_t d6) {
    const int n = G >> 2, k4 = G & 3;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        g.ql[t] = *reinterpret_cast<const uint2 *>(img + 16 * n + 8 * (k4 & 1) + 32 * t);
        g.qh[t] = *reinterpret_cast<const uint2 *>(img + 128 + 8 * n + 16 * t);
    }
    g.sc = *reinterpret_cast<const uint16_t *>(img + 192 + 8 * n + 2 * k4);
    g.d = d6;
}

// The chains of one pass of activation rows for a wave's 64 weight rows, advanced by a 32-wide group: lane l
// holds weight row l's decoded elements y[e] (the B operand) and reads the activations (the A operand) from the
// wave's 16 x 32 LDS tile. Both instructions are K = 1 outer products, each output one fma(a, b, c) with a single
// rounding (checked bit for bit against fmaf, subnormal, signed-zero and non-finite operands included).
//   MT = 0: v_mfma_f32_16x16x1f32, four blocks of 16 x 16: lane l supplies A(l / 16, l % 16) and B(l / 16, l % 16);
//           D(b, m, n) comes back in lane 16 (m / 4) + n, register 4 b + m % 4. A = x[l % 16] in every block: one
//           instruction advances 16 activation rows x 64 weight rows.
//   MT > 0: MT x v_mfma_f32_4x4x1f32, sixteen blocks of 4 x 4: lane l supplies A(l / 4, l % 4) and B(l / 4, l % 4);
//           D(b, m, n) comes back in lane 4 b + n, register m. Tile t takes A = x[4 t + l % 4]: 4 activation rows x
//           64 weight rows per instruction, and lane l collects its own row's results. At 9 cycles against 32.5 it
//           costs a quarter of the 16-row instruction for up to 4 rows.
template <int MT>
struct Tiles;

template <>
struct Tiles<0> {
    static constexpr int kRows = 16;
    v16f acc;
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = 0.0f;
    }
    __device__ __forceinline__ void step(const float *xs, int lane, const float y[32]) {
        const float *xr = xs + (lane & 15) * kXPitch;
        f32x4 xa[8];
#pragma unroll
        for (int q = 0; q < 8; q++) xa[q] = *reinterpret_cast<const f32x4 *>(xr + 4 * q);
#pragma unroll
        for (int e = 0; e < 32; e++) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(xa[e >> 2][e & 3], y[e], acc, 0, 0, 0);
    }
    __device__ __forceinline__ void store(float *res, int lane) const {  // res[m][row]
#pragma unroll
        for (int v = 0; v < 16; v++) res[(4 * (lane >> 4) + (v & 3)) * kRPitch + 16 * (v >> 2) + (lane & 15)] = acc[v];
    }
    // pp[m * ld + row] for m < mb, row < nrows
    __device__ __forceinline__ void store_global(float *pp, int64_t ld, int64_t mb, int64_t nrows, int lane) const {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = 4 * (lane >> 4) + (v & 3), row = 16 * (v >> 2) + (lane & 15);
            if (m < mb && row < nrows) pp[m * ld + row] = acc[v];
        }
    }
};

template <int MT>
struct Tiles {
    static constexpr int kRows = 4 * MT;
    v4f acc[MT];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[t][v] = 0.0f;
    }
    __device__ __forceinline__ void step(const float *xs, int lane, const float y[32]) {
        f32x4 xa[MT][8];
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int q = 0; q < 8; q++)
                xa[t][q] = *reinterpret_cast<const f32x4 *>(xs + (4 * t + (lane & 3)) * kXPitch + 4 * q);
#pragma unroll
        for (int e = 0; e < 32; e++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(xa[t][e >> 2][e & 3], y[e], acc[t], 0, 0, 0);
    }
    __device__ __forceinline__ void store(float *res, int lane) const {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) res[(4 * t + v) * kRPitch + lane] = acc[t][v];
    }
    __device__ __forceinline__ void store_global(float *pp, int64_t ld, int64_t mb, int64_t nrows, int lane) const {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (4 * t + v < mb && lane < nrows) pp[(4 * t + v) * ld + lane] = acc[t][v];
    }
};

// Element types of x and c (TRHIP_F32, or 16-bit ones widened exactly on use and rounded once; c is fp32 where x is), and
// c (+)=.
struct RowsIo {
    int x, c;
    bool acc;
};
__device__ __forceinline__ f32x4 widened(f32x4 v, int) { return v; }
__device__ __forceinline__ f32x4 widened(u32x2 v, int io) {
    return (f32x4){h16_to_f32(v.x & 0xFFFFu, io), h16_to_f32(v.x >> 16, io), h16_to_f32(v.y & 0xFFFFu, io),
                   h16_to_f32(v.y >> 16, io)};
}
template <bool X16>
__device__ __forceinline__ void put_c(void *c, int64_t i, float v, const RowsIo &io) {
    if (!X16 || io.c == TRHIP_F32) {
        float *o = static_cast<float *>(c) + i;
        *o = io.acc ? *o + v : v;
    } else {
        uint16_t *o = static_cast<uint16_t *>(c) + i;
        *o = (uint16_t)f32_to_h16(io.acc ? h16_to_f32(*o, io.c) + v : v, io.c);
    }
}

// Two-tile workgroups of four waves in q4_0 and q4_k are held to two waves a SIMD (left alone they take 297 registers and
// run one: 8192 x 8192, M = 200 488 us against 348 in seven workgroups a slice); q8_0 and q6_k would spill a hundred
// (4096 x 4096, M = 17 q8_0 25 us against 36).
template <int DT, int MT, int W>
constexpr int rows_waves() { return W == kStageWaves || (MT < 0 && (DT == kQ4 || DT == kQ4K)) ? 2 : 1; }

// The same chains on the matrix cores, a pass of Tiles<MT>::kRows activation rows at a time, in ascending k from +0
// as the CPU kernel does. Activation rows past M repeat row M - 1; their results are dropped.
//
// Workgroup (blockIdx.x, blockIdx.y, blockIdx.z) covers rows 64 blockIdx.x .. +63, chunks [cps blockIdx.y, + cps) and
// every gridDim.z-th pass from blockIdx.z. MT = -1: passes of 32 rows, two 16-row tiles on one decoding of the weights
// (the tiles share the LDS tile of activations in turn, so the LDS is that of one). A wave
// stages its chunk's weight images in LDS (loaded during its previous chunk) and each 32-wide group of activations
// (loaded a few groups ahead) in a 16 x 32 LDS tile that its lanes read back as A operands. With partial == null
// the workgroup covers every chunk and adds the chain results to `part` in chunk order in LDS; otherwise each
// chain result goes to partial[chunk][m][row] for sum_chunks_kernel.
template <int DT, bool X16, int MT, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(rows_waves<DT, MT, W>()))) void gemm_rows_mfma(
    const Planes p, const void *__restrict__ xv, void *__restrict__ c, float *__restrict__ partial, int64_t N, int64_t row0,
    int64_t M, int64_t K, int64_t cps, RowsIo io) {
    using XT = std::conditional_t<X16, uint16_t, float>;
    using XP = std::conditional_t<X16, u32x2, f32x4>;  // four activations as loaded
    const XT *x = static_cast<const XT *>(xv);
    using I = Image<DT>;
    using TL = Tiles<MT < 0 ? 0 : MT>;
    constexpr int NT = MT < 0 ? 2 : 1, MP = NT * TL::kRows;  // tiles and activation rows of a pass
    // activation groups in flight (larger images and two tiles leave fewer registers)
    constexpr int XD = DT == kQ8 ? 1 : DT == kQ6K || NT == 2 ? 2 : 4;
    static_assert(NT * 16 * kRPitch * 4 <= 64 * I::kPitch, "chain results reuse the wave's image space");
    __shared__ __align__(16) uint8_t wsl[W][64 * I::kPitch];
    __shared__ __align__(16) float xsl[W][16 * kXPitch];
    const int lane = threadIdx.x & 63;
    const int cw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tm = threadIdx.x >> 6;  // summing role: activation rows tm + W j of the pass, weight row `lane`
    const int64_t rbase = (int64_t)blockIdx.x * 64;
    const int64_t r = rbase + lane;
    const int64_t nchunks = (K + 255) / 256;
    const int64_t cb = (int64_t)blockIdx.y * cps, ce = cb + cps < nchunks ? cb + cps : nchunks;
    uint8_t *ws = wsl[cw];
    float *xs = xsl[cw];
    const uint8_t *img = ws + lane * I::kPitch;
    for (int64_t m0 = (int64_t)blockIdx.z * MP; m0 < M; m0 += (int64_t)gridDim.z * MP) {
        const int64_t mb = (M - m0) < MP ? (M - m0) : MP;
        const bool two = NT == 2 && mb > 16;  // the pass has rows for its second tile
        const XT *xp[2 * NT];  // x piece P = 64 i + lane: activation row P / 8, floats 4 (P % 8) .. +3 of a group
#pragma unroll
        for (int i = 0; i < 2 * NT; i++) {
            const int P = 64 * i + lane, m = P >> 3;
            xp[i] = x + (m0 + (m < mb ? m : mb - 1)) * K + 4 * (P & 7);
        }
        XP xg[XD][2 * NT];  // activations of the next XD groups; group g of every chunk uses slot g % XD
        auto fetch = [&](XP(&v)[2 * NT], int64_t k) {
#pragma unroll
            for (int i = 0; i < 2 * NT; i++)
                if (i < 2 || two) v[i] = *reinterpret_cast<const XP *>(xp[i] + k);
        };
        constexpr int PR = 16 * NT / W;
        float part[PR];
#pragma unroll
        for (int j = 0; j < PR; j++) part[j] = 0.0f;
        Stage<DT> st;
        if (cb + cw < ce) {
            st.load(p, row0, rbase, N, cb + cw, lane);
            const int64_t k0 = (cb + cw) * 256;
            const int ng0 = (int)(((K - k0) < 256 ? (K - k0) : 256) / 32);
#pragma unroll
            for (int g = 0; g < XD; g++)
                if (g < ng0) fetch(xg[g], k0 + 32 * g);
        }
        for (int64_t c0 = cb; c0 < ce; c0 += W) {
            const int64_t pc = c0 + cw;
            if (pc < ce) {  // wave-uniform
                st.store(ws, lane);
                const uint32_t d6 = st.d6;
                const int64_t k0 = pc * 256;
                const int ngroups = (int)(((K - k0) < 256 ? (K - k0) : 256) / 32);
                const bool more = pc + W < ce;
                const int64_t kx = (pc + W) * 256;  // the wave's next chunk
                const int ngx = more ? (int)(((K - kx) < 256 ? (K - kx) : 256) / 32) : 0;
                TL tl[NT];
#pragma unroll
                for (int h = 0; h < NT; h++) tl[h].zero();
                static_for<0, 8>([&](auto G) {
                    constexpr int gi = decltype(G)::value;
                    constexpr int sl = gi % XD;
                    if (gi < ngroups) {
                        auto put_x = [&](int h) {  // tile h's activations of this group
                            __builtin_amdgcn_wave_barrier();
#pragma unroll
                            for (int i = 0; i < 2; i++) {
                                const int P = 64 * i + lane;
                                *reinterpret_cast<f32x4 *>(xs + (P >> 3) * kXPitch + 4 * (P & 7)) = widened(xg[sl][2 * h + i], io.x);
                            }
                        };
                        // the activations XD groups on, then (once a chunk) the next chunk's weights, are in flight
                        // during the arithmetic of the groups before them
                        auto next_x = [&]() {
                            constexpr int gn = gi + XD;
                            if (gn < ngroups || gn - ngroups < ngx)
                                fetch(xg[sl], gn < ngroups ? k0 + 32 * gn : kx + 32 * (gn - ngroups));
                        };
                        put_x(0);
                        if (NT == 1) next_x();
                        if (gi == 0 && more) st.load(p, row0, rbase, N, pc + W, lane);
                        __builtin_amdgcn_wave_barrier();
                        Group<DT> g;
                        group_from_image<DT>(g, img, gi, d6);
                        float y[32];
                        g.decode(gi, y);
                        tl[0].step(xs, lane, y);
                        if constexpr (NT == 2) {
                            if (two) {
                                put_x(1);
                                __builtin_amdgcn_wave_barrier();
                                tl[1].step(xs, lane, y);
                            }
                            next_x();
                        }
                    }
                });
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int h = 0; h < NT; h++) {
                    if (partial)
                        tl[h].store_global(partial + (pc * M + m0 + 16 * h) * N + rbase, N, mb - 16 * h, N - rbase, lane);
                    else
                        tl[h].store(reinterpret_cast<float *>(ws) + 16 * h * kRPitch, lane);
                }
            }
            if (!partial) {  // kernel-uniform
                __syncthreads();
                const int ng = (int)((ce - c0) < W ? (ce - c0) : W);
                for (int i = 0; i < ng; i++) {
                    const float *res = reinterpret_cast<const float *>(wsl[i]);
#pragma unroll
                    for (int j = 0; j < PR; j++)
                        if (tm + W * j < MP) part[j] = part[j] + res[(tm + W * j) * kRPitch + lane];
                }
                __syncthreads();
            }
        }
        if (!partial && r < N) {
#pragma unroll
            for (int j = 0; j < PR; j++)
                if (tm + W * j < mb) put_c<X16>(c, (m0 + tm + W * j) * N + r, part[j], io);
        }
    }
}

// c[i] (+)= (((0 + partial[0][i]) + partial[1][i]) + ...) over the chunks in order, i < M N.
template <bool X16>
__global__ void sum_chunks_kernel(const float *__restrict__ partial, void *__restrict__ c, int64_t MN, int64_t nchunks,
                                  RowsIo io) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < MN; i += (int64_t)gridDim.x * blockDim.x) {
        float part = 0.0f;
        for (int64_t ch = 0; ch < nchunks; ch += 8) {  // up to eight loads in flight, added in chunk order
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = ch + u < nchunks ? partial[(ch + u) * MN + i] : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (ch + u < nchunks) part = part + v[u];
        }
        put_c<X16>(c, i, part, io);
    }
}


// How a call is cut into workgroups: chunks of a row block in nslices slices of cps (1: a workgroup of kStageWaves covers
// them all), passes of 16 or, two, 32 activation rows dealt over pz workgroups per row block and slice.
struct RowsPlan {
    int64_t nslices, cps, pz;
    bool two;
};

struct RowsCall {
    trhip_ctx *ctx;
    const trhip_wstore *w;
    int64_t row0, N, M;
    const void *x;
    void *c;
    float *partial;
    RowsPlan plan;
    RowsIo io;
};

template <int DT, int MT, int W>
int run_tiles(const RowsCall &r) {
    dim3 grid((unsigned)((r.N + 63) / 64), (unsigned)r.plan.nslices, (unsigned)r.plan.pz), block(64 * W);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, block, 0, r.ctx->stream, r.w->planes(), r.x, r.c, r.partial, r.N, r.row0, r.M,
                           r.w->K, r.plan.cps, r.io);
    };
    if (r.io.x == TRHIP_F32) go(gemm_rows_mfma<DT, false, MT, W>);
    else go(gemm_rows_mfma<DT, true, MT, W>);
    return launch_check(r.ctx, "gemm_rows");
}

// Up to 4 activation rows: one 4-row tile; up to 8: two; more: passes of 16 or 32 rows.
template <int DT, int W>
int run_w(const RowsCall &r) {
    if (r.M <= 4) return run_tiles<DT, 1, W>(r);
    if (r.M <= 8) return run_tiles<DT, 2, W>(r);
    return r.plan.two ? run_tiles<DT, -1, W>(r) : run_tiles<DT, 0, W>(r);
}

template <int DT>
int run_dt(const RowsCall &r) {
    return r.partial ? run_w<DT, kSplitWaves>(r) : run_w<DT, kStageWaves>(r);
}

// Up to 16 activation rows (one pass): one workgroup of kStageWaves waves per 64-row block covers all of its chunks when
// there are enough row blocks to occupy the device; otherwise the chunks are split into slices of kSplitWaves chunks
// (about two workgroups per CU in all) whose chain results are added in chunk order by sum_chunks_kernel.
//
// More rows: the plan of least estimated time, unless the walked one (16-row passes, one workgroup a row block and slice) is
// within 4% of it. The costs below are fitted to the measured times of every plan at 2948 sizes (four formats, 256 to 32768
// rows, 17 to 2048 activation rows, cold weights): the plan taken is 1.2% over the best one in the mean, and over the
// walked one by more than 3% at 10 of them, 10% at most. (Turns of one workgroup of kStageWaves or two of kSplitWaves a
// CU for every format, in whole rounds of the device, had put it over the walked plan by up to 32%: 4096 x 4096, M = 77,
// q8_0 55 -> 73 us.)
//
// A CU holds one workgroup of kStageWaves, and of kSplitWaves as many as their registers leave: two for q4_0 and q4_k, one
// for q8_0 and q6_k (more than 256 registers a wave). Passes dealt over workgroups instead of walked by one fill the device
// where row blocks are few: q4_k 4096 x 4096, M = 77 53 us walked, 41 in two workgroups per slice; 1024 x 4096, M = 300 172
// walked, 48 dealt; 14336 x 4096, M = 512 864 walked in 16s, 661 dealt in 32s.
struct TurnCost {                        // us for a turn on 16 and on 32 activation rows (whose weights are decoded once)
    double whole[2], alone[2], pair[2];  // a workgroup of kStageWaves; of kSplitWaves, one and two on a CU
    double start[2], slice_start, pass;  // the start of a workgroup of kStageWaves, of kSplitWaves; of a pass
    double later, half;                  // share of a start that shows after the first; of a tile that a half pass saves
    double sums, l2_rate, rate;          // the partial sums' launch; MB / us of those that the L2s hold, of the rest
};
TurnCost turn_cost(int dtype) {
    if (dtype == kQ8) return {{14.2, 25.7}, {7.62, 13}, {0, 0}, {6.73, 17.7}, 1.4, 1.5, 0.71, 0.538, 6.68, 5.49, 2.03};
    if (dtype == kQ6K) return {{16.2, 29.1}, {9.24, 14.8}, {0, 0}, {5.81, 12.6}, 0.884, 1.24, 0.729, 0.564, 6.71, 3.98, 2.37};
    return {{10.8, 18.4}, {6.24, 10.1}, {8.66, 17.1}, {4.03, 5.21}, 0.857, 0.862, 0.334, 0.749, 6.89, 5.52, 2.3};
}
constexpr bool two_split_workgroups(int dtype) { return dtype == kQ4 || dtype == kQ4K; }

// Workgroups are dealt in order over the shader engines (8 CUs each) and stay there, so that a plan lasts as long as the
// engine with the most of them: 276 on 256 CUs leave one engine nine on eight CUs (q4_0 2944 x 1536, M = 343 in 32s: 73 us
// in six workgroups a row block, 52 in eleven).
constexpr int64_t kEngineCus = 8;

// Passes one after another until the last of an engine's n workgroups ends, `slots` at a time in grid order; `heavy` of them,
// the first, take q + 1 passes, the others q.
int64_t passes_in_turn(int64_t n, int64_t heavy, int64_t q, int64_t slots) {
    const int64_t f = heavy / slots, l = heavy % slots, rest = n - f * slots, t = f * (q + 1);
    if (rest <= 0) return t;
    const int64_t r = (rest + slots - 1) / slots, last = rest - (r - 1) * slots;
    if (l == 0) return t + r * q;
    if (r == 1) return t + q + 1;
    if (last > slots - l) return t + q + 1 + (r - 1) * q;
    return t + (r * q > q + 1 + (r - 2) * q ? r * q : q + 1 + (r - 2) * q);
}

double plan_time(const RowsPlan &p, const TurnCost &cost, int dtype, int64_t M, int64_t N, int64_t nchunks, int64_t cus) {
    const bool cut = p.nslices > 1;
    const int64_t nrb = (N + 63) / 64, B = nrb * p.nslices, waves = cut ? kSplitWaves : kStageWaves;
    const int64_t np = (M + (p.two ? 31 : 15)) / (p.two ? 32 : 16), turns = (p.cps + waves - 1) / waves;
    const int64_t engines = cus > kEngineCus ? cus / kEngineCus : 1, n = (B * p.pz + engines - 1) / engines;
    const bool pair = cut && two_split_workgroups(dtype) && n > kEngineCus;
    // (up to kSplitWaves chunks leave a workgroup of kStageWaves one wave a SIMD)
    const double *turn = pair ? cost.pair : cut || nchunks <= kSplitWaves ? cost.alone : cost.whole;
    const int64_t slots = pair ? 2 * kEngineCus : kEngineCus, rounds = (n + slots - 1) / slots;
    const int64_t heavy = (np % p.pz * B + engines - 1) / engines, passes = passes_in_turn(n, heavy, np / p.pz, slots);
    double t = (double)passes * ((double)turns * turn[p.two] + cost.pass);
    // (a start after the first overlaps the other workgroups' work in part)
    t += (1.0 + cost.later * (double)(rounds - 1)) * (cut ? cost.slice_start : cost.start[p.two]);
    // half a last pass: in every round where passes are walked, in its share of the rounds where each has its workgroup
    const double halves = p.pz == 1 ? (double)rounds : p.pz == np ? (double)B / (double)(slots * engines) : 0.0;
    if (p.two && M - 32 * (np - 1) <= 16) t -= cost.half * halves * (double)turns * (turn[1] - turn[0]);
    if (cut) {
        const double mb = (double)(nchunks * M * N) * 4e-6, l2 = mb < 32.0 ? mb : 32.0;
        t += cost.sums + l2 / cost.l2_rate + (mb - l2) / cost.rate;
    }
    return t;
}

// uncut: only plans without partial sums
RowsPlan rows_plan(int dtype, int64_t M, int64_t N, int64_t nchunks, int64_t cus, const int *force = nullptr,
                   bool uncut = false) {
    const int64_t nrb = (N + 63) / 64;
    RowsPlan split = {1, nchunks, 1, false};
    if (nchunks > kSplitWaves && !uncut) {
        const int64_t want = (512 + nrb - 1) / nrb;  // slices per row block for about 512 workgroups
        const int64_t maxs = (nchunks + kSplitWaves - 1) / kSplitWaves;
        const int64_t ns = want < maxs ? want : maxs, cps = (nchunks + ns - 1) / ns;
        split.cps = (cps + kSplitWaves - 1) / kSplitWaves * kSplitWaves;
        split.nslices = (nchunks + split.cps - 1) / split.cps;
    }
    const RowsPlan whole = {1, nchunks, 1, false}, walked = nrb < 160 ? split : whole;
    if (M <= 16) return walked;
    if (force && force[0]) {
        RowsPlan p = force[0] == 2 ? split : whole;
        p.two = force[1] == 32;
        const int64_t np = (M + force[1] - 1) / force[1];
        p.pz = force[2] < np ? force[2] : np;
        return p;
    }
    const TurnCost cost = turn_cost(dtype);
    RowsPlan best = walked;
    double least = 0.96 * plan_time(walked, cost, dtype, M, N, nchunks, cus);
    for (int cut = 0; cut < (split.nslices > 1 ? 2 : 1); cut++)
        for (int two = 0; two < 2; two++) {
            RowsPlan p = cut ? split : whole;
            p.two = two != 0;
            const int64_t np = (M + (two ? 31 : 15)) / (two ? 32 : 16);
            for (int64_t z = 1; z <= 65535;) {  // the fewest workgroups for each number of passes one may take
                p.pz = z;
                const double t = plan_time(p, cost, dtype, M, N, nchunks, cus);
                if (t < least) {
                    least = t;
                    best = p;
                }
                const int64_t most = (np + z - 1) / z;
                if (most == 1) break;
                z = (np + most - 2) / (most - 1);
            }
        }
    return best;
}

}  // namespace

// (the fitted costs rank plans; the time they give is 2% short for q8_0 and 15% for q4_0)
double gemm_rows_time(int dtype, int64_t M, int64_t N, int64_t K, int64_t cus) {
    const int64_t nchunks = (K + 255) / 256;
    const RowsPlan p = rows_plan(dtype, M, N, nchunks, cus);
    return plan_time(p, turn_cost(dtype), dtype, M, N, nchunks, cus) * (dtype == kQ8 ? 1.02 : 1.15);
}

void gemm_rows_cut(int dtype, int64_t M, int64_t N, int64_t K, int64_t cus, int64_t plan[3]) {
    const RowsPlan p = rows_plan(dtype, M, N, (K + 255) / 256, cus);
    plan[0] = p.nslices;
    plan[1] = p.two ? 32 : 16;
    plan[2] = p.pz;
}

int launch_gemm_rows(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const void *x, void *c, int64_t M,
                     bool acc, int xio, int cio) {
    if (N == 0 || M == 0) return TRHIP_OK;
    const int64_t K = w->K, nchunks = (K + 255) / 256;
    const int64_t cus = ctx->sm_count > 0 ? ctx->sm_count : 256;
    RowsPlan pl = rows_plan(w->dtype, M, N, nchunks, cus, ctx->force_rows);
    // the kernel reads x four elements at a time
    const size_t xel = xio == TRHIP_F32 ? sizeof(float) : sizeof(uint16_t);
    const bool copy_x = reinterpret_cast<uintptr_t>(x) % (4 * xel) != 0;
    const size_t xbytes = copy_x ? ((size_t)(M * K) * xel + 255) / 256 * 256 : 0;
    // A captured call cannot grow the workspace. From 160 row blocks the chunks need no slices, so that such a call needs
    // none for them either.
    if (pl.nslices > 1 && N > 159 * 64 && xbytes + (size_t)(nchunks * M * N) * sizeof(float) > ctx->ws_bytes && capturing(ctx))
        pl = rows_plan(w->dtype, M, N, nchunks, cus, ctx->force_rows, true);
    const size_t pbytes = pl.nslices > 1 ? (size_t)(nchunks * M * N) * sizeof(float) : 0;
    int st = TRHIP_OK;
    uint8_t *ws = nullptr;
    if (xbytes + pbytes > 0) {
        ws = static_cast<uint8_t *>(workspace(ctx, xbytes + pbytes, &st));
        if (!ws) return st;
    }
    RowsCall r = {ctx, w, row0, N, M, x, c, nullptr, pl, {xio, cio, acc}};
    if (copy_x) {
        hipError_t e = hipMemcpyAsync(ws, x, (size_t)(M * K) * xel, hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "gemm_rows: align x");
        r.x = ws;
    }
    if (pl.nslices > 1) r.partial = reinterpret_cast<float *>(ws + xbytes);
    switch (w->dtype) {
    case kQ8: st = run_dt<kQ8>(r); break;
    case kQ4: st = run_dt<kQ4>(r); break;
    case kQ4K: st = run_dt<kQ4K>(r); break;
    case kQ6K: st = run_dt<kQ6K>(r); break;
    default: return fail(ctx, TRHIP_ERR_INVALID, "gemm_rows: bad dtype");
    }
    if (st != TRHIP_OK || !r.partial) return st;
    const int64_t MN = M * N;
    const unsigned blocks = (unsigned)((MN + 255) / 256 < 4096 ? (MN + 255) / 256 : 4096);
    auto sum = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, ctx->stream, r.partial, c, MN, nchunks, r.io);
    };
    if (xio == TRHIP_F32) sum(sum_chunks_kernel<false>);
    else sum(sum_chunks_kernel<true>);
    return launch_check(ctx, "sum_chunks");
}

}  // namespace trhip
