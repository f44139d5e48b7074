// fastg.hip -- fast-mode (tolerance) product of fp32 activations for more than 16 rows, every weight format, on 16-bit
// matrix cores: trhip_gemm_q(TRHIP_MODE_FAST). The reference's GPU runs these as dequantized tiles through a float GEMM
// (gpu/backend_quant.go:43-134), a tolerance path too.
//
// Activations: x is scaled by a power of two, x' = x 2^(80 - E) or x 2^(14 - E), and split into terms.
//   q8_0, q4_0: 2^E > max|x| of the row; three bf16 terms of eight bits, which add up to x' exactly, whatever the range of the row (bf16 has fp32's
//     exponents; elements below 2^-182 of the row's largest would lose low bits). Two f16 terms, exact to 2^-39 of the row's
//     largest only, were 10-30% faster (4096 x 14336, M = 300 136 against 176 us) and lost every element beside one 2^40
//     times larger.
//   q4_k, q6_k: 2^E > max|x| of the row's 256-element block, which each block is multiplied back by where it is folded (one
//     exponent a row loses the other blocks of a row that holds an outlier: a row of order 1 with one element of 1e8 was
//     off by 9e-4). Two f16 terms, hi = f16(x') and lo = f16(x' - hi): exact to 2^-23 of each element, and to 2^-39 of
//     the block's largest where lo is subnormal (the f16 MFMAs keep subnormals).
// Weights: the integer part of every format is exact in the terms' type,
//   q8_0, q4_0: the code (q4 - 8);   q4_k: q4 sc - o;   q6_k: (q6 - 32) (sc & ~1) and (q6 - 32) (sc & 1), two planes
// so each product is exact and only fp32 sums round. Per block (32 elements for q8_0 and q4_0, 256 for the k-quants)
//   acc += d D,   D = sum w x'   (over the terms);   q4_k: acc += d D + sum_j v_j S_j,   v_j = d o_j - dmin m_j
// with S_j the sub-block sums of x' as three f16 terms and v_j, scaled by a power of two per block, as two. o_j is an
// integer near dmin m_j / d, so that the code and minimum terms, several times the result, cancel in no sum. (q4_k, error
// against float64 at K = 4096: 1.6e-7; with o_j = 8 sc_j 3.0e-7; the exact mode's 3.0e-7, the int8 digits' 2.2e-7.)
//
// Tiles. A workgroup is 8 waves over 32 WM activation rows and 256 weight rows. The weights of 64 elements are expanded
// once per workgroup, by all threads, into LDS in operand order (two buffers, one barrier per 64 elements); a wave
// multiplies 32 activation rows by 32 CT of the columns, so each B operand read from LDS serves an MFMA per term and
// each A operand, read straight from the split activations in L2, CT of them. (Weights expanded into each wave's own
// registers would leave an A operand one MFMA at 32 columns a wave, and the A reads alone would fill the LDS bandwidth.)
//
// What bounds it: the matrix cores' rate under load and what is added to it. A plain f16 product reaches 1.38 PFLOP/s here
// (24 ns per MFMA and SIMD, against 17 for int8), so the two products of 14336 x 4096 at M = 512 (q4_k) cannot take less
// than 87 us; beside its 2176 MFMAs a wave issues 9300 VALU, most of them the expansion and the fold (counters of both
// kernels: profiles/fast_gemm_and_actq_blocks.txt). Operand reads, expansion and folding each added their own time when
// put back one by one, whether the two waves of a SIMD worked in step or in opposite phases: 148 us a call (digits kernel
// 196). Multiplying before expanding, in each step, measured 143.8 against 152.6 us (with one exponent a row). q8_0 (exact
// K = 1 products before): 14336 x 4096, M = 300 606 -> 195; 4096 x 14336, M = 300 725 -> 176.
#include "trhip_internal.hpp"
#include "mfma_util.hpp"

#include <cfloat>

namespace trhip {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

constexpr int FG_W = 8, FG_THREADS = 64 * FG_W, FG_TN = 256;

template <int DT>
struct Fg {
    static constexpr bool KQ = DT == kQ4K || DT == kQ6K;
    static constexpr int TERMS = KQ ? 2 : 3;                  // of an activation
    static constexpr int E = KQ ? 14 : 80;                    // |x'| < 2^E
    static constexpr int PL = DT == kQ6K ? 2 : 1;             // planes per weight
    static constexpr int B = PL * 4 * 8 * 1024;               // operands of a step: [plane][step][column tile][lane][16]
    static constexpr int DS = KQ ? 0 : 2 * FG_TN * 4;         // d of the step's two blocks
    static constexpr int BUF = B + DS;
    static constexpr int CO = DT == kQ4K ? FG_TN * 64 : 0;     // q4_k: v_j 2^-q as two f16 terms; the code constants
    static constexpr int DK = KQ ? FG_TN * 8 : 0;             // per column d and (q4_k) 2^(q + 6), S_j being scaled 2^-6
    static constexpr int BLK = CO + DK;                       // per block, two buffers
    static constexpr size_t LDS = 2 * BUF + 2 * BLK;
};
static_assert(Fg<kQ6K>::LDS <= 160 * 1024 && Fg<kQ4K>::LDS <= 160 * 1024, "one workgroup per CU");

// ---- activations ----

// Largest |x| of each 1024-element piece of a row, one wave a piece: pm[m][piece], infinity if it holds NaN / Inf
// (k-quants); FINITE (q8_0, q4_0): of its finite elements.
template <bool FINITE>
__global__ __launch_bounds__(256) void row_max_kernel(const float *__restrict__ x, int64_t M, int64_t K, int64_t np,
                                                      float *__restrict__ pm) {
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= M * np) return;  // wave-uniform
    const int64_t m = t / np, k0 = (t % np) * 1024;
    float a = 0.0f;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t k = k0 + 256 * i + 4 * lane;
        const float4 v = *reinterpret_cast<const float4 *>(x + m * K + (k < K ? k : 0));
        if (k >= K) continue;
        if (FINITE) {
            const float e[4] = {fabsf(v.x), fabsf(v.y), fabsf(v.z), fabsf(v.w)};
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (e[j] <= FLT_MAX) a = fmaxf(a, e[j]);
        } else {
            a = fmaxf(a, amax4(v));
            bad |= non_finite4(v) != 0;
        }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) a = fmaxf(a, __shfl_xor(a, o));
    bad = __any(bad);
    if (lane == 0) pm[t] = bad ? __builtin_inff() : a;
}

// The split activations: per 32-row tile and 16-element step, 1 KB of operands of each term, largest term first (lane
// r + 32 h: row r, elements 8 h .. + 7 of the step, each four as 0, 2, 1, 3: the order in which nibbles and bytes pair up
// in a dword). q8_0 / q4_0: three bf16 terms cut off x' in turn, eight bits each, so that they add up to x' exactly; a NaN
// or Inf is its first term.
// K is padded with zeros to a multiple of 64, rows to 32. q4_k: the sub-block sums S_j 2^-6 as three f16 terms, per tile
// and 256-element block two operands [P0 | P1], [P0 | P2] (times [vh | vh], [vl | vh] of the weights). Workgroup (tile,
// 256-element chunk); ex[m] = E of the row less Fg::E, bad[m], sx[tile][chunk][row] = 2^(the block's E - the row's).
template <int DT>
__global__ __launch_bounds__(256) void split_kernel(const float *__restrict__ x, int64_t M, int64_t K, int64_t np,
                                                    const float *__restrict__ pm, uint8_t *__restrict__ rec,
                                                    uint8_t *__restrict__ srec, float *__restrict__ sx,
                                                    int *__restrict__ ex, int *__restrict__ bad) {
    constexpr bool SUMS = DT == kQ4K;
    constexpr int TERMS = Fg<DT>::TERMS;
    const int tid = threadIdx.x, r = tid >> 3, s8 = tid & 7;
    const int64_t nch = (K + 255) / 256, mt = blockIdx.x / nch, ch = blockIdx.x % nch;
    const int64_t m = 32 * mt + r, KS = (K + 63) / 64 * 4;
    const bool row = m < M;
    float a = 0.0f;
    for (int64_t i = s8; i < np; i += 8) a = fmaxf(a, pm[(row ? m : 0) * np + i]);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) a = fmaxf(a, __shfl_xor(a, o));
    const bool inf = a > FLT_MAX;
    int E = 0;
    if (!inf && a > 0.0f) (void)frexpf(a, &E);
    if (ch == 0 && s8 == 0 && row) {
        ex[m] = E - Fg<DT>::E;
        if (Fg<DT>::KQ) bad[m] = inf ? 1 : 0;
    }
    const bool use = row && !inf;
    float4 in4[4][2];
    auto load = [&](int j) {
        const int64_t k = 256 * ch + 64 * j + 8 * s8;
        const float4 *p = reinterpret_cast<const float4 *>(x + (use && k < K ? m * K + k : 0));
        in4[j][0] = p[0];
        in4[j][1] = p[1];
    };
    if (Fg<DT>::KQ) {  // the block's own exponent (K is a multiple of 256)
        float b = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            load(j);
            b = fmaxf(b, fmaxf(amax4(in4[j][0]), amax4(in4[j][1])));
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) b = fmaxf(b, __shfl_xor(b, o));
        int eb = E - 120;
        if (use && b > 0.0f) {
            int e = 0;
            (void)frexpf(b, &e);
            if (e > eb) eb = e;
        }
        if (s8 == 0) sx[(mt * nch + ch) * 32 + r] = ldexpf(1.0f, eb - E);
        E = eb;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t k = 256 * ch + 64 * j + 8 * s8;
        if (k - 8 * s8 >= 16 * KS) break;  // past the padded row (uniform)
        float v[8];
        const bool in = use && k < K;
        if (!Fg<DT>::KQ) load(j);
        const float4 v0 = in4[j][0], v1 = in4[j][1];
        const float raw[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        uint16_t tm[TERMS][8];
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = in ? ldexpf(raw[i], Fg<DT>::E - E) : 0.0f;
            if constexpr (TERMS == 3) {
                const uint32_t u = __builtin_bit_cast(uint32_t, v[i]);
                const bool fin = (u & 0x7F800000u) != 0x7F800000u;
                float rest = v[i];
#pragma unroll
                for (int t = 0; t < 3; t++) {
                    const uint32_t top = __builtin_bit_cast(uint32_t, rest) & 0xFFFF0000u;
                    tm[t][i] = (uint16_t)(top >> 16);
                    rest = fin ? rest - __builtin_bit_cast(float, top) : 0.0f;
                }
                if (!fin && (u & 0x007FFFFFu)) tm[0][i] |= 0x40;  // a NaN whose payload is all in the cut bits
            } else {
                const _Float16 h = (_Float16)v[i];
                tm[0][i] = __builtin_bit_cast(uint16_t, h);
                tm[1][i] = __builtin_bit_cast(uint16_t, (_Float16)(v[i] - (float)h));
            }
            if (SUMS) s += (double)v[i];
        }
        auto pack = [](const uint16_t (&u)[8]) {
            return make_uint4(u[0] | (uint32_t)u[2] << 16, u[1] | (uint32_t)u[3] << 16, u[4] | (uint32_t)u[6] << 16,
                              u[5] | (uint32_t)u[7] << 16);
        };
        uint8_t *o = rec + ((mt * KS + (k >> 4)) * TERMS) * 1024 + (r + 32 * (s8 & 1)) * 16;
#pragma unroll
        for (int t = 0; t < TERMS; t++) *reinterpret_cast<uint4 *>(o + 1024 * t) = pack(tm[t]);
        if (SUMS) {
            s += __shfl_xor(s, 1);
            s += __shfl_xor(s, 2);
            if ((s8 & 3) == 0) {  // sub-block 2 j + s8 / 4
                const int jj = 2 * j + (s8 >> 2);
                s *= 0x1p-6;
                const _Float16 p0 = (_Float16)(float)s;
                s -= (double)(float)p0;
                const _Float16 p1 = (_Float16)(float)s;
                s -= (double)(float)p1;
                _Float16 *so = reinterpret_cast<_Float16 *>(srec + (mt * nch + ch) * 2048);
                so[8 * r + jj] = p0;
                so[8 * (r + 32) + jj] = p1;
                so[512 + 8 * r + jj] = p0;
                so[512 + 8 * (r + 32) + jj] = (_Float16)(float)s;
            }
        }
    }
}

// ---- weights ----
//
// Thread (column c = tid % 256, half h = tid / 256) expands half of its column's 64 elements of a step: whole 16-element
// operand steps, in the record's order. Registers are refilled for the next use as soon as they are expanded.

// Two codes of a dword as an f16 pair. 0x6400 | v is 1024 + v; the constant sits in a register (`k64`), so that masking and
// or-ing are one v_and_or_b32.
__device__ __forceinline__ h2 pair_f16(uint32_t w, uint32_t mask, uint32_t k64, _Float16 mul, _Float16 add) {
    const h2 v = __builtin_bit_cast(h2, (w & mask) | k64);
    return __builtin_elementwise_fma(v, (h2){mul, mul}, (h2){add, add});
}
__device__ __forceinline__ uint32_t bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// The four signed bytes of a dword as bf16 pairs, bytes 0, 2 and 1, 3: the upper halves of the integers' fp32 values, which
// hold them exactly (eight significant bits).
__device__ __forceinline__ void bytes4(uint32_t w, uint32_t &p02, uint32_t &p13) {
    uint32_t f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) f[i] = __builtin_bit_cast(uint32_t, (float)(int8_t)(w >> (8 * i)));
    p02 = __builtin_amdgcn_perm(f[2], f[0], 0x07060302u);
    p13 = __builtin_amdgcn_perm(f[3], f[1], 0x07060302u);
}

// (1024 + 16 q) m + a for the eight nibbles q of a dword, each at bits 4..7 of a half word: with m = s / 16 and an integer
// a near -64 s this is q s + 64 s + a, exactly. The pairs are bytes 0, 2 and 1, 3.
__device__ __forceinline__ void nibbles8(uint32_t w, uint32_t k64, _Float16 ml, _Float16 al, _Float16 mh, _Float16 ah,
                                         uint32_t (&lo)[2], uint32_t (&hi)[2]) {
    lo[0] = bits(pair_f16(w << 4, 0x00F000F0u, k64, ml, al));
    lo[1] = bits(pair_f16(w >> 4, 0x00F000F0u, k64, ml, al));
    hi[0] = bits(pair_f16(w, 0x00F000F0u, k64, mh, ah));
    hi[1] = bits(pair_f16(w >> 8, 0x00F000F0u, k64, mh, ah));
}

template <int DT>
struct ColW;

template <>
struct ColW<kQ8> {
    uint4 a[2][2];  // steps in flight, parity s & 1
    uint32_t d[2];
    __device__ __forceinline__ void load(const Planes &p, int64_t row, int s, int h, int i) {
        int64_t b = 2 * (int64_t)s + h;
        const bool in = b < p.nb;
        b = row * p.nb + (in ? b : p.nb - 1);
        const uint4 *q = reinterpret_cast<const uint4 *>(p.qs + b * 32);
        a[i][0] = q[0];
        a[i][1] = q[1];
        d[i] = p.d[b];
    }
    __device__ __forceinline__ void expand(uint8_t *buf, int c, int h, int i) {
        uint8_t *o = buf + ((2 * h) * 8 + (c >> 5)) * 1024 + (c & 31) * 16;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const uint32_t w[4] = {a[i][ks].x, a[i][ks].y, a[i][ks].z, a[i][ks].w};
            uint32_t v[8];
#pragma unroll
            for (int e = 0; e < 4; e++) bytes4(w[e], v[2 * e], v[2 * e + 1]);
            *reinterpret_cast<uint4 *>(o + ks * 8192) = make_uint4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<uint4 *>(o + ks * 8192 + 512) = make_uint4(v[4], v[5], v[6], v[7]);
        }
        reinterpret_cast<float *>(buf + Fg<kQ8>::B)[FG_TN * h + c] = f16_to_f32((uint16_t)d[i]);
    }
};

template <>
struct ColW<kQ4> {
    uint4 a[2];
    uint32_t d[2];
    __device__ __forceinline__ void load(const Planes &p, int64_t row, int s, int h, int i) {
        int64_t b = 2 * (int64_t)s + h;
        b = row * p.nb + (b < p.nb ? b : p.nb - 1);
        a[i] = *reinterpret_cast<const uint4 *>(p.qs + b * 16);
        d[i] = p.d[b];
    }
    __device__ __forceinline__ void expand(uint8_t *buf, int c, int h, int i) {
        // byte j holds elements j (low nibble, operand step 2 h) and j + 16 (high, step 2 h + 1)
        uint8_t *o = buf + ((2 * h) * 8 + (c >> 5)) * 1024 + (c & 31) * 16;
        const uint32_t w[4] = {a[i].x, a[i].y, a[i].z, a[i].w};
        uint32_t lo[4][2], hi[4][2];
#pragma unroll
        for (int e = 0; e < 4; e++) {  // q - 8 as signed bytes: (q + 120) ^ 128, no carry between bytes
            bytes4(((w[e] & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u, lo[e][0], lo[e][1]);
            bytes4((((w[e] >> 4) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u, hi[e][0], hi[e][1]);
        }
        *reinterpret_cast<uint4 *>(o) = make_uint4(lo[0][0], lo[0][1], lo[1][0], lo[1][1]);
        *reinterpret_cast<uint4 *>(o + 512) = make_uint4(lo[2][0], lo[2][1], lo[3][0], lo[3][1]);
        *reinterpret_cast<uint4 *>(o + 8192) = make_uint4(hi[0][0], hi[0][1], hi[1][0], hi[1][1]);
        *reinterpret_cast<uint4 *>(o + 8192 + 512) = make_uint4(hi[2][0], hi[2][1], hi[3][0], hi[3][1]);
        reinterpret_cast<float *>(buf + Fg<kQ4>::B)[FG_TN * h + c] = f16_to_f32((uint16_t)d[i]);
    }
};

template <>
struct ColW<kQ4K> {
    uint4 q[4], hdr;
    // piece g of half h: elements 64 g + 16 h .. + 15 (low nibbles) and 64 g + 32 + 16 h .. (high)
    __device__ __forceinline__ void load(const Planes &p, int64_t row, int b, int h, int g) {
        q[g] = *(reinterpret_cast<const uint4 *>(p.qs + (row * p.nb + b) * 128 + 64 * h) + g);
    }
    __device__ __forceinline__ void load_hdr(const Planes &p, int64_t row, int b) {
        hdr = *reinterpret_cast<const uint4 *>(p.aux + (row * p.nb + b) * 16);
    }
    // The block's constants, a step before its first expansion: thread h takes sub-blocks 4 h .. + 3. Per sub-block the
    // multiplier s / 16 and addend -(64 s + o) of the codes, o an integer in [0, 15 s] near dmin m / d (any is right; a
    // close one keeps v small), 64 s + o as f16 holds it; v = d o - dmin m scaled by 2^-q, |v 2^-q| < 2^10.
    __device__ __forceinline__ void constants(uint8_t *blk, int c, int h) {
        uint32_t sc[2], mn[2];
        q4k_scales(hdr.y, hdr.z, hdr.w, sc[0], sc[1], mn[0], mn[1]);
        const uint32_t scw = h ? sc[1] : sc[0], mnw = h ? mn[1] : mn[0];
        const float d = f16_to_f32((uint16_t)(hdr.x & 0xFFFF)), dmin = f16_to_f32((uint16_t)(hdr.x >> 16));
        int e = 0;
        (void)frexpf(fmaxf(fabsf(d), fabsf(dmin)), &e);
        const float r = dmin * __builtin_amdgcn_rcpf(d), de = ldexpf(d, -e), dm = ldexpf(dmin, -e);
        _Float16 vh[4], vl[4];
        h2 ma[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float s = ubyte_f(scw, j), m = ubyte_f(mnw, j);
            const _Float16 o64 = (_Float16)rintf(fmaf(64.0f, s, fminf(fmaxf(r * m, 0.0f), 15.0f * s)));
            ma[j] = (h2){(_Float16)(s * 0.0625f), -o64};
            const float v = fmaf(de, (float)o64 - 64.0f * s, -(dm * m));
            vh[j] = (_Float16)v;
            vl[j] = (_Float16)(v - (float)vh[j]);
        }
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<h4 *>(blk + 16 * c + 8 * h) = (h4){vh[0], vh[1], vh[2], vh[3]};
        *reinterpret_cast<h4 *>(blk + FG_TN * 16 + 16 * c + 8 * h) = (h4){vl[0], vl[1], vl[2], vl[3]};
        // (pairs of sub-blocks, [pair][column][2])
        *reinterpret_cast<uint2 *>(blk + FG_TN * 32 + (2 * h) * FG_TN * 8 + 8 * c) = make_uint2(bits(ma[0]), bits(ma[1]));
        *reinterpret_cast<uint2 *>(blk + FG_TN * 32 + (2 * h + 1) * FG_TN * 8 + 8 * c) = make_uint2(bits(ma[2]), bits(ma[3]));
        reinterpret_cast<float *>(blk + Fg<kQ4K>::CO)[FG_TN * h + c] = h ? ldexpf(1.0f, e + 6) : d;
    }
    __device__ __forceinline__ void expand(uint8_t *buf, const uint8_t *blk, int c, int h, int g, uint32_t k64) {
        const uint2 cc = *reinterpret_cast<const uint2 *>(blk + FG_TN * 32 + g * FG_TN * 8 + 8 * c);
        const h2 c0 = __builtin_bit_cast(h2, cc.x), c1 = __builtin_bit_cast(h2, cc.y);
        const uint32_t w[4] = {q[g].x, q[g].y, q[g].z, q[g].w};
        uint32_t lo[4][2], hi[4][2];
#pragma unroll
        for (int e = 0; e < 4; e++) nibbles8(w[e], k64, c0.x, c0.y, c1.x, c1.y, lo[e], hi[e]);
        uint8_t *o = buf + (h * 8 + (c >> 5)) * 1024 + (c & 31) * 16;  // operand steps h and 2 + h
        *reinterpret_cast<uint4 *>(o) = make_uint4(lo[0][0], lo[0][1], lo[1][0], lo[1][1]);
        *reinterpret_cast<uint4 *>(o + 512) = make_uint4(lo[2][0], lo[2][1], lo[3][0], lo[3][1]);
        *reinterpret_cast<uint4 *>(o + 16384) = make_uint4(hi[0][0], hi[0][1], hi[1][0], hi[1][1]);
        *reinterpret_cast<uint4 *>(o + 16384 + 512) = make_uint4(hi[2][0], hi[2][1], hi[3][0], hi[3][1]);
    }
};

template <>
struct ColW<kQ6K> {
    uint2 ql[4][2];  // chunk pair g: elements 64 g + 16 h .. (chunk 2 g) and 64 g + 32 + 16 h .. (2 g + 1)
    uint4 qh[2], scv;
    uint32_t d;
    // In the lane-sliced planes (trhip_internal.hpp), 8-byte pieces t = 2 h, 2 h + 1: ql at 32 t + 16 n + 8 (chunk % 2)
    // with n = g / 2, low nibbles for g even, high for odd; qh at 16 t + 8 n, bit pair chunk % 4.
    __device__ __forceinline__ void load(const Planes &p, int64_t row, int b, int h, int g) {
        const int64_t bi = row * p.nb + b;
        if (!(g & 1)) {  // pieces of chunks 2 g .. 2 g + 3 (both nibbles)
            const uint4 *l = reinterpret_cast<const uint4 *>(p.qs + bi * 128 + 64 * h + 16 * (g >> 1));
            const uint4 u0 = l[0], u1 = l[2];
            ql[g][0] = make_uint2(u0.x, u0.y);      // t = 2 h, even chunk
            ql[g][1] = make_uint2(u0.z, u0.w);      // t = 2 h, odd chunk
            ql[g + 1][0] = make_uint2(u1.x, u1.y);  // t = 2 h + 1
            ql[g + 1][1] = make_uint2(u1.z, u1.w);
        }
        if (g == 0) {
            const uint4 *u = reinterpret_cast<const uint4 *>(p.aux + bi * 64 + 32 * h);
            qh[0] = u[0];
            qh[1] = u[1];
            scv = *reinterpret_cast<const uint4 *>(p.sc + bi * 16);
            d = p.d[bi];
        }
    }
    __device__ __forceinline__ void expand(uint8_t *buf, uint8_t *blk, int c, int h, int g, uint32_t k64) {
        if (g == 0 && h == 0) reinterpret_cast<float *>(blk)[c] = f16_to_f32((uint16_t)d);
        const int n2 = g >> 1, hw = g & 1;
        const uint32_t sw = g == 0 ? scv.x : g == 1 ? scv.y : g == 2 ? scv.z : scv.w;  // sub-blocks 4 g .. 4 g + 3
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {  // chunk 2 g + kk: 16 elements, sub-block 4 g + 2 kk + h
            const int sc = __builtin_amdgcn_sbfe((int)sw, 16 * kk + 8 * h, 8);
            const _Float16 se = (_Float16)(float)(sc & ~1), so = (_Float16)(float)(sc & 1);
            uint32_t ve[8], vo[8];
#pragma unroll
            for (int e = 0; e < 4; e++) {  // dword e & 1 of piece t = 2 h + e / 2
                const uint2 lq = ql[2 * n2 + (e >> 1)][kk];
                const uint4 hq = qh[e >> 1];
                const uint32_t lw = ((e & 1) ? lq.y : lq.x) >> (4 * hw);
                const uint32_t hd = n2 ? ((e & 1) ? hq.w : hq.z) : ((e & 1) ? hq.y : hq.x);
                const uint32_t C = (lw & 0x0F0F0F0Fu) | (((hd >> (4 * hw + 2 * kk)) & 0x03030303u) << 4);
                const h2 p0 = pair_f16(C, 0x00FF00FFu, k64, (_Float16)1.0f, (_Float16)-1056.0f);  // q - 32
                const h2 p1 = pair_f16(C >> 8, 0x00FF00FFu, k64, (_Float16)1.0f, (_Float16)-1056.0f);
                ve[2 * e] = bits(p0 * (h2){se, se});
                ve[2 * e + 1] = bits(p1 * (h2){se, se});
                vo[2 * e] = bits(p0 * (h2){so, so});
                vo[2 * e + 1] = bits(p1 * (h2){so, so});
            }
            uint8_t *o = buf + ((2 * kk + h) * 8 + (c >> 5)) * 1024 + (c & 31) * 16;
            *reinterpret_cast<uint4 *>(o) = make_uint4(ve[0], ve[1], ve[2], ve[3]);
            *reinterpret_cast<uint4 *>(o + 512) = make_uint4(ve[4], ve[5], ve[6], ve[7]);
            *reinterpret_cast<uint4 *>(o + 32768) = make_uint4(vo[0], vo[1], vo[2], vo[3]);
            *reinterpret_cast<uint4 *>(o + 32768 + 512) = make_uint4(vo[4], vo[5], vo[6], vo[7]);
        }
    }
};

// Workgroup (tile, slice): 32 WM activation rows x 256 weight rows over the 256-element chunks [cps y, + cps). With
// partial the slice's products go to partial[y][m][n], else to c.
template <int DT, int WM, int CT>
__global__ __launch_bounds__(FG_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void fast_gemm(
    const Planes p, int64_t N, int64_t row0, int64_t M, int64_t K, const float *__restrict__ x,
    const uint8_t *__restrict__ rec, const uint8_t *__restrict__ srec, const float *__restrict__ sx,
    const int *__restrict__ ex, const int *__restrict__ bad, int64_t cps, float *__restrict__ c, float *__restrict__ partial, int acc_c) {
    using L = Fg<DT>;
    constexpr bool KQ = L::KQ;
    constexpr int TM = 32 * WM, PL = L::PL, TERMS = L::TERMS;
    static_assert(FG_W / WM * CT * 32 == FG_TN, "the waves cover the tile");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w % WM, wn = w / WM;
    int64_t tmi, tni;
    tile_of(blockIdx.x, (M + TM - 1) / TM, (N + FG_TN - 1) / FG_TN, tmi, tni);
    const int64_t n0 = tni * FG_TN, m0 = tmi * TM, mtiles = (M + 31) / 32;
    const int64_t mt = m0 / 32 + wm < mtiles ? m0 / 32 + wm : mtiles - 1;  // (a repeated last tile is not stored)
    const int ns = (int)((K + 63) / 64), nch = (ns + 3) / 4;
    const int ch0 = (int)(blockIdx.y * cps), ch1 = (int)(ch0 + cps < nch ? ch0 + cps : nch);
    const int col = tid & 255, h = tid >> 8;
    const int64_t wrow = row0 + (n0 + col < N ? n0 + col : N - 1);
    auto bufp = [&](int i) { return lds + i * L::BUF; };
    auto blkp = [&](int i) { return lds + 2 * L::BUF + i * L::BLK; };
    const uint8_t *arec = rec + mt * (4 * (int64_t)ns) * (TERMS * 1024);  // wave-uniform
    const uint32_t l16 = 16 * (uint32_t)lane;
    auto clamp_s = [&](int s) { return s < ns ? s : ns - 1; };
    auto clamp_c = [&](int ch) { return ch < nch ? ch : nch - 1; };

    const uint32_t k64 = hide(0x64006400u);
    ColW<DT> W;
    v8h A[4][TERMS];
    if constexpr (KQ) {
#pragma unroll
        for (int g = 0; g < 4; g++) W.load(p, wrow, ch0, h, g);
        if constexpr (DT == kQ4K) {
            W.load_hdr(p, wrow, ch0);
            W.constants(blkp(ch0 & 1), col, h);
            lds_barrier();
            W.load_hdr(p, wrow, clamp_c(ch0 + 1));
        }
        W.expand(bufp(0), blkp(ch0 & 1), col, h, 0, k64);
        if (DT == kQ4K) W.load(p, wrow, clamp_c(ch0 + 1), h, 0);
    } else {
        W.load(p, wrow, 4 * ch0, h, 0);
        W.load(p, wrow, clamp_s(4 * ch0 + 1), h, 1);
        W.expand(bufp(0), col, h, 0);
        W.load(p, wrow, clamp_s(4 * ch0 + 2), h, 0);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
        for (int t = 0; t < TERMS; t++)
            A[ks][t] = *reinterpret_cast<const v8h *>(arec + (int64_t)((16 * ch0 + ks) * TERMS + t) * 1024 + l16);

    float acc[CT][16];
#pragma unroll
    for (int t = 0; t < CT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.0f;
    v16f D[KQ ? CT : 1];
    // the registers of operand step ks are refilled with the next step's as soon as they have been multiplied
    auto refill = [&](int ks, int s) {
        const uint8_t *an = arec + (int64_t)((4 * clamp_s(s + 1) + ks) * TERMS) * 1024;
#pragma unroll
        for (int t = 0; t < TERMS; t++) A[ks][t] = *reinterpret_cast<const v8h *>(an + 1024 * t + l16);
    };

    // Fold block ch (k-quants) into the sums: its value times the power of two of (activation row, block).
    auto fold = [&](int ch) {
        const uint8_t *kb = blkp(ch & 1);
        const float4 *xp = reinterpret_cast<const float4 *>(sx + (mt * nch + ch) * 32) + (lane >> 5);
        float s8[16];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 u = xp[2 * q];
            s8[4 * q] = u.x, s8[4 * q + 1] = u.y, s8[4 * q + 2] = u.z, s8[4 * q + 3] = u.w;
        }
        const float *dk = reinterpret_cast<const float *>(kb + L::CO) + 32 * CT * wn + (lane & 31);
        if constexpr (DT == kQ4K) {
            const v8h *so = reinterpret_cast<const v8h *>(srec + (mt * nch + ch) * 2048) + lane;
            const v8h S0 = so[0], S1 = so[64];
            const v8h *co = reinterpret_cast<const v8h *>(kb) + 32 * CT * wn + (lane & 31);
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const v8h vh = co[32 * t], vl = co[FG_TN + 32 * t];
                v16f V = __builtin_amdgcn_mfma_f32_32x32x16_f16(S1, lane < 32 ? vl : vh, (v16f){0.0f}, 0, 0, 0);
                V = __builtin_amdgcn_mfma_f32_32x32x16_f16(S0, vh, V, 0, 0, 0);
                const float dv = dk[32 * t], sv = dk[FG_TN + 32 * t];
#pragma unroll
                for (int v = 0; v < 16; v++) acc[t][v] = fmaf(fmaf(dv, D[t][v], sv * V[v]), s8[v], acc[t][v]);
            }
        } else if constexpr (DT == kQ6K) {
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const float dv = dk[32 * t];
#pragma unroll
                for (int v = 0; v < 16; v++) acc[t][v] = fmaf(dv, D[t][v] * s8[v], acc[t][v]);
            }
        }
    };
    for (int ch = ch0; ch < ch1; ch++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int s = 4 * ch + g;
            if (!KQ && s >= ns) break;  // workgroup-uniform: the ragged tail of q8_0 / q4_0
            lds_barrier();  // step s is in buffer g & 1, and nobody reads the other one any more
            if (KQ && g == 0 && ch > ch0) fold(ch - 1);
            // The products, (operand step, plane) pairs in turn with the next pair's B operands in flight. q8_0 / q4_0:
            // column tile by column tile within a block, each tile's d D folded in under the next one's MFMAs; the first
            // terms are summed apart from the small ones, for a sum over all of them rounds at full size six times a block
            // (error against float64 at 14336 x 2048 1.77e-7, two f16 terms 1.57e-7, apart 1.42e-7, for 3% of the time).
            const uint8_t *bb = bufp(g & 1) + (wn * CT) * 1024 + 16 * lane;
            if constexpr (KQ) {
                v8h B[2][CT];
                auto load_b = [&](int i) {
#pragma unroll
                    for (int t = 0; t < CT; t++)
                        B[i & 1][t] = *reinterpret_cast<const v8h *>(bb + (i % PL) * 32768 + (i / PL) * 8192 + t * 1024);
                };
                load_b(0);
#pragma unroll
                for (int i = 0; i < 4 * PL; i++) {
                    const int ks = i / PL;
                    if (i + 1 < 4 * PL) load_b(i + 1);
#pragma unroll
                    for (int q = 0; q < 2; q++)
#pragma unroll
                        for (int t = 0; t < CT; t++)
                            D[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                A[ks][q], B[i & 1][t], g == 0 && i == 0 && q == 0 ? (v16f){0.0f} : D[t], 0, 0, 0);
                    if (i % PL == PL - 1) refill(ks, s);
                }
            } else {
                const float *ds = reinterpret_cast<const float *>(bufp(g & 1) + L::B) + 32 * CT * wn + (lane & 31);
                v8h B[2][2];  // [tile parity][step of the block]
                auto load_b = [&](int i) {  // tile i % CT of block i / CT
#pragma unroll
                    for (int k = 0; k < 2; k++)
                        B[i & 1][k] = *reinterpret_cast<const v8h *>(bb + (2 * (i / CT) + k) * 8192 + (i % CT) * 1024);
                };
                v16f E[2];
                float dv[2];
                load_b(0);
#pragma unroll
                for (int i = 0; i < 2 * CT; i++) {
                    const int blk = i / CT, t = i % CT;
                    if (i + 1 < 2 * CT) load_b(i + 1);
                    dv[i & 1] = ds[FG_TN * blk + 32 * t];
                    v16f e = (v16f){0.0f}, rest = (v16f){0.0f};
#pragma unroll
                    for (int q = TERMS - 1; q >= 0; q--)
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            v16f &o = q ? rest : e;
                            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, A[2 * blk + k][q]),
                                                                        __builtin_bit_cast(v8b, B[i & 1][k]), o, 0, 0, 0);
                        }
#pragma unroll
                    for (int v = 0; v < 16; v++) E[i & 1][v] = e[v] + rest[v];
                    if (t == CT - 1) {
                        refill(2 * blk, s);
                        refill(2 * blk + 1, s);
                    }
                    if (i) {
                        const int u = (i - 1) % CT;
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[u][v] = fmaf(dv[(i - 1) & 1], E[(i - 1) & 1][v], acc[u][v]);
                    }
                }
#pragma unroll
                for (int v = 0; v < 16; v++) acc[CT - 1][v] = fmaf(dv[1], E[1][v], acc[CT - 1][v]);
            }
            {  // expand step s + 1, and request what follows it
                uint8_t *nb = bufp((g + 1) & 1);
                if constexpr (KQ) {
                    const int gn = (g + 1) & 3;
                    W.expand(nb, blkp((g == 3 ? ch + 1 : ch) & 1), col, h, gn, k64);
                    if constexpr (DT == kQ4K) {
                        W.load(p, wrow, clamp_c(g == 3 ? ch + 2 : ch + 1), h, gn);
                        if (g == 2) {
                            W.constants(blkp((ch + 1) & 1), col, h);
                            W.load_hdr(p, wrow, clamp_c(ch + 2));
                        }
                    } else if (g == 2) {
#pragma unroll
                        for (int q = 0; q < 4; q++) W.load(p, wrow, clamp_c(ch + 1), h, q);
                    }
                } else {
                    W.expand(nb, col, h, (g + 1) & 1);
                    W.load(p, wrow, clamp_s(s + 3), h, (g + 1) & 1);
                }
            }
        }
    }
    if (KQ) fold(ch1 - 1);

    float *dst = partial ? partial + (int64_t)blockIdx.y * M * N : c;
    const bool add = acc_c && !partial;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int64_t m = m0 + 32 * wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const int e = ex[m < M ? m : M - 1];
        const bool ok = m < M && (!KQ || !bad[m < M ? m : M - 1]);
#pragma unroll
        for (int t = 0; t < CT; t++) {
            const int64_t n = n0 + 32 * (CT * wn + t) + (lane & 31);
            if (ok && n < N) {
                const float y = ldexpf(acc[t][v], e);
                float *o = dst + m * N + n;
                *o = add ? *o + y : y;
            }
        }
    }
    if constexpr (!KQ) return;  // (NaN and Inf are ordinary terms there)
    // rows holding NaN/Inf: exact float dot products (in the first slice; the others add +0); rare
    if (!__syncthreads_or(tid < TM && m0 + tid < M && bad[m0 + tid])) return;
    for (int i = tid; i < TM * FG_TN; i += FG_THREADS) {
        const int64_t m = m0 + i / FG_TN, n = n0 + i % FG_TN;
        if (m >= M || n >= N || !bad[m]) continue;
        const float y = blockIdx.y == 0 ? exact_dot_row<DT>(p, row0 + n, x + m * K, K) : 0.0f;
        float *o = dst + m * N + n;
        *o = add ? *o + y : y;
    }
}

// c[i] (+)= the slices' sum in slice order; or, swi: out[m, i] = silu(g) u over [gate | up] columns (N = 2 I).
template <bool SWI>
__global__ __launch_bounds__(256) void slice_sum(const float *__restrict__ partial, float *__restrict__ c, int64_t M,
                                                 int64_t N, int64_t ns, int acc) {
    const int64_t MN = M * N, W = SWI ? N / 2 : N, total = M * W;
    auto at = [&](int64_t i) {
        float s = partial[i];
        for (int64_t k = 1; k < ns; k++) s = s + partial[k * MN + i];
        return s;
    };
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (int64_t)gridDim.x * 256) {
        if (SWI) {
            const int64_t m = t / W, i = m * N + t % W;
            c[t] = silu_ref(at(i)) * at(i + W);
        } else {
            const float s = at(t);
            c[t] = acc ? c[t] + s : s;
        }
    }
}

template <int DT, int WM, int CT>
int run(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, const uint8_t *rec,
        const uint8_t *srec, const float *sx, const int *ex, const int *bad, int64_t cps, int64_t nsl, float *c, float *partial, int64_t M,
        bool acc) {
    const auto kern = &fast_gemm<DT, WM, CT>;
    const int st = allow_dyn_lds(ctx, reinterpret_cast<const void *>(kern), Fg<DT>::LDS, "fast_gemm: LDS size");
    if (st != TRHIP_OK) return st;
    const int64_t tiles = ((M + 32 * WM - 1) / (32 * WM)) * ((N + FG_TN - 1) / FG_TN);
    if (tiles >= ((int64_t)1 << 31)) return fail(ctx, TRHIP_ERR_UNSUPPORTED, "fast_gemm: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)nsl), dim3(FG_THREADS), Fg<DT>::LDS, ctx->stream, w->planes(),
                       N, row0, M, w->K, x, rec, srec, sx, ex, bad, cps, c, partial, acc ? 1 : 0);
    return launch_check(ctx, "fast_gemm");
}

template <int DT>
int run_dt(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, const uint8_t *rec,
           const uint8_t *srec, const float *sx, const int *ex, const int *bad, int64_t cps, int64_t nsl, float *c, float *partial,
           int64_t M, bool acc, int wm) {
    if (wm == 1) return run<DT, 1, 1>(ctx, w, row0, N, x, rec, srec, sx, ex, bad, cps, nsl, c, partial, M, acc);
    if (wm == 2) return run<DT, 2, 2>(ctx, w, row0, N, x, rec, srec, sx, ex, bad, cps, nsl, c, partial, M, acc);
    return run<DT, 4, 4>(ctx, w, row0, N, x, rec, srec, sx, ex, bad, cps, nsl, c, partial, M, acc);
}

}  // namespace

namespace {

// Row-tile height (in 32s) and K slices: as many slices as still fit one workgroup per CU, of at least two chunks.
struct Tiling {
    int wm;
    int64_t tiles, nch, nsl, cps;
    double us;  // estimated
};

// Estimated time, fitted to measured ones (four formats, 256 to 128256 weight rows, K 256 to 14336, 17 to 2048 activation
// rows, cold weights; within 7% rms).
Tiling tiling_of(int wm, int dtype, int64_t M, int64_t N, int64_t K, int64_t cus) {
    Tiling t;
    t.wm = wm;
    t.tiles = ((M + 32 * wm - 1) / (32 * wm)) * ((N + FG_TN - 1) / FG_TN);
    t.nch = (K + 255) / 256;
    t.nsl = cus / t.tiles;
    if (t.nsl > t.nch / 2) t.nsl = t.nch / 2;
    if (t.nsl < 1) t.nsl = 1;
    t.cps = (t.nch + t.nsl - 1) / t.nsl;
    t.nsl = (t.nch + t.cps - 1) / t.cps;
    static constexpr double chunk[4][3] = {{7.0, 8.6, 11.7}, {5.4, 7.0, 10.6}, {3.9, 4.9, 8.0}, {6.4, 8.5, 12.7}};
    const double c = chunk[dtype == kQ8 ? 0 : dtype == kQ4 ? 1 : dtype == kQ4K ? 2 : 3][wm / 2];
    const int64_t rounds = (t.tiles * t.nsl + cus - 1) / cus;
    t.us = (double)rounds * (17.0 + (double)t.cps * c) + (double)(M * K) * 4e-6 / 3.0;
    if (t.nsl > 1) t.us += 3.5 + (double)(t.nsl * M * N) * 8e-6 / 4.0;
    return t;
}
Tiling tiling(int dtype, int64_t M, int64_t N, int64_t K, int64_t cus) {
    const int wm = M <= 32 ? 1 : M <= 64 ? 2 : 4;
    const Tiling t = tiling_of(wm, dtype, M, N, K, cus);
    if (wm == 1) return t;
    // half the height where that saves padded rows or fills the CUs (q4_k 20000 x 2048, 192 rows: 83 us in 128s, 66 in 64s)
    // and leaves no fewer slices: longer sums round more (q8_0 10240 x 4096, 192 rows, two slices for three: error against
    // float64 1.50e-7 for 1.43e-7)
    const Tiling half = tiling_of(wm / 2, dtype, M, N, K, cus);
    return half.us < 0.95 * t.us && half.cps <= t.cps ? half : t;
}

}  // namespace

// Where the two splitting launches and the 256-column tiles pay. q8_0 / q4_0, exact below: by estimated time (us, exact
// against this: 1024 x 4096, 64 rows q8_0 17, 38; 4096 x 4096, 64 rows 38, 41; 14336 x 4096, 32 rows 78, 54; 300 rows 575,
// 195). q4_k, int8 digits below: from 7.5e9 multiply-adds (128 rows: 14336 x 4096 69, 68; 4096 x 4096 30, 44). q6_k,
// 16-row f16 tiles below: from 4e9 (128 rows of 4096 x 4096 39, 52; 256 rows 59, 62). Past their lines a few shapes of the
// k-quants would still be faster on the kernels below (20000 x 2048, 400 rows q4_k 157 here, 122), which are further from
// float64 (4096 x 4096, 512 rows, x with a mean of 1, q4_k 1.5e-7 here, 1.1e-6). Rows below 256 elements stay exact: with
// so few sums the exact chain is nearer to float64 (K = 32: 4.9e-8 against 5.4e-8).
bool fast_gemm_pays(int dtype, int64_t M, int64_t N, int64_t K, int64_t cus) {
    if (M <= 16 || K < 256) return false;
    const double macs = (double)M * (double)N * (double)K;
    if (dtype == kQ4K) return macs >= 7.5e9;
    if (dtype == kQ6K) return macs >= 4e9;
    return tiling(dtype, M, N, K, cus).us < 0.95 * gemm_rows_time(dtype, M, N, K, cus);
}

bool fast_gemm_applies(const trhip_ctx *ctx, int dtype, int64_t M, int64_t N, int64_t K) {
    if (ctx->force_fast_gemm) return ctx->force_fast_gemm == 1 && M > 16 && K >= 256;
    return fast_gemm_pays(dtype, M, N, K, ctx->sm_count > 0 ? ctx->sm_count : 256);
}

int launch_fast_gemm(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, float *c, int64_t M,
                     bool acc, float *swi) {
    const int64_t K = w->K, np = (K + 1023) / 1024, mt = (M + 31) / 32, KS = (K + 63) / 64 * 4;
    const Tiling tl = tiling(w->dtype, M, N, K, ctx->sm_count > 0 ? ctx->sm_count : 256);
    const int64_t nch = tl.nch, nsl = tl.nsl, cps = tl.cps;
    const int wm = tl.wm;
    auto al = [](size_t v) { return (v + 255) / 256 * 256; };
    const bool copy_x = reinterpret_cast<uintptr_t>(x) % 16 != 0;
    const bool kq = w->dtype == kQ4K || w->dtype == kQ6K;
    const size_t o_s = al((size_t)(mt * KS) * (kq ? 2048 : 3072));
    const size_t o_sx = al(o_s + (w->dtype == kQ4K ? (size_t)(mt * nch) * 2048 : 0));
    const size_t o_pm = al(o_sx + (kq ? (size_t)(mt * nch) * 32 * sizeof(float) : 0));
    const size_t o_ex = al(o_pm + (size_t)(M * np) * sizeof(float)), o_bad = al(o_ex + (size_t)M * sizeof(int));
    const size_t o_x = al(o_bad + (size_t)M * sizeof(int));
    const size_t o_p = al(o_x + (copy_x ? (size_t)(M * K) * sizeof(float) : 0));
    const size_t total = o_p + (nsl > 1 ? (size_t)(nsl * M * N) * sizeof(float) : 0);
    if (total > ctx->ws_bytes && capturing(ctx)) return -1;
    int st = TRHIP_OK;
    uint8_t *ws = static_cast<uint8_t *>(workspace(ctx, total, &st));
    if (!ws) return st;
    const float *xa = x;
    if (copy_x) {
        hipError_t e = hipMemcpyAsync(ws + o_x, x, (size_t)(M * K) * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) return hip_fail(ctx, e, "fast_gemm: align x");
        xa = reinterpret_cast<const float *>(ws + o_x);
    }
    float *pm = reinterpret_cast<float *>(ws + o_pm), *sx = reinterpret_cast<float *>(ws + o_sx);
    int *ex = reinterpret_cast<int *>(ws + o_ex), *bad = reinterpret_cast<int *>(ws + o_bad);
    auto split = [&](auto max_kernel, auto split_kernel) {
        hipLaunchKernelGGL(max_kernel, dim3((unsigned)((M * np + 3) / 4)), dim3(256), 0, ctx->stream, xa, M, K, np, pm);
        hipLaunchKernelGGL(split_kernel, dim3((unsigned)(mt * nch)), dim3(256), 0, ctx->stream, xa, M, K, np, pm, ws,
                           ws + o_s, sx, ex, bad);
    };
    if (w->dtype == kQ4K) split(row_max_kernel<false>, split_kernel<kQ4K>);
    else if (w->dtype == kQ6K) split(row_max_kernel<false>, split_kernel<kQ6K>);
    else split(row_max_kernel<true>, split_kernel<kQ8>);  // (as for kQ4)
    if ((st = launch_check(ctx, "fast_gemm: split")) != TRHIP_OK) return st;
    float *partial = nsl > 1 ? reinterpret_cast<float *>(ws + o_p) : nullptr;
#define TRHIP_FG(DT) st = run_dt<DT>(ctx, w, row0, N, xa, ws, ws + o_s, sx, ex, bad, cps, nsl, c, partial, M, acc, wm)
    switch (w->dtype) {
    case kQ8: TRHIP_FG(kQ8); break;
    case kQ4: TRHIP_FG(kQ4); break;
    case kQ4K: TRHIP_FG(kQ4K); break;
    case kQ6K: TRHIP_FG(kQ6K); break;
    default: return fail(ctx, TRHIP_ERR_INVALID, "fast_gemm: bad dtype");
    }
#undef TRHIP_FG
    if (st != TRHIP_OK) return st;
    if (!partial) return swi ? launch_swiglu(ctx, c, M, N / 2, swi) : TRHIP_OK;
    const int64_t outs = swi ? M * (N / 2) : M * N;
    const unsigned blocks = (unsigned)((outs + 255) / 256 < 4096 ? (outs + 255) / 256 : 4096);
    if (swi)
        hipLaunchKernelGGL(slice_sum<true>, dim3(blocks), dim3(256), 0, ctx->stream, partial, swi, M, N, nsl, 0);
    else
        hipLaunchKernelGGL(slice_sum<false>, dim3(blocks), dim3(256), 0, ctx->stream, partial, c, M, N, nsl, acc ? 1 : 0);
    return launch_check(ctx, "slice_sum");
}

}  // namespace trhip
