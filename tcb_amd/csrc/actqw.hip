// actqw.hip -- act-quant product for q4_k and q6_k weights with the blocks of a row dealt over the waves of a
// workgroup, bit-identical to dotQ4KQ8Go / dotQ6KQ8Go (tensor/cpu_quant_q8.go:91-116, 378-407). Taken where the 128 x 256
// tiles of prefill.hip would not fill the device, decode (M = 1) up to a few hundred rows; q4_k grids between the two, of
// 160 tiles of 64 x 128 and more, stay on actq_mfma.hip (actq_blocks_applies).
//
// Per block b and output (m, n) the reference adds one fp32 value, blocks in order: acc = fl(acc + v_b) with
//   q4_k: v_b = fl(fl(fl(d fl(isum)) - fl(dmin fl(msum))) d8)      q6_k: v_b = fl(fl(d fl(X)) d8)
// (isum, msum, X exact integers; see prefill.hip for the two int8 planes they are built from). Only the sum is ordered:
// the v_b are independent. So a workgroup owns 32 weight rows and 32 MT activation rows, its W waves compute the v_b
// of W consecutive blocks at once, each for the whole tile, and leave them in LDS, where every output is then advanced
// by W additions in block order.
//
// Why this split. A kernel whose waves own outputs walks all blocks of a row in turn, and its grid is the output's
// tiles: q6_k 4096 x 14336 at 130 rows ran 96 workgroups of 56 serial blocks, each wave expanding its weights for 64
// activation rows only (366 us), and M = 1 ran a thread per output (q4_k 14336 x 4096 23 us). Here the grid is N / 32
// tiles times 4 to 8 waves whatever K is, a weight block is expanded once for up to 96 activation rows, and the exchange
// costs 8 KB of LDS traffic per 32 x 32 tile and block, beside 16 int8 MFMAs and about 100 VALU: 49.7 and 11.9 us. What
// bounds it: VALU issue and the waits for it at two waves per SIMD (q6_k at 130 rows: 814 VALU per block, 440 of them the
// expansion; of a SIMD's time VALU is active half, MFMA 19%: profiles/fast_gemm_and_actq_blocks.txt); at M = 1 the start of
// each workgroup, then the weight bytes.
#include "trhip_internal.hpp"
#include "mfma_util.hpp"

#include <type_traits>

namespace trhip {
namespace {

constexpr int AW_TN = 32;  // weight rows per wave (one MFMA column tile)

// A wave's weight block of R rows on its way through LDS. The matrix operands want a row per lane, and loads in that
// shape touch 64 cache lines per instruction, which bounds a CU by its line rate well below HBM (M = 1, 14336 x 4096:
// 16 us). So lanes load 16-byte pieces of the rows' images in order (piece P = 64 i + lane is piece P % PIECES of row
// P / PIECES, whole lines per instruction), the wave writes them to its own part of LDS and each lane reads its row
// back. The pitch (an odd number of 16-byte units) puts 16 consecutive rows on distinct banks.
template <int DT, int R>
struct Raw {
    static constexpr int PIECES = DT == kQ4K ? 9 : 13;  // q4_k: 8 code pieces, the header; q6_k: 8 ql, 4 qh, the scales
    static constexpr int PITCH = 16 * PIECES;
    static constexpr int BYTES = R * PITCH;
    static constexpr int LOADS = (R * PIECES + 63) / 64;
    v4i v[LOADS];
    uint32_t d;  // q6_k: the fp16 scale of row lane % R
    // rows n0 .. n0 + R - 1 of a slice of N rows starting at store row row0; rows past the slice repeat its last
    __device__ __forceinline__ void load(const Planes &p, int64_t row0, int64_t n0, int64_t N, int b, int lane) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            int P = 64 * i + lane;
            P = P < R * PIECES ? P : R * PIECES - 1;
            const int rr = P / PIECES, q = P % PIECES;
            const int64_t bi = (row0 + (n0 + rr < N ? n0 + rr : N - 1)) * p.nb + b;
            const uint8_t *s;
            if (DT == kQ4K) s = q < 8 ? p.qs + bi * 128 + 16 * q : p.aux + bi * 16;
            else s = q < 8 ? p.qs + bi * 128 + 16 * q : q < 12 ? p.aux + bi * 64 + 16 * (q - 8) : p.sc + bi * 16;
            v[i] = *reinterpret_cast<const v4i *>(s);
        }
        if (DT == kQ6K) {
            const int64_t n = n0 + lane % R;
            d = p.d[(row0 + (n < N ? n : N - 1)) * p.nb + b];
        }
    }
    __device__ __forceinline__ void store(uint8_t *l, int lane) const {
#pragma unroll
        for (int i = 0; i < LOADS; i++)
            if (64 * (i + 1) <= R * PIECES || 64 * i + lane < R * PIECES)
                *reinterpret_cast<v4i *>(l + 16 * (64 * i + lane)) = v[i];
    }
};

// Both int8 planes of a block of 32 weight rows, their d (and q4_k: dmin and the msum operand), from the images: lane
// (r = lane % 32, h = lane / 32) takes row r's elements 16 h .. + 15 of every 32-element group, contiguous in the
// lane-sliced planes. q4_k: isum = A.lo + 8 A.hi; q6_k: X = A.lo + 128 A.hi.
template <int DT>
__device__ __forceinline__ void expand_block(const uint8_t *img, int h, uint32_t d16, v4i (&lo)[8], v4i (&hi)[8],
                                             float &dd, float &dm, v8h &bm) {
    uint4 q[4];
#pragma unroll
    for (int g = 0; g < 4; g++) q[g] = *reinterpret_cast<const uint4 *>(img + 64 * h + 16 * g);
    if constexpr (DT == kQ4K) {
        const uint4 hdr = *reinterpret_cast<const uint4 *>(img + 128);
        uint32_t sc_lo, sc_hi, m_lo, m_hi;
        q4k_scales(hdr.y, hdr.z, hdr.w, sc_lo, sc_hi, m_lo, m_hi);
        dd = f16_to_f32((uint16_t)(hdr.x & 0xFFFF));
        dm = f16_to_f32((uint16_t)(hdr.x >> 16));
#pragma unroll
        for (int kc = 0; kc < 8; kc++) {
            const uint4 raw = q[kc >> 1];
            const uint4 nib = (kc & 1) ? make_uint4((raw.x >> 4) & 0x0F0F0F0Fu, (raw.y >> 4) & 0x0F0F0F0Fu,
                                                    (raw.z >> 4) & 0x0F0F0F0Fu, (raw.w >> 4) & 0x0F0F0F0Fu)
                                       : make_uint4(raw.x & 0x0F0F0F0Fu, raw.y & 0x0F0F0F0Fu, raw.z & 0x0F0F0F0Fu,
                                                    raw.w & 0x0F0F0F0Fu);
            const uint32_t sc = ((kc < 4 ? sc_lo : sc_hi) >> (8 * (kc & 3))) & 0xFF;
            lo[kc] = mul16(nib, sc & 7);
            hi[kc] = mul16(nib, sc >> 3);
        }
        bm = small_f16x8(m_lo, m_hi, h ? (_Float16)1.0f : (_Float16)64.0f);
    } else {
        uint4 qh[2];
        qh[0] = *reinterpret_cast<const uint4 *>(img + 128 + 32 * h);
        qh[1] = *reinterpret_cast<const uint4 *>(img + 144 + 32 * h);
        const uint4 sc = *reinterpret_cast<const uint4 *>(img + 192);
        dd = f16_to_f32((uint16_t)d16);
#pragma unroll
        for (int kc = 0; kc < 8; kc++) {
            const int n2 = kc >> 2, k = kc & 3, kk = k & 1;
            uint32_t L[4], H[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint4 lq = q[n2 + 2 * (e >> 1)], hq = qh[e >> 1];
                const int ld = 2 * kk + (e & 1), hd = 2 * n2 + (e & 1);
                L[e] = ld == 0 ? lq.x : ld == 1 ? lq.y : ld == 2 ? lq.z : lq.w;
                H[e] = hd == 0 ? hq.x : hd == 1 ? hq.y : hd == 2 ? hq.z : hq.w;
            }
            const uint32_t sw = (kc >> 1) == 0 ? sc.x : (kc >> 1) == 1 ? sc.y : (kc >> 1) == 2 ? sc.z : sc.w;
            q6_planes(L, H, k, __builtin_amdgcn_sbfe((int)sw, 16 * (kc & 1) + 8 * h, 8), lo[kc], hi[kc]);
        }
    }
}

// Activation operands of one 32-row tile and block in the tiled layout (trhip_internal.hpp): codes, the q4_k msum
// operand and the scales of the lane's output rows. Lanes of rows past the tile's rows read row 0's (their outputs are
// not stored; at M = 1 the other 31 rows would be 8 KB of padding per block).
template <int DT>
struct BlockA {
    v4i a[8];
    v8h s;
    float4 d8[4];
    __device__ __forceinline__ void load(const int8_t *qt, const float *dt, const uint16_t *st, int64_t tb, int rows,
                                         int lane) {
        const int r = lane & 31, h = lane >> 5, l = r < rows ? lane : 32 * h;
        const v4i *q = reinterpret_cast<const v4i *>(qt + tb * 8192) + l;
#pragma unroll
        for (int kc = 0; kc < 8; kc++) a[kc] = q[64 * kc];
        if (DT == kQ4K) s = *(reinterpret_cast<const v8h *>(st + tb * 512) + l);
        const float *dr = dt + tb * 32 + 4 * h;
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) d8[q4] = *reinterpret_cast<const float4 *>(dr + 8 * q4);
    }
};

// The value of output (row 8 q + 4 h + i, column c) of tile t and wave w is component i of ex[w][(8 t + 2 q + h) 32 + c]:
// one 16-byte store per four outputs, whole 1 KB runs per wave, and the same for the reads of the sums.
template <int DT, int MT, int W, int CW>
struct Aw {
    static constexpr int BW = W / CW;                      // blocks a round
    static constexpr int TN = AW_TN * CW;                   // weight rows per workgroup
    static constexpr int SLOTS = MT * 256;                  // float4 slots of a wave's tile
    // a wave's region, in float4: its block's images first, then (those read) its values
    static constexpr int REG = SLOTS * 16 > Raw<DT, 32>::BYTES ? SLOTS : Raw<DT, 32>::BYTES / 16;
    static constexpr int BUF = W * REG * 32 <= 131072 ? 2 : 1;  // two buffers (one barrier per round) where they fit
    static constexpr int AHEAD = MT == 1 ? 2 : 1;           // rounds the weights are requested ahead
    static constexpr int OWN = (CW * SLOTS + 64 * W - 1) / (64 * W);  // slots each thread sums
    static constexpr size_t EX = (size_t)BUF * W * REG * 16;
    static constexpr size_t LDS = EX + (32 * MT + 1) * sizeof(int);
};

// FAST (q4_k): the same integer sums, the two products of the epilogue fused (tolerance mode).
template <int DT, int MT, int W, int CW, bool FAST>
__global__ __launch_bounds__(64 * W) void actq_blocks(const Planes p, int64_t N, int64_t row0, int64_t M, int64_t K,
                                                      const float *__restrict__ x, const int8_t *__restrict__ qt,
                                                      const float *__restrict__ dt, const uint16_t *__restrict__ st,
                                                      const uint8_t *__restrict__ bad_blk, float *__restrict__ c,
                                                      int acc) {
    using T = Aw<DT, MT, W, CW>;
    extern __shared__ __align__(16) uint8_t lds[];
    float4 *ex = reinterpret_cast<float4 *>(lds);
    int *rowstate = reinterpret_cast<int *>(lds + T::EX);  // [32 MT] 0 ok, 1 NaN/Inf row, 2 outside M
    int *anybad = rowstate + 32 * MT;
    const int nb = (int)p.nb;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int64_t tmi, tni;
    tile_of(blockIdx.x, (M + 32 * MT - 1) / (32 * MT), (N + T::TN - 1) / T::TN, tmi, tni);
    const int bw = w / CW, cw = w % CW;  // this wave's block of a round, column tile
    const int64_t n0 = tni * T::TN, m0 = tmi * 32 * MT, mt0 = m0 >> 5;
    const int r = lane & 31, h = lane >> 5;
    const int mrows = (int)(M - m0 < 32 * MT ? M - m0 : 32 * MT), nt = (mrows + 31) >> 5;  // valid rows, tiles

    // Weights are requested two rounds ahead into two register sets taken in turn, the first tile's activations one
    // round ahead, in this order: loads complete in order, so a tile's activations never wait for weights requested
    // after them. Every load is unconditional (past the end: the last block or tile again), so every wait count is
    // static; a guarded one makes the compiler wait for everything in flight, a memory latency per round.
    Raw<DT, 32> w0, w1;
    const int64_t nw = n0 + AW_TN * cw;  // this wave's first weight row
    BlockA<DT> A;
    auto clamp_b = [&](int b) { return b < nb ? b : nb - 1; };
    w0.load(p, row0, nw, N, clamp_b(bw), lane);
    A.load(qt, dt, st, mt0 * nb + clamp_b(bw), mrows, lane);
    if (T::AHEAD == 2) w1.load(p, row0, nw, N, clamp_b(bw + T::BW), lane);
    tile_row_flags<32 * MT, 64 * W>(bad_blk, m0, M, nb, rowstate, anybad);

    float4 sum[T::OWN];
#pragma unroll
    for (int i = 0; i < T::OWN; i++) sum[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);

    auto round = [&](Raw<DT, 32> &wn, int r0, int buf) {
        const int b = clamp_b(r0 + bw);
        float4 *xw = ex + (size_t)(buf * W + w) * T::REG;
        uint8_t *img = reinterpret_cast<uint8_t *>(xw);
        wn.store(img, lane);
        __builtin_amdgcn_wave_barrier();
        v4i lo[8], hi[8];
        float dd, dm = 0.0f;
        v8h bm = (v8h){0};
        expand_block<DT>(img + r * Raw<DT, 32>::PITCH, h, wn.d, lo, hi, dd, dm, bm);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < MT; t++) {
            if (t < nt) {
                v16i c0 = (v16i){0}, c1 = (v16i){0};
                v16f cm = (v16f){0.0f};
                if (DT == kQ4K) cm = __builtin_amdgcn_mfma_f32_32x32x16_f16(A.s, bm, cm, 0, 0, 0);
#pragma unroll
                for (int kc = 0; kc < 8; kc++) {
                    c0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(A.a[kc], lo[kc], c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(A.a[kc], hi[kc], c1, 0, 0, 0);
                }
                float4 d8[4];
#pragma unroll
                for (int q = 0; q < 4; q++) d8[q] = A.d8[q];
                const bool last = t + 1 == MT || t + 1 == nt;  // the next round's first tile, or this one's next
                const int64_t nx = last ? mt0 * nb + clamp_b(r0 + T::BW + bw) : (mt0 + t + 1) * nb + b;
                A.load(qt, dt, st, nx, last ? mrows : mrows - 32 * (t + 1), lane);
                if (t + 1 == MT) wn.load(p, row0, nw, N, clamp_b(r0 + T::AHEAD * T::BW + bw), lane);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float s8[4] = {d8[q].x, d8[q].y, d8[q].z, d8[q].w};
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int e = 4 * q + i;
                        float tt;
                        if (DT == kQ6K) tt = dd * (float)(c0[e] + 128 * c1[e]);
                        else if (FAST) tt = fmaf(-dm, cm[e], dd * (float)(c0[e] + 8 * c1[e]));
                        else tt = (dd * (float)(c0[e] + 8 * c1[e])) - (dm * cm[e]);
                        v[i] = tt * s8[i];
                    }
                    xw[(8 * t + 2 * q + h) * 32 + r] = make_float4(v[0], v[1], v[2], v[3]);
                }
            } else if (t + 1 == MT) {
                wn.load(p, row0, nw, N, clamp_b(r0 + T::AHEAD * T::BW + bw), lane);
            }
        }
        lds_barrier();
        const int n = nb - r0 < T::BW ? nb - r0 : T::BW;
#pragma unroll
        for (int i = 0; i < T::OWN; i++) {
            const int s = tid + 64 * W * i;
            const float4 *e = ex + (size_t)(buf * W + s / T::SLOTS) * T::REG + s % T::SLOTS;
            auto add = [&](const float4 &v) {
                sum[i].x = sum[i].x + v.x;
                sum[i].y = sum[i].y + v.y;
                sum[i].z = sum[i].z + v.z;
                sum[i].w = sum[i].w + v.w;
            };
            if (s < CW * T::SLOTS) {
                if (n == T::BW) {  // a full round: every read in flight before the first addition
                    float4 v[T::BW];
#pragma unroll
                    for (int k = 0; k < T::BW; k++) v[k] = e[(size_t)k * CW * T::REG];
#pragma unroll
                    for (int k = 0; k < T::BW; k++) add(v[k]);
                } else {
                    for (int k = 0; k < n; k++) add(e[(size_t)k * CW * T::REG]);
                }
            }
        }
        if (T::BUF == 1) lds_barrier();  // the one buffer is rewritten next
    };
    for (int r0 = 0; r0 < nb; r0 += 2 * T::BW) {
        round(w0, r0, 0);
        if (r0 + T::BW >= nb) break;  // workgroup-uniform
        round(T::AHEAD == 2 ? w1 : w0, r0 + T::BW, T::BUF - 1);
    }

#pragma unroll
    for (int i = 0; i < T::OWN; i++) {
        const int s = tid + 64 * W * i;
        const int64_t gn = n0 + AW_TN * (s / T::SLOTS) + (s & 31);
        const int ts = s % T::SLOTS, t = ts / 256, ml = 32 * t + 4 * ((ts >> 5) % 8);
        if (s < CW * T::SLOTS && t < nt && gn < N) {
            const float v[4] = {sum[i].x, sum[i].y, sum[i].z, sum[i].w};
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (rowstate[ml + k] == 0) {
                    float *o = c + (m0 + ml + k) * N + gn;
                    *o = acc ? *o + v[k] : v[k];
                }
        }
    }
    // rows holding NaN/Inf take the exact fp32 path (quantGemv) on their own; rare
    if (!*anybad) return;
    for (int i = tid; i < 32 * MT * T::TN; i += 64 * W) {
        const int ml = i / T::TN, nl = i % T::TN;
        const int64_t gn2 = n0 + nl;
        if (rowstate[ml] != 1 || gn2 >= N) continue;
        const int64_t gm = m0 + ml;
        const float v = exact_dot_row<DT>(p, row0 + gn2, x + gm * K, K);
        float *o = c + gm * N + gn2;
        *o = acc ? *o + v : v;
    }
}

template <int DT, int MT, int W, int CW, bool FAST>
int go(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, float *c, int64_t M, bool acc,
       const int8_t *qt, const float *dt, const uint16_t *st, const uint8_t *bad) {
    using T = Aw<DT, MT, W, CW>;
    static_assert(T::LDS <= 160 * 1024, "one workgroup per CU");
    const int64_t wgs = ((M + 32 * MT - 1) / (32 * MT)) * ((N + T::TN - 1) / T::TN);
    if (wgs >= ((int64_t)1 << 31)) return fail(ctx, TRHIP_ERR_UNSUPPORTED, "actq_blocks: grid too large");
    const auto kern = &actq_blocks<DT, MT, W, CW, FAST>;
    const int s = allow_dyn_lds(ctx, reinterpret_cast<const void *>(kern), T::LDS, "actq_blocks: LDS size");
    if (s != TRHIP_OK) return s;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * W), T::LDS, ctx->stream, w->planes(), N, row0, M, w->K, x, qt,
                       dt, st, bad, c, acc ? 1 : 0);
    return launch_check(ctx, "actq_blocks");
}

// ---- up to 16 activation rows: 16x16x64 products ----
//
// A 32 x 32 tile computes 32 activation rows whatever M is and holds 64 registers of weight planes. With few rows the
// weight bytes are what has to move, so here a wave takes CT tiles of 16 weight rows through v_mfma_i32_16x16x64_i8 (a
// result is four registers), which leaves room for four waves per SIMD: enough in flight while others expand.
//
// Lane (n = lane % 16, g = lane / 16) is weight row n (B) and activation row n (A) in k-slice g of a 64-element window;
// result register v is activation row 4 g + v of weight row n (the layout of actq.hip's oracle checks).
// A operand of window i from a row's 256 codes (row: a 256-byte row in element order, or the tiled layout).
template <int DT>
__device__ __forceinline__ v4i few_a_row(const int8_t *row, int i, int g) {
    if (DT == kQ6K) return *reinterpret_cast<const v4i *>(row + 64 * i + 16 * g);
    const uint2 a = *reinterpret_cast<const uint2 *>(row + 64 * i + 8 * g);
    const uint2 b = *reinterpret_cast<const uint2 *>(row + 64 * i + 32 + 8 * g);
    return (v4i){(int)a.x, (int)a.y, (int)b.x, (int)b.y};
}
template <int DT>
__device__ __forceinline__ v4i few_a_tiled(const int8_t *tile, int m, int i, int g) {
    if (DT == kQ6K) return *reinterpret_cast<const v4i *>(tile + 1024 * (2 * i + (g >> 1)) + 16 * (m + 32 * (g & 1)));
    const int8_t *t = tile + 2048 * i + 16 * (m + 32 * (g >> 1)) + 8 * (g & 1);
    const uint2 a = *reinterpret_cast<const uint2 *>(t), b = *reinterpret_cast<const uint2 *>(t + 1024);
    return (v4i){(int)a.x, (int)a.y, (int)b.x, (int)b.y};
}

typedef float v4ff __attribute__((ext_vector_type(4)));

// FQ (M = 1): the wave quantizes its block of x itself, so that a decode step's product is one launch.
template <int DT, int CT, int W>
struct Few {
    static constexpr int REG = Raw<DT, 16 * CT>::BYTES / 16;  // a wave's region, in float4: images, then values
    static_assert(REG >= 64 * CT, "the values fit the images' place");
    static constexpr size_t EX = (size_t)2 * W * REG * 16;
    static constexpr int QROW = 256 + 32 + 16;  // a wave's codes and msum operand
    static constexpr size_t QB = (size_t)W * QROW;
    static constexpr size_t LDS = EX + QB + 17 * sizeof(int);
};

// Largest lane value of a non-negative, NaN-free a, in every lane: four rotations inside the 16-lane rows, then the
// four rows' values as scalars (the bits of such floats order as integers).
__device__ __forceinline__ float wave_max(float a) {
    auto rot = [&](auto ctrl) {
        const int o = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a), decltype(ctrl)::value, 0xF, 0xF, true);
        a = fmaxf(a, __builtin_bit_cast(float, o));
    };
    rot(std::integral_constant<int, 0x128>{});  // row_ror:8
    rot(std::integral_constant<int, 0x124>{});
    rot(std::integral_constant<int, 0x122>{});
    rot(std::integral_constant<int, 0x121>{});
    const uint32_t u = __builtin_bit_cast(uint32_t, a);
    auto at = [&](int l) { return (uint32_t)__builtin_amdgcn_readlane((int)u, l); };
    const uint32_t lo = at(0) > at(16) ? at(0) : at(16), hi = at(32) > at(48) ? at(32) : at(48);
    return __builtin_bit_cast(float, lo > hi ? lo : hi);
}
// Sum over the eight lanes of a group: xor 1, xor 2 inside quads, then the mirrored half row.
__device__ __forceinline__ int group8_sum(int s) {
    s += __builtin_amdgcn_update_dpp(0, s, 0xB1, 0xF, 0xF, true);   // quad_perm [1, 0, 3, 2]
    s += __builtin_amdgcn_update_dpp(0, s, 0x4E, 0xF, 0xF, true);   // quad_perm [2, 3, 0, 1]
    s += __builtin_amdgcn_update_dpp(0, s, 0x141, 0xF, 0xF, true);  // row_half_mirror
    return s;
}

template <int DT, int CT, int W, bool FQ, bool FAST>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(DT == kQ6K ? 3 : 4, 4))) void actq_few(
    const Planes p, int64_t N, int64_t row0, int64_t M, int64_t K, const float *__restrict__ x,
    const int8_t *__restrict__ qt, const float *__restrict__ dt, const uint16_t *__restrict__ st,
    const uint8_t *__restrict__ bad_blk, float *__restrict__ c, int acc) {
    using T = Few<DT, CT, W>;
    constexpr int TN = 16 * CT, NT = 64 * W;
    extern __shared__ __align__(16) uint8_t lds[];
    float4 *ex = reinterpret_cast<float4 *>(lds);
    int *rowstate = reinterpret_cast<int *>(lds + T::EX + T::QB);  // [16] 0 ok, 1 NaN/Inf row, 2 outside M
    int *anybad = rowstate + 16;
    const int nb = (int)p.nb;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *qw = lds + T::EX + w * T::QROW;
    const int64_t n0 = (int64_t)blockIdx.x * TN;
    const int ma = n < M ? n : 0;  // rows past M repeat row 0; their outputs are not stored
    auto clamp_b = [&](int b) { return b < nb ? b : nb - 1; };

    // Requested in the order the loop requests them: (the row flags,) a round's weights, its activations, the next
    // round's weights. Loads complete in order and all of these are unconditional, so the waits are the same static
    // counts on every pass (another order here would make the first use of w0 wait for w1 on every pass).
    const int nflags = FQ ? 0 : (int)M * nb;
    uint32_t fl[2] = {0, 0};
    if (!FQ) {
#pragma unroll
        for (int i = 0; i < 2; i++) fl[i] = bad_blk[tid + NT * i < nflags ? tid + NT * i : 0];
    }
    v4i A[4];
    v8h S = (v8h){0};
    float4 d8, xv;
    auto load_act = [&](int b) {
        if (FQ) {
            xv = *(reinterpret_cast<const float4 *>(x + 256 * (int64_t)b) + lane);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) A[i] = few_a_tiled<DT>(qt + (int64_t)b * 8192, ma, i, g);
            if (DT == kQ4K) S = *(reinterpret_cast<const v8h *>(st + (int64_t)b * 512) + ma + 32 * (g & 1));
            d8 = *reinterpret_cast<const float4 *>(dt + (int64_t)b * 32 + 4 * g);
        }
    };
    Raw<DT, 16 * CT> w0, w1;
    w0.load(p, row0, n0, N, clamp_b(w), lane);
    load_act(clamp_b(w));
    w1.load(p, row0, n0, N, clamp_b(W + w), lane);
    if (tid < 16) rowstate[tid] = tid < M ? 0 : 2;
    if (tid == 16) *anybad = 0;
    lds_barrier();
    if (!FQ) {
        auto flag = [&](int i, uint32_t f) {
            if (i < nflags && f) {
                atomicOr(&rowstate[i / nb], 1);
                *anybad = 1;
            }
        };
        flag(tid, fl[0]);
        flag(tid + NT, fl[1]);
        for (int i = tid + 2 * NT; i < nflags; i += NT) flag(i, bad_blk[i]);  // K above 16384 (or W = 4)
    }

    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto round = [&](Raw<DT, 16 * CT> &wn, int r0, int buf) {
        float4 *xw = ex + (buf * W + w) * T::REG;
        uint8_t *img = reinterpret_cast<uint8_t *>(xw);
        if (FQ) {
            int s4;
            const bool bad = __any(non_finite4(xv));
            float d;
            const uint32_t codes = q8_codes(xv, wave_max(amax4(xv)), d, s4);
            d8 = make_float4(d, d, d, d);
            reinterpret_cast<uint32_t *>(qw)[lane] = codes;
            if (DT == kQ4K) {
                s4 = group8_sum(s4);
                if ((lane & 7) == 0) {  // 32-element sums S_j = 64 Sh + Sl as f16
                    _Float16 *o = reinterpret_cast<_Float16 *>(qw + 256);
                    o[lane >> 3] = (_Float16)(float)(s4 >> 6);
                    o[8 + (lane >> 3)] = (_Float16)(float)(s4 & 63);
                }
            }
            if (bad && lane == 0) rowstate[0] = *anybad = 1;
            __builtin_amdgcn_wave_barrier();
            const int8_t *qr = reinterpret_cast<const int8_t *>(qw);
#pragma unroll
            for (int i = 0; i < 4; i++) A[i] = few_a_row<DT>(qr, i, g);
            if (DT == kQ4K) S = *reinterpret_cast<const v8h *>(qr + 256 + 16 * (g & 1));
            __builtin_amdgcn_wave_barrier();
            load_act(clamp_b(r0 + W + w));
        }
        if (DT == kQ4K) S = g < 2 ? S : (v8h){0};  // the product's k-slices 2 and 3 are zero
        wn.store(img, lane);
        __builtin_amdgcn_wave_barrier();
        float4 vals[CT];  // written once every lane has read the images they replace
        const float s8[4] = {d8.x, d8.y, d8.z, d8.w};
#pragma unroll
        for (int t = 0; t < CT; t++) {
            v4i c0 = (v4i){0}, c1 = (v4i){0};
            float v[4];
            const uint8_t *im = img + (16 * t + n) * Raw<DT, 16 * CT>::PITCH;
            if constexpr (DT == kQ4K) {
                // window i, slice g: bytes 32 i + 8 g .. + 7 of the GGUF block, elements 64 i + 8 g .. (low nibbles)
                // and 64 i + 32 + 8 g .. (high)
                const uint4 h = *reinterpret_cast<const uint4 *>(im + 128);
                const uint8_t *qp = im + 64 * (g >> 1) + 8 * (g & 1);
                uint32_t sc_lo, sc_hi, m_lo, m_hi;
                q4k_scales(h.y, h.z, h.w, sc_lo, sc_hi, m_lo, m_hi);
                const float dd = f16_to_f32((uint16_t)(h.x & 0xFFFF)), dm = f16_to_f32((uint16_t)(h.x >> 16));
                const v4ff cm = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    S, small_f16x8(m_lo, m_hi, g ? (_Float16)1.0f : (_Float16)64.0f), (v4ff){0.0f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t sw = i < 2 ? sc_lo : sc_hi, sa = (sw >> (16 * (i & 1))) & 0xFF,
                                   sb = (sw >> (16 * (i & 1) + 8)) & 0xFF;
                    const uint2 q = *reinterpret_cast<const uint2 *>(qp + 16 * i);
                    const uint32_t l0 = q.x & 0x0F0F0F0Fu, l1 = q.y & 0x0F0F0F0Fu, u0 = (q.x >> 4) & 0x0F0F0F0Fu,
                                   u1 = (q.y >> 4) & 0x0F0F0F0Fu;
                    const v4i B0 = (v4i){(int)mul4(l0, sa & 7), (int)mul4(l1, sa & 7), (int)mul4(u0, sb & 7), (int)mul4(u1, sb & 7)};
                    const v4i B1 = (v4i){(int)mul4(l0, sa >> 3), (int)mul4(l1, sa >> 3), (int)mul4(u0, sb >> 3), (int)mul4(u1, sb >> 3)};
                    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[i], B0, c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[i], B1, c1, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float is = (float)(c0[e] + 8 * c1[e]);
                    v[e] = (FAST ? fmaf(-dm, cm[e], dd * is) : (dd * is) - (dm * cm[e])) * s8[e];
                }
            } else {
                // window i, slice g: elements 64 i + 16 g .. + 15 (sub-block 4 i + g), half g % 2 of chunk 2 i + g / 2
                const float dd = f16_to_f32((uint16_t)__shfl((int)wn.d, 16 * t + n));
                const uint4 sc = *reinterpret_cast<const uint4 *>(im + 192);
                uint2 ql[4];
                uint4 qh[2];
#pragma unroll
                for (int i = 0; i < 4; i++)  // i = n2 + 2 tt
                    ql[i] = *reinterpret_cast<const uint2 *>(im + 64 * (g & 1) + 8 * (g >> 1) + 16 * i);
                qh[0] = *reinterpret_cast<const uint4 *>(im + 128 + 32 * (g & 1));
                qh[1] = *reinterpret_cast<const uint4 *>(im + 144 + 32 * (g & 1));
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    // chunk 2 i + g / 2: ql nibble half i % 2, qh bit pair 2 (i % 2) + g / 2, sub-block 4 i + g
                    const int n2 = i >> 1;
                    uint32_t L[4], H[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint2 lq = ql[n2 + 2 * (e >> 1)];
                        const uint4 hq = qh[e >> 1];
                        L[e] = (e & 1) ? lq.y : lq.x;
                        const uint32_t hw = n2 ? ((e & 1) ? hq.w : hq.z) : ((e & 1) ? hq.y : hq.x);
                        H[e] = hw >> (2 * (g >> 1));  // bit pair 2 (i % 2) + g / 2 at bit 4 (i % 2)
                    }
                    const uint32_t sw = i == 0 ? sc.x : i == 1 ? sc.y : i == 2 ? sc.z : sc.w;
                    v4i B0, B1;
                    q6_planes(L, H, 2 * (i & 1), (int)(int8_t)(sw >> (8 * g)), B0, B1);
                    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[i], B0, c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[i], B1, c1, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = (dd * (float)(c0[e] + 128 * c1[e])) * s8[e];
            }
            vals[t] = make_float4(v[0], v[1], v[2], v[3]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < CT; t++) xw[64 * t + lane] = vals[t];
        if (!FQ) load_act(clamp_b(r0 + W + w));
        wn.load(p, row0, n0, N, clamp_b(r0 + 2 * W + w), lane);
        lds_barrier();
        if (tid < 64 * CT) {
            const int k1 = nb - r0 < W ? nb - r0 : W;
            const float4 *e = ex + buf * W * T::REG + tid;
            float4 u[W];
#pragma unroll
            for (int k = 0; k < W; k++) u[k] = e[k * T::REG];
#pragma unroll
            for (int k = 0; k < W; k++)
                if (k < k1) {
                    sum.x = sum.x + u[k].x;
                    sum.y = sum.y + u[k].y;
                    sum.z = sum.z + u[k].z;
                    sum.w = sum.w + u[k].w;
                }
        }
    };
    for (int r0 = 0; r0 < nb; r0 += 2 * W) {
        round(w0, r0, 0);
        if (r0 + W >= nb) break;  // workgroup-uniform
        round(w1, r0 + W, 1);
    }

    if (tid < 64 * CT) {
        const int64_t gn = n0 + 16 * (tid >> 6) + n;
        const float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (gn < N && rowstate[4 * g + e] == 0) {
                float *o = c + (4 * g + e) * N + gn;
                *o = acc ? *o + v[e] : v[e];
            }
    }
    // rows holding NaN/Inf take the exact fp32 path (quantGemv) on their own; rare
    if (!*anybad) return;
    for (int i = tid; i < 16 * TN; i += NT) {
        const int ml = i / TN;
        const int64_t gn2 = n0 + i % TN;
        if (rowstate[ml] != 1 || gn2 >= N) continue;
        const float v = exact_dot_row<DT>(p, row0 + gn2, x + ml * K, K);
        float *o = c + ml * N + gn2;
        *o = acc ? *o + v : v;
    }
}

template <int DT, int CT, int W, bool FQ, bool FAST>
int go_few(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, float *c, int64_t M, bool acc,
           const int8_t *qt, const float *dt, const uint16_t *st, const uint8_t *bad) {
    using T = Few<DT, CT, W>;
    const int64_t wgs = (N + 16 * CT - 1) / (16 * CT);
    if (wgs >= ((int64_t)1 << 31)) return fail(ctx, TRHIP_ERR_UNSUPPORTED, "actq_few: grid too large");
    const auto kern = &actq_few<DT, CT, W, FQ, FAST>;
    const int s = allow_dyn_lds(ctx, reinterpret_cast<const void *>(kern), T::LDS, "actq_few: LDS size");
    if (s != TRHIP_OK) return s;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * W), T::LDS, ctx->stream, w->planes(), N, row0, M, w->K, x, qt,
                       dt, st, bad, c, acc ? 1 : 0);
    return launch_check(ctx, "actq_few");
}

template <int DT, bool FAST>
int pick(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, float *c, int64_t M, bool acc,
         const int8_t *qt, const float *dt, const uint16_t *st, const uint8_t *bad) {
#define TRHIP_AW(kern, ...) kern<__VA_ARGS__, FAST>(ctx, w, row0, N, x, c, M, acc, qt, dt, st, bad)
    const int64_t cus = ctx->sm_count > 0 ? ctx->sm_count : 256;
    // Grids of at least one 32-row workgroup per CU take four-wave workgroups (several to a CU, one's start overlapping
    // another's products), smaller ones eight waves, so that a row's blocks need fewer rounds. Cold, us: q4_k M = 1
    // 14336 x 4096 12.7 against 13.2, 4096 x 14336 22.5 against 13.8; q6_k, whose two tiles of images a wave would
    // spill, one tile: 18.4 against 20.2, 21.5 against 18.2.
    const bool wide = N >= 32 * cus;
    if (M == 1) {
        if (!wide) return TRHIP_AW(go_few, DT, 1, 8, true);
        return TRHIP_AW(go_few, DT, (DT == kQ4K ? 2 : 1), 4, true);
    }
    if (M <= 16) {
        if (!wide) return TRHIP_AW(go_few, DT, 1, 8, false);
        return TRHIP_AW(go_few, DT, (DT == kQ4K ? 2 : 1), 4, false);
    }
    if (M <= 32) {
        if (!wide) return TRHIP_AW(go, DT, 1, 8, 1);
        return TRHIP_AW(go, DT, 1, 8, 2);
    }
    // One workgroup fits a CU. While two-tile workgroups make one pass over the CUs they win (q4_k 128 rows, 4096 x
    // 14336: 37 us against 49 on three tiles); then three-tile ones while those do (130 rows: 50 against 59); beyond,
    // two column tiles per workgroup halve what each block's activations are read (256 rows: 63 against 66 and 87).
    const int64_t cols = (N + AW_TN - 1) / AW_TN;
    if (cols * ((M + 63) / 64) <= cus) return TRHIP_AW(go, DT, 2, 8, 1);
    if (cols * ((M + 95) / 96) <= cus) return TRHIP_AW(go, DT, 3, 8, 1);
    return TRHIP_AW(go, DT, 2, 8, 2);
#undef TRHIP_AW
}

}  // namespace

// q4_k: up to 32 rows always, more while the 64-row tiles of actq_mfma.hip would leave CUs idle (fewer than 160
// workgroups; 128 rows, us: 4096 x 14336 37 against 70, 14336 x 4096, 224 tiles, 39 against 37). q6_k: always.
bool actq_blocks_applies(int dtype, int64_t M, int64_t N) {
    if (dtype == kQ6K) return true;
    return dtype == kQ4K && (M <= 32 || ((M + 63) / 64) * ((N + 127) / 128) < 160);
}

bool actq_blocks_quantizes(int64_t M) { return M == 1; }

int launch_actq_blocks(trhip_ctx *ctx, const trhip_wstore *w, int64_t row0, int64_t N, const float *x, float *c,
                       int64_t M, bool acc, const int8_t *qt, const float *dt, const uint16_t *st, const uint8_t *bad,
                       bool fast) {
    if (w->dtype == kQ6K) return pick<kQ6K, false>(ctx, w, row0, N, x, c, M, acc, qt, dt, st, bad);
    if (w->dtype != kQ4K) return fail(ctx, TRHIP_ERR_UNSUPPORTED, "actq_blocks: q4_k or q6_k");
    return fast ? pick<kQ4K, true>(ctx, w, row0, N, x, c, M, acc, qt, dt, st, bad)
                : pick<kQ4K, false>(ctx, w, row0, N, x, c, M, acc, qt, dt, st, bad);
}

}  // namespace trhip
