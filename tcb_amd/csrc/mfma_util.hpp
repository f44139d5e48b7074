// mfma_util.hpp -- helpers shared by the matrix-core kernels (actq_mfma.hip, prefill.hip, actqw.hip): operand
// vector types, the two-plane weight expansions, f16 packing of small integers, tile row states and the XCD-aware
// workgroup-to-tile mapping.
#pragma once

#include "trhip_internal.hpp"

namespace trhip {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Four bytes (each < 16) times s (< 8) with one packed 16-bit multiply: the products (< 128) stay in
// their bytes, so nothing carries into the neighbour.
__device__ __forceinline__ uint32_t mul4(uint32_t nib4, uint32_t s) {
    us2 a = __builtin_bit_cast(us2, nib4);
    us2 r = a * (us2){(unsigned short)s, (unsigned short)s};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ v4i mul16(uint4 nib, uint32_t s) {
    return (v4i){(int)mul4(nib.x, s), (int)mul4(nib.y, s), (int)mul4(nib.z, s), (int)mul4(nib.w, s)};
}

__device__ __forceinline__ uint32_t pack_h2(uint32_t a, uint32_t b) {  // two small integers as f16 bits
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)a) |
           ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)b) << 16);
}

// Eight integers below 64 (the bytes of lo, then hi) times c (1 or 64) as f16: v_perm_b32 places each byte under
// 0x64, giving the f16 value 1024 + v; subtracting 1024 and multiplying by c are both exact (v c <= 4032). (A fused
// (1024 + v) c - 1024 c is not usable: -1024 * 64 is beyond the f16 range.)
__device__ __forceinline__ v8h small_f16x8(uint32_t lo, uint32_t hi, _Float16 c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 cc = (h2){c, c}, off = (h2){(_Float16)(-1024.0f), (_Float16)(-1024.0f)};
    auto pair = [&](uint32_t v, uint32_t sel) {
        const h2 x = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, sel));
        return __builtin_bit_cast(uint32_t, (x + off) * cc);
    };
    return __builtin_bit_cast(v8h, make_uint4(pair(lo, 0x04010400u), pair(lo, 0x04030402u), pair(hi, 0x04010400u),
                                              pair(hi, 0x04030402u)));
}

typedef short pf_s2 __attribute__((ext_vector_type(2)));

// Chunk kc's two B operands for lane (r, h): elements 32 kc + 16 h .. + 15 of the row, the four 4-element groups
// e = 2 tt + hh (tt, hh in 0..1) from ql dword L[e] (nibble half k / 2) and qh dword H[e] (bit pair k = kc % 4), all
// in sub-block 2 kc + h with signed scale sc. Per group: the codes c as bytes, spread to 16-bit pairs, v = c sc - 32 sc
// by packed 16-bit multiply-adds, then the bytes of v >> 7 (h) and of v & 127 (l).
__device__ __forceinline__ void q6_planes(const uint32_t (&L)[4], const uint32_t (&H)[4], int k, int sc, v4i &lo,
                                          v4i &hi) {
    const pf_s2 S = (pf_s2){(short)sc, (short)sc}, O = (pf_s2){(short)(-32 * sc), (short)(-32 * sc)};
    uint32_t lb[4], hb[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t lw = (k >> 1) ? (L[e] >> 4) : L[e];
        const uint32_t hw = k == 0 ? (H[e] << 4) : k == 1 ? (H[e] << 2) : k == 2 ? H[e] : (H[e] >> 2);
        const uint32_t C = (lw & 0x0F0F0F0Fu) | (hw & 0x30303030u);  // codes 0..63
        const pf_s2 c01 = __builtin_bit_cast(pf_s2, __builtin_amdgcn_perm(0u, C, 0x0c010c00u));
        const pf_s2 c23 = __builtin_bit_cast(pf_s2, __builtin_amdgcn_perm(0u, C, 0x0c030c02u));
        const uint32_t v01 = __builtin_bit_cast(uint32_t, c01 * S + O), v23 = __builtin_bit_cast(uint32_t, c23 * S + O);
        lb[e] = __builtin_amdgcn_perm(v23, v01, 0x06040200u) & 0x7F7F7F7Fu;  // low bytes, low 7 bits: v & 127
        hb[e] = __builtin_amdgcn_perm(v23 >> 7, v01 >> 7, 0x06040200u);     // bits 7..14 of each v: v >> 7
    }
    lo = (v4i){(int)lb[0], (int)lb[1], (int)lb[2], (int)lb[3]};
    hi = (v4i){(int)hb[0], (int)hb[1], (int)hb[2], (int)hb[3]};
}

// Row states of a tile of TM activation rows from per-(row, block) NaN/Inf flags flags[row * nb + b]:
// st[r] = 0 (finite), 1 (some block flagged) or 2 (row m0 + r is past M), *any = 1 if some row is 1. Every thread
// takes a share of the flags, so the loads are independent rather than one chain per row. Ends with a barrier.
template <int TM, int THREADS>
__device__ __forceinline__ void tile_row_flags(const uint8_t *__restrict__ flags, int64_t m0, int64_t M, int nb,
                                               int *st, int *any) {
    const int tid = threadIdx.x;
    if (tid < TM) st[tid] = m0 + tid < M ? 0 : 2;
    if (tid == 0) *any = 0;
    __syncthreads();
    constexpr int P = THREADS / TM;  // threads per row
    const int r = tid % TM, part = tid / TM;
    if (m0 + r < M) {
        const uint8_t *f = flags + (m0 + r) * nb;
        int v = 0;
#pragma unroll 8
        for (int b = part; b < nb; b += P) v |= f[b];
        if (v) {
            atomicOr(&st[r], 1);
            *any = 1;
        }
    }
    __syncthreads();
}

// Workgroup -> tile: workgroups are dealt to the 8 XCDs round-robin, so when the tile count allows, XCD x takes a
// contiguous run of column tiles with all their row tiles next to each other: a weight tile is fetched into that
// XCD's L2 once and reused by every row tile.
__device__ __forceinline__ void tile_of(int64_t wg, int64_t mt, int64_t nt, int64_t &tm, int64_t &tn) {
    const int64_t total = mt * nt;
    int64_t t = wg;
    if (total % 8 == 0) t = (wg & 7) * (total / 8) + (wg >> 3);
    tm = t % mt;
    tn = t / mt;
}

}  // namespace
}  // namespace trhip
