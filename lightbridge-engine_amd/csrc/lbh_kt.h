// lbh_kt.h — Q4_K / Q5_K rows against 16-token tiles on the f16 matrix cores, one
// wave per 16 rows and tile, bit-identical to the reference's per-row
// dot (dot_q4_or_q5_k, crates/bridge-quant-layout/src/q8_k.rs:247-327).
//
// Per block the eight lane sums (residues mod 8) are one
// v_mfma_f32_16x16x32_f16 each: operand A holds 16 tokens, operand B 16 rows,
// lane 16 q + c the row / token c and the 8 elements of residue t in sub-blocks
// 2q, 2q + 1, the weights pre-multiplied by their 6-bit scale (sc * q <= 1953).
// The minimum sum is one v_mfma_f32_16x16x16_f16 of (128 mn, mn) against the
// bsums pairs split (bh, bl).  All operands are integers an f16 holds and
// every partial sum an integer below 2^24 (32 * 1953 * 128 < 2^23), so the f32
// results are the exact integer sums converted; result i of a lane is (token
// 4q + i, row c).  The nine f32 chains run in the reference's block order,
// result = minimum chain + chain 0 + ... + chain 7.
//
// The weights come from a tile copy (k_kt_pack), per 16 rows x block and in
// lane order: Q4_K 32 bytes a lane (the residue-major dwords of group q: both
// its sub-blocks), Q5_K 64 bytes a lane (the quants as bytes: rebuilding the
// fifth bit from its plane cost as many instructions as the products), then
// the f16 scales and minimums of the lane's sub-blocks (8 bytes) and the rows'
// (d, dmin).  The tokens come as f16 operands (kt_store_piece) from L1 / L2.
//
// What bounds it: VALU issue, 80 instructions per token tile (16 per f32 chain
// step pair and the scales) and about 80 for the weights of a step.
#pragma once
#include "lbh_dev.h"

namespace lbh {

typedef _Float16 kt_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 kt_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 kt_h8 __attribute__((ext_vector_type(8)));
typedef float kt_f4 __attribute__((ext_vector_type(4)));

// Token operand tile (16 tokens, block b): eight residue operands of 64 lanes x
// 16 bytes, the minimum operand of 64 lanes x 8 bytes, the tokens' d8.
constexpr int KT_MIN = 8 * 1024, KT_D8 = KT_MIN + 512, KT_TOK_TILE = KT_D8 + 64;
// Weight tile (16 rows, block b).
template <int TY>
struct KtTile {
    static constexpr int PIECES = TY == T_Q5_K ? 4 : 2;   // 16-byte quant pieces per lane
    static constexpr int SCALES = PIECES * 1024, DD = SCALES + 512, BYTES = DD + 64;
};
__host__ __device__ constexpr size_t kt_w_bytes(int ty, int rows, int nb) {
    return (size_t)(rows / 16) * nb * (ty == T_Q5_K ? KtTile<T_Q5_K>::BYTES : KtTile<T_Q4_K>::BYTES);
}
__host__ __device__ constexpr size_t kt_tok_bytes(int n_tokens, int nb) {
    return (size_t)((n_tokens + 15) / 16) * nb * KT_TOK_TILE;
}

__device__ __forceinline__ kt_h2 kt_pair(uint32_t v) { return __builtin_bit_cast(kt_h2, v); }
__device__ __forceinline__ uint32_t kt_bits(kt_h2 v) { return __builtin_bit_cast(uint32_t, v); }

// One lane's weights of a step.
template <int TY>
struct KtW {
    uint4 x[KtTile<TY>::PIECES];
    uint2 sc;      // f16 scales (low) and minimums of sub-blocks 2q, 2q + 1
    uint32_t dd;   // the row's f16 d, dmin
};

template <int TY>
__device__ __forceinline__ void kt_load(const Planes &P, uint32_t tile, int lane, KtW<TY> &w) {
    const uint32_t base = tile * (uint32_t)KtTile<TY>::BYTES;
#pragma unroll
    for (int p = 0; p < KtTile<TY>::PIECES; ++p) w.x[p] = bld128(P, 16u * lane, base + 1024u * p);
    w.sc = bld64(P, 8u * lane, base + KtTile<TY>::SCALES);
    w.dd = bld32(P, 4u * (lane & 15), base + KtTile<TY>::DD);
}

// The scaled weights of residue t: (1024 + q) * sc - 1024 sc, one fused step
// (exact: every value is an integer below 2^17, the result below 2048; the
// high nibbles stay in place as 1024 + 16 q against sc / 16).
struct KtScales {
    kt_h2 s0, m0, s1, m1;
};
template <int TY>
__device__ __forceinline__ KtScales kt_scales(const KtW<TY> &w) {
    constexpr _Float16 f = TY == T_Q4_K ? (_Float16)0.0625f : (_Float16)1.0f, n = (_Float16)-1024.0f;
    const kt_h2 both = {n, n}, fac = {f, f};
    KtScales k;
    k.s0 = kt_pair(perm(w.sc.x, w.sc.x, 0x01000100u));
    k.s1 = kt_pair(perm(w.sc.x, w.sc.x, 0x03020302u)) * fac;
    k.m0 = k.s0 * both;
    k.m1 = k.s1 * both;
    return k;
}
template <int TY>
__device__ __forceinline__ kt_h8 kt_weights(const KtW<TY> &w, const KtScales &k, int t) {
    uint32_t h[4];
    if constexpr (TY == T_Q4_K) {
        const uint4 v = w.x[t >> 2];
        const uint32_t x = (t & 3) == 0 ? v.x : (t & 3) == 1 ? v.y : (t & 3) == 2 ? v.z : v.w, y = x >> 8;
        h[0] = (x & 0x000f000fu) | 0x64006400u, h[1] = (y & 0x000f000fu) | 0x64006400u;
        h[2] = (x & 0x00f000f0u) | 0x64006400u, h[3] = (y & 0x00f000f0u) | 0x64006400u;
    } else {
        const uint4 v = w.x[t >> 1];
        const uint32_t x = t & 1 ? v.z : v.x, y = t & 1 ? v.w : v.y;
        h[0] = perm(0x64646464u, x, 0x04010400u), h[1] = perm(0x64646464u, x, 0x04030402u);
        h[2] = perm(0x64646464u, y, 0x04010400u), h[3] = perm(0x64646464u, y, 0x04030402u);
    }
    struct {
        uint32_t v[4];
    } o;
    o.v[0] = kt_bits(__builtin_elementwise_fma(kt_pair(h[0]), k.s0, k.m0));
    o.v[1] = kt_bits(__builtin_elementwise_fma(kt_pair(h[1]), k.s0, k.m0));
    o.v[2] = kt_bits(__builtin_elementwise_fma(kt_pair(h[2]), k.s1, k.m1));
    o.v[3] = kt_bits(__builtin_elementwise_fma(kt_pair(h[3]), k.s1, k.m1));
    return __builtin_bit_cast(kt_h8, o);
}
template <int TY>
__device__ __forceinline__ kt_h4 kt_mins(const KtW<TY> &w) {
    const kt_h2 f = {(_Float16)128.0f, (_Float16)1.0f};
    struct {
        uint32_t v[2];
    } o = {{kt_bits(kt_pair(perm(w.sc.y, w.sc.y, 0x01000100u)) * f), kt_bits(kt_pair(perm(w.sc.y, w.sc.y, 0x03020302u)) * f)}};
    return __builtin_bit_cast(kt_h4, o);
}

// Row tile rt (16 rows) of a tile copy (K = 256 nb) against the 16-token tile at tok:
// out(token in the tile, row in the tile, value).  The weights of the next block
// and the token operands of the next RING residues are in flight while a residue
// is computed.
template <int TY, class Out>
__device__ __forceinline__ void kt_rows(const uint8_t *w, size_t w_bytes, int rt, int nb, const uint8_t *tok, Out out) {
    constexpr int RING = 4;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    Planes P;
    P.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(w), (short)0, (int)(uint32_t)w_bytes, 0x00020000);
    KtW<TY> wa, wb;
    kt_h8 ring[RING];
    kt_h4 mn;
    float4 d8;
    float acc[9][4];
#pragma unroll
    for (int c = 0; c < 9; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][i] = 0.0f;
    auto fetch = [&](int t, int b) {   // residue t (static) of block b
        ring[t % RING] = *reinterpret_cast<const kt_h8 *>(tok + (size_t)b * KT_TOK_TILE + 1024 * t + 16 * lane);
    };
    auto fetch_rest = [&](int b) {
        const uint8_t *p = tok + (size_t)b * KT_TOK_TILE;
        mn = *reinterpret_cast<const kt_h4 *>(p + KT_MIN + 8 * lane);
        d8 = *reinterpret_cast<const float4 *>(p + KT_D8 + 16 * q);
    };
    const kt_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto block = [&](int b, const KtW<TY> &cur, KtW<TY> &next) {
        const int bn = b + 1 < nb ? b + 1 : b;   // past the end: reloads the last block, never used
        kt_load<TY>(P, (uint32_t)(rt * nb + bn), lane, next);
        const KtScales k = kt_scales<TY>(cur);
        const float d = f16_to_f32(cur.dd & 0xffffu), dmin = f16_to_f32(cur.dd >> 16);
        float s[4];
        const kt_f4 m = __builtin_amdgcn_mfma_f32_16x16x16f16(mn, kt_mins<TY>(cur), zero, 0, 0, 0);
        const float e[4] = {d8.x, d8.y, d8.z, d8.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = __fmul_rn(d, e[i]);
            acc[8][i] = __fsub_rn(acc[8][i], __fmul_rn(__fmul_rn(dmin, e[i]), m[i]));
        }
        fetch_rest(bn);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const kt_h8 wt = kt_weights<TY>(cur, k, t);
            const kt_f4 r = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[t % RING], wt, zero, 0, 0, 0);
            if (t + RING < 8) fetch(t + RING, b);
            else fetch(t + RING - 8, bn);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][i] = __fadd_rn(acc[t][i], __fmul_rn(s[i], r[i]));
        }
    };
    kt_load<TY>(P, (uint32_t)(rt * nb), lane, wa);
    fetch_rest(0);
#pragma unroll
    for (int t = 0; t < RING; ++t) fetch(t, 0);
    for (int b = 0; b < nb; b += 2) {
        block(b, wa, wb);
        if (b + 1 >= nb) break;
        block(b + 1, wb, wa);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = acc[8][i];
#pragma unroll
        for (int t = 0; t < 8; ++t) v = __fadd_rn(v, acc[t][i]);   // q8_k.rs:323-325
        out(4 * q + i, lane & 15, v);
    }
}

// The token operand pieces of one quantized block (292 Q8_K bytes at blk, LDS)
// of token t, block b of nb: piece k < 32 is lane quarter k % 4 of residue
// k / 4 (elements r, r + 16, r + 8, r + 24 of both sub-blocks), 32 <= k < 36 the
// minimum operand's quarters; piece 32 also writes d8.
__device__ __forceinline__ void kt_store_piece(uint8_t *tok, long long t, int b, int nb, const uint8_t *blk, int k) {
    uint8_t *dst = tok + ((t >> 4) * nb + b) * (long long)KT_TOK_TILE;
    const int c = (int)(t & 15), q = k & 3;
    if (k < 32) {
        const int r = k >> 2;
        kt_h8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            constexpr int at[4] = {0, 16, 8, 24};
            o[e] = (_Float16)(int)(int8_t)blk[4 + 64 * q + 32 * (e >> 2) + at[e & 3] + r];
        }
        *reinterpret_cast<kt_h8 *>(dst + 1024 * r + 16 * (16 * q + c)) = o;
    } else {
        kt_h4 o;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t w = ld_u32(blk + 260 + 4 * (2 * q + e));
            const int bsp = (int)(int16_t)(w & 0xffff) + (int)(int16_t)(w >> 16);
            o[2 * e] = (_Float16)(bsp >> 7), o[2 * e + 1] = (_Float16)(bsp & 127);
        }
        *reinterpret_cast<kt_h4 *>(dst + KT_MIN + 8 * (16 * q + c)) = o;
        if (q == 0) reinterpret_cast<uint32_t *>(dst + KT_D8)[c] = ld_u32(blk);
    }
}
constexpr int KT_STORE_PIECES = 36;

// Tile copy of a Q4_K / Q5_K matrix (rows % 16 == 0): one thread per lane slice.
template <int TY>
__global__ void k_kt_pack(MatView m, uint8_t *dst) {
    const long long n = m.units * 4, U = m.units;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const long long tile = i >> 6;
        const int lane = (int)(i & 63), q = lane >> 4, c = lane & 15;
        const long long u = ((tile / m.nb) * 16 + c) * m.nb + tile % m.nb;
        auto chunk = [&](int k) { return ld_u128(m.planes + ((long long)k * U + u) * 16); };
        constexpr int QS0 = TY == T_Q5_K ? 3 : 1;
        uint8_t *t = dst + tile * KtTile<TY>::BYTES;
        const uint4 hdr = chunk(0), a = chunk(QS0 + 2 * q), b = chunk(QS0 + 2 * q + 1);
        const uint32_t x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        if constexpr (TY == T_Q4_K) {
            reinterpret_cast<uint4 *>(t)[lane] = a;
            reinterpret_cast<uint4 *>(t + 1024)[lane] = b;
        } else {
            const uint4 h0 = chunk(1), h1 = chunk(2);
            const uint32_t qh[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                uint32_t o[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int r = 2 * p + (k >> 1), sub = k & 1;   // residue, sub-block 2q + sub
                    const uint32_t v = ((x[r] >> (4 * sub)) & 0x0f0f0f0fu) | (((qh[r] >> (2 * q + sub)) & 0x01010101u) << 4);
                    o[k] = perm(v, v, 0x03010200u);   // elements r, r + 16, r + 8, r + 24
                }
                reinterpret_cast<uint4 *>(t + 1024 * p)[lane] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
        int32_t sc[2], mn[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) scale_min_of(hdr.y, hdr.z, hdr.w, 2 * q + e, sc[e], mn[e]);
        const kt_h4 s = {(_Float16)sc[0], (_Float16)sc[1], (_Float16)mn[0], (_Float16)mn[1]};
        reinterpret_cast<kt_h4 *>(t + KtTile<TY>::SCALES)[lane] = s;
        if (q == 0) reinterpret_cast<uint32_t *>(t + KtTile<TY>::DD)[c] = hdr.x;
    }
}

}  // namespace lbh
