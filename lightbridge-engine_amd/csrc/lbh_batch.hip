// lbh_batch.hip — batched decode of a batch of tokens through the MoE layer.
//
// Per token the result is bit-identical to moe_routed_by_id_into
// (crates/bridge-kernels-reference/src/moe.rs:64-147), which the reference
// runs one token at a time (crates/bridge-runtime/src/hy3_scalar.rs:504-650).
// Here the batch's (token, routed expert) pairs are sorted by expert, so each
// selected expert's weights stream from HBM once per chunk of its tokens and
// are decoded once into registers for all of them:
//
//   k_mb_prep     counting sort of the pairs by expert (ascending token order
//                 inside an expert) into a chunk table; Q8_K of every token and
//                 its matrix-core operands;
//   k_mx_gate_up  per (chunk, row tile) on the int8 matrix cores: gate and up
//                 rows against the chunk's tokens, folded in the reference's
//                 block order; the same launch holds the shared expert's
//                 K-quant gate and up (lbh_kt.h);
//   k_mb_quant_h  SwiGLU and the Q8_K operands of every h row (the down
//                 projections' inputs, gemv.rs:161-163);
//   k_mx_down     per (chunk, row tile): the down rows against the chunk's h,
//                 and the shared expert's down;
//   k_mb_combine  per token and output row, in the reference's order:
//                 y = ((0 + c_0 d_0) + c_1 d_1) + ... + 1.0 * d_shared.
//
// k_mb_gate_up / k_mb_down are the same streams on the VALU integer dots, for
// the chunks below a caller's matrix-core threshold
// (lbh_moe_set_batch_engine).  By default every chunk runs on the matrix cores,
// also those of one token: a 16-token tile decodes its weights at the VALU cost
// of a one-token dot (measured, 192 experts of hidden 4096, width 1536, top-8:
// 64 tokens with tile copies 255 us per step, 295 with the one-token chunks on
// the VALU beside; 5 tokens without copies 112 and 143 us).
//
// Several workgroups read the same expert rows (one per chunk of its tokens),
// so the weight loads keep the default cache policy here.
#define LBH_WEIGHT_CPOL 0
#include "lbh_internal.h"
#include "lbh_kt.h"
#include "lbh_math.h"
#include "lbh_router.h"
#include "lbh_rows.h"

namespace lbh {

constexpr int MB_THREADS = 256;
constexpr int MB_WAVES = MB_THREADS / 64;

// A staged Q8_K block in LDS: d at 0, qs at 16, bsums at 272 (16-byte aligned
// quants so a lane's slice is a run of 16-byte reads).
constexpr int Q8L = 304;

// Matrix-core operand copy of Q8_K rows, written beside the GGML bytes by the
// quantize kernels: block k's 256 quants at q + 256 k, its scale at d[k].  Dword
// 16 m + 4 p + i is dword 4 m + i of lane quarter p, so that the four lanes of a
// token read 64 contiguous bytes at a time: elements 64 p + 16 m + 4 i .. + 3 for
// IQ2_S, for IQ3_S (split) elements 32 g + 8 p + 4 h .. + 3 with 2 g + h = 4 m + i.
struct MxRows {
    uint8_t *q;
    float *d;
    bool split;
};

__host__ __device__ constexpr int al16(int v) { return (v + 15) & ~15; }

// ------------------------------------------------------------ activations

template <int G>
__device__ __forceinline__ void load_act_lds(const uint8_t *blk, int p, ActIQ<G> &a) {
    a.d8 = __uint_as_float(*reinterpret_cast<const uint32_t *>(blk));
    const uint4 *q = reinterpret_cast<const uint4 *>(blk + 16 + 32 * G * p);
#pragma unroll
    for (int i = 0; i < 2 * G; ++i) {
        const uint4 v = q[i];
        a.q[4 * i] = v.x, a.q[4 * i + 1] = v.y, a.q[4 * i + 2] = v.z, a.q[4 * i + 3] = v.w;
    }
}

// K-quant consumers read residue-major qs (dword t of a 32-byte group holds
// bytes t, t + 8, t + 16, t + 24): the ActKQ layout, so no transpose here.
template <int G>
__device__ __forceinline__ void load_act_lds(const uint8_t *blk, int p, ActKQ<G> &a) {
    a.d8 = __uint_as_float(*reinterpret_cast<const uint32_t *>(blk));
    const uint4 *q = reinterpret_cast<const uint4 *>(blk + 16 + 64 * G * p);
#pragma unroll
    for (int j = 0; j < 2 * G; ++j) {
        const uint4 v0 = q[2 * j], v1 = q[2 * j + 1];
        a.t[j][0] = v0.x, a.t[j][1] = v0.y, a.t[j][2] = v0.z, a.t[j][3] = v0.w;
        a.t[j][4] = v1.x, a.t[j][5] = v1.y, a.t[j][6] = v1.z, a.t[j][7] = v1.w;
    }
    const uint32_t *bs = reinterpret_cast<const uint32_t *>(blk + 272 + 8 * G * p);
#pragma unroll
    for (int j = 0; j < 2 * G; ++j) {
        const uint32_t w = bs[j];
        a.bsp[j] = (int32_t)(int16_t)(w & 0xffff) + (int32_t)(int16_t)(w >> 16);
    }
}

// ------------------------------------------------------- decoded weights
//
// IQ2_S / IQ3_S: the slice's signed int8 weights and the integer scale of
// each 16-element half group (IQ2_S: 1 + 2 * nibble per half, q8_k.rs:355-362;
// IQ3_S: 2 * nibble + 1 for the whole group, q8_k.rs:389-427), so the block
// sum is sum over halves of scale * dot(16 weights, 16 quants): the same
// integer as the reference's (integer addition is exact in any order).
template <int LPU>
struct DecIQ {
    static constexpr int G = 8 / LPU;
    uint32_t w[8 * G];
    int32_t s[2 * G];
    float d;
};

// Q4_K / Q5_K: unsigned quants of each sub-block j in residue-major dwords,
// sub-block scale and min (scale_min, k_quants.rs:231-240), d and dmin.
template <int LPU>
struct DecKQ {
    static constexpr int G = 4 / LPU;
    uint32_t q[2 * G][8];
    int32_t sc[2 * G], mn[2 * G];
    float d, dmin;
};

template <int TY, int LPU>
using DecOf = typename std::conditional<Traits<TY>::KQ, DecKQ<LPU>, DecIQ<LPU>>::type;

template <int LPU>
__device__ __forceinline__ void decode(const WSlice<T_IQ2_S, LPU> &w, const void *gridp, int, DecIQ<LPU> &o) {
    constexpr int G = 8 / LPU;
    const GridRef<T_IQ2_S> grid(gridp);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const Iq2sGroup q = iq2s_group(w, g);
        const uint32_t sc = byte_of(g < 4 ? w.sc : w.sc2, g & 3);
#pragma unroll
        for (int lg = 0; lg < 4; ++lg) {
            const uint2 code = grid.code_at(q.addr(lg));
            const uint32_t sel_lo = q.sel(2 * lg) | code.x;
            const uint32_t sel_hi = q.sel(2 * lg + 1) | code.y;
            o.w[8 * g + 2 * lg] = perm(IQ2S_NEG, IQ2S_POS, sel_lo);
            o.w[8 * g + 2 * lg + 1] = perm(IQ2S_NEG, IQ2S_POS, sel_hi);
        }
        o.s[2 * g] = (int32_t)(1 + 2 * (sc & 15u));
        o.s[2 * g + 1] = (int32_t)(1 + 2 * (sc >> 4));
    }
    o.d = f16_to_f32(w.d);
}

template <int LPU>
__device__ __forceinline__ void decode(const WSlice<T_IQ3_S, LPU> &w, const void *gridp, int, DecIQ<LPU> &o) {
    constexpr int G = 8 / LPU;
    const GridRef<T_IQ3_S> grid(gridp);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int32_t sc = (int32_t)(2 * ((w.sc >> (4 * g)) & 15u) + 1);
        uint32_t ad[8];
        iq3_group_addrs(w.qs[2 * g], w.qs[2 * g + 1], byte_of(g < 4 ? w.qh : w.qh2, g & 3), ad);
#pragma unroll
        for (int lg = 0; lg < 4; ++lg) {
            const uint2 sm = grid.sel(byte_of(w.sg[g], lg));
            o.w[8 * g + 2 * lg] = iq3_signed(grid.pair(ad[2 * lg]), sm.x);
            o.w[8 * g + 2 * lg + 1] = iq3_signed(grid.pair(ad[2 * lg + 1]), sm.y);
        }
        o.s[2 * g] = sc;
        o.s[2 * g + 1] = sc;
    }
    o.d = f16_to_f32(w.d);
}

template <int TY, int LPU>
__device__ __forceinline__ void decode(const WSliceKQ<TY, LPU> &w, const void *, int p, DecKQ<LPU> &o) {
    constexpr int G = 4 / LPU;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int gg = G * p + g;
        int32_t sc0, mn0, sc1, mn1;
        scale_min_of(w.hdr.y, w.hdr.z, w.hdr.w, 2 * gg, sc0, mn0);
        scale_min_of(w.hdr.y, w.hdr.z, w.hdr.w, 2 * gg + 1, sc1, mn1);
        o.sc[2 * g] = sc0, o.mn[2 * g] = mn0, o.sc[2 * g + 1] = sc1, o.mn[2 * g + 1] = mn1;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            uint32_t lo = w.q[g][t] & 0x0f0f0f0fu;
            uint32_t hi = (w.q[g][t] >> 4) & 0x0f0f0f0fu;
            if constexpr (TY == T_Q5_K) {
                lo |= ((w.qh[t] >> (2 * gg)) & 0x01010101u) << 4;
                hi |= ((w.qh[t] >> (2 * gg + 1)) & 0x01010101u) << 4;
            }
            o.q[2 * g][t] = lo;
            o.q[2 * g + 1][t] = hi;
        }
    }
    o.d = f16_to_f32(w.hdr.x & 0xffffu);
    o.dmin = f16_to_f32(w.hdr.x >> 16);
}

// Integer stage of one token against a decoded slice: IQ -> v[0] = the
// slice's share of the block sum; K-quants -> v[0..7] lane sums, v[8] the
// minimum sum (q8_k.rs:288-312, :337-364, :380-428).
template <int LPU>
__device__ __forceinline__ void token_ints(const DecIQ<LPU> &o, const ActIQ<8 / LPU> &a, int32_t *v) {
    constexpr int G = 8 / LPU;
    int32_t bs = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        int32_t p0 = 0, p1 = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) p0 = dot4(o.w[8 * g + k], a.q[8 * g + k], p0);
#pragma unroll
        for (int k = 4; k < 8; ++k) p1 = dot4(o.w[8 * g + k], a.q[8 * g + k], p1);
        bs = mul24(o.s[2 * g], p0) + bs;
        bs = mul24(o.s[2 * g + 1], p1) + bs;
    }
    v[0] = bs;
}

template <int LPU>
__device__ __forceinline__ void token_ints(const DecKQ<LPU> &o, const ActKQ<4 / LPU> &a, int32_t *v) {
    constexpr int G = 4 / LPU;
    int32_t ms = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = 0;
#pragma unroll
    for (int j = 0; j < 2 * G; ++j) {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = mul24(o.sc[j], dot4(o.q[j][t], a.t[j][t], 0)) + v[t];
        ms = mul24(o.mn[j], a.bsp[j]) + ms;
    }
    v[8] = ms;
}

// ------------------------------------------------------------ one wave step
//
// The decoded rows of NM matrices (rpw rows, one per slot) against n staged
// tokens.  Tokens go in fold batches of FB: the integer stage of every token
// of a batch writes its per-block f32 terms to the wave's LDS table, then the
// wave's lanes fold the (matrix, token, row, chain) chains in parallel, each
// chain in the reference's sequential block order (lbh_rows.h fold_terms),
// and lanes (token, row) combine the chains (K-quants: sum = minimum chain,
// then += lane chains 0..7, q8_k.rs:314-326; IQ2_S: x 0.125, q8_k.rs:369) and
// call out(token, slot, values[NM]).  Every lane of the wave must call it.
template <int TY, int LPU, int NM, int FB, class Out>
__device__ __forceinline__ void batch_step(const DecOf<TY, LPU> (&dec)[NM], bool on, const LaneMap<LPU> &L, int nb,
                                           const uint8_t *s_act, int n, float *terms, float *chains, Out out) {
    using Tr = Traits<TY>;
    constexpr int NCH = Tr::NCH;
    const int tstr = nb + 1;
    const int lane = threadIdx.x & 63;
    const int rpw = L.rpw;
    for (int i0 = 0; i0 < n; i0 += FB) {
        const int nf = n - i0 < FB ? n - i0 : FB;
        for (int f = 0; f < nf; ++f) {
            ActOf<TY, LPU> act;
            load_act_lds(s_act + ((i0 + f) * nb + L.b) * Q8L, L.part, act);
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                int32_t v[NCH];
                token_ints(dec[m], act, v);
#pragma unroll
                for (int c = 0; c < NCH; ++c) v[c] = unit_reduce<LPU>(v[c]);
                if (on && L.part == 0) {
                    float *t = terms + (((m * FB + f) * rpw + L.slot) * NCH) * tstr + L.b;
                    if constexpr (Tr::KQ) {
                        const float s = __fmul_rn(dec[m].d, act.d8);
                        const float ms = __fmul_rn(dec[m].dmin, act.d8);
#pragma unroll
                        for (int c = 0; c < 8; ++c) t[c * tstr] = __fmul_rn(s, (float)v[c]);
                        t[8 * tstr] = __fmul_rn(ms, (float)v[8]);
                    } else {
                        t[0] = __fmul_rn(__fmul_rn(dec[m].d, act.d8), (float)v[0]);
                    }
                }
            }
        }
        wave_sync();
        const int tasks = NM * nf * rpw * NCH;
        for (int k = lane; k < tasks; k += 64) {
            const int c = k % NCH;
            int r = k / NCH;
            const int slot = r % rpw;
            r /= rpw;
            const int f = r % nf, m = r / nf;
            const int idx = ((m * FB + f) * rpw + slot) * NCH + c;
            chains[idx] = fold_terms(terms + idx * tstr, nb, Tr::KQ && c == 8);
        }
        wave_sync();
        for (int k = lane; k < nf * rpw; k += 64) {
            const int f = k % nf, slot = k / nf;
            float res[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const float *ch = chains + ((m * FB + f) * rpw + slot) * NCH;
                float s;
                if constexpr (Tr::KQ) {
                    s = ch[8];
#pragma unroll
                    for (int l = 0; l < 8; ++l) s = __fadd_rn(s, ch[l]);
                } else {
                    s = ch[0];
                    if (TY == T_IQ2_S) s = __fmul_rn(0.125f, s);
                }
                res[m] = s;
            }
            out(i0 + f, slot, res);
        }
        wave_sync();
    }
}

// Fold batch per type: IQ chains are short work per token, so their folds
// wait for up to eight tokens; K-quants carry nine chains per row and fold
// after every token (a small term table).
template <int TY>
constexpr int fold_batch() {
    return Traits<TY>::KQ ? 1 : 8;
}

// LDS floats of one wave's term table and chain results.
template <int TY, int NM>
__host__ __device__ constexpr int wave_fold_floats(int rpw, int nb) {
    return NM * fold_batch<TY>() * rpw * Traits<TY>::NCH * (nb + 2);
}

__host__ __device__ constexpr int rows_per_step(int lpu, int nb) { return (64 / lpu) / nb; }

// Rows [r0, r1) of NM matrices against the n tokens staged in s_act.  The
// wave's first weight loads are issued before `prologue` (codebook fill and
// activation staging, ended by a workgroup barrier), so their latency
// overlaps it; then a software pipeline keeps the next step's loads in flight.
// FUSED (chunks of one token): each row is the matvec's row dot (lbh_rows.h
// row_dot, the same terms and block-order fold as batch_step) on the staged
// token, with no decoded copy of the slice held for reuse, which a single
// token never needs; the wave's fold table holds its FoldLDS.
template <int TY, int LPU, int NM, bool FUSED = false, class Prologue, class Out>
__device__ __forceinline__ void batch_rows(const MatView (&mv)[NM], int r0, int r1, const uint8_t *s_act, int n,
                                           const void *grid, float *fold_lds, Prologue prologue, Out out) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int nb = mv[0].nb;
    const LaneMap<LPU> L(lane, nb);
    using W = WOf<TY, LPU>;
    Planes P[NM];
    uint32_t po[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        P[m] = make_planes(mv[m].planes, mv[m].units, mv[m].bytes);
        po[m] = part_offset<TY, LPU>(P[m], L.part);
    }
    const int rpw = L.rpw;
    float *terms = fold_lds + wid * wave_fold_floats<TY, NM>(rpw, nb);
    float *chains = terms + NM * fold_batch<TY>() * rpw * Traits<TY>::NCH * (nb + 1);
    const int steps = (r1 - r0 + rpw - 1) / rpw;
    // Lanes past the tile (or past the wave's last whole row) load and decode
    // the tile's last row: every register is defined, and `on` gates the writes.
    // The loads are unconditional (a step past the end reloads the tile's last
    // row, never used), so the wait before a step's use leaves the next step's
    // loads in flight.
    auto issue = [&](int j, W (&w)[NM]) {
        int r = r0 + j * rpw + L.slot;
        r = L.lane_on && r < r1 ? r : r1 - 1;
#pragma unroll
        for (int m = 0; m < NM; ++m) load_slice(P[m], (uint32_t)(r * nb + L.b), po[m], L.part, w[m]);
    };
    ActOf<TY, LPU> act1;   // FUSED: the staged token
    auto process = [&](int j, const W (&w)[NM]) {
        const int r = r0 + j * rpw + L.slot;
        const bool on = L.lane_on && r < r1;
        if constexpr (FUSED) {
            FoldLDS<TY> &fl = *reinterpret_cast<FoldLDS<TY> *>(terms);
            float res[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m) res[m] = row_dot<TY, LPU>(w[m], act1, on, L, grid, fl, nullptr, 0);
            if (on && L.leader()) out(0, r, res);
            return;
        }
        DecOf<TY, LPU> dec[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) decode(w[m], grid, L.part, dec[m]);
        batch_step<TY, LPU, NM, fold_batch<TY>()>(dec, on, L, nb, s_act, n, terms, chains,
                                                  [&](int i, int slot, const float *res) {
                                                      const int rr = r0 + j * rpw + slot;
                                                      if (rr < r1) out(i, rr, res);
                                                  });
    };
    int j = wid;
    W wa[NM], wb[NM];
    issue(j, wa);
    prologue();
    if constexpr (FUSED) load_act_lds(s_act + L.b * Q8L, L.part, act1);
    while (j < steps) {
        issue(j + MB_WAVES, wb);
        process(j, wa);
        j += MB_WAVES;
        if (j >= steps) break;
        issue(j + MB_WAVES, wa);
        process(j, wb);
        j += MB_WAVES;
    }
}

// Copies n x nb GGML Q8_K blocks (block (i, b) at src_of(i) + 292 * b) into
// the padded LDS layout, all threads of the workgroup.
template <class Src>
__device__ __forceinline__ void stage_q8(uint8_t *s_act, int n, int nb, Src src_of) {
    const int total = n * nb * 73;
    for (int k = threadIdx.x; k < total; k += blockDim.x) {
        const int blk = k / 73, w = k - blk * 73;
        const int i = blk / nb, b = blk - i * nb;
        const uint32_t v = *reinterpret_cast<const uint32_t *>(src_of(i) + b * 292 + 4 * w);
        const int off = w == 0 ? 0 : w <= 64 ? 16 + 4 * (w - 1) : 272 + 4 * (w - 65);
        *reinterpret_cast<uint32_t *>(s_act + blk * Q8L + off) = v;
    }
}

// LDS of a stream workgroup: the codebook (a static array, static_grid), then,
// dynamic, [staged activations][fold tables].
template <int TY, int NM>
__host__ __device__ constexpr int stream_lds(int tc, int nb, int lpu) {
    return al16(tc * nb * Q8L) + al16(GridLDS<TY>::BYTES) + MB_WAVES * 4 * wave_fold_floats<TY, NM>(rows_per_step(lpu, nb), nb);
}

template <int TY>
constexpr int mb_lpu() {
    return 2;
}

// ------------------------------------------------------------------ kernels

// Q8_K of one block by one wave, lane l holding elements 4l .. 4l + 3 (v), in
// the forms the consumers read: block `blk` of the GGML bytes (plain != NULL),
// of the copy with residue-major qs (rm != NULL), of the matrix-core operand
// copy (mx.q != NULL), and of the f16 operand tiles of the K-quant rows (kt !=
// NULL, rows of nb blocks; lbh_kt.h).  lds: 292 bytes of the wave.
//
// These kernels are latency-bound: a block per wave with four elements a lane
// and one coalesced dword a lane per copy took the 64-token (256-token) h
// quantization from 13 (34) us, at four blocks per wave and 16 elements a lane
// copied out of LDS, to 7 (16) us.
__device__ __forceinline__ void quantize_block_out(const float4 v, long long blk, uint8_t *plain, uint8_t *rm, uint8_t *lds,
                                                   MxRows mx, uint8_t *kt, int nb) {
    const int lane = threadIdx.x & 63;
    const float e[4] = {v.x, v.y, v.z, v.w};
    // the lane's largest |x| and the value at its first index, then the lowest
    // lane holding the wave's (q8_k.rs:43-49: the first index on ties)
    uint32_t am = __float_as_uint(fabsf(e[0]));
    float mv = e[0];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
        const uint32_t b = __float_as_uint(fabsf(e[i]));
        if (b > am) am = b, mv = e[i];
    }
    const uint32_t amax = wave_max_u32(am);
    const int owner = (int)__builtin_ctzll(__ballot(am == amax));
    const float maxv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mv), owner));
    uint32_t q = 0;
    int32_t sum = 0;
    float d = 0.0f;
    if (amax != 0) {
        const float iscale = -127.0f / maxv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int32_t x = nearest_int(__fmul_rn(iscale, e[i]));
            x = x < 127 ? x : 127;
            q |= (uint32_t)(uint8_t)(int8_t)x << (8 * i);
            sum += (int8_t)x;
        }
        d = 1.0f / iscale;
    }
    // bsums of 16 elements (four lanes), and the next group's
    sum += (int32_t)dpp_row<0xB1>((uint32_t)sum);
    sum += (int32_t)dpp_row<0x4E>((uint32_t)sum);
    const int32_t after = __builtin_amdgcn_update_dpp(0, sum, 0x104, 0xf, 0xf, false);   // row_shl:4
    const uint32_t pair = (uint32_t)(uint16_t)(int16_t)sum | ((uint32_t)(uint16_t)(int16_t)after << 16);
    if (mx.q) {
        // element dword `lane` as dword o of lane quarter p (MxRows)
        const int p = mx.split ? (lane >> 1) & 3 : lane >> 4, o = mx.split ? 2 * (lane >> 3) + (lane & 1) : lane & 15;
        reinterpret_cast<uint32_t *>(mx.q)[blk * 64 + 16 * (o >> 2) + 4 * p + (o & 3)] = q;
        if (lane == 0) mx.d[blk] = d;
    }
    auto store = [&](uint8_t *b) {
        uint32_t *o = reinterpret_cast<uint32_t *>(b);
        if (lane == 0) o[0] = __float_as_uint(d);
        o[1 + lane] = q;
        if ((lane & 7) == 0) o[65 + (lane >> 3)] = pair;
    };
    if (plain) store(plain + blk * 292);
    if (!kt && !rm) return;
    store(lds);
    wave_sync();
    if (kt && lane < KT_STORE_PIECES) {
        const long long t = blk / nb;
        kt_store_piece(kt, t, (int)(blk - t * nb), nb, lds, lane);
    }
    if (rm) {
        uint32_t *o = reinterpret_cast<uint32_t *>(rm + blk * 292);
        const uint8_t *src = lds + 4 + 32 * (lane >> 3) + (lane & 7);
        o[1 + lane] = (uint32_t)src[0] | ((uint32_t)src[8] << 8) | ((uint32_t)src[16] << 16) | ((uint32_t)src[24] << 24);
        if (lane == 0) o[0] = __float_as_uint(d);
        if ((lane & 7) == 0) o[65 + (lane >> 3)] = pair;
    }
}

// Sort of the batch's pairs by expert (workgroup 0) and Q8_K of every token
// (the other workgroups, a block per wave).
__global__ void __launch_bounds__(MB_THREADS) k_mb_prep(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    if (blockIdx.x > 0) {
        const int nb = a.hidden / 256;
        const long long blk = (long long)(blockIdx.x - 1) * MB_WAVES + (tid >> 6);
        if (blk >= (long long)a.n_tokens * nb) return;
        const bool rm = a.has_shared && !a.shared_kt && (a.shared.gate.type == T_Q4_K || a.shared.gate.type == T_Q5_K);
        const float4 v = reinterpret_cast<const float4 *>(a.x + blk * 256)[tid & 63];
        quantize_block_out(v, blk, a.valu ? a.q8x : nullptr, rm ? a.q8x_rm : nullptr, smem + (tid >> 6) * 304,
                           MxRows{a.mx ? a.xq_mx : nullptr, a.xd_mx, false}, a.shared_kt ? a.kt_x : nullptr, nb);
        return;
    }
    const int NE = a.n_experts, T = a.n_tokens, K = a.top_k, TC = a.tc;
    const int W = (T + 31) / 32;
    uint32_t *bm = reinterpret_cast<uint32_t *>(smem);              // [NE][W] token bitmaps
    int32_t *cnt = reinterpret_cast<int32_t *>(bm + NE * W);       // [NE]
    int32_t *off = cnt + NE;                                       // [NE] first sorted pair
    int32_t *coff = off + NE;                                      // [NE] first chunk
    int32_t *part = coff + NE;                                     // [MB_WAVES] scan partials
    int32_t *flags = part + MB_WAVES;
    // the thread's pairs tid, tid + 256, ..: every load in flight at once
    constexpr int PAIRS = BATCH_MAX_TOKENS * MOE_MAX_ROUTED / MB_THREADS;
    uint32_t ids[PAIRS];
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) ids[i] = i * MB_THREADS + tid < T * K ? a.ids[i * MB_THREADS + tid] : 0u;
    for (int i = tid; i < NE * W; i += MB_THREADS) bm[i] = 0;
    if (tid == 0) flags[0] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
        const int p = i * MB_THREADS + tid;
        if (p >= T * K) break;
        const int t = p / K;
        const uint32_t e = ids[i];
        if (e >= (uint32_t)NE) {
            atomicOr(&flags[0], 1);
            continue;
        }
        const uint32_t bit = 1u << (t & 31);
        const uint32_t old = atomicOr(&bm[e * W + (t >> 5)], bit);
        if (old & bit) atomicOr(&flags[0], 2);
    }
    __syncthreads();
    // Per-expert counts and chunk counts; each thread owns a run of experts.
    const int per = (NE + MB_THREADS - 1) / MB_THREADS;
    const int e0 = tid * per, e1 = e0 + per < NE ? e0 + per : NE;
    int sc = 0, sk = 0;
    for (int e = e0; e < e1; ++e) {
        int c = 0;
        for (int w = 0; w < W; ++w) c += __popc(bm[e * W + w]);
        cnt[e] = c;
        sc += c;
        sk += (c + TC - 1) / TC;
    }
    // Exclusive scan of (pairs, chunks), both at most 4096, as one word.
    static_assert(BATCH_MAX_TOKENS * MOE_MAX_ROUTED < 0x8000, "two sums share a word");
    uint32_t sum = (uint32_t)sc << 16 | (uint32_t)sk;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)sum, d, 64);
        if ((tid & 63) >= d) sum += o;
    }
    if ((tid & 63) == 63) part[tid >> 6] = (int32_t)sum;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < MB_WAVES; ++w) {
        if (w < tid >> 6) before += (uint32_t)part[w];
        total += (uint32_t)part[w];
    }
    {
        const uint32_t at = before + sum - ((uint32_t)sc << 16 | (uint32_t)sk);
        int o = (int)(at >> 16), ko = (int)(at & 0xffffu);
        for (int e = e0; e < e1; ++e) {
            off[e] = o;
            coff[e] = ko;
            o += cnt[e];
            ko += (cnt[e] + TC - 1) / TC;
        }
    }
    __syncthreads();
    const bool bad = flags[0] != 0;
    if (!bad) {
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) {
            const int p = i * MB_THREADS + tid;
            if (p >= T * K) break;
            const int t = p / K;
            const uint32_t e = ids[i];
            int rank = __popc(bm[e * W + (t >> 5)] & ((1u << (t & 31)) - 1u));
            for (int w = 0; w < (t >> 5); ++w) rank += __popc(bm[e * W + w]);
            const int pos = off[e] + rank;
            a.pair_token[pos] = t;
            a.pair_of[p] = pos;
        }
        for (int e = e0; e < e1; ++e) {
            const int c = cnt[e];
            for (int j = 0; j * TC < c; ++j) {
                const int ch = coff[e] + j;
                a.chunk_expert[ch] = e;
                a.chunk_p0[ch] = off[e] + j * TC;
                a.chunk_n[ch] = c - j * TC < TC ? c - j * TC : TC;
            }
        }
    }
    if (tid == 0) {
        a.plan[0] = bad ? 0 : (int32_t)(total & 0xffffu);
        a.plan[1] = flags[0];
    }
}

// A chunk of n tokens of a TY stream belongs to the matrix-core kernels.
template <int TY>
__device__ __forceinline__ bool mx_takes(const BatchArgs &a, int n) {
    return (TY == T_IQ2_S || TY == T_IQ3_S) && a.mx && n >= a.mx_min;
}

// Tokens a VALU stream of type ty stages at most: the chunks the matrix cores
// leave to it (IQ types with mx on), else whole chunks.
__host__ __device__ inline int valu_cap(const BatchArgs &a, int ty) {
    return a.mx && (ty == T_IQ2_S || ty == T_IQ3_S) ? a.vc : a.tc;
}

// Gate/up, SwiGLU (activation.rs:170-178) -> h, one launch per stream:
// SHARED: workgroup (token chunk, row tile) of the shared expert; else
// workgroup (routed chunk, row tile), idle past the sort's chunk count.
// PART (routed IQ streams beside the matrix cores): 0 every VALU chunk, 1
// the chunks of one token (the FUSED rows of batch_rows: 116 instead of 170
// VGPRs, four waves per SIMD instead of two), 2 the other VALU chunks.
template <int TY, bool SHARED, int PART = 0>
__global__ void __launch_bounds__(MB_THREADS) k_mb_gate_up(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    if (a.plan[1]) return;
    const int nb = a.hidden / 256;
    constexpr int LPU = mb_lpu<TY>();
    uint8_t *s_act = smem;
    uint8_t *grid = static_grid<TY>();
    float *fold = reinterpret_cast<float *>(smem + al16(valu_cap(a, TY) * nb * Q8L));
    if constexpr (SHARED) {
        const int tiles = (a.ffn_s + a.rt_gu_s - 1) / a.rt_gu_s;
        const int c = blockIdx.x / tiles, tile = blockIdx.x - c * tiles;
        const int t0 = c * a.tc;
        const int n = a.n_tokens - t0 < a.tc ? a.n_tokens - t0 : a.tc;
        if (mx_takes<TY>(a, n)) return;
        const int r0 = tile * a.rt_gu_s, r1 = r0 + a.rt_gu_s < a.ffn_s ? r0 + a.rt_gu_s : a.ffn_s;
        const uint8_t *src = Traits<TY>::KQ ? a.q8x_rm : a.q8x;
        const MatView mv[2] = {a.shared.gate, a.shared.up};
        batch_rows<TY, LPU, 2>(
            mv, r0, r1, s_act, n, grid, fold,
            [&]() {
                fill_grid<TY>(grid);
                stage_q8(s_act, n, nb, [&](int i) { return src + (long long)(t0 + i) * nb * 292; });
                __syncthreads();
            },
            [&](int i, int r, const float *res) {
                const long long o = (long long)(t0 + i) * a.ffn_s + r;
                a.g_s[o] = res[0];
                a.u_s[o] = res[1];
            });
    } else {
        const int tiles = (a.ffn_r + a.rt_gu_r - 1) / a.rt_gu_r;
        const int c = blockIdx.x / tiles, tile = blockIdx.x - c * tiles;
        if (c >= a.plan[0]) return;
        const int e = a.chunk_expert[c], p0 = a.chunk_p0[c], n = a.chunk_n[c];
        if (mx_takes<TY>(a, n)) return;
        if ((PART == 1 && n != 1) || (PART == 2 && n == 1)) return;
        const int r0 = tile * a.rt_gu_r, r1 = r0 + a.rt_gu_r < a.ffn_r ? r0 + a.rt_gu_r : a.ffn_r;
        const MatView mv[2] = {a.experts[e].gate, a.experts[e].up};
        batch_rows<TY, LPU, 2, PART == 1>(
            mv, r0, r1, s_act, n, grid, fold,
            [&]() {
                fill_grid<TY>(grid);
                stage_q8(s_act, n, nb, [&](int i) { return a.q8x + (long long)a.pair_token[p0 + i] * nb * 292; });
                __syncthreads();
            },
            [&](int i, int r, const float *res) {
                const long long o = (long long)(p0 + i) * a.ffn_r + r;
                a.g_r[o] = res[0];
                a.u_r[o] = res[1];
            });
    }
}

// h = SwiGLU(gate, up) (activation.rs:170-178) and its Q8_K (quantize_row_q8_k_into
// of each down projection's input, gemv.rs:161-163) for every routed pair row
// [0, pairs), then the shared rows.  The gate/up streams leave gate and up
// apart, so no exp runs inside their weight loops (its table load would wait
// for every weight load in flight).  shared_mode 0: the shared copy is GGML
// bytes plus the matrix-core operand copy (IQ down); 1: residue-major qs only
// (VALU K-quant down); 2: the f16 operand tiles (matrix-core K-quant down).
__global__ void __launch_bounds__(MB_THREADS) k_mb_quant_h(BatchArgs a, int shared_mode) {
    __shared__ __align__(16) uint8_t lds[MB_WAVES][304];
    __shared__ uint64_t exp_tab[32];
    if (threadIdx.x < 32) exp_tab[threadIdx.x] = c_expf_tab[threadIdx.x];
    const int nbr = a.ffn_r / 256, nbs = a.ffn_s / 256;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const long long br = (long long)a.n_tokens * a.top_k * nbr;
    const long long bs = a.has_shared ? (long long)a.n_tokens * nbs : 0;
    long long blk = (long long)blockIdx.x * MB_WAVES + wid;   // routed blocks, then the shared ones
    const bool routed = blk < br, on = blk < br + bs;
    if (!routed) blk -= br;
    float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f), u = g;
    if (on) {
        g = reinterpret_cast<const float4 *>((routed ? a.g_r : a.g_s) + blk * 256)[lane];
        u = reinterpret_cast<const float4 *>((routed ? a.u_r : a.u_s) + blk * 256)[lane];
    }
    __syncthreads();
    if (!on || a.plan[1]) return;
    const float4 h = make_float4(swiglu_ref(g.x, u.x, exp_tab), swiglu_ref(g.y, u.y, exp_tab),
                                 swiglu_ref(g.z, u.z, exp_tab), swiglu_ref(g.w, u.w, exp_tab));
    if (routed)
        quantize_block_out(h, blk, a.valu ? a.q8h_r : nullptr, nullptr, lds[wid],
                           MxRows{a.mx ? a.hq_mx_r : nullptr, a.hd_mx_r, a.type_down_r == T_IQ3_S}, nullptr, nbr);
    else
        quantize_block_out(h, blk, shared_mode == 0 ? a.q8h_s : nullptr, shared_mode == 1 ? a.q8h_s : nullptr, lds[wid],
                           MxRows{a.mx && shared_mode == 0 ? a.hq_mx_s : nullptr, a.hd_mx_s, a.shared.down.type == T_IQ3_S},
                           shared_mode == 2 ? a.kt_h : nullptr, nbs);
}

// Down rows -> d, one launch per stream (as k_mb_gate_up; PART 1: every
// chunk has one token, the FUSED rows of batch_rows).
template <int TY, bool SHARED, int PART = 0>
__global__ void __launch_bounds__(MB_THREADS) k_mb_down(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    if (a.plan[1]) return;
    constexpr int LPU = mb_lpu<TY>();
    uint8_t *s_act = smem;
    if constexpr (SHARED) {
        const int nb = a.ffn_s / 256;
        const int tiles = (a.hidden + a.rt_d_s - 1) / a.rt_d_s;
        const int c = blockIdx.x / tiles, tile = blockIdx.x - c * tiles;
        const int t0 = c * a.tc;
        const int n = a.n_tokens - t0 < a.tc ? a.n_tokens - t0 : a.tc;
        if (mx_takes<TY>(a, n)) return;
        const int r0 = tile * a.rt_d_s, r1 = r0 + a.rt_d_s < a.hidden ? r0 + a.rt_d_s : a.hidden;
        uint8_t *grid = static_grid<TY>();
        float *fold = reinterpret_cast<float *>(smem + al16(valu_cap(a, TY) * nb * Q8L));
        const MatView mv[1] = {a.shared.down};
        batch_rows<TY, LPU, 1>(
            mv, r0, r1, s_act, n, grid, fold,
            [&]() {
                fill_grid<TY>(grid);
                stage_q8(s_act, n, nb, [&](int i) { return a.q8h_s + (long long)(t0 + i) * nb * 292; });
                __syncthreads();
            },
            [&](int i, int r, const float *res) { a.d_s[(long long)(t0 + i) * a.hidden + r] = res[0]; });
    } else {
        const int nb = a.ffn_r / 256;
        const int tiles = (a.hidden + a.rt_d_r - 1) / a.rt_d_r;
        const int c = blockIdx.x / tiles, tile = blockIdx.x - c * tiles;
        if (c >= a.plan[0]) return;
        const int e = a.chunk_expert[c], p0 = a.chunk_p0[c], n = a.chunk_n[c];
        if (mx_takes<TY>(a, n)) return;
        const int r0 = tile * a.rt_d_r, r1 = r0 + a.rt_d_r < a.hidden ? r0 + a.rt_d_r : a.hidden;
        uint8_t *grid = static_grid<TY>();
        float *fold = reinterpret_cast<float *>(smem + al16(valu_cap(a, TY) * nb * Q8L));
        const MatView mv[1] = {a.experts[e].down};
        batch_rows<TY, LPU, 1, PART == 1>(
            mv, r0, r1, s_act, n, grid, fold,
            [&]() {
                fill_grid<TY>(grid);
                stage_q8(s_act, n, nb, [&](int i) { return a.q8h_r + (long long)(p0 + i) * nb * 292; });
                __syncthreads();
            },
            [&](int i, int r, const float *res) { a.d_r[(long long)(p0 + i) * a.hidden + r] = res[0]; });
    }
}

// ==================================================== IQ streams on the matrix cores
//
// The IQ2_S / IQ3_S gate/up and down streams as int8 matrix-core products,
// bit-identical to the dot4 streams above: per (row, token, block) the integer
// block sum is formed exactly and folded in the reference's order.
//
// Wave tile: the chunk's tokens (up to 16, operand A) x 16 weight rows
// (operand B) per block.  Lane l = 16 q + c supplies token c of A and row c of
// B for the same elements of the block, so an instruction contracts identical
// elements whatever its internal k order; result i of the lane is (token
// 4q + i, row c), so the row's d and scales are the lane's own.
//   IQ2_S: v_mfma_i32_16x16x64_i8; instruction m contracts the lane's 16
//     elements 64q + 16m .. + 15, one scale (half group).  The scaled weight
//     +-{8, 25, 43} (1 + 2 nibble) is split as 256 hi + lo into two signed
//     bytes, each a v_perm by the weight's code and sign from a table of the
//     scale (16 entries x 16 bytes in LDS): two chains over the whole block,
//     bsum = 256 sum_hi + sum_lo, no multiply per scale.
//   IQ3_S: v_mfma_i32_16x16x32_i8; instruction g contracts group g (lane:
//     elements 32g + 8q .. + 7), whose scale multiplies the 32-bit result
//     (bsum += (2 nibble + 1) * result: 24-bit operands).  The signed bytes
//     come from the 32 KiB signed table, one word per four weights.
// The sums are int32 throughout, hence exact in any order, and equal the
// reference's (q8_k.rs:337-364, :380-428).  The fold is the one of
// lbh_rows.h: term = (d * d8) * (float)bsum, chain += term in block order,
// IQ2_S result = 0.125 * chain.
//
// What bounds it: VALU issue (about 118 instructions per IQ2_S matrix, 16 rows
// and block, 128 for IQ3_S; busy 72% and 62% of the time), beside the codebook
// reads of the LDS.  As f16 products (v_mfma_f32_16x16x32_f16 on pre-scaled f16
// weights) the same tile took about twice the VALU work: f16 signs and scales
// for the weights, f16 conversions of the quants.  Measured on 192 experts of
// hidden 4096, width 1536, top-8 Zipf(1.1), tile copies, kernel times:
//   64 tokens   gate/up 159 -> 88 us, down 91 -> 61 us (step 417 -> 355 us)
//   256 tokens  gate/up 375 -> 222 us, down 242 -> 143 us (step 832 -> 626 us)

typedef int mx_i4 __attribute__((ext_vector_type(4)));

constexpr int MX_THREADS = 256;
constexpr int MX_WAVES = MX_THREADS / 64;
constexpr int MX_MAX_NB = 64;

// IQ2_S scaled weights by scale nibble n: bytes 0-2 of {lo+, lo-, hi+, hi-} are
// the split +-m (1 + 2n) = 256 hi + lo (lo signed) of m = 8, 25, 43.
struct alignas(16) MxProducts {
    uint32_t v[16][4];
    constexpr MxProducts() : v{} {
        const int mag[3] = {8, 25, 43};
        for (int n = 0; n < 16; ++n)
            for (int sg = 0; sg < 2; ++sg)
                for (int c = 0; c < 3; ++c) {
                    const int p = (sg ? -1 : 1) * mag[c] * (1 + 2 * n);
                    const int low = p & 0xff, lo = low >= 128 ? low - 256 : low, hi = (p - lo) / 256;
                    v[n][sg] |= (uint32_t)low << (8 * c);
                    v[n][2 + sg] |= (uint32_t)(hi & 0xff) << (8 * c);
                }
    }
};
static __constant__ MxProducts c_mx_products = MxProducts();

// LDS tables of a stream: IQ2_S the byte codes (GridLDS image) and the scaled
// weights, IQ3_S the signed table.
template <int TY>
struct MxTab {
    static constexpr int GRID = TY == T_IQ2_S ? GridLDS<T_IQ2_S>::BYTES : GridLDS<T_IQ3S_SGN>::BYTES;
    static constexpr int BYTES = GRID + (TY == T_IQ2_S ? 256 : 0);
};

// Copies TY's tables into LDS (all threads; the caller synchronises).
template <int TY>
__device__ __forceinline__ void mx_fill(uint8_t *tab) {
    const uint4 *g = grid_image<TY == T_IQ2_S ? T_IQ2_S : T_IQ3S_SGN>();
    uint4 *o = reinterpret_cast<uint4 *>(tab);
#pragma unroll
    for (int i = 0; i < MxTab<TY>::GRID / 16 / MX_THREADS; ++i) o[threadIdx.x + i * MX_THREADS] = g[threadIdx.x + i * MX_THREADS];
    static_assert(alignof(MxProducts) % 16 == 0, "read as uint4");
    if (TY == T_IQ2_S && threadIdx.x < 16)
        o[MxTab<TY>::GRID / 16 + threadIdx.x] = reinterpret_cast<const uint4 *>(&c_mx_products.v[0][0])[threadIdx.x];
}

// One lane's 64 weights of its row's block, in the order of the tile copies:
//   IQ2_S  w: qs of its two groups, sg: their sign dwords, e: byte j the
//          groups' qh fields of lookup j (low nibble) and the scale nibble of
//          half group j (high nibble).
//   IQ3_S  w: lookup bytes of four quads: the lane's lookups are 2q and 2q + 1 of
//          every group; quad 0 / 1 holds lookup 2q / 2q + 1 of groups 0, 1, 4, 5,
//          quad 2 / 3 those of groups 2, 3, 6, 7 (byte i: the i-th listed
//          group).  sg[j] byte i: the sign byte q of the i-th group of quads
//          2j, 2j + 1.  qh, sc: the row's qh bytes and scale nibbles.
template <int TY>
struct MxW;
template <>
struct MxW<T_IQ2_S> {
    uint32_t w[2], sg[2], e, d;
};
template <>
struct MxW<T_IQ3_S> {
    uint32_t w[4], sg[2], qh[2], sc, d;
};

typedef uint32_t mx_u3 __attribute__((ext_vector_type(3)));

// The row's own bytes of unit u: d, and for IQ3_S qh and the scales.
__device__ __forceinline__ void mx_load_row(const Planes &P, uint32_t u, MxW<T_IQ2_S> &o) { o.d = bld16(P, u * 2, 5 * P.U16); }
__device__ __forceinline__ void mx_load_row(const Planes &P, uint32_t u, MxW<T_IQ3_S> &o) {
    const mx_u3 t = __builtin_bit_cast(mx_u3, __builtin_amdgcn_raw_buffer_load_b96(P.rsrc, u * 12, 6 * P.U16, WEIGHT_CPOL));
    o.qh[0] = t.x, o.qh[1] = t.y, o.sc = t.z;
    o.d = bld16(P, u * 2, 6 * P.U16 + 12 * P.U);
}

__device__ __forceinline__ void mx_set_row(MxW<T_IQ2_S> &o, const MxW<T_IQ2_S> &r) { o.d = r.d; }
__device__ __forceinline__ void mx_set_row(MxW<T_IQ3_S> &o, const MxW<T_IQ3_S> &r) {
    o.qh[0] = r.qh[0], o.qh[1] = r.qh[1], o.sc = r.sc, o.d = r.d;
}

// Slice of a tile copy (k_units_to_tiles): u is the tile's first unit.
__device__ __forceinline__ void mx_load(const Planes &P, uint32_t u, int lane, MxW<T_IQ2_S> &o) {
    const uint4 a = bld128(P, u * 64 + 16u * lane, 0);
    o.w[0] = a.x, o.w[1] = a.y, o.sg[0] = a.z, o.sg[1] = a.w;
    o.e = bld32(P, u * 16 + 4u * lane, 4 * P.U16);
    mx_load_row(P, u + (lane & 15), o);
}
__device__ __forceinline__ void mx_load(const Planes &P, uint32_t u, int lane, MxW<T_IQ3_S> &o) {
    const uint4 a = bld128(P, u * 64 + 16u * lane, 0);
    const uint2 s = bld64(P, u * 32 + 8u * lane, 4 * P.U16);
    o.w[0] = a.x, o.w[1] = a.y, o.w[2] = a.z, o.w[3] = a.w;
    o.sg[0] = s.x, o.sg[1] = s.y;
    mx_load_row(P, u + (lane & 15), o);
}

// Row-major matrices: lane (q, c) reads whole block b0 + q of row c (u: its
// unit), so each load covers 64 contiguous bytes of 16 rows; the four lanes of a
// row exchange quarters for blocks (v_permlane32_swap / 16_swap, a 4 x 4
// transposition), after which slice j is block b0 + j in the order above.
// Eight blocks at a time: load set h gives lane (q, c) block b0 + 2q + c / 8 of
// row 8h + c % 8, 128 contiguous bytes of eight rows; lanes c and c ^ 8 swap
// across the sets (mx_rows8), set p then holds block b0 + 2q + p of row c and
// its slice j block b0 + 2j + p.
template <int TY>
struct MxRaw {
    uint32_t v[TY == T_IQ2_S ? 20 : 24];   // IQ2_S qs, signs, qh, scales; IQ3_S qs, signs
};
template <int TY>
__device__ __forceinline__ void mx_load_raw(const Planes &P, uint32_t u, MxRaw<TY> &o) {
#pragma unroll
    for (int k = 0; k < (TY == T_IQ2_S ? 5 : 6); ++k) {
        const uint4 a = bld128(P, u * 16, k * P.U16);
        o.v[4 * k] = a.x, o.v[4 * k + 1] = a.y, o.v[4 * k + 2] = a.z, o.v[4 * k + 3] = a.w;
    }
}

__device__ __forceinline__ void mx_rows8(uint32_t &a, uint32_t &b) {
    const int x = (int)a, y = (int)b;   // row_ror:8 into lanes 8-15 / 0-7 of each row of 16
    a = (uint32_t)__builtin_amdgcn_update_dpp(x, y, 0x128, 0xf, 0xc, false);
    b = (uint32_t)__builtin_amdgcn_update_dpp(y, x, 0x128, 0xf, 0x3, false);
}
// t[k] of lane quarter q becomes t[q] of lane quarter k.
__device__ __forceinline__ void mx_exchange(uint32_t &t0, uint32_t &t1, uint32_t &t2, uint32_t &t3) {
    auto r = __builtin_amdgcn_permlane32_swap(t0, t2, false, false);
    t0 = r[0], t2 = r[1];
    r = __builtin_amdgcn_permlane32_swap(t1, t3, false, false);
    t1 = r[0], t3 = r[1];
    r = __builtin_amdgcn_permlane16_swap(t0, t1, false, false);
    t0 = r[0], t1 = r[1];
    r = __builtin_amdgcn_permlane16_swap(t2, t3, false, false);
    t2 = r[0], t3 = r[1];
}
// 4 x 4 byte transposition: byte i of o[k] = byte k of (a, b, c, d)[i].
__device__ __forceinline__ void mx_bytes4(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&o)[4]) {
    const uint32_t ab0 = perm(b, a, 0x05010400u), ab1 = perm(b, a, 0x07030602u);   // a0 b0 a1 b1, a2 b2 a3 b3
    const uint32_t cd0 = perm(d, c, 0x05010400u), cd1 = perm(d, c, 0x07030602u);
    o[0] = perm(cd0, ab0, 0x05040100u), o[1] = perm(cd0, ab0, 0x07060302u);
    o[2] = perm(cd1, ab1, 0x05040100u), o[3] = perm(cd1, ab1, 0x07060302u);
}
__device__ __forceinline__ void mx_slices(const MxRaw<T_IQ2_S> &r, MxW<T_IQ2_S> (&o)[4]) {
    uint32_t e[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {   // quarter k of the lane's block
        const uint32_t qh = (r.v[16 + (k >> 1)] >> (4 * (k & 1))) & 0x0f0f0f0fu;
        const uint32_t sc = perm(0u, r.v[18 + (k >> 1)], k & 1 ? 0x03030202u : 0x01010000u);
        e[k] = qh | (((sc << 4) & 0x00f000f0u) | (sc & 0xf000f000u));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t w[4] = {r.v[i], r.v[2 + i], r.v[4 + i], r.v[6 + i]};
        uint32_t s[4] = {r.v[8 + i], r.v[10 + i], r.v[12 + i], r.v[14 + i]};
        mx_exchange(w[0], w[1], w[2], w[3]);
        mx_exchange(s[0], s[1], s[2], s[3]);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j].w[i] = w[j], o[j].sg[i] = s[j];
    }
    mx_exchange(e[0], e[1], e[2], e[3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j].e = e[j];
}
__device__ __forceinline__ void mx_slices(const MxRaw<T_IQ3_S> &r, MxW<T_IQ3_S> (&o)[4]) {
    // qs bytes of group g: v[2g], v[2g + 1]; lane quarter k takes bytes 2k, 2k + 1
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int g0 = 4 * j / 2;   // quads 2j, 2j + 1: groups 2j, 2j + 1, 2j + 4, 2j + 5
        uint32_t lo[4], hi[4], s[4], q0[4], q1[4];
        mx_bytes4(r.v[2 * g0], r.v[2 * g0 + 2], r.v[2 * g0 + 8], r.v[2 * g0 + 10], lo);       // lookups 0-3
        mx_bytes4(r.v[2 * g0 + 1], r.v[2 * g0 + 3], r.v[2 * g0 + 9], r.v[2 * g0 + 11], hi);   // lookups 4-7
        mx_bytes4(r.v[16 + g0], r.v[17 + g0], r.v[20 + g0], r.v[21 + g0], s);
        q0[0] = lo[0], q0[1] = lo[2], q0[2] = hi[0], q0[3] = hi[2];   // even lookups of quarters 0-3
        q1[0] = lo[1], q1[1] = lo[3], q1[2] = hi[1], q1[3] = hi[3];
        mx_exchange(q0[0], q0[1], q0[2], q0[3]);
        mx_exchange(q1[0], q1[1], q1[2], q1[3]);
        mx_exchange(s[0], s[1], s[2], s[3]);
#pragma unroll
        for (int b = 0; b < 4; ++b) o[b].w[2 * j] = q0[b], o[b].w[2 * j + 1] = q1[b], o[b].sg[j] = s[b];
    }
}

// The tile copy of a matrix (the slices' layout at MxW): the same bits with the
// units in 16-row tile order and, inside a tile (16 rows of one block), the chunk
// bytes of the streams' 64 lanes side by side, lane 16 q + c holding what it reads
// of row c:
//   IQ2_S  first 64 U bytes: 16 per lane, the qs and the sign dwords of groups
//          2q, 2q + 1; next 16 U: 4 per lane, byte j the groups' qh fields of
//          lookup j (low nibble) and the scale nibble of half group j; d plane.
//   IQ3_S  first 64 U bytes: 16 per lane, dword k byte i the qs byte of lookup
//          2q + k % 2 of the i-th of groups 0, 1, 4, 5 (k < 2) or 2, 3, 6, 7;
//          next 32 U: 8 per lane, dword j byte i the sign byte q of the i-th of
//          the same groups; tail and d planes in unit order.
// A wave takes four blocks of 16 rows as the row-major streams do, 64 contiguous
// bytes of each row per load: 3.8 us for 4096 x 1536 of either type.  One lane
// slice a thread, gathered byte by byte, took 7.0 for IQ3_S.
template <int TY>
__global__ void __launch_bounds__(MX_THREADS) k_units_to_tiles(MatView m, uint8_t *dst) {
    constexpr TypeLayout L = layout_of(TY);
    const Planes P = make_planes(m.planes, m.units, m.bytes);
    const long long U = m.units, base = L.nchunk * U * 16;
    const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15, nb = m.nb, groups = (nb + 3) / 4;
    const int n = m.rows / 16 * groups;
    for (int i = (int)blockIdx.x * MX_WAVES + (int)(threadIdx.x >> 6); i < n; i += (int)gridDim.x * MX_WAVES) {
        const int rt = i / groups, b0 = (i - rt * groups) * 4, b = b0 + q < nb ? b0 + q : nb - 1;
        const uint32_t u = (uint32_t)((16 * rt + c) * nb + b);
        MxRaw<TY> raw;
        mx_load_raw(P, u, raw);
        MxW<TY> row, w[4];
        mx_load_row(P, u, row);
        mx_slices(raw, w);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (b0 + j >= nb) break;
            const long long at = ((long long)rt * nb + b0 + j) * 64 + lane;
            if constexpr (TY == T_IQ2_S) {
                reinterpret_cast<uint4 *>(dst)[at] = make_uint4(w[j].w[0], w[j].w[1], w[j].sg[0], w[j].sg[1]);
                reinterpret_cast<uint32_t *>(dst + 64 * U)[at] = w[j].e;
            } else {
                reinterpret_cast<uint4 *>(dst)[at] = make_uint4(w[j].w[0], w[j].w[1], w[j].w[2], w[j].w[3]);
                reinterpret_cast<uint2 *>(dst + 64 * U)[at] = make_uint2(w[j].sg[0], w[j].sg[1]);
            }
        }
        if (b0 + q < nb) {
            const long long ut = ((long long)rt * nb + b) * 16 + c;
            if constexpr (TY == T_IQ3_S) {
                uint32_t *t = reinterpret_cast<uint32_t *>(dst + base) + 3 * ut;
                t[0] = row.qh[0], t[1] = row.qh[1], t[2] = row.sc;
            }
            reinterpret_cast<uint16_t *>(dst + base + L.tail * U)[ut] = (uint16_t)row.d;
        }
    }
}

// Integer block sums bs[i] of (token 4q + i, row c) from the lane's weights
// and its 64 quants of token c (tok[m]: 16 bytes).
__device__ __forceinline__ void mx_block(const MxW<T_IQ2_S> &o, const uint4 (&tok)[4], const uint8_t *tab, int,
                                         int32_t (&bs)[4]) {
    const GridRef<T_IQ2_S> grid(tab);
    mx_i4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const Iq2sGroup g = Iq2sGroup::make(o.w[m >> 1], o.e, m >> 1, o.sg[m >> 1]);
        const uint4 t = *reinterpret_cast<const uint4 *>(tab + MxTab<T_IQ2_S>::GRID + ((o.e >> (8 * m)) & 0xf0u));
        mx_i4 bl, bh;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int lg = 2 * (m & 1) + k;
            const uint2 code = grid.code_at(g.addr(lg));
            const uint32_t s0 = g.sel(2 * lg) | code.x, s1 = g.sel(2 * lg + 1) | code.y;
            bl[2 * k] = (int)perm(t.y, t.x, s0), bl[2 * k + 1] = (int)perm(t.y, t.x, s1);
            bh[2 * k] = (int)perm(t.w, t.z, s0), bh[2 * k + 1] = (int)perm(t.w, t.z, s1);
        }
        const mx_i4 a = __builtin_bit_cast(mx_i4, tok[m]);
        lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bl, lo, 0, 0, 0);
        hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bh, hi, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) bs[i] = (hi[i] << 8) + lo[i];
}

__device__ __forceinline__ void mx_block(const MxW<T_IQ3_S> &o, const uint4 (&tok)[4], const uint8_t *tab, int lane,
                                         int32_t (&bs)[4]) {
    const Iq3SignedRef grid(tab);
    // bits 0, 1 of byte i: the high index bits of lookups 2q, 2q + 1
    const uint32_t ta = o.qh[0] >> (2 * (lane >> 4)), tb = o.qh[1] >> (2 * (lane >> 4));
    const uint32_t hb[2] = {perm(tb, ta, 0x05040100u), perm(tb, ta, 0x07060302u)};
    uint32_t word[2][8];   // [even, odd lookup][group]
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int j = k >> 1, odd = k & 1;
        // iq3_signed_offset = x + 256 y per byte
        const uint32_t h = (odd ? hb[j] << 1 : hb[j] << 2) & 0x04040404u;
        const uint32_t s = (odd ? o.sg[j] >> 1 : o.sg[j] << 3) & 0x78787878u;
        const uint32_t x = o.w[k] & 0xfcfcfcfcu, y = (o.w[k] & 0x03030303u) | h | s;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            word[odd][(i & 1) + 4 * (i >> 1) + 2 * j] = grid.word(perm(y, x, 0x0c0c0000u | ((4u + i) << 8) | (uint32_t)i));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) bs[i] = 0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const uint4 v = tok[g >> 1];
        const uint2 a = (g & 1) ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y);
        const uint2 b = make_uint2(word[0][g], word[1][g]);
        const mx_i4 zero = {0, 0, 0, 0};
        const mx_i4 r = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b),
                                                              zero, 0, 0, 0);
        const int32_t ls = (int32_t)(((g == 0 ? o.sc << 1 : o.sc >> (4 * g - 1)) & 0x1eu) | 1u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bs[i] += mul24(r[i], ls);
            asm("" : "+v"(bs[i]));   // one v_mad_i32_i24 each, not two products and a three-way add
        }
    }
}

// LDS of a matrix-core stream workgroup: the tables and the token scales.
__host__ __device__ constexpr int mx_lds_bytes(int ty) {
    return (ty == T_IQ2_S ? MxTab<T_IQ2_S>::BYTES : MxTab<T_IQ3_S>::BYTES) + MX_MAX_NB * 16 * 4;
}

// The wave's f32 chains of one tile: the lane's four (token 4q + i, row c)
// results of NM matrices (or row tiles), blocks added in order.
template <int TY, int NM>
struct MxChains {
    float c[NM][4];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int t = 0; t < NM; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) c[t][i] = 0.0f;
    }
    __device__ __forceinline__ void add(int t, const MxW<TY> &w, const uint4 (&tok)[4], const float4 &d8, const uint8_t *tab,
                                        int lane) {
        int32_t bs[4];
        mx_block(w, tok, tab, lane, bs);
        const float d = f16_to_f32(w.d), e[4] = {d8.x, d8.y, d8.z, d8.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) c[t][i] = __fadd_rn(c[t][i], __fmul_rn(__fmul_rn(d, e[i]), (float)bs[i]));
    }
    template <class Out>
    __device__ __forceinline__ void finish(int q, int row, Out &out) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float res[NM];
#pragma unroll
            for (int t = 0; t < NM; ++t) res[t] = TY == T_IQ2_S ? __fmul_rn(0.125f, c[t][i]) : c[t][i];   // q8_k.rs:369
            out(4 * q + i, row, res);
        }
        clear();
    }
};

// Rows [r0, r1) (a multiple of 16) of NM tiles per step against the chunk's
// tokens: the NM matrices mv (gate and up), or, PAIR, NM adjacent 16-row tiles
// of the one matrix mv[0], which share the step's token operands.  The waves
// take tiles r0 + RW wid, + 4 RW, ... (RW = 16 or 16 NM rows) to r1, every
// block of a tile in order; s_d8[16 b + i] is the scale of token i's block b,
// bq the lane's token operand row.  out(token column, row, values) is called
// once per (token, row).  The first loads are issued before `prologue` (tables
// and scales to LDS, ended by a workgroup barrier); then a step's loads are in
// flight while the one before is computed.
//   TILE: tile copies, one block per step.
//   else: row-major matrices, four blocks (IQ2_S) or eight (IQ3_S, whose rows
//   are short) per load step, exchanged into slices (mx_slices).  Loading 16
//   bytes of each line at a time, block by block, took 1.5 to 2 times the tile
//   copies' time; four blocks still fetch half of the lines twice from beyond
//   L2, and eight with no spare registers to load ahead measured slower (64
//   tokens, gate/up: 231 us with four, 265 us with eight).
template <int TY, int NM, bool TILE, bool PAIR, class Prologue, class Out>
__device__ __forceinline__ void mx_tiles(const MatView *mv, int r0, int r1, int nb, const uint8_t *bq, const uint8_t *tab,
                                         const float *s_d8, Prologue prologue, Out out) {
    constexpr int NP = PAIR ? 1 : NM, RW = PAIR ? 16 * NM : 16, RG = RW * MX_WAVES;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, q = lane >> 4;
    const int rt0 = r0 + RW * wid;
    const int tiles = rt0 < r1 ? (r1 - rt0 + RG - 1) / RG : 0;
    Planes P[NP];
#pragma unroll
    for (int t = 0; t < NP; ++t) P[t] = make_planes(mv[t].planes, mv[t].units, mv[t].bytes);
    const uint8_t *tp = bq + 16 * q;
    auto tokens = [&](int b, uint4 (&tok)[4]) {
        const uint4 *src = reinterpret_cast<const uint4 *>(tp + b * 256);
#pragma unroll
        for (int k = 0; k < 4; ++k) tok[k] = src[4 * k];
    };
    auto scales = [&](int b) { return *reinterpret_cast<const float4 *>(s_d8 + 16 * b + 4 * q); };
    MxChains<TY, NM> ch;
    ch.clear();
    // The loads are unconditional: a step past the wave's last one reloads the
    // last (in bounds, never used), so the compiler's wait before a step's use
    // counts exactly the younger step's loads.
    int ir = rt0 < r1 ? rt0 : r0, ib = 0;   // next tile row and block to load
    int pr = rt0, pb = 0;                   // tile row and block of the step being computed
    if constexpr (TILE) {
        const int steps = tiles * nb;
        struct Step {
            MxW<TY> w[NM];
            uint4 tok[4];
        };
        auto issue = [&](Step &st) {
#pragma unroll
            for (int t = 0; t < NM; ++t)
                mx_load(P[PAIR ? 0 : t], (uint32_t)((PAIR ? ir + 16 * t : ir) * nb + 16 * ib), lane, st.w[t]);
            tokens(ib, st.tok);
            if (ib + 1 < nb)
                ++ib;
            else if (ir + RG < r1)
                ir += RG, ib = 0;
        };
        auto process = [&](const Step &st) {
            const float4 d8 = scales(pb);
#pragma unroll
            for (int t = 0; t < NM; ++t) ch.add(t, st.w[t], st.tok, d8, tab, lane);
            if (++pb == nb) {
                ch.finish(q, pr + c, out);
                pr += RG, pb = 0;
            }
        };
        Step sa, sb;
        issue(sa);
        prologue();
        for (int s = 0; s < steps; s += 2) {
            issue(sb);
            process(sa);
            if (s + 1 >= steps) break;
            issue(sa);
            process(sb);
        }
    } else {
        static_assert(!PAIR || NM == 1, "row-major streams take one row tile per step");
        constexpr int G = TY == T_IQ2_S ? 4 : 8, H = G / 4;   // blocks per group, register sets of four
        const int groups = tiles * ((nb + G - 1) / G);
        MxRaw<TY> raw[H][NM];
        auto issue = [&](int h) {
            const int b = G == 8 ? ib + 2 * q + (c >> 3) : ib + q, r = G == 8 ? 8 * h + (c & 7) : c;
#pragma unroll
            for (int t = 0; t < NM; ++t) mx_load_raw(P[t], (uint32_t)((ir + r) * nb + (b < nb ? b : nb - 1)), raw[h][t]);
        };
#pragma unroll
        for (int h = 0; h < H; ++h) issue(h);
        prologue();
        for (int s = 0; s < groups; ++s) {
            const int b0 = pb, n = nb - b0 < G ? nb - b0 : G;
            uint4 tok[2][4];
            MxW<TY> row[2][NM];   // the rows' own bytes of the block
            auto next = [&](int k) {
                const int b = b0 + k < nb ? b0 + k : nb - 1;
                tokens(b, tok[k & 1]);
#pragma unroll
                for (int t = 0; t < NM; ++t) mx_load_row(P[t], (uint32_t)((pr + c) * nb + b), row[k & 1][t]);
            };
            next(0);
            MxW<TY> w[H][NM][4];
            if constexpr (G == 8) {
#pragma unroll
                for (int k = 0; k < (int)(sizeof(raw[0][0].v) / 4); ++k)
#pragma unroll
                    for (int t = 0; t < NM; ++t) mx_rows8(raw[0][t].v[k], raw[H - 1][t].v[k]);
            }
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int t = 0; t < NM; ++t) mx_slices(raw[h][t], w[h][t]);
            if (ib + G < nb)
                ib += G;
            else if (ir + RG < r1)
                ir += RG, ib = 0;
            if (G == 4) issue(0);
#pragma unroll
            for (int k = 0; k < G; ++k) {
                if (k < n) {
                    next(k + 1);
                    const float4 d8 = scales(b0 + k);
#pragma unroll
                    for (int t = 0; t < NM; ++t) {
                        MxW<TY> &x = w[G == 8 ? k & 1 : 0][t][G == 8 ? k >> 1 : k];
                        mx_set_row(x, row[k & 1][t]);
                        ch.add(t, x, tok[k & 1], d8, tab, lane);
                    }
                }
                if (G == 8 && k == 3) issue(0);   // half of the set registers are free again
            }
            if (G == 8) issue(H - 1);
            pb += G;
            if (pb >= nb) {
                ch.finish(q, pr + c, out);
                pr += RG, pb = 0;
            }
        }
    }
}

// Tables and token scales of a matrix-core workgroup into LDS.
template <int TY, class D8>
__device__ __forceinline__ void mx_prologue(uint8_t *tab, float *s_d8, int n, int nb, D8 d8_of) {
    mx_fill<TY>(tab);
    for (int k = threadIdx.x; k < 16 * nb; k += MX_THREADS) {
        const int i = k & 15;
        s_d8[k] = i < n ? d8_of(i)[k >> 4] : 0.0f;
    }
    __syncthreads();
}

// The shared expert's K-quant rows in a stage launch (lbh_kt.h): workgroup wg of
// kt_wgs(): 64 rows (one 16-row tile per wave) of matrix m against one token tile;
// the token tiles of a row quad are neighbours, so its weights are fetched once.
// Two tiles a wave hold registers that the routed streams of the launch then lack
// (steps of 5 / 64 / 256 tokens: 103 / 246 / 502 us with one, 114 / 260 / 518 with
// two).
template <int TY>
__device__ __forceinline__ void kt_workgroup(const uint8_t *w, int rows, int nb, const uint8_t *tok, int n_tokens, float *y,
                                             int wg) {
    const int n_tt = (n_tokens + 15) / 16, quad = wg / n_tt, tt = wg - quad * n_tt;
    const int rt = 4 * quad + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    kt_rows<TY>(w, kt_w_bytes(TY, rows, nb), rt, nb, tok + (size_t)tt * nb * KT_TOK_TILE, [&](int i, int r, float v) {
        const int t = 16 * tt + i;
        if (t < n_tokens) y[(long long)t * rows + rt * 16 + r] = v;
    });
}

// Gate/up on the matrix cores (as k_mb_gate_up): workgroup (chunk, row tile).
// TILE: the chunks whose expert has tile copies, else the others.  NM: gate and
// up in one workgroup (2) or in two (1: few chunks of row-major matrices).  KTY: the
// first kt_wgs workgroups run the shared expert's gate and up (K-quant type
// KTY), so that one launch holds all of the stage's work.
template <int TY, bool SHARED, bool TILE, int NM, int KTY = 0>
__global__ void __launch_bounds__(MX_THREADS) k_mx_gate_up(BatchArgs a, int kt_wgs) {
    __shared__ __align__(16) uint8_t tab[MxTab<TY>::BYTES];
    __shared__ __align__(16) float s_d8[MX_MAX_NB * 16];
    if (a.plan[1]) return;
    const int nb = a.hidden / 256;
    if constexpr (KTY != 0) {
        if ((int)blockIdx.x < kt_wgs) {
            const int half = kt_wgs / 2, up = (int)blockIdx.x >= half;
            kt_workgroup<KTY>(a.kt_w[up], a.ffn_s, nb, a.kt_x, a.n_tokens, up ? a.u_s : a.g_s, (int)blockIdx.x - up * half);
            return;
        }
    }
    const int wg = (int)blockIdx.x - kt_wgs;
    // NM = 1: gate and up of a row tile are neighbouring workgroups.
    const int ffn = SHARED ? a.ffn_s : a.ffn_r, rt = a.mx_rows_gu;
    const int tiles = (ffn + rt - 1) / rt * (3 - NM);
    const int ci = wg / tiles, up = NM == 1 ? (wg - ci * tiles) & 1 : 0, tile = (wg - ci * tiles) / (3 - NM);
    const int r0 = tile * rt, r1 = r0 + rt < ffn ? r0 + rt : ffn;
    int p0, n;
    MatView mv[2];
    if constexpr (SHARED) {
        p0 = ci * a.tc;
        n = a.n_tokens - p0 < a.tc ? a.n_tokens - p0 : a.tc;
        mv[0] = a.shared.gate, mv[1] = a.shared.up;
    } else {
        if (ci >= a.plan[0]) return;
        p0 = a.chunk_p0[ci], n = a.chunk_n[ci];
        const ExpertDev &E = a.experts_mx[a.chunk_expert[ci]];
        mv[0] = E.gate, mv[1] = E.up;
    }
    if (n < a.mx_min || (mv[0].order == MAT_TILE16) != TILE) return;
    auto token = [&](int i) {
        i = i < n ? i : n - 1;
        return SHARED ? (long long)(p0 + i) : (long long)a.pair_token[p0 + i];
    };
    auto d8_of = [&](int i) { return a.xd_mx + token(i) * nb; };
    float *g = SHARED ? a.g_s : a.g_r, *u = SHARED ? a.u_s : a.u_r;
    if (up) g = u, mv[0] = mv[1];
    mx_tiles<TY, NM, TILE, false>(
        mv, r0, r1, nb, a.xq_mx + token(threadIdx.x & 15) * nb * 256, tab, s_d8,
        [&]() { mx_prologue<TY>(tab, s_d8, n, nb, d8_of); },
        [&](int i, int r, const float *res) {
            if (i < n) {
                const long long o = (long long)(p0 + i) * ffn + r;
                g[o] = res[0];
                if constexpr (NM == 2) u[o] = res[1];
            }
        });
}

// Down on the matrix cores (as k_mb_down); over tile copies each wave takes two
// adjacent 16-row tiles a step, which share the token operands.
template <int TY, bool SHARED, bool TILE, int KTY = 0>
__global__ void __launch_bounds__(MX_THREADS) k_mx_down(BatchArgs a, int kt_wgs) {
    __shared__ __align__(16) uint8_t tab[MxTab<TY>::BYTES];
    __shared__ __align__(16) float s_d8[MX_MAX_NB * 16];
    if (a.plan[1]) return;
    if constexpr (KTY != 0) {
        if ((int)blockIdx.x < kt_wgs) {
            kt_workgroup<KTY>(a.kt_w[2], a.hidden, a.ffn_s / 256, a.kt_h, a.n_tokens, a.d_s, (int)blockIdx.x);
            return;
        }
    }
    const int wg = (int)blockIdx.x - kt_wgs;
    const int nb = (SHARED ? a.ffn_s : a.ffn_r) / 256;
    const int rt = a.mx_rows_d;
    const int tiles = (a.hidden + rt - 1) / rt;
    const int ci = wg / tiles, tile = wg - ci * tiles;
    const int r0 = tile * rt, r1 = r0 + rt < a.hidden ? r0 + rt : a.hidden;
    int p0, n;
    MatView mv[1];
    if constexpr (SHARED) {
        p0 = ci * a.tc;
        n = a.n_tokens - p0 < a.tc ? a.n_tokens - p0 : a.tc;
        mv[0] = a.shared.down;
    } else {
        if (ci >= a.plan[0]) return;
        p0 = a.chunk_p0[ci], n = a.chunk_n[ci];
        mv[0] = a.experts_mx[a.chunk_expert[ci]].down;
    }
    if (n < a.mx_min || (mv[0].order == MAT_TILE16) != TILE) return;
    const uint8_t *hq = SHARED ? a.hq_mx_s : a.hq_mx_r;
    const float *hd = SHARED ? a.hd_mx_s : a.hd_mx_r;
    const int c = (int)(threadIdx.x & 15) < n ? (int)(threadIdx.x & 15) : n - 1;
    auto d8_of = [&](int i) { return hd + (long long)(p0 + (i < n ? i : n - 1)) * nb; };
    float *d = SHARED ? a.d_s : a.d_r;
    constexpr int NM = TILE ? 2 : 1;
    mx_tiles<TY, NM, TILE, true>(
        mv, r0, r1, nb, hq + (long long)(p0 + c) * nb * 256, tab, s_d8,
        [&]() { mx_prologue<TY>(tab, s_d8, n, nb, d8_of); },
        [&](int i, int r, const float *res) {
            if (i < n) {
#pragma unroll
                for (int t = 0; t < NM; ++t) d[(long long)(p0 + i) * a.hidden + r + 16 * t] = res[t];
            }
        });
}

// The shared expert's K-quant rows alone (a batch whose routed chunks all run
// on the VALU).
template <int TY>
__global__ void __launch_bounds__(MX_THREADS) k_kt_rows(const uint8_t *w0, const uint8_t *w1, int rows, int nb,
                                                        const uint8_t *tok, int n_tokens, float *y0, float *y1, int half) {
    const int second = (int)blockIdx.x >= half;
    kt_workgroup<TY>(second ? w1 : w0, rows, nb, tok, n_tokens, second ? y1 : y0, (int)blockIdx.x - second * half);
}

// Ordered combine of one token's routed outputs in its slot (ascending id)
// order, then the shared expert at 1.0 (moe.rs:141-146).
// Workgroup (1024 rows, token): the token's pairs are scalar reads, and the
// rows of eight experts are in flight at once (64 / 256 tokens: 9.0 / 20 -> 5.0 /
// 9.0 us against one row a thread with each expert's loads behind the last's).
// y is the caller's: floats, at any multiple of four bytes.
typedef float y_f4 __attribute__((ext_vector_type(4), aligned(4)));
__global__ void __launch_bounds__(MB_THREADS) k_mb_combine(BatchArgs a) {
    if (a.plan[1]) return;
    const int t = blockIdx.y, r = (int)(blockIdx.x * MB_THREADS + threadIdx.x) * 4;
    if (r >= a.hidden) return;
    const long long at = (long long)t * a.hidden + r;
    float4 sh = make_float4(0.0f, 0.0f, 0.0f, 0.0f), y = sh, acc = sh;
    if (a.has_shared) sh = *reinterpret_cast<const float4 *>(a.d_s + at);
    if (a.residual) {
        const y_f4 v = *reinterpret_cast<const y_f4 *>(a.y + at);
        y = make_float4(v.x, v.y, v.z, v.w);
    }
    for (int s0 = 0; s0 < a.top_k; s0 += 8) {
        float4 d[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (s0 + s < a.top_k)
                d[s] = *reinterpret_cast<const float4 *>(a.d_r + (long long)a.pair_of[t * a.top_k + s0 + s] * a.hidden + r);
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (s0 + s < a.top_k) {
                const float c = a.coefs[t * a.top_k + s0 + s];
                acc.x = __fadd_rn(acc.x, __fmul_rn(c, d[s].x));
                acc.y = __fadd_rn(acc.y, __fmul_rn(c, d[s].y));
                acc.z = __fadd_rn(acc.z, __fmul_rn(c, d[s].z));
                acc.w = __fadd_rn(acc.w, __fmul_rn(c, d[s].w));
            }
    }
    if (a.has_shared) {
        acc.x = __fadd_rn(acc.x, __fmul_rn(1.0f, sh.x));
        acc.y = __fadd_rn(acc.y, __fmul_rn(1.0f, sh.y));
        acc.z = __fadd_rn(acc.z, __fmul_rn(1.0f, sh.z));
        acc.w = __fadd_rn(acc.w, __fmul_rn(1.0f, sh.w));
    }
    if (a.residual) acc = make_float4(__fadd_rn(y.x, acc.x), __fadd_rn(y.y, acc.y), __fadd_rn(y.z, acc.z), __fadd_rn(y.w, acc.w));
    *reinterpret_cast<y_f4 *>(a.y + at) = y_f4{acc.x, acc.y, acc.z, acc.w};
}

// Top-k selection of every token of a batch from finished logits, one wave per token.
__global__ void __launch_bounds__(64) k_route_batch(RouteBatchArgs a) {
    const int t = blockIdx.x;
    RouterArgs r = a.r;
    r.logits = const_cast<float *>(a.logits) + (long long)t * r.n_experts;
    MoeRoute out;
    unsigned long long bad;
    select_route(r, out, bad);
    // out is the same in every lane: lane s writes slot s.
#pragma unroll
    for (int s = 0; s < MOE_MAX_ROUTED; ++s) {
        if (s < r.top_k && (int)threadIdx.x == s) {
            a.ids[(long long)t * r.top_k + s] = out.ids[s];
            a.coefs[(long long)t * r.top_k + s] = out.coefs[s];
        }
    }
    if (threadIdx.x == 0 && a.status && bad != ~0ull) atomicMin(a.status, ((unsigned long long)t << 32) | bad);
}

// ---------------------------------------------------------------- launchers

static inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

// LDS bytes of a VALU stream launch of type ty (nm matrices, nb blocks per row).
static int stream_lds_of(int ty, int nm, int tc, int nb) {
    switch (ty) {
    case T_IQ2_S: return nm == 2 ? stream_lds<T_IQ2_S, 2>(tc, nb, 2) : stream_lds<T_IQ2_S, 1>(tc, nb, 2);
    case T_IQ3_S: return nm == 2 ? stream_lds<T_IQ3_S, 2>(tc, nb, 2) : stream_lds<T_IQ3_S, 1>(tc, nb, 2);
    case T_Q4_K: return nm == 2 ? stream_lds<T_Q4_K, 2>(tc, nb, 2) : stream_lds<T_Q4_K, 1>(tc, nb, 2);
    case T_Q5_K: return nm == 2 ? stream_lds<T_Q5_K, 2>(tc, nb, 2) : stream_lds<T_Q5_K, 1>(tc, nb, 2);
    default: return 1 << 30;
    }
}

// LDS of the launches of one stream: the VALU kernel's where some chunk can run
// there (past any limit where a row's units do not fit a wave, which leaves no row
// step), and the matrix-core kernel's when it runs that type.
static int stream_max(const BatchArgs &a, int ty, int nm, int nb) {
    const bool mx = a.mx && (ty == T_IQ2_S || ty == T_IQ3_S);
    const int m = mx ? mx_lds_bytes(ty) : 0;
    if (mx && a.mx_min <= 1) return m;
    const int v = rows_per_step(2, nb) < 1 ? 1 << 30 : stream_lds_of(ty, nm, valu_cap(a, ty), nb);
    return v > m ? v : m;
}

// stage 0: sort + quantize; 1/2: routed / shared gate-up; 3/4: routed / shared down.
int batch_lds_bytes(const BatchArgs &a, int stage) {
    const int nbh = a.hidden / 256, nbr = a.ffn_r / 256, nbs = a.ffn_s / 256;
    // Q4_K / Q5_K shared rows run on the matrix cores (lbh_kt.h) and keep the limit
    // of the VALU kernel's staging alone.
    const bool kt = a.has_shared && a.shared.gate.type == T_Q4_K && a.shared.down.type == T_Q5_K;
    switch (stage) {
    case 0: {
        const int W = (a.n_tokens + 31) / 32;
        const int sort = (a.n_experts * W + 3 * a.n_experts + MB_WAVES + 4) * 4;
        return sort > MB_WAVES * 304 ? sort : MB_WAVES * 304;
    }
    case 1: return stream_max(a, a.type_gate_r, 2, nbh);
    case 2: return kt ? stream_lds_of(T_Q4_K, 2, a.tc, nbh) : a.has_shared ? stream_max(a, a.shared.gate.type, 2, nbh) : 0;
    case 3: return stream_max(a, a.type_down_r, 1, nbr);
    default: return kt ? stream_lds_of(T_Q5_K, 1, a.tc, nbs) : a.has_shared ? stream_max(a, a.shared.down.type, 1, nbs) : 0;
    }
}

template <class K>
static hipError_t allow_lds(K kernel, int lds) {
    if (lds <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
}

// The VALU kernels hold the codebook statically, the rest is dynamic.
template <int TY, bool SHARED>
static hipError_t gate_up_typed(const BatchArgs &a, hipStream_t s) {
    const int lds = stream_lds<TY, 2>(valu_cap(a, TY), a.hidden / 256, 2) - al16(GridLDS<TY>::BYTES);
    const int grid = SHARED ? cdiv(a.n_tokens, a.tc) * cdiv(a.ffn_s, a.rt_gu_s) : a.max_chunks * cdiv(a.ffn_r, a.rt_gu_r);
    // Routed IQ chunks left to the VALU beside the matrix cores: one-token
    // chunks in their own launch, then the rest (64 tokens, chunks below four on
    // the VALU beside the f16 form of the matrix-core streams: 378.7 -> 369.8 us
    // per step; the fused rows for two-token chunks too measured slower, 405 us).
    if constexpr (!SHARED && (TY == T_IQ2_S || TY == T_IQ3_S)) {
        if (a.mx) {
            hipError_t e = allow_lds(k_mb_gate_up<TY, SHARED, 1>, lds);
            if (e == hipSuccess) e = allow_lds(k_mb_gate_up<TY, SHARED, 2>, lds);
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL((k_mb_gate_up<TY, SHARED, 1>), dim3(grid), dim3(MB_THREADS), lds, s, a);
            if ((e = hipGetLastError()) != hipSuccess || a.mx_min <= 2) return e;   // no chunk of 2+ left
            hipLaunchKernelGGL((k_mb_gate_up<TY, SHARED, 2>), dim3(grid), dim3(MB_THREADS), lds, s, a);
            return hipGetLastError();
        }
    }
    hipError_t e = allow_lds(k_mb_gate_up<TY, SHARED>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_mb_gate_up<TY, SHARED>), dim3(grid), dim3(MB_THREADS), lds, s, a);
    return hipGetLastError();
}

template <int TY, bool SHARED>
static hipError_t down_typed(const BatchArgs &a, hipStream_t s) {
    const int lds = stream_lds<TY, 1>(valu_cap(a, TY), (SHARED ? a.ffn_s : a.ffn_r) / 256, 2) - al16(GridLDS<TY>::BYTES);
    const int grid = SHARED ? cdiv(a.n_tokens, a.tc) * cdiv(a.hidden, a.rt_d_s) : a.max_chunks * cdiv(a.hidden, a.rt_d_r);
    // Routed IQ downs beside the matrix cores taking every chunk of 2+ tokens:
    // the VALU chunks all hold one token and run the fused rows (64 tokens, as
    // above: 365.5 -> 359-362 us per step; with 2-token chunks also left to the
    // VALU, a second launch for them made the split slower, 382 against 370 us).
    if constexpr (!SHARED && (TY == T_IQ2_S || TY == T_IQ3_S)) {
        if (a.mx && a.mx_min <= 2) {
            const hipError_t e = allow_lds(k_mb_down<TY, SHARED, 1>, lds);
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL((k_mb_down<TY, SHARED, 1>), dim3(grid), dim3(MB_THREADS), lds, s, a);
            return hipGetLastError();
        }
    }
    hipError_t e = allow_lds(k_mb_down<TY, SHARED>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_mb_down<TY, SHARED>), dim3(grid), dim3(MB_THREADS), lds, s, a);
    return hipGetLastError();
}

// Workgroups of the shared expert's K-quant rows (kt_workgroup).
static int kt_wgs(const BatchArgs &a, int rows) { return rows / 64 * cdiv(a.n_tokens, 16); }

// KTY: the launch also holds the shared expert's K-quant gate and up / down.
template <int TY, bool SHARED, bool TILE, int NM, int KTY = 0>
static hipError_t mx_gate_up_launch(const BatchArgs &a, hipStream_t s) {
    const int kt = KTY ? 2 * kt_wgs(a, a.ffn_s) : 0;
    const int grid = (SHARED ? cdiv(a.n_tokens, a.tc) : a.max_chunks) * cdiv(SHARED ? a.ffn_s : a.ffn_r, a.mx_rows_gu) * (3 - NM);
    hipLaunchKernelGGL((k_mx_gate_up<TY, SHARED, TILE, NM, KTY>), dim3(kt + grid), dim3(MX_THREADS), 0, s, a, kt);
    return hipGetLastError();
}

template <int TY, bool SHARED, bool TILE, int KTY = 0>
static hipError_t mx_down_launch(const BatchArgs &a, hipStream_t s) {
    const int kt = KTY ? kt_wgs(a, a.hidden) : 0;
    const int grid = (SHARED ? cdiv(a.n_tokens, a.tc) : a.max_chunks) * cdiv(a.hidden, a.mx_rows_d);
    hipLaunchKernelGGL((k_mx_down<TY, SHARED, TILE, KTY>), dim3(kt + grid), dim3(MX_THREADS), 0, s, a, kt);
    return hipGetLastError();
}

// One launch for the experts with tile copies, one for the others (a layer
// with copies of some experts only needs both); the shared expert's K-quant
// rows go with the stage's first launch.
template <int TY, bool SHARED>
static hipError_t mx_gate_up_launches(const BatchArgs &a, hipStream_t s) {
    if constexpr (SHARED) {
        // Gate and up apart while that takes no more than a workgroup per CU (whole
        // steps, apart / together, shared width 4096: 16 tokens, 64 workgroups, 80 /
        // 87 us, 48 tokens, 192 workgroups, 99.6 / 95.4; width 1536: 64 tokens, 96
        // workgroups, 144 / 145, 96 tokens, 144 workgroups, 174 / 167).
        if (cdiv(a.n_tokens, a.tc) * cdiv(a.ffn_s, a.mx_rows_gu) <= 128) return mx_gate_up_launch<TY, true, false, 1>(a, s);
        return mx_gate_up_launch<TY, true, false, 2>(a, s);
    } else {
        hipError_t e = hipSuccess;
        bool kt = a.shared_kt;
        if (a.mx_copies) {
            e = kt ? mx_gate_up_launch<TY, false, true, 2, T_Q4_K>(a, s) : mx_gate_up_launch<TY, false, true, 2>(a, s);
            kt = false;
        }
        if (e != hipSuccess || a.mx_copies == 2) return e;
        // Row-major: with few workgroups gate and up apart fill the waves more
        // evenly (step of 5 tokens of top-8: 112 against 120 us, 16 tokens 190
        // against 196), with many the shared token loads count (64 tokens: 368
        // against 356 us).
        if ((long long)a.max_chunks * cdiv(a.ffn_r, a.mx_rows_gu) < 4096)
            return kt ? mx_gate_up_launch<TY, false, false, 1, T_Q4_K>(a, s) : mx_gate_up_launch<TY, false, false, 1>(a, s);
        return kt ? mx_gate_up_launch<TY, false, false, 2, T_Q4_K>(a, s) : mx_gate_up_launch<TY, false, false, 2>(a, s);
    }
}

template <int TY, bool SHARED>
static hipError_t mx_down_launches(const BatchArgs &a, hipStream_t s) {
    if constexpr (SHARED) {
        // A tile per wave instead of four, one after the other, while the default
        // rows give less than a workgroup per CU (hidden 4096 from IQ3_S 1536: 16
        // workgroups for up to 16 tokens; step of 5 tokens with copies 90 -> 81 us,
        // from 4096 105 -> 78).
        BatchArgs b = a;
        if (cdiv(a.n_tokens, a.tc) * cdiv(a.hidden, a.mx_rows_d) < 256 && a.mx_rows_d > 64) b.mx_rows_d = 64;
        return mx_down_launch<TY, true, false>(b, s);
    } else {
        hipError_t e = hipSuccess;
        bool kt = a.shared_kt;
        if (a.mx_copies) {
            e = kt ? mx_down_launch<TY, false, true, T_Q5_K>(a, s) : mx_down_launch<TY, false, true>(a, s);
            kt = false;
        }
        if (e == hipSuccess && a.mx_copies != 2)
            e = kt ? mx_down_launch<TY, false, false, T_Q5_K>(a, s) : mx_down_launch<TY, false, false>(a, s);
        return e;
    }
}

// An IQ stream with the matrix cores on: the matrix-core launch when some
// chunk can reach mx_min tokens, then the VALU launch when some chunk can stay
// below it (each kernel returns early on the other's chunks).
template <int TY, bool SHARED>
static hipError_t mx_gate_up_typed(const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    if (a.mx_min <= a.tc) {
        const hipError_t e = mx_gate_up_launches<TY, SHARED>(a, s_mx);
        if (e != hipSuccess) return e;
    }
    return a.mx_min > 1 ? gate_up_typed<TY, SHARED>(a, s_valu) : hipSuccess;
}

template <int TY, bool SHARED>
static hipError_t mx_down_typed(const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    if (a.mx_min <= a.tc) {
        const hipError_t e = mx_down_launches<TY, SHARED>(a, s_mx);
        if (e != hipSuccess) return e;
    }
    return a.mx_min > 1 ? down_typed<TY, SHARED>(a, s_valu) : hipSuccess;
}

// The matrix-core part of an IQ stream goes to s_mx, its VALU part to s_valu.
template <bool SHARED>
static hipError_t gate_up_any(int ty, const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    const hipStream_t s = s_valu;
    switch (ty) {
    case T_IQ2_S:
        return a.mx ? mx_gate_up_typed<T_IQ2_S, SHARED>(a, s_mx, s_valu) : gate_up_typed<T_IQ2_S, SHARED>(a, s);
    case T_Q4_K: return gate_up_typed<T_Q4_K, SHARED>(a, s);
    default: return hipErrorInvalidValue;
    }
}

template <bool SHARED>
static hipError_t down_any(int ty, const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    const hipStream_t s = s_valu;
    switch (ty) {
    case T_IQ2_S: return a.mx ? mx_down_typed<T_IQ2_S, SHARED>(a, s_mx, s_valu) : down_typed<T_IQ2_S, SHARED>(a, s);
    case T_IQ3_S: return a.mx ? mx_down_typed<T_IQ3_S, SHARED>(a, s_mx, s_valu) : down_typed<T_IQ3_S, SHARED>(a, s);
    case T_Q5_K: return down_typed<T_Q5_K, SHARED>(a, s);
    default: return hipErrorInvalidValue;
    }
}

bool batch_types_supported(int gate_r, int down_r, int gate_s, int down_s) {
    return gate_r == T_IQ2_S && (down_r == T_IQ3_S || down_r == T_IQ2_S) && (gate_s == T_IQ2_S || gate_s == T_Q4_K) &&
           (down_s == T_IQ2_S || down_s == T_IQ3_S || down_s == T_Q5_K);
}

hipError_t launch_moe_batch(const BatchArgs &a, hipStream_t s, const BatchStreams *streams) {
    if (a.n_tokens < 1 || a.n_tokens > BATCH_MAX_TOKENS || a.top_k < 1 || a.top_k > MOE_MAX_ROUTED ||
        a.n_experts < 1 || a.n_experts > BATCH_MAX_EXPERTS || a.tc < 1 || a.tc > BATCH_MAX_TC)
        return hipErrorInvalidValue;
    const int tsg = a.has_shared ? a.shared.gate.type : T_IQ2_S;
    const int tsd = a.has_shared ? a.shared.down.type : T_IQ3_S;
    if (!batch_types_supported(a.type_gate_r, a.type_down_r, tsg, tsd)) return hipErrorInvalidValue;
    int lds[5];
    for (int i = 0; i < 5; ++i) {
        lds[i] = batch_lds_bytes(a, i);
        if (lds[i] > 160 * 1024) return hipErrorInvalidValue;
    }
    const int nbh = a.hidden / 256;
    hipError_t e = allow_lds(k_mb_prep, lds[0]);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mb_prep, dim3(1 + cdiv((long long)a.n_tokens * nbh, MB_WAVES)), dim3(MB_THREADS), lds[0],
                       s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // Stage 1 (gate/up) and stage 2 (down) each fork the side stream after the
    // main stream's last dependency and join it before the next dependent launch.
    // With every chunk on the matrix cores a stage is one launch (two for an IQ
    // shared expert or copies of some experts only) and stays on the main
    // stream: a fork and join cost 10-20 us per stage.
    const bool two = streams && streams->side && !(a.mx && a.mx_min <= 1);
    const hipStream_t s2 = two ? streams->side : s;
    auto fork = [&](int i) -> hipError_t {
        if (!two) return hipSuccess;
        hipError_t r = hipEventRecord(streams->fork[i], s);
        return r == hipSuccess ? hipStreamWaitEvent(s2, streams->fork[i], 0) : r;
    };
    auto join = [&](int i) -> hipError_t {
        if (!two) return hipSuccess;
        hipError_t r = hipEventRecord(streams->join[i], s2);
        return r == hipSuccess ? hipStreamWaitEvent(s, streams->join[i], 0) : r;
    };
    // The shared expert's K-quant rows ride in the routed matrix-core launch;
    // without one (every chunk on the VALU) they run in a launch of their own.
    const bool mx_launch = a.mx && a.mx_min <= a.tc;
    if ((e = fork(0)) != hipSuccess) return e;
    if (a.shared_kt && !mx_launch) {
        const int n = kt_wgs(a, a.ffn_s);
        hipLaunchKernelGGL(k_kt_rows<T_Q4_K>, dim3(2 * n), dim3(MX_THREADS), 0, s2, a.kt_w[0], a.kt_w[1], a.ffn_s, nbh,
                           a.kt_x, a.n_tokens, a.g_s, a.u_s, n);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    } else if (a.has_shared && !a.shared_kt && (e = gate_up_any<true>(tsg, a, s2, s2)) != hipSuccess) {
        return e;
    }
    if ((e = gate_up_any<false>(a.type_gate_r, a, s2, s)) != hipSuccess) return e;
    if ((e = join(0)) != hipSuccess) return e;

    const bool rm = tsd == T_Q4_K || tsd == T_Q5_K;
    const int mode = !a.has_shared ? 0 : a.shared_kt ? 2 : rm ? 1 : 0;
    const long long br = (long long)a.n_tokens * a.top_k * (a.ffn_r / 256);
    const long long bs = a.has_shared ? (long long)a.n_tokens * (a.ffn_s / 256) : 0;
    hipLaunchKernelGGL(k_mb_quant_h, dim3(cdiv(br + bs, MB_WAVES)), dim3(MB_THREADS), 0, s, a, mode);
    if ((e = hipGetLastError()) != hipSuccess) return e;

    if ((e = fork(1)) != hipSuccess) return e;
    if (a.shared_kt && !mx_launch) {
        const int n = kt_wgs(a, a.hidden);
        hipLaunchKernelGGL(k_kt_rows<T_Q5_K>, dim3(n), dim3(MX_THREADS), 0, s2, a.kt_w[2], nullptr, a.hidden, a.ffn_s / 256,
                           a.kt_h, a.n_tokens, a.d_s, nullptr, n);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    } else if (a.has_shared && !a.shared_kt && (e = down_any<true>(tsd, a, s2, s2)) != hipSuccess) {
        return e;
    }
    if ((e = down_any<false>(a.type_down_r, a, s2, s)) != hipSuccess) return e;
    if ((e = join(1)) != hipSuccess) return e;

    hipLaunchKernelGGL(k_mb_combine, dim3(cdiv(a.hidden, 4 * MB_THREADS), a.n_tokens), dim3(MB_THREADS), 0, s, a);
    return hipGetLastError();
}

size_t kt_weight_bytes(int ty, int rows, int nb) { return kt_w_bytes(ty, rows, nb); }
size_t kt_token_bytes(int n_tokens, int nb) { return kt_tok_bytes(n_tokens, nb); }

hipError_t launch_kt_pack(const MatView &m, uint8_t *dst, hipStream_t s) {
    if (m.rows % 16) return hipErrorInvalidValue;
    int grid = cdiv(m.units * 4, 256);
    grid = grid > 8192 ? 8192 : grid;
    if (m.type == T_Q4_K)
        hipLaunchKernelGGL(k_kt_pack<T_Q4_K>, dim3(grid), dim3(256), 0, s, m, dst);
    else if (m.type == T_Q5_K)
        hipLaunchKernelGGL(k_kt_pack<T_Q5_K>, dim3(grid), dim3(256), 0, s, m, dst);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_units_to_tiles(const MatView &m, uint8_t *dst, hipStream_t s) {
    if (m.rows % 16 != 0) return hipErrorInvalidValue;
    int grid = cdiv((long long)(m.rows / 16) * cdiv(m.nb, 4), MX_WAVES);
    grid = grid > 8192 ? 8192 : grid;
    switch (m.type) {
    case T_IQ2_S:
        hipLaunchKernelGGL(k_units_to_tiles<T_IQ2_S>, dim3(grid), dim3(MX_THREADS), 0, s, m, dst);
        break;
    case T_IQ3_S:
        hipLaunchKernelGGL(k_units_to_tiles<T_IQ3_S>, dim3(grid), dim3(MX_THREADS), 0, s, m, dst);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_route_batch(const RouteBatchArgs &a, hipStream_t s) {
    if (a.n_tokens < 1 || a.r.n_experts < 1 || a.r.n_experts > 256 || a.r.top_k < 1 || a.r.top_k > MOE_MAX_ROUTED ||
        a.r.top_k > a.r.n_experts)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_route_batch, dim3(a.n_tokens), dim3(64), 0, s, a);
    return hipGetLastError();
}

}  // namespace lbh
