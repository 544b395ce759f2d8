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
//                 inside an expert) into a chunk table; Q8_K of every token;
//   k_mb_gate_up  per (chunk, row tile): the chunk's Q8_K activations staged
//                 in LDS, gate and up rows decoded once, integer dots against
//                 every staged token, per-(row, token) folds in the
//                 reference's block order, SwiGLU -> h;
//   k_mb_quant_h  Q8_K of every h row (the down projections' inputs,
//                 gemv.rs:161-163);
//   k_mb_down     per (chunk, row tile): the down rows against every staged h;
//   k_mb_combine  per token and output row, in the reference's order:
//                 y = ((0 + c_0 d_0) + c_1 d_1) + ... + 1.0 * d_shared.
//
// The shared expert is one more "expert" that every token selects.
//
// Several workgroups read the same expert rows (one per chunk of its tokens),
// so the weight loads keep the default cache policy here.
#define LBH_WEIGHT_CPOL 0
#include "lbh_internal.h"
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
// quantize kernels: block k's 256 quants at q + 256 k, its scale at d[k].
// split: in the order of the IQ3_S instructions (dword 2g + h of lane quarter
// p holds elements 32g + 8p + 4h .. + 3), else in element order (IQ2_S).
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

// Sort of the batch's pairs by expert (workgroup 0) and Q8_K of every token
// (the other workgroups, four blocks per wave).
__device__ __forceinline__ void quantize_rows_out(const float *x, long long nblocks, long long first, uint8_t *plain,
                                                  uint8_t *rm, uint8_t *lds_wave, MxRows mx = MxRows{}) {
    // Blocks [first, first + 4) (x points at block `first`) into the wave's
    // LDS, then out to global memory: the GGML bytes, (rm != NULL) the copy
    // with residue-major qs, and (mx.q != NULL) the matrix-core operand copy.
    const int lane = threadIdx.x & 63;
    const long long cnt = nblocks - first < 4 ? nblocks - first : 4;
    quantize_blocks_wave(x, lds_wave, 0, cnt);
    wave_sync();
    if (mx.q) {
        for (int k = lane; k < (int)cnt * 64; k += 64) {
            const int blk = k >> 6, w = k & 63;
            // w: destination dword, from source dword sw
            const int sw = mx.split ? 8 * ((w >> 1) & 7) + 2 * (w >> 4) + (w & 1) : w;
            reinterpret_cast<uint32_t *>(mx.q)[(first + blk) * 64 + w] =
                *reinterpret_cast<const uint32_t *>(lds_wave + blk * 292 + 4 + 4 * sw);
        }
        if (lane < cnt) mx.d[first + lane] = *reinterpret_cast<const float *>(lds_wave + lane * 292);
    }
    const int dw = (int)cnt * 73;
    for (int k = lane; k < dw; k += 64) {
        const int blk = k / 73, w = k - blk * 73;
        const uint8_t *sb = lds_wave + blk * 292;
        const uint32_t v = *reinterpret_cast<const uint32_t *>(sb + 4 * w);
        if (plain) *reinterpret_cast<uint32_t *>(plain + (first + blk) * 292 + 4 * w) = v;
        if (rm) {
            uint32_t r = v;
            if (w >= 1 && w <= 64) {
                const int q = w - 1, g = q >> 3, t = q & 7;
                const uint8_t *src = sb + 4 + 32 * g + t;
                r = (uint32_t)src[0] | ((uint32_t)src[8] << 8) | ((uint32_t)src[16] << 16) | ((uint32_t)src[24] << 24);
            }
            *reinterpret_cast<uint32_t *>(rm + (first + blk) * 292 + 4 * w) = r;
        }
    }
    wave_sync();
}

__global__ void __launch_bounds__(MB_THREADS) k_mb_prep(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    if (blockIdx.x > 0) {
        const int nb = a.hidden / 256;
        const long long nblocks = (long long)a.n_tokens * nb;
        const long long first = ((long long)(blockIdx.x - 1) * MB_WAVES + (tid >> 6)) * 4;
        const bool rm = a.has_shared && !a.shared_gemm && (a.shared.gate.type == T_Q4_K || a.shared.gate.type == T_Q5_K);
        if (first < nblocks)
            quantize_rows_out(a.x + first * 256, nblocks, first, a.q8x, rm ? a.q8x_rm : nullptr,
                              smem + (tid >> 6) * 4 * 292, MxRows{a.mx ? a.xq_mx : nullptr, a.xd_mx, false});
        return;
    }
    const int NE = a.n_experts, T = a.n_tokens, K = a.top_k, TC = a.tc;
    const int W = (T + 31) / 32;
    uint32_t *bm = reinterpret_cast<uint32_t *>(smem);              // [NE][W] token bitmaps
    int32_t *cnt = reinterpret_cast<int32_t *>(bm + NE * W);       // [NE]
    int32_t *off = cnt + NE;                                       // [NE] first sorted pair
    int32_t *coff = off + NE;                                      // [NE] first chunk
    int32_t *part = coff + NE;                                     // [2][MB_THREADS] scan partials
    int32_t *flags = part + 2 * MB_THREADS;
    for (int i = tid; i < NE * W; i += MB_THREADS) bm[i] = 0;
    if (tid == 0) flags[0] = 0;
    __syncthreads();
    for (int p = tid; p < T * K; p += MB_THREADS) {
        const int t = p / K;
        const uint32_t e = a.ids[p];
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
    part[tid] = sc;
    part[MB_THREADS + tid] = sk;
    __syncthreads();
    // Inclusive scan of the partials (Hillis-Steele), then exclusive offsets.
    for (int d = 1; d < MB_THREADS; d <<= 1) {
        const int v0 = tid >= d ? part[tid - d] : 0;
        const int v1 = tid >= d ? part[MB_THREADS + tid - d] : 0;
        __syncthreads();
        part[tid] += v0;
        part[MB_THREADS + tid] += v1;
        __syncthreads();
    }
    {
        int o = part[tid] - sc, ko = part[MB_THREADS + tid] - sk;
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
        for (int p = tid; p < T * K; p += MB_THREADS) {
            const int t = p / K;
            const uint32_t e = a.ids[p];
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
        a.plan[0] = bad ? 0 : part[2 * MB_THREADS - 1];
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
// (VALU K-quant down); 2: GGML bytes (K-quant GEMM down).
__global__ void __launch_bounds__(MB_THREADS) k_mb_quant_h(BatchArgs a, int shared_mode) {
    __shared__ __align__(16) uint8_t lds[MB_WAVES * 4 * 292];
    __shared__ __align__(16) float hbuf[MB_WAVES][4 * 256];
    if (a.plan[1]) return;
    const int nbr = a.ffn_r / 256, nbs = a.ffn_s / 256;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const long long br = (long long)a.n_tokens * a.top_k * nbr;
    const long long brp = (br + 3) & ~3ll;   // chunks of four never straddle the two ranges
    const long long bs = a.has_shared ? (long long)a.n_tokens * nbs : 0;
    const long long chunk = ((long long)blockIdx.x * MB_WAVES + wid) * 4;
    uint8_t *lw = lds + wid * 4 * 292;
    // Lane (block first + lane / 16, elements 16 (lane % 16) ..) forms the
    // sixteen values it quantizes below.
    auto swiglu_blocks = [&](const float *g, const float *u, long long first, long long nblocks) {
        const long long blk = first + (lane >> 4);
        if (blk < nblocks) {
            const long long base = blk * 256 + 16 * (lane & 15);
            float *hb = &hbuf[wid][(lane >> 4) * 256 + 16 * (lane & 15)];
#pragma unroll
            for (int i = 0; i < 16; ++i) hb[i] = swiglu_ref(g[base + i], u[base + i]);
        }
        wave_sync();
    };
    if (chunk < br) {
        swiglu_blocks(a.g_r, a.u_r, chunk, br);
        quantize_rows_out(&hbuf[wid][0], br, chunk, a.q8h_r, nullptr, lw, MxRows{a.mx ? a.hq_mx_r : nullptr, a.hd_mx_r, a.type_down_r == T_IQ3_S});
    } else if (chunk >= brp && chunk - brp < bs) {
        const long long f = chunk - brp;
        swiglu_blocks(a.g_s, a.u_s, f, bs);
        quantize_rows_out(&hbuf[wid][0], bs, f, shared_mode == 1 ? nullptr : a.q8h_s, shared_mode == 1 ? a.q8h_s : nullptr,
                          lw, MxRows{a.mx && shared_mode == 0 ? a.hq_mx_s : nullptr, a.hd_mx_s, a.shared.down.type == T_IQ3_S});
    }
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
//   64 tokens   gate/up 159 -> 88 us, down 91 -> 61 us (step 417 -> 354 us)
//   256 tokens  gate/up 375 -> 222 us, down 242 -> 143 us (step 832 -> 611 us)

typedef int mx_i4 __attribute__((ext_vector_type(4)));

constexpr int MX_THREADS = 256;
constexpr int MX_WAVES = MX_THREADS / 64;
constexpr int MX_MAX_NB = 64;

// IQ2_S scaled weights by scale nibble n: bytes 0-2 of {lo+, lo-, hi+, hi-} are
// the split +-m (1 + 2n) = 256 hi + lo (lo signed) of m = 8, 25, 43.
struct MxProducts {
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
    if (TY == T_IQ2_S && threadIdx.x < 16)
        o[MxTab<TY>::GRID / 16 + threadIdx.x] = reinterpret_cast<const uint4 *>(&c_mx_products.v[0][0])[threadIdx.x];
}

// One lane's 64 weights of its row's block.
//   IQ2_S  w: qs of its two groups, sg: their sign dwords, e: low nibble of
//          byte j the groups' qh fields of lookup j; TILE: high nibble of byte
//          j the scale nibble of half group j, else sc holds the four nibbles.
//   IQ3_S  w: lookup bytes of four quads (below), sg: their sign dwords;
//          qh, sc: the row's qh bytes and scale nibbles, all groups.
template <int TY>
struct MxW;
template <>
struct MxW<T_IQ2_S> {
    uint32_t w[2], sg[2], e, sc, d;
};
template <>
struct MxW<T_IQ3_S> {
    uint32_t w[4], sg[2], qh[2], sc, d;
};

typedef uint32_t mx_u3 __attribute__((ext_vector_type(3)));

// TILE: the matrix is a 16-row tile copy (k_units_to_tiles), whose lane slices
// lie in lane order: u is the tile's first unit.  Else the row-major device
// layout: u is the lane's unit.
template <bool TILE>
__device__ __forceinline__ void mx_load(const Planes &P, uint32_t u, int lane, MxW<T_IQ2_S> &o) {
    const int q = lane >> 4;
    if constexpr (TILE) {
        const uint4 a = bld128(P, u * 64 + 16u * lane, 0);
        o.w[0] = a.x, o.w[1] = a.y, o.sg[0] = a.z, o.sg[1] = a.w;
        o.e = bld32(P, u * 16 + 4u * lane, 4 * P.U16);
        o.d = bld16(P, u * 2 + 2u * (lane & 15), 5 * P.U16);
        o.sc = 0;
    } else {
        const uint32_t u16 = u * 16, po = (uint32_t)(q >> 1) * P.U16 + 8u * (uint32_t)(q & 1);
        const uint2 a = bld64(P, u16 + po, 0), c = bld64(P, u16 + po, 2 * P.U16);
        o.w[0] = a.x, o.w[1] = a.y, o.sg[0] = c.x, o.sg[1] = c.y;
        o.e = bld32(P, u16 + 4u * (uint32_t)(q >> 1), 4 * P.U16);
        o.sc = bld16(P, u16 + 8u + 2u * (uint32_t)q, 4 * P.U16);
        o.d = bld16(P, u * 2, 5 * P.U16);
    }
}
template <bool TILE>
__device__ __forceinline__ void mx_load(const Planes &P, uint32_t u, int lane, MxW<T_IQ3_S> &o) {
    const int q = lane >> 4;
    uint4 a;
    uint2 s;
    if constexpr (TILE) {
        a = bld128(P, u * 64 + 16u * lane, 0);
        s = bld64(P, u * 32 + 8u * lane, 4 * P.U16);
        u += lane & 15;
    } else {
        a = bld128(P, u * 16 + (uint32_t)q * P.U16, 0);
        s = bld64(P, u * 16 + (uint32_t)(q >> 1) * P.U16 + 8u * (uint32_t)(q & 1), 4 * P.U16);
    }
    const mx_u3 t = __builtin_bit_cast(mx_u3, __builtin_amdgcn_raw_buffer_load_b96(P.rsrc, u * 12, 6 * P.U16, WEIGHT_CPOL));
    o.w[0] = a.x, o.w[1] = a.y, o.w[2] = a.z, o.w[3] = a.w;
    o.sg[0] = s.x, o.sg[1] = s.y;
    o.qh[0] = t.x, o.qh[1] = t.y, o.sc = t.z;
    o.d = bld16(P, u * 2, 6 * P.U16 + 12 * P.U);
}

__device__ __forceinline__ void lanes32_swap(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void lanes16_swap(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}

// Integer block sums bs[i] of (token 4q + i, row c) from the lane's weights
// and its 64 quants of token c (tok[m]: 16 bytes).
template <bool TILE>
__device__ __forceinline__ void mx_block(const MxW<T_IQ2_S> &o, const uint4 (&tok)[4], const uint8_t *tab, int lane,
                                         int32_t (&bs)[4]) {
    const GridRef<T_IQ2_S> grid(tab);
    // row-major: the lane's qh fields are fields 2 (q & 1), + 1 of its dword
    const uint32_t e = TILE ? o.e : o.e >> (4 * ((lane >> 4) & 1));
    mx_i4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const Iq2sGroup g = Iq2sGroup::make(o.w[m >> 1], e, m >> 1, o.sg[m >> 1]);
        const uint32_t na = TILE ? (e >> (8 * m)) & 0xf0u
                                 : (m == 0 ? o.sc << 4 : o.sc >> (4 * m - 4)) & 0xf0u;
        const uint4 t = *reinterpret_cast<const uint4 *>(tab + MxTab<T_IQ2_S>::GRID + na);
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

// IQ3_S quads: the lane's lookups are 2q and 2q + 1 of every group; quad 0 / 1
// holds lookup 2q / 2q + 1 of groups 0, 1, 4, 5, quad 2 / 3 those of groups 2,
// 3, 6, 7 (byte i: the i-th listed group).  Sign dword j: byte i the sign byte
// q of the i-th group of quads 2j, 2j + 1.  A tile copy holds them so; the
// row-major slice of lane q is groups 2q, 2q + 1 whole, and the four lanes of
// a row exchange 4 x 4 pieces (v_permlane32_swap / 16_swap).
__device__ __forceinline__ void mx_iq3_exchange(const MxW<T_IQ3_S> &o, uint32_t (&qd)[4], uint32_t (&sg)[2]) {
    // t[j]: the lookups 2j, 2j + 1 of both groups, for the row's lane j
    uint32_t t[4] = {perm(o.w[2], o.w[0], 0x05040100u), perm(o.w[2], o.w[0], 0x07060302u),
                     perm(o.w[3], o.w[1], 0x05040100u), perm(o.w[3], o.w[1], 0x07060302u)};
    lanes32_swap(t[0], t[2]);
    lanes32_swap(t[1], t[3]);
    lanes16_swap(t[0], t[1]);
    lanes16_swap(t[2], t[3]);
    qd[0] = perm(t[2], t[0], 0x06040200u), qd[1] = perm(t[2], t[0], 0x07050301u);
    qd[2] = perm(t[3], t[1], 0x06040200u), qd[3] = perm(t[3], t[1], 0x07050301u);
    uint32_t w0 = perm(o.sg[1], o.sg[0], 0x05010400u), w1 = perm(o.sg[1], o.sg[0], 0x07030602u);
    lanes32_swap(w0, w1);
    sg[0] = perm(w1, w0, 0x05040100u), sg[1] = perm(w1, w0, 0x07060302u);
    lanes16_swap(sg[0], sg[1]);
}

template <bool TILE>
__device__ __forceinline__ void mx_block(const MxW<T_IQ3_S> &o, const uint4 (&tok)[4], const uint8_t *tab, int lane,
                                         int32_t (&bs)[4]) {
    const Iq3SignedRef grid(tab);
    uint32_t qd[4] = {o.w[0], o.w[1], o.w[2], o.w[3]}, sg[2] = {o.sg[0], o.sg[1]};
    if constexpr (!TILE) mx_iq3_exchange(o, qd, sg);
    // bits 0, 1 of byte i: the high index bits of lookups 2q, 2q + 1
    const uint32_t ta = o.qh[0] >> (2 * (lane >> 4)), tb = o.qh[1] >> (2 * (lane >> 4));
    const uint32_t hb[2] = {perm(tb, ta, 0x05040100u), perm(tb, ta, 0x07060302u)};
    uint32_t word[2][8];   // [even, odd lookup][group]
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int j = k >> 1, odd = k & 1;
        // iq3_signed_offset = x + 256 y per byte
        const uint32_t h = (odd ? hb[j] << 1 : hb[j] << 2) & 0x04040404u;
        const uint32_t s = (odd ? sg[j] >> 1 : sg[j] << 3) & 0x78787878u;
        const uint32_t x = qd[k] & 0xfcfcfcfcu, y = (qd[k] & 0x03030303u) | h | s;
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

// One wave step's inputs: NM slices of the lane's rows and its quants of
// token c.
template <int TY, int NM>
struct MxStep {
    MxW<TY> w[NM];
    uint4 tok[4];
};

// Dynamic LDS of a matrix-core stream workgroup (beside its static tables and
// scales): with split > 1, per tile the f32 terms [matrix][block][token][row].
__host__ __device__ constexpr int mx_dyn_lds(int nm, int split, int nb) {
    return split > 1 ? (MX_WAVES / split) * nm * nb * 256 * 4 : 0;
}
__host__ __device__ constexpr int mx_lds_bytes(int ty, int nm, int split, int nb) {
    return (ty == T_IQ2_S ? MxTab<T_IQ2_S>::BYTES : MxTab<T_IQ3_S>::BYTES) +
           (split > 1 ? mx_dyn_lds(nm, split, nb) : MX_MAX_NB * 16 * 4);
}

// Rows [r0, r1) (multiples of 16 NM') of NM tiles per step against the chunk's
// tokens: the NM matrices mv (gate and up), or, PAIR, NM adjacent 16-row tiles
// of the one matrix mv[0], which share the step's token operands.
//   S = 1: the waves take tiles r0 + RW wid, + 4 RW, ... (RW = 16 or 16 NM
//     rows) to r1, computing every block of a tile in order, the chains of
//     the lane's four (token, row) results in registers; s_d8[16 b + i] is the
//     scale of token i's block b.
//   S > 1: the workgroup holds MX_WAVES / S tiles, the S waves of a tile take
//     its blocks j, j + S, ... and write the f32 term (d * d8) * (float)bsum of
//     each (row, token, block) to LDS; after a workgroup barrier one thread
//     per (tile, token, row) folds its terms in block order (lbh_rows.h: chain =
//     0 + t_0 + t_1 + ...) and calls out(token column, row, values).  bd: the
//     scales of the lane's tokens, d8_of(i)[b].
// bq: the lane's token operand row.  The first step's loads are issued before
// `prologue` (tables and scales to LDS, ended by a workgroup barrier); then
// each step's loads are in flight while the one before is computed.
template <int TY, int NM, int S, bool TILE, bool PAIR, class Prologue, class D8, class Out>
__device__ __forceinline__ void mx_tiles(const MatView *mv, int r0, int r1, int nb, const uint8_t *bq, const uint8_t *tab,
                                         const float *s_d8, float *terms, Prologue prologue, D8 d8_of, Out out) {
    constexpr int NP = PAIR ? 1 : NM, RW = PAIR ? 16 * NM : 16;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, q = lane >> 4;
    const int tl = wid / S, j = wid - tl * S;
    const int rt0 = r0 + RW * tl;
    // steps of the wave: its blocks of one tile (S > 1), or its tiles' blocks (S = 1)
    const int tiles = S > 1 ? 1 : (r1 - rt0 + RW * MX_WAVES - 1) / (RW * MX_WAVES);
    const int steps = rt0 < r1 ? (S > 1 ? (j < nb ? (nb - j + S - 1) / S : 0) : tiles * nb) : 0;
    Planes P[NP];
#pragma unroll
    for (int t = 0; t < NP; ++t) P[t] = make_planes(mv[t].planes, mv[t].units, mv[t].bytes);
    const uint8_t *tp = bq + 64 * q;
    // The loads are unconditional: a step past the wave's last one reloads the
    // last (in bounds, never used), so the compiler's wait before a step's use
    // counts exactly the younger step's loads.
    int ir = rt0 < r1 ? rt0 : r0, ib = S > 1 ? (j < nb ? j : nb - 1) : 0;   // next tile row and block to load
    auto issue = [&](MxStep<TY, NM> &st) {
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            const int r = PAIR ? ir + 16 * t : ir;
            const uint32_t u = TILE ? (uint32_t)(r * nb + 16 * ib) : (uint32_t)((r + c) * nb + ib);
            mx_load<TILE>(P[PAIR ? 0 : t], u, lane, st.w[t]);
        }
        const uint4 *src = reinterpret_cast<const uint4 *>(tp + ib * 256);
#pragma unroll
        for (int k = 0; k < 4; ++k) st.tok[k] = src[k];
        if constexpr (S > 1) {
            ib = ib + S < nb ? ib + S : ib;
        } else if (++ib == nb) {
            if (ir + RW * MX_WAVES < r1)
                ir += RW * MX_WAVES, ib = 0;
            else
                ib = nb - 1;
        }
    };
    float chain[NM][4];   // S == 1
#pragma unroll
    for (int t = 0; t < NM; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) chain[t][i] = 0.0f;
    int pr = rt0, pb = S > 1 ? j : 0;   // tile row and block of the step being computed
    auto process = [&](const MxStep<TY, NM> &st) {
        float d8[4];
        if constexpr (S == 1) {
            const float4 v = *reinterpret_cast<const float4 *>(s_d8 + 16 * pb + 4 * q);
            d8[0] = v.x, d8[1] = v.y, d8[2] = v.z, d8[3] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) d8[i] = d8_of(4 * q + i)[pb];
        }
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            int32_t bs[4];
            mx_block<TILE>(st.w[t], st.tok, tab, lane, bs);
            const float d = f16_to_f32(st.w[t].d);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float term = __fmul_rn(__fmul_rn(d, d8[i]), (float)bs[i]);
                if constexpr (S == 1)
                    chain[t][i] = __fadd_rn(chain[t][i], term);   // blocks in order
                else
                    terms[((tl * NM + t) * nb + pb) * 256 + 16 * (4 * q + i) + c] = term;
            }
        }
        if constexpr (S > 1) {
            pb += S;
        } else if (++pb == nb) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float res[NM];
#pragma unroll
                for (int t = 0; t < NM; ++t) {
                    res[t] = TY == T_IQ2_S ? __fmul_rn(0.125f, chain[t][i]) : chain[t][i];   // q8_k.rs:369
                    chain[t][i] = 0.0f;
                }
                out(4 * q + i, pr + c, res);
            }
            pr += RW * MX_WAVES, pb = 0;
        }
    };
    MxStep<TY, NM> sa, sb;
    issue(sa);
    prologue();
    for (int s = 0; s < steps; s += 2) {
        issue(sb);
        process(sa);
        if (s + 1 >= steps) break;
        issue(sa);
        process(sb);
    }
    if constexpr (S > 1) {
        __syncthreads();
        for (int p = threadIdx.x; p < (MX_WAVES / S) * 256; p += MX_THREADS) {
            const int ptl = p >> 8, cc = (p >> 4) & 15, row = p & 15;
            const float *src = terms + ptl * NM * nb * 256 + cc * 16 + row;
            float res[NM];
#pragma unroll
            for (int t = 0; t < NM; ++t) {
                float ch = 0.0f;
                for (int b = 0; b < nb; ++b) ch = __fadd_rn(ch, src[(t * nb + b) * 256]);
                res[t] = TY == T_IQ2_S ? __fmul_rn(0.125f, ch) : ch;  // q8_k.rs:369
            }
            out(cc, r0 + 16 * ptl + row, res);
        }
    }
}

// Tables and token scales of a matrix-core workgroup into LDS.
template <int TY, int S, class D8>
__device__ __forceinline__ void mx_prologue(uint8_t *tab, float *s_d8, int n, int nb, D8 d8_of) {
    mx_fill<TY>(tab);
    if constexpr (S == 1)
        for (int k = threadIdx.x; k < 16 * nb; k += MX_THREADS) {
            const int i = k & 15;
            s_d8[k] = i < n ? d8_of(i)[k >> 4] : 0.0f;
        }
    __syncthreads();
}

// Gate/up on the matrix cores (as k_mb_gate_up): workgroup (chunk, row tile).
// TILE: the chunks whose expert has tile copies, else the others.
template <int TY, bool SHARED, int S, bool TILE>
__global__ void __launch_bounds__(MX_THREADS) k_mx_gate_up(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ __align__(16) uint8_t tab[MxTab<TY>::BYTES];
    __shared__ __align__(16) float s_d8[S == 1 ? MX_MAX_NB * 16 : 4];
    if (a.plan[1]) return;
    const int nb = a.hidden / 256;
    const int ffn = SHARED ? a.ffn_s : a.ffn_r, rt = S == 1 ? a.mx_rows_gu : 16 * MX_WAVES / S;
    const int tiles = (ffn + rt - 1) / rt;
    const int ci = blockIdx.x / tiles, tile = blockIdx.x - ci * tiles;
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
    mx_tiles<TY, 2, S, TILE, false>(
        mv, r0, r1, nb, a.xq_mx + token(threadIdx.x & 15) * nb * 256, tab, s_d8, reinterpret_cast<float *>(smem),
        [&]() { mx_prologue<TY, S>(tab, s_d8, n, nb, d8_of); }, d8_of,
        [&](int i, int r, const float *res) {
            if (i < n) {
                const long long o = (long long)(p0 + i) * ffn + r;
                g[o] = res[0];
                u[o] = res[1];
            }
        });
}

// Down on the matrix cores (as k_mb_down); with S = 1 each wave takes two
// adjacent 16-row tiles a step, which share the token operands.
template <int TY, bool SHARED, int S, bool TILE>
__global__ void __launch_bounds__(MX_THREADS) k_mx_down(BatchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ __align__(16) uint8_t tab[MxTab<TY>::BYTES];
    __shared__ __align__(16) float s_d8[S == 1 ? MX_MAX_NB * 16 : 4];
    if (a.plan[1]) return;
    const int nb = (SHARED ? a.ffn_s : a.ffn_r) / 256;
    const int rt = S == 1 ? a.mx_rows_d : 16 * MX_WAVES / S;
    const int tiles = (a.hidden + rt - 1) / rt;
    const int ci = blockIdx.x / tiles, tile = blockIdx.x - ci * tiles;
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
    constexpr int NM = S == 1 ? 2 : 1;
    mx_tiles<TY, NM, S, TILE, true>(
        mv, r0, r1, nb, hq + (long long)(p0 + c) * nb * 256, tab, s_d8, reinterpret_cast<float *>(smem),
        [&]() { mx_prologue<TY, S>(tab, s_d8, n, nb, d8_of); }, d8_of,
        [&](int i, int r, const float *res) {
            if (i < n) {
#pragma unroll
                for (int t = 0; t < NM; ++t) d[(long long)(p0 + i) * a.hidden + r + 16 * t] = res[t];
            }
        });
}

// Ordered combine of one token's routed outputs in its slot (ascending id)
// order, then the shared expert at 1.0 (moe.rs:141-146).
__global__ void __launch_bounds__(MB_THREADS) k_mb_combine(BatchArgs a) {
    if (a.plan[1]) return;
    const long long total = (long long)a.n_tokens * a.hidden;
    for (long long k = (long long)blockIdx.x * MB_THREADS + threadIdx.x; k < total;
         k += (long long)gridDim.x * MB_THREADS) {
        const int t = (int)(k / a.hidden), r = (int)(k - (long long)t * a.hidden);
        float acc = 0.0f;
        for (int s = 0; s < a.top_k; ++s) {
            const int p = a.pair_of[t * a.top_k + s];
            acc = __fadd_rn(acc, __fmul_rn(a.coefs[t * a.top_k + s], a.d_r[(long long)p * a.hidden + r]));
        }
        if (a.has_shared) acc = __fadd_rn(acc, __fmul_rn(1.0f, a.d_s[(long long)t * a.hidden + r]));
        a.y[k] = a.residual ? __fadd_rn(a.y[k], acc) : acc;
    }
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

// LDS bytes of a stream launch of type ty (nm matrices, nb blocks per row).
static int stream_lds_of(int ty, int nm, int tc, int nb) {
    switch (ty) {
    case T_IQ2_S: return nm == 2 ? stream_lds<T_IQ2_S, 2>(tc, nb, 2) : stream_lds<T_IQ2_S, 1>(tc, nb, 2);
    case T_IQ3_S: return nm == 2 ? stream_lds<T_IQ3_S, 2>(tc, nb, 2) : stream_lds<T_IQ3_S, 1>(tc, nb, 2);
    case T_Q4_K: return nm == 2 ? stream_lds<T_Q4_K, 2>(tc, nb, 2) : stream_lds<T_Q4_K, 1>(tc, nb, 2);
    case T_Q5_K: return nm == 2 ? stream_lds<T_Q5_K, 2>(tc, nb, 2) : stream_lds<T_Q5_K, 1>(tc, nb, 2);
    default: return 1 << 30;
    }
}

// LDS of the launches of one stream: the VALU kernel's, and the matrix-core
// kernel's when it runs that type.
static int stream_max(const BatchArgs &a, int ty, int nm, int nb, int split) {
    const int v = stream_lds_of(ty, nm, valu_cap(a, ty), nb);
    if (!a.mx || (ty != T_IQ2_S && ty != T_IQ3_S)) return v;
    const int m = mx_lds_bytes(ty, nm, split < 1 ? 1 : split, nb);
    return v > m ? v : m;
}

// stage 0: sort + quantize; 1/2: routed / shared gate-up; 3/4: routed / shared down.
int batch_lds_bytes(const BatchArgs &a, int stage) {
    const int nbh = a.hidden / 256, nbr = a.ffn_r / 256, nbs = a.ffn_s / 256;
    switch (stage) {
    case 0: {
        const int W = (a.n_tokens + 31) / 32;
        const int sort = (a.n_experts * W + 3 * a.n_experts + 2 * MB_THREADS + 4) * 4;
        return sort > MB_WAVES * 4 * 292 ? sort : MB_WAVES * 4 * 292;
    }
    case 1: return stream_max(a, a.type_gate_r, 2, nbh, a.mx_split_gu);
    case 2: return a.has_shared ? stream_max(a, a.shared.gate.type, 2, nbh, a.mx_split_gu) : 0;
    case 3: return stream_max(a, a.type_down_r, 1, nbr, a.mx_split_d);
    default: return a.has_shared ? stream_max(a, a.shared.down.type, 1, nbs, a.mx_split_d) : 0;
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
    // chunks in their own launch, then the rest (measured on MI355X at the
    // configs[3] shapes: 378.7 -> 369.8 us per step; the fused rows for
    // two-token chunks too measured slower, 405 us).
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
    // the VALU chunks all hold one token and run the fused rows (measured on
    // MI355X at the configs[3] shapes: 365.5 -> 359-362 us per step; with
    // 2-token chunks also left to the VALU, a second launch for them made the
    // split slower, 382 against 370 us).
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

template <int TY, bool SHARED, int S, bool TILE>
static hipError_t mx_gate_up_launch(const BatchArgs &a, hipStream_t s) {
    const int lds = mx_dyn_lds(2, S, a.hidden / 256), rows = S == 1 ? a.mx_rows_gu : 16 * MX_WAVES / S;
    const hipError_t e = allow_lds(k_mx_gate_up<TY, SHARED, S, TILE>, lds);
    if (e != hipSuccess) return e;
    const int grid = (SHARED ? cdiv(a.n_tokens, a.tc) : a.max_chunks) * cdiv(SHARED ? a.ffn_s : a.ffn_r, rows);
    hipLaunchKernelGGL((k_mx_gate_up<TY, SHARED, S, TILE>), dim3(grid), dim3(MX_THREADS), lds, s, a);
    return hipGetLastError();
}

template <int TY, bool SHARED, int S, bool TILE>
static hipError_t mx_down_launch(const BatchArgs &a, hipStream_t s) {
    const int nb = (SHARED ? a.ffn_s : a.ffn_r) / 256;
    const int lds = mx_dyn_lds(1, S, nb), rows = S == 1 ? a.mx_rows_d : 16 * MX_WAVES / S;
    const hipError_t e = allow_lds(k_mx_down<TY, SHARED, S, TILE>, lds);
    if (e != hipSuccess) return e;
    const int grid = (SHARED ? cdiv(a.n_tokens, a.tc) : a.max_chunks) * cdiv(a.hidden, rows);
    hipLaunchKernelGGL((k_mx_down<TY, SHARED, S, TILE>), dim3(grid), dim3(MX_THREADS), lds, s, a);
    return hipGetLastError();
}

// One launch for the experts with tile copies, one for the others (a layer
// with copies of some experts only needs both).
template <int TY, bool SHARED, int S>
static hipError_t mx_gate_up_split(const BatchArgs &a, hipStream_t s) {
    hipError_t e = hipSuccess;
    if (SHARED || a.mx_copies != 2) e = mx_gate_up_launch<TY, SHARED, S, false>(a, s);
    if constexpr (!SHARED)
        if (e == hipSuccess && a.mx_copies) e = mx_gate_up_launch<TY, SHARED, S, true>(a, s);
    return e;
}

template <int TY, bool SHARED, int S>
static hipError_t mx_down_split(const BatchArgs &a, hipStream_t s) {
    hipError_t e = hipSuccess;
    if (SHARED || a.mx_copies != 2) e = mx_down_launch<TY, SHARED, S, false>(a, s);
    if constexpr (!SHARED)
        if (e == hipSuccess && a.mx_copies) e = mx_down_launch<TY, SHARED, S, true>(a, s);
    return e;
}

// An IQ stream with the matrix cores on: the matrix-core launch when some
// chunk can reach mx_min tokens, then the VALU launch when some chunk can stay
// below it (each kernel returns early on the other's chunks).  mx_split_* is
// the number of waves that share a 16-row tile (1, 2 or 4).
template <int TY, bool SHARED>
static hipError_t mx_gate_up_typed(const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    if (a.mx_min <= a.tc) {
        const hipError_t e = a.mx_split_gu == 4   ? mx_gate_up_split<TY, SHARED, 4>(a, s_mx)
                             : a.mx_split_gu == 2 ? mx_gate_up_split<TY, SHARED, 2>(a, s_mx)
                                                  : mx_gate_up_split<TY, SHARED, 1>(a, s_mx);
        if (e != hipSuccess) return e;
    }
    return a.mx_min > 1 ? gate_up_typed<TY, SHARED>(a, s_valu) : hipSuccess;
}

template <int TY, bool SHARED>
static hipError_t mx_down_typed(const BatchArgs &a, hipStream_t s_mx, hipStream_t s_valu) {
    if (a.mx_min <= a.tc) {
        const hipError_t e = a.mx_split_d == 4   ? mx_down_split<TY, SHARED, 4>(a, s_mx)
                             : a.mx_split_d == 2 ? mx_down_split<TY, SHARED, 2>(a, s_mx)
                                                 : mx_down_split<TY, SHARED, 1>(a, s_mx);
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
    hipLaunchKernelGGL(k_mb_prep, dim3(1 + cdiv((long long)a.n_tokens * nbh, 4 * MB_WAVES)), dim3(MB_THREADS), lds[0],
                       s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // Stage 1 (gate/up) and stage 2 (down) each fork the side stream after the
    // main stream's last dependency and join it before the next dependent launch.
    const bool two = streams && streams->side;
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
    if ((e = fork(0)) != hipSuccess) return e;
    if (a.has_shared && a.shared_gemm) {
        // shared gate/up on the matrix cores: they only need Q8_K(x)
        GemmArgs gm{};
        gm.b = a.bx;
        gm.nb = nbh;
        gm.n_tokens = a.n_tokens;
        gm.shape = a.gemm_shape;
        gm.n_mat = 2;
        gm.mat[0] = a.sg;
        gm.mat[1] = a.su;
        if ((e = launch_prep_b(a.q8x, a.n_tokens, nbh, a.bx, s2)) != hipSuccess) return e;
        if ((e = launch_kq_gemm(gm, s2)) != hipSuccess) return e;
    } else if (a.has_shared && (e = gate_up_any<true>(tsg, a, s2, s2)) != hipSuccess) {
        return e;
    }
    if ((e = gate_up_any<false>(a.type_gate_r, a, s2, s)) != hipSuccess) return e;
    if ((e = join(0)) != hipSuccess) return e;

    const bool rm = tsd == T_Q4_K || tsd == T_Q5_K;
    const int mode = !a.has_shared ? 0 : a.shared_gemm ? 2 : rm ? 1 : 0;
    const long long br = (long long)a.n_tokens * a.top_k * (a.ffn_r / 256);
    const long long bs = a.has_shared ? (long long)a.n_tokens * (a.ffn_s / 256) : 0;
    hipLaunchKernelGGL(k_mb_quant_h, dim3(cdiv(((br + 3) & ~3ll) + bs, 4 * MB_WAVES)), dim3(MB_THREADS), 0, s, a, mode);
    if ((e = hipGetLastError()) != hipSuccess) return e;

    if ((e = fork(1)) != hipSuccess) return e;
    if (a.has_shared && a.shared_gemm) {
        const int nbs = a.ffn_s / 256;
        GemmArgs gm{};
        gm.b = a.bh;
        gm.nb = nbs;
        gm.n_tokens = a.n_tokens;
        gm.shape = a.gemm_shape;
        gm.n_mat = 1;
        gm.mat[0] = a.sd;
        if ((e = launch_prep_b(a.q8h_s, a.n_tokens, nbs, a.bh, s2)) != hipSuccess) return e;
        if ((e = launch_kq_gemm(gm, s2)) != hipSuccess) return e;
    } else if (a.has_shared && (e = down_any<true>(tsd, a, s2, s2)) != hipSuccess) {
        return e;
    }
    if ((e = down_any<false>(a.type_down_r, a, s2, s)) != hipSuccess) return e;
    if ((e = join(1)) != hipSuccess) return e;

    const long long total = (long long)a.n_tokens * a.hidden;
    int g = cdiv(total, MB_THREADS);
    g = g > 4096 ? 4096 : g;
    hipLaunchKernelGGL(k_mb_combine, dim3(g), dim3(MB_THREADS), 0, s, a);
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
