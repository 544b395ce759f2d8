// lbh_gemm.hip — Q4_K / Q5_K x Q8_K for a batch of tokens on the f16 matrix
// cores (v_mfma_f32_16x16x32_f16, 32x32x16), bit-identical to the reference's per-row
// dot (dot_q4_or_q5_k, crates/bridge-quant-layout/src/q8_k.rs:247-327) for
// every (row, token):
//
//   lane_sums[l] = sum_j sc_j * sum_{k<4} q[32j + 8k + l] * a[32j + 8k + l]
//   minimum_sum  = sum_j mn_j * (bsums[2j] + bsums[2j + 1])
//   per block:  sums[l] += (d * d8) * lane_sums[l];  sum -= (dmin * d8) * minimum_sum
//   result = sum + sums[0] + ... + sums[7]
//
// The integer stage runs on the matrix cores, the f32 chains on the VALU in
// the reference's block order.  Exactness: the A operand holds the weight
// pre-scaled by its sub-block scale, w = sc * q <= 63 * 31 = 1953, and the B
// operand the Q8_K byte, both integers an f16 holds exactly; every product
// and every partial sum of one lane sum is an integer below 2^24
// (32 * 1953 * 128 < 2^23), so the f32 accumulation inside the instruction
// is exact in any order and the result equals lane_sums[l] converted to f32
// (which the reference's `as f32` also does exactly).  Each lane sum (the 32
// elements of residue l) is one K = 32 instruction on an operand pair, or two
// K = 16 ones, the second accumulating onto the first.  The minimum sum is a
// K = 16 instruction on the 6-bit mins
// against the pair sums of bsums split as 128 * bh + bl: A holds
// (128 mn_j, mn_j), B holds (bh_j, bl_j), |partial sums| < 8 * 63 * 8128.
//
// Layouts (built once per matrix by k_prep_a, per call by k_prep_b):
//   A tile (32 rows, block b): 17 operands x 64 lanes x 16 B, operand o at
//     position op_pos(o) (0-3, 16, 4-15: a pass of the three-pass form reads
//     consecutive ones), then the 32 rows' d, -dmin, d, d as f32 (the last two
//     keep the tile a multiple of 512 B).
//     Operand 2l + p, lane j: row j % 32, the 8 f16 of sub-blocks
//     4p + 2 (j / 32) + e / 4, element 8 (e % 4) + l.
//     Operand 16, lane j: sub-blocks 4 (j / 32) + e / 2, (128 mn, mn).
//   B tile (32 tokens, block b): the same operands for token j % 32 (Q8_K
//     bytes; operand 16 = (bh, bl)), then the 32 tokens' d8.
//   A and B use the same slot <-> element convention, so the contraction
//   pairs identical elements whatever the instruction's internal k order.
#include "lbh_internal.h"
#include "lbh_rows.h"

namespace lbh {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int OPS = 17;                          // 8 residues x 2 halves + the minimum
constexpr int OP_BYTES = 1024;                   // 64 lanes x 8 f16
constexpr int A_TILE = OPS * OP_BYTES + 32 * 16; // + the rows' scales: d, -dmin, d, d (32 f32 each)
constexpr int B_TILE = OPS * OP_BYTES + 32 * 4;  // + d8 of the tile's tokens
constexpr int PIECES = OPS + 1;                  // 1 KiB staging units per tile (the last one partial)

// Position of operand o in a tile: residue operands 0-3, the minimum operand,
// residue operands 4-15.
__host__ __device__ constexpr int op_pos(int o) { return o < 4 ? o : o == 16 ? 4 : o + 1; }

__device__ __forceinline__ uint32_t pack_f16(_Float16 lo, _Float16 hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
}

// ------------------------------------------------------------ A preparation
//
// One wave per (row tile, block).  Reads the block from the chunk-major
// device layout (lbh_layout.h): Q4_K chunk 0 header, chunks 1-8 residue-major
// qs; Q5_K chunk 0 header, 1-2 residue-major qh, 3-10 residue-major qs.
template <int TY>
__global__ void __launch_bounds__(64) k_prep_a(MatView m, uint8_t *a_out) {
    const int lane = threadIdx.x;
    const int nb = m.nb;
    const int tile = blockIdx.x / nb, b = blockIdx.x - tile * nb;
    const int h = lane >> 5;
    const int row = tile * 32 + (lane & 31);
    const bool valid = row < m.rows;
    const long long U = m.units, u = (long long)row * nb + b;
    constexpr int QS0 = TY == T_Q5_K ? 3 : 1;
    constexpr int NCH = TY == T_Q5_K ? 11 : 9;
    uint8_t blk[NCH * 16];
    for (int c = 0; c < NCH; ++c) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (valid) v = *reinterpret_cast<const uint4 *>(m.planes + ((long long)c * U + u) * 16);
        *reinterpret_cast<uint4 *>(blk + 16 * c) = v;
    }
    int sc[8], mn[8];
    {
        const uint32_t s0 = *reinterpret_cast<const uint32_t *>(blk + 4);
        const uint32_t s1 = *reinterpret_cast<const uint32_t *>(blk + 8);
        const uint32_t s2 = *reinterpret_cast<const uint32_t *>(blk + 12);
        for (int j = 0; j < 8; ++j) scale_min_of(s0, s1, s2, j, sc[j], mn[j]);
    }
    uint8_t *tile_base = a_out + ((long long)tile * nb + b) * A_TILE;
    uint8_t *dst = tile_base + lane * 16;
    for (int l = 0; l < 8; ++l) {
        for (int p = 0; p < 2; ++p) {
            uint32_t o[4];
            for (int e = 0; e < 8; e += 2) {
                int w[2];
                for (int f = 0; f < 2; ++f) {
                    const int jj = 4 * p + 2 * h + ((e + f) >> 2), k = (e + f) & 3;
                    // residue-major: dword l of qs group jj / 2 holds elements l + 8k
                    const int pos = 4 * l + k;
                    const uint8_t qb = blk[16 * (QS0 + 2 * (jj >> 1)) + pos];
                    int v = (jj & 1) ? (qb >> 4) : (qb & 15);
                    if (TY == T_Q5_K) v += ((blk[16 + pos] >> jj) & 1) << 4;
                    w[f] = sc[jj] * v;
                }
                o[e >> 1] = pack_f16((_Float16)w[0], (_Float16)w[1]);
            }
            *reinterpret_cast<uint4 *>(dst + op_pos(2 * l + p) * OP_BYTES) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
    {
        uint32_t o[4];
        for (int e = 0; e < 8; e += 2) {
            const int jj = 4 * h + (e >> 1);
            o[e >> 1] = pack_f16((_Float16)(128 * mn[jj]), (_Float16)mn[jj]);
        }
        *reinterpret_cast<uint4 *>(dst + op_pos(16) * OP_BYTES) = make_uint4(o[0], o[1], o[2], o[3]);
    }
    if (lane < 32) {
        float2 v = make_float2(0.0f, 0.0f);
        if (valid) {
            const uint32_t hdr = *reinterpret_cast<const uint32_t *>(blk);
            v = make_float2(f16_to_f32(hdr & 0xffffu), f16_to_f32(hdr >> 16));
        }
        // -dmin: the minimum term is added, sum + (-dmin * d8) * minimum_sum,
        // the same f32 value as the reference's sum - (dmin * d8) * minimum_sum
        // (x - y is x + (-y), and (-a) * b is -(a * b) under round to nearest).
        float *dm = reinterpret_cast<float *>(tile_base + OPS * OP_BYTES);
        dm[lane] = v.x;
        dm[32 + lane] = -v.y;
        dm[64 + lane] = v.x;
        dm[96 + lane] = v.x;
    }
}

// ------------------------------------------------------------ B preparation
//
// One wave per (token tile, block) from GGML Q8_K bytes (d @0, qs @4,
// bsums @260; block (t, b) at q8 + (t * nb + b) * 292).  Lane j needs the
// four sub-blocks 2 (j / 32) + {0, 1, 4, 5} of token j % 32.
__global__ void __launch_bounds__(64) k_prep_b(const uint8_t *q8, int n_tokens, int nb, uint8_t *b_out) {
    const int lane = threadIdx.x;
    const int tile = blockIdx.x / nb, b = blockIdx.x - tile * nb;
    const int h = lane >> 5;
    const int t = tile * 32 + (lane & 31);
    const bool valid = t < n_tokens;
    const uint8_t *blk = q8 + ((long long)(valid ? t : 0) * nb + b) * 292;
    uint8_t *tile_base = b_out + ((long long)tile * nb + b) * B_TILE;
    uint8_t *dst = tile_base + lane * 16;
    // qs of sub-blocks 2h, 2h + 1 (p = 0) and 4 + 2h, 5 + 2h (p = 1): 64 bytes each
    uint32_t q[2][16];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (valid) v = *reinterpret_cast<const uint4 *>(blk + 4 + 32 * (4 * p + 2 * h) + 16 * i);
            q[p][4 * i] = v.x, q[p][4 * i + 1] = v.y, q[p][4 * i + 2] = v.z, q[p][4 * i + 3] = v.w;
        }
#pragma unroll
    for (int l = 0; l < 8; ++l) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                _Float16 x[2];
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    // element 8k + l of sub-block 4p + 2h + (e + f) / 4: byte 32 * ((e + f) / 4) + 8k + l
                    const int k = (e + f) & 3, byte = 32 * ((e + f) >> 2) + 8 * k + l;
                    x[f] = (_Float16)(int)(int8_t)(q[p][byte >> 2] >> (8 * (byte & 3)));
                }
                o[e >> 1] = pack_f16(x[0], x[1]);
            }
            *reinterpret_cast<uint4 *>(dst + op_pos(2 * l + p) * OP_BYTES) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
    {
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const int jj = 4 * h + (e >> 1);
            int bsp = 0;
            if (valid)
                bsp = (int)*reinterpret_cast<const int16_t *>(blk + 260 + 4 * jj) +
                      (int)*reinterpret_cast<const int16_t *>(blk + 262 + 4 * jj);
            o[e >> 1] = pack_f16((_Float16)(bsp >> 7), (_Float16)(bsp & 127));
        }
        *reinterpret_cast<uint4 *>(dst + op_pos(16) * OP_BYTES) = make_uint4(o[0], o[1], o[2], o[3]);
    }
    if (lane < 32)
        reinterpret_cast<float *>(tile_base + OPS * OP_BYTES)[lane] = valid ? *reinterpret_cast<const float *>(blk) : 0.0f;
}

// ------------------------------------------------------------------ GEMM
//
// Three forms, chosen by their counts of workgroups (launch_kq_gemm).  All run
// the f32 chains on the VALU in the reference's block order, 8 instructions per
// chain, 16 x 16 pairs and block, besides the scales.
//
//   k_kq_gemm_split  16 rows x 16 NT tokens per workgroup of three waves, each
//     running three of the nine chains, both operands from L1 / L2: a short
//     pass for launches of few pairs, bound by the operands' traffic from L2.
//     77 tokens x 4096 rows x 4096 (Q4_K): 19 us with NT = 3, 21 with NT = 2
//     (330 MB), 29 with the 2 x 2 form; 1024 rows: 16 us where that took 31.
//   k_kq_gemm_2x2    64 rows x 64 tokens, both operands in LDS: 31-35 us for any
//     count of workgroups up to the 256 CUs (LDS reads and staging latency).
//   k_kq_gemm_lds    128 rows x 64 tokens, a wave 16 rows x 64 tokens in three
//     passes over K of three chains each (64 accumulators: four waves fit a
//     SIMD).  The row operands go straight from L2 to registers, one block
//     ahead, each serving the wave's four token tiles; the token operands are
//     staged in LDS two blocks at a time (direct buffer-to-LDS loads).  512
//     tokens x 12288 rows x 4096 (Q5_K): 112 us, of which 68 are the issue of
//     the VALU and matrix instructions, 58 the LDS reads and 16 the row
//     operands' way past L2; with both operands in LDS and one 32 x 32 tile per
//     wave, which reads LDS twice as much, 137.  All nine chains at once with 16
//     x 64 pairs (two waves per SIMD, the tokens read once) took 136, four-wave
//     workgroups of 64 rows 124, plain workgroup order 133, row operands and
//     staging two blocks ahead 113.
//
// The split and LDS forms use v_mfma_f32_16x16x32_f16 with tokens as operand A
// and rows as operand B: lane 16 q + c supplies token / row c and the 8
// elements that tile lane (row c, half q & 1) holds in operand 2l + q / 2, so
// one instruction gives a lane sum of 16 x 16 pairs, result i of the lane being
// (token 4q + i, row c): the row's d is the lane's own and the four tokens' d8
// one 16-byte read.

typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Lane 16 q + c's place in a 32-row tile's operand pair 2l, 2l + 1 (rows 16 half
// + c), in its minimum operand, and in its scale rows.
__device__ __forceinline__ uint32_t op_lane(int lane, int half) {
    const int q = lane >> 4, c = lane & 15;
    return (uint32_t)((q >> 1) * OP_BYTES + (16 * half + c + 32 * (q & 1)) * 16);
}
__device__ __forceinline__ uint32_t min_lane(int lane, int half) {
    const int q = lane >> 4, c = lane & 15;
    return (uint32_t)(op_pos(16) * OP_BYTES + (16 * half + c + 32 * (q >> 1)) * 16 + 8 * (q & 1));
}

// The row operands of one wave: 16 rows of an A tile row, every block.
struct RowSrc {
    __amdgpu_buffer_rsrc_t r;
    uint32_t op, mn, sc;   // lane offsets: operands, minimum operand, d / -dmin
    __device__ __forceinline__ RowSrc(const uint8_t *a, int tile, int half, int nb, int lane) {
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a + (long long)tile * nb * A_TILE), (short)0, nb * A_TILE,
                                              0x00020000);
        op = op_lane(lane, half);
        mn = min_lane(lane, half);
        sc = (uint32_t)(OPS * OP_BYTES + (16 * half + (lane & 15)) * 4);
    }
    __device__ __forceinline__ v8h residue(int b, int l) const {
        return __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(r, op, (uint32_t)(b * A_TILE + op_pos(2 * l) * OP_BYTES), 0));
    }
    __device__ __forceinline__ v4h minimum(int b) const {
        return __builtin_bit_cast(v4h, __builtin_amdgcn_raw_buffer_load_b64(r, mn, (uint32_t)(b * A_TILE), 0));
    }
    __device__ __forceinline__ float d(int b) const {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, sc, (uint32_t)(b * A_TILE), 0));
    }
    __device__ __forceinline__ float neg_dmin(int b) const {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, sc, (uint32_t)(b * A_TILE + 128), 0));
    }
};

// acc += (scale * d8) * sum for one chain of one token tile.
__device__ __forceinline__ void fold4(float (&acc)[4], const float (&s)[4], const v4f &r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn(s[i], r[i]));
}

// ---- 2 x 2 tiles in LDS
//
// Workgroup: 2 x 2 tiles of 32 rows x 32 tokens (v_mfma_f32_32x32x16_f16, two
// per lane sum), two waves per tile: wave half 0 runs residues 0-3 and the
// minimum, half 1 residues 4-7, so a wave keeps 16 (row, token) pairs x 4 or 5
// f32 chains in registers and two waves share each SIMD.  Per block the
// workgroup stages its two A tiles and two B tiles (70 KiB) in LDS,
// double-buffered, through registers two blocks ahead: block b + 2 is loaded
// into one register set while block b is computed, and the set loaded during
// block b - 1 is written to LDS after it (140 KiB in flight per CU).
constexpr int RG = 2, TG = 2;                 // row tiles, token tiles per workgroup
constexpr int NW = 2 * RG * TG;               // waves
constexpr int UNITS = (RG + TG) * PIECES;     // 1 KiB staging units per block
constexpr int UPW = UNITS / NW;               // units per wave (9)
static_assert(UNITS % NW == 0, "every wave stages the same number of units");

// LDS tiles are PIECES whole KiB: the partial last piece is staged with all
// 64 lanes (no divergent loads or stores, so the compiler's wait counts stay
// exact); the bytes past the tile's data are never read.
constexpr int LDS_TILE = PIECES * OP_BYTES;
struct GemmLDS {
    uint8_t a[2][RG][LDS_TILE];
    uint8_t b[2][TG][LDS_TILE];
};

// Where staging unit k of wave `wid` lives: unit u = wid + NW k is piece
// u % PIECES of tile u / PIECES (A tiles first).  Tiles past the matrix or
// the batch are clamped to the last one (their results are not stored).
struct Unit {
    bool is_a;
    int tile, piece;
};
__device__ __forceinline__ Unit unit_of(int wid, int k) {
    const int u = wid + NW * k;
    Unit x;
    x.tile = u / PIECES;
    x.piece = u - x.tile * PIECES;
    x.is_a = x.tile < RG;
    if (!x.is_a) x.tile -= RG;
    return x;
}

struct StageSrc {
    __amdgpu_buffer_rsrc_t ra, rb;   // this workgroup's A tiles / B tiles (all blocks)
    int last_a, last_b;              // last valid tile, relative to the workgroup's first
};

// Byte offset of unit x of block b in its descriptor (all operands uniform,
// so the offset is a scalar operand of the load).
__device__ __forceinline__ uint32_t unit_offset(const StageSrc &src, const Unit &x, int nb, int b) {
    if (x.is_a) {
        const int t = x.tile < src.last_a ? x.tile : src.last_a;
        return (uint32_t)((t * nb + b) * A_TILE + x.piece * OP_BYTES);
    }
    const int t = x.tile < src.last_b ? x.tile : src.last_b;
    return (uint32_t)((t * nb + b) * B_TILE + x.piece * OP_BYTES);
}
__device__ __forceinline__ uint8_t *unit_dst(GemmLDS &S, const Unit &x, int buf) {
    return (x.is_a ? S.a[buf][x.tile] : S.b[buf][x.tile]) + x.piece * OP_BYTES;
}

// Loads block b's units of this wave into R; for b >= nb the lane offset is
// pushed past the descriptors' ranges (< 2^31 bytes), so the loads return
// zeros and read no memory.
__device__ __forceinline__ void stage_regs(const StageSrc &src, uint4 (&R)[UPW], int nb, int b, int wid, int lane) {
    const uint32_t vo = (uint32_t)lane * 16 + (b < nb ? 0u : 0x80000000u);
    const int bc = b < nb ? b : nb - 1;
#pragma unroll
    for (int k = 0; k < UPW; ++k) {
        const Unit x = unit_of(wid, k);
        R[k] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(x.is_a ? src.ra : src.rb, vo,
                                                                               unit_offset(src, x, nb, bc), 0));
    }
}
__device__ __forceinline__ void store_regs(GemmLDS &S, const uint4 (&R)[UPW], int buf, int wid, int lane) {
#pragma unroll
    for (int k = 0; k < UPW; ++k) {
        const Unit x = unit_of(wid, k);
        reinterpret_cast<uint4 *>(unit_dst(S, x, buf))[lane] = R[k];
    }
}
// Both MFMAs of residue l (operands 2l, 2l + 1), or the minimum (l = 8).
__device__ __forceinline__ v16f residue_mfma(const v8h *Av, const v8h *Bv, int l) {
    const v16f zero = {};
    if (l == 8) {
        v8h a = Av[op_pos(16) * 64], b = Bv[op_pos(16) * 64];
        asm volatile("" : "+v"(a), "+v"(b));
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, zero, 0, 0, 0);
    }
    const int p0 = op_pos(2 * l), p1 = op_pos(2 * l + 1);
    v8h a0 = Av[p0 * 64], b0 = Bv[p0 * 64], a1 = Av[p1 * 64], b1 = Bv[p1 * 64];
    asm volatile("" : "+v"(a0), "+v"(b0), "+v"(a1), "+v"(b1));
    const v16f c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b0, zero, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b1, c, 0, 0, 0);
}

// The f32 chains of one wave.  The lane's pair i (0..15) is row
// 8 (i / 4) + 4 (lane / 32) + i % 4 of the tile, token lane % 32.
template <int HV>
struct Chains {
    float c[16][4];   // residues 4 HV + r
    float msum[16];   // the minimum chain (HV 0)
};

// One block of one wave: HV 0 folds residues 0-3 and the minimum, HV 1
// residues 4-7, each in the reference's order within its chain.
template <int HV>
__device__ __forceinline__ void fold_block(Chains<HV> &ch, const uint8_t *At, const uint8_t *Bt, int lane) {
    const int h = lane >> 5;
    const v8h *Av = reinterpret_cast<const v8h *>(At) + lane;
    const v8h *Bv = reinterpret_cast<const v8h *>(Bt) + lane;
    const float d8 = reinterpret_cast<const float *>(Bt + OPS * OP_BYTES)[lane & 31];
    // d of rows 8q + 4h + 0..3 (the lane's pairs 4q..4q + 3): one 16-byte read per q
    const float4 *dv = reinterpret_cast<const float4 *>(At + OPS * OP_BYTES);
    float sc[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 d = dv[2 * q + h];
        sc[4 * q] = __fmul_rn(d.x, d8);
        sc[4 * q + 1] = __fmul_rn(d.y, d8);
        sc[4 * q + 2] = __fmul_rn(d.z, d8);
        sc[4 * q + 3] = __fmul_rn(d.w, d8);
    }
    // The MFMAs of step r + 1 go out before step r is folded; the empty asm
    // statements (no instructions) keep the compiler from hoisting every
    // step's MFMAs (16 result registers each) above the folds.
    v16f cn = residue_mfma(Av, Bv, 4 * HV);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const v16f c = cn;
        if (r < 3) cn = residue_mfma(Av, Bv, 4 * HV + r + 1);
        else if (HV == 0) cn = residue_mfma(Av, Bv, 8);
#pragma unroll
        for (int i = 0; i < 16; ++i) ch.c[i][r] = __fadd_rn(ch.c[i][r], __fmul_rn(sc[i], c[i]));
        asm volatile("" : "+v"(ch.c[0][r]), "+v"(ch.c[1][r]), "+v"(ch.c[2][r]), "+v"(ch.c[3][r]),
                     "+v"(ch.c[4][r]), "+v"(ch.c[5][r]), "+v"(ch.c[6][r]), "+v"(ch.c[7][r]),
                     "+v"(ch.c[8][r]), "+v"(ch.c[9][r]), "+v"(ch.c[10][r]), "+v"(ch.c[11][r]),
                     "+v"(ch.c[12][r]), "+v"(ch.c[13][r]), "+v"(ch.c[14][r]), "+v"(ch.c[15][r]));
    }
    if (HV == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 m = dv[8 + 2 * q + h];   // -dmin
            const float ms[4] = {__fmul_rn(m.x, d8), __fmul_rn(m.y, d8), __fmul_rn(m.z, d8), __fmul_rn(m.w, d8)};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                ch.msum[4 * q + e] = __fadd_rn(ch.msum[4 * q + e], __fmul_rn(ms[e], cn[4 * q + e]));
        }
    }
}

template <int HV>
__device__ __forceinline__ void gemm_tile(const GemmArgs &g, GemmLDS &S, const StageSrc &src,
                                          int rg, int tg, int tw, int wid, int lane, int rt0, int tt0) {
    const int nb = g.nb;
    Chains<HV> ch;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        ch.msum[i] = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) ch.c[i][r] = 0.0f;
    }
    // Block j: loaded into R[j % 2] during block j - 2, written to LDS
    // buffer j % 2 after block j - 1, computed as block j.  Every load
    // is unconditional, so the compiler's wait before each LDS store
    // leaves the younger set's loads in flight; loads past the last
    // block are sent out of the descriptor's range (they return zeros
    // without touching memory).
    uint4 R0[UPW], R1[UPW];
    stage_regs(src, R0, nb, 0, wid, lane);
    stage_regs(src, R1, nb, 1, wid, lane);
    store_regs(S, R0, 0, wid, lane);
    __syncthreads();
    for (int b = 0; b < nb; b += 2) {
        stage_regs(src, R0, nb, b + 2, wid, lane);
        fold_block<HV>(ch, S.a[0][rg], S.b[0][tg], lane);
        if (b + 1 < nb) store_regs(S, R1, 1, wid, lane);
        __syncthreads();
        if (b + 1 >= nb) break;
        stage_regs(src, R1, nb, b + 3, wid, lane);
        fold_block<HV>(ch, S.a[1][rg], S.b[1][tg], lane);
        if (b + 2 < nb) store_regs(S, R0, 0, wid, lane);
        __syncthreads();
    }

    // result = minimum chain + sums[0] + ... + sums[7]: half 0 adds its four
    // chains onto the minimum chain and hands the partial to half 1 through
    // LDS (the staging buffers are free after the last barrier).
    const int h = lane >> 5;
    float *xch = reinterpret_cast<float *>(&S) + tw * 16 * 64;
    if (HV == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v = ch.msum[i];
#pragma unroll
            for (int r = 0; r < 4; ++r) v = __fadd_rn(v, ch.c[i][r]);
            xch[i * 64 + lane] = v;
        }
    }
    __syncthreads();
    if (HV == 1) {
        const int t = (tt0 + tg) * 32 + (lane & 31);
        if (t >= g.n_tokens) return;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = (rt0 + rg) * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
            float v = xch[i * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) v = __fadd_rn(v, ch.c[i][r]);
            if (row < g.rows) g.y[(long long)t * g.rows + row] = v;
        }
    }
}

__global__ void __launch_bounds__(64 * NW) k_kq_gemm_2x2(GemmArgs g) {
    extern __shared__ __align__(16) uint8_t smem[];
    GemmLDS &S = *reinterpret_cast<GemmLDS *>(smem);
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // waves w and w + RG * TG (the two halves of one tile) land on the same SIMD
    const int tw = wid % (RG * TG), hv = wid / (RG * TG);
    const int rg = tw % RG, tg = tw / RG;
    const int n_rt = (g.rows + 31) / 32, n_tt = (g.n_tokens + 31) / 32;
    const int row_wgs = (n_rt + RG - 1) / RG, tok_wgs = (n_tt + TG - 1) / TG;
    // XCD-aware order: workgroups are dealt to the eight XCDs round robin;
    // consecutive workgroups of one XCD share a row tile, so each A tile is
    // fetched into that XCD's L2 once for all of its token tiles.  Within an
    // XCD's range the token tiles are taken in two phases (the first half of
    // the token workgroups over all of the XCD's row bands, then the second
    // half): half the activation tiles are live in the XCD's 4 MB L2 at a
    // time, for every A band read twice (measured 2-4% faster than one phase).
    const int nwg = row_wgs * tok_wgs;
    const int id = (int)blockIdx.x;
    if (id >= nwg) return;
    const int nfull = nwg & ~7;
    int lin = id < nfull ? (id % 8) * (nfull / 8) + id / 8 : id;   // a bijection of [0, nwg)
    {
        constexpr int PHASES = 2;
        const int per = nfull / 8;
        if (id < nfull && tok_wgs % PHASES == 0 && per % tok_wgs == 0) {
            const int x = lin / per, i = lin - x * per;
            const int tq = tok_wgs / PHASES, bands = per / tok_wgs;
            const int ph = i / (bands * tq), rem = i - ph * bands * tq;
            lin = x * per + (rem / tq) * tok_wgs + ph * tq + rem % tq;   // still a bijection of the XCD's range
        }
    }
    const int wrt = lin / tok_wgs, wtt = lin - wrt * tok_wgs;
    const int rt0 = wrt * RG, tt0 = wtt * TG;

    // The descriptors span only the workgroup's valid tiles: the partial last
    // staging piece of the last tile then reads zeros past it, never memory
    // past the allocation.
    StageSrc src;
    src.last_a = n_rt - 1 - rt0 < RG - 1 ? n_rt - 1 - rt0 : RG - 1;
    src.last_b = n_tt - 1 - tt0 < TG - 1 ? n_tt - 1 - tt0 : TG - 1;
    src.ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(g.a + (long long)rt0 * g.nb * A_TILE), (short)0,
                                               (src.last_a + 1) * g.nb * A_TILE, 0x00020000);
    src.rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(g.b + (long long)tt0 * g.nb * B_TILE), (short)0,
                                               (src.last_b + 1) * g.nb * B_TILE, 0x00020000);

    if (hv == 0)
        gemm_tile<0>(g, S, src, rg, tg, tw, wid, lane, rt0, tt0);
    else
        gemm_tile<1>(g, S, src, rg, tg, tw, wid, lane, rt0, tt0);
}

// ---- tokens in LDS

constexpr int GL_WAVES = 8, GL_NT = 4;
constexpr int GL_PASS_OPS = 6;                       // operand positions of a pass (pass 0: five)
constexpr int GL_TILE = GL_PASS_OPS * OP_BYTES;      // one 32-token tile's operands of a pass
constexpr int GL_BLOCK = 2 * GL_TILE + 256;          // two tiles, then the 64 tokens' d8
// Two distinct arrays: the compiler's wait before a read of one leaves the
// loads into the other in flight.
__shared__ __align__(16) uint8_t gl_lds0[2 * GL_BLOCK];
__shared__ __align__(16) uint8_t gl_lds1[2 * GL_BLOCK];

#define GL_FENCE __builtin_amdgcn_sched_barrier(0)

typedef __attribute__((address_space(3))) void lds_void;

template <int BUF>
__device__ __forceinline__ uint8_t *gl_buffer() {
    return BUF == 0 ? gl_lds0 : gl_lds1;
}

// Blocks b and b + 1 (clamped) of the token tiles, operand positions op0 .. op0
// + 5: 24 pieces of 1 KiB, three per wave, and each block's d8 by one wave.
template <int BUF>
__device__ __forceinline__ void gl_stage(__amdgpu_buffer_rsrc_t rb, int last, int nb, int b, int op0, int wid, int lane) {
    uint8_t *buf = gl_buffer<BUF>();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int u = wid + GL_WAVES * k, blk = u / 12, t = (u / 6) & 1, piece = u % 6;
        const int bb = b + blk < nb ? b + blk : nb - 1;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void *)(buf + blk * GL_BLOCK + t * GL_TILE + piece * OP_BYTES), 16, lane * 16,
                                                 (uint32_t)(((t < last ? t : last) * nb + bb) * B_TILE + (op0 + piece) * OP_BYTES), 0, 0);
    }
    if (wid < 2) {
        const int bb = b + wid < nb ? b + wid : nb - 1, t = lane >> 5;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void *)(buf + wid * GL_BLOCK + 2 * GL_TILE), 4,
                                                 (t < last ? t : last) * nb * B_TILE + (lane & 31) * 4,
                                                 (uint32_t)(bb * B_TILE + OPS * OP_BYTES), 0, 0);
    }
}

// Three chains of a pass and its running operands.  MIN (pass 0): the minimum
// chain (slot 2) and lane chains 0, 1; otherwise three lane chains from l0.
template <bool MIN>
struct GlPass {
    float c[3][GL_NT][4];
    v8h a[3];
    float d, ndm;

    __device__ __forceinline__ void load(const RowSrc &A, int b, int l0, int k) {
        if (MIN && k == 2) a[2] = __builtin_bit_cast(v8h, __builtin_shufflevector(A.minimum(b), A.minimum(b), 0, 1, 2, 3, 0, 1, 2, 3));
        else a[k] = A.residue(b, l0 + k);
    }
    __device__ __forceinline__ void load_scales(const RowSrc &A, int b) {
        d = A.d(b);
        if (MIN) ndm = A.neg_dmin(b);
    }

    __device__ __forceinline__ void block(const uint8_t *buf, const RowSrc &A, int bn, int l0, int lane) {
        const int q = lane >> 4;
        const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
        // step 2 k + p: chain k, the token tiles of the 32-token tile p
        v8h x[2][2];
        auto tokens = [&](int st) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uint8_t *t = buf + (st & 1) * GL_TILE;
                if (MIN && st >= 4) {
                    const v4h h = *reinterpret_cast<const v4h *>(t + min_lane(lane, n));
                    x[st & 1][n] = __builtin_shufflevector(h, h, 0, 1, 2, 3, 0, 1, 2, 3);
                } else {
                    x[st & 1][n] = *reinterpret_cast<const v8h *>(t + (st & ~1) * OP_BYTES + op_lane(lane, n));
                }
            }
        };
        float4 e[GL_NT];
#pragma unroll
        for (int n = 0; n < GL_NT; ++n) e[n] = *reinterpret_cast<const float4 *>(buf + 2 * GL_TILE + (16 * n + 4 * q) * 4);
        tokens(0);
        GL_FENCE;
        float s[GL_NT][4], m[MIN ? GL_NT : 1][4];
#pragma unroll
        for (int n = 0; n < GL_NT; ++n) {
            const float d8[4] = {e[n].x, e[n].y, e[n].z, e[n].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[n][i] = __fmul_rn(d, d8[i]);
                if (MIN) m[n][i] = __fmul_rn(ndm, d8[i]);
            }
        }
        load_scales(A, bn);
#pragma unroll
        for (int st = 0; st < 6; ++st) {
            const int k = st >> 1, p = st & 1;
            v4f r[2];
            if (st < 5) tokens(st + 1);
            GL_FENCE;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                if (MIN && k == 2)
                    r[n] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_shufflevector(x[p][n], x[p][n], 0, 1, 2, 3),
                                                                 __builtin_shufflevector(a[2], a[2], 0, 1, 2, 3), zero, 0, 0, 0);
                else
                    r[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[p][n], a[k], zero, 0, 0, 0);
            }
            if (p == 1) load(A, bn, l0, k);
            GL_FENCE;
#pragma unroll
            for (int n = 0; n < 2; ++n) fold4(c[k][2 * p + n], MIN && k == 2 ? m[2 * p + n] : s[2 * p + n], r[n]);
        }
    }
};

// One pass over the blocks: v = ((v + c) + c') + c''.
template <bool MIN>
__device__ __forceinline__ void gl_pass(float (&v)[GL_NT][4], const RowSrc &A, __amdgpu_buffer_rsrc_t rb, int last, int nb, int l0,
                                        int wid, int lane) {
    const int op0 = MIN ? 0 : op_pos(4) + 2 * (l0 - 2);
    GlPass<MIN> p;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < GL_NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) p.c[c][n][i] = 0.0f;
    gl_stage<0>(rb, last, nb, 0, op0, wid, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k) p.load(A, 0, l0, k);
    p.load_scales(A, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int b = 0; b < nb; b += 4) {
        // the next two blocks' tokens go to the other buffer meanwhile
        gl_stage<1>(rb, last, nb, b + 2, op0, wid, lane);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (b + h < nb) p.block(gl_buffer<0>() + h * GL_BLOCK, A, b + h + 1 < nb ? b + h + 1 : nb - 1, l0, lane);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        gl_stage<0>(rb, last, nb, b + 4, op0, wid, lane);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (b + 2 + h < nb) p.block(gl_buffer<1>() + h * GL_BLOCK, A, b + h + 3 < nb ? b + h + 3 : nb - 1, l0, lane);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
#pragma unroll
    for (int n = 0; n < GL_NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (MIN) v[n][i] = __fadd_rn(__fadd_rn(p.c[2][n][i], p.c[0][n][i]), p.c[1][n][i]);
            else v[n][i] = __fadd_rn(__fadd_rn(__fadd_rn(v[n][i], p.c[0][n][i]), p.c[1][n][i]), p.c[2][n][i]);
        }
}

__global__ void __launch_bounds__(64 * GL_WAVES, 4) k_kq_gemm_lds(GemmArgs g) {
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = g.nb;
    const int n_rt = (g.rows + 31) / 32, n_tt = (g.n_tokens + 31) / 32;
    const int row_wgs = (n_rt + 3) / 4, tok_wgs = (n_tt + 1) / 2;
    // XCD-aware order: workgroups are dealt to the eight XCDs round robin; each
    // XCD takes a contiguous run of row groups with all their token groups, so
    // a row group's operands are fetched into one XCD's L2 once.
    const int nwg = row_wgs * tok_wgs;
    const int id = (int)blockIdx.x;
    if (id >= nwg) return;
    const int nfull = nwg & ~7;
    const int lin = id < nfull ? (id % 8) * (nfull / 8) + id / 8 : id;   // a bijection of [0, nwg)
    const int wrt = lin / tok_wgs, tt0 = (lin - wrt * tok_wgs) * 2;
    const int rt = wrt * 4 + (wid >> 1), half = wid & 1;
    const RowSrc A(g.a, rt < n_rt ? rt : n_rt - 1, half, nb, lane);   // rows past the matrix: never stored
    const int last = n_tt - 1 - tt0 < 1 ? n_tt - 1 - tt0 : 1;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(g.b + (long long)tt0 * nb * B_TILE), (short)0, (last + 1) * nb * B_TILE, 0x00020000);
    float v[GL_NT][4];
    gl_pass<true>(v, A, rb, last, nb, 0, wid, lane);
    for (int l0 = 2; l0 < 8; l0 += 3) gl_pass<false>(v, A, rb, last, nb, l0, wid, lane);
    const int row = rt * 32 + 16 * half + (lane & 15);
    if (row >= g.rows) return;
#pragma unroll
    for (int n = 0; n < GL_NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = tt0 * 32 + 16 * n + 4 * (lane >> 4) + i;
            if (t < g.n_tokens) g.y[(long long)t * g.rows + row] = v[n][i];
        }
}

// ---- chains split over three waves, tokens from L1 / L2

constexpr int GS_WAVES = 3;

// Wave W's chains: 0: the minimum and lane chains 0, 1; 1: 2, 3, 4; 2: 5, 6, 7
// (slot k: residue first + k, slot 2 of wave 0 the minimum).
template <int NT, int W>
__device__ __forceinline__ void gs_chains(const RowSrc &A, const GemmArgs &g, int tt0, int lane, float (&acc)[3][NT][4]) {
    constexpr int L0 = W == 0 ? 0 : 3 * W - 1, NL = W == 0 ? 2 : 3;
    const int nb = g.nb, q = lane >> 4;
    const int n16 = (g.n_tokens + 15) / 16;
    const uint8_t *tp[NT];
    int th[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int t = tt0 + n < n16 ? tt0 + n : n16 - 1;   // tiles past the batch: never stored
        tp[n] = g.b + (long long)(t >> 1) * nb * B_TILE;
        th[n] = t & 1;
    }
    struct Step {
        v8h a[NL], b[NL][NT];
        v4h am, bm[NT];
        float d, ndm;
        float4 e[NT];
    };
    auto load = [&](int b, Step &x) {
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            x.a[l] = A.residue(b, L0 + l);
#pragma unroll
            for (int n = 0; n < NT; ++n)
                x.b[l][n] = *reinterpret_cast<const v8h *>(tp[n] + (long long)b * B_TILE + op_pos(2 * (L0 + l)) * OP_BYTES +
                                                           op_lane(lane, th[n]));
        }
        x.d = A.d(b);
#pragma unroll
        for (int n = 0; n < NT; ++n)
            x.e[n] = *reinterpret_cast<const float4 *>(tp[n] + (long long)b * B_TILE + OPS * OP_BYTES + (16 * th[n] + 4 * q) * 4);
        if constexpr (W == 0) {
            x.am = A.minimum(b), x.ndm = A.neg_dmin(b);
#pragma unroll
            for (int n = 0; n < NT; ++n)
                x.bm[n] = *reinterpret_cast<const v4h *>(tp[n] + (long long)b * B_TILE + min_lane(lane, th[n]));
        }
    };
    auto compute = [&](const Step &x) {
        const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const float d8[4] = {x.e[n].x, x.e[n].y, x.e[n].z, x.e[n].w};
            float s[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = __fmul_rn(x.d, d8[i]);
#pragma unroll
            for (int l = 0; l < NL; ++l)
                fold4(acc[l][n], s, __builtin_amdgcn_mfma_f32_16x16x32_f16(x.b[l][n], x.a[l], zero, 0, 0, 0));
            if constexpr (W == 0) {
                float m[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) m[i] = __fmul_rn(x.ndm, d8[i]);
                fold4(acc[2][n], m, __builtin_amdgcn_mfma_f32_16x16x16f16(x.bm[n], x.am, zero, 0, 0, 0));
            }
        }
    };
    Step sa, sb;
    load(0, sa);
    for (int b = 0; b < nb; b += 2) {
        load(b + 1 < nb ? b + 1 : b, sb);
        compute(sa);
        if (b + 1 >= nb) break;
        load(b + 2 < nb ? b + 2 : b + 1, sa);
        compute(sb);
    }
}

template <int NT>
__global__ void __launch_bounds__(64 * GS_WAVES) k_kq_gemm_split(GemmArgs g) {
    __shared__ __align__(16) float s_ch[9][NT][4][64];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = (g.rows + 15) / 16, tg = ((g.n_tokens + 15) / 16 + NT - 1) / NT;
    const int r16 = (int)blockIdx.x / tg, tt0 = ((int)blockIdx.x - r16 * tg) * NT;
    if (r16 >= n16) return;
    const RowSrc A(g.a, r16 >> 1, r16 & 1, g.nb, lane);
    float acc[3][NT][4];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[c][n][i] = 0.0f;
    if (wid == 0) gs_chains<NT, 0>(A, g, tt0, lane, acc);
    else if (wid == 1) gs_chains<NT, 1>(A, g, tt0, lane, acc);
    else gs_chains<NT, 2>(A, g, tt0, lane, acc);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int c = wid == 0 ? (k == 2 ? 8 : k) : 3 * wid - 1 + k;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) s_ch[c][n][i][lane] = acc[k][n][i];
    }
    __syncthreads();
    // result = minimum chain + lane chains 0..7 (q8_k.rs:320-326)
    for (int o = threadIdx.x; o < NT * 256; o += 64 * GS_WAVES) {
        const int n = o >> 8, i = (o >> 6) & 3, l = o & 63;
        float v = s_ch[8][n][i][l];
#pragma unroll
        for (int c = 0; c < 8; ++c) v = __fadd_rn(v, s_ch[c][n][i][l]);
        const int t = 16 * (tt0 + n) + 4 * (l >> 4) + i, row = 16 * r16 + (l & 15);
        if (t < g.n_tokens && row < g.rows) g.y[(long long)t * g.rows + row] = v;
    }
}

// ---------------------------------------------------------------- launchers

static inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

size_t gemm_a_bytes(int rows, int nb) { return (size_t)cdiv(rows, 32) * nb * A_TILE; }
size_t gemm_b_bytes(int n_tokens, int nb) { return (size_t)cdiv(n_tokens, 32) * nb * B_TILE; }

hipError_t launch_prep_a(const MatView &m, uint8_t *a, hipStream_t s) {
    const int grid = cdiv(m.rows, 32) * m.nb;
    if (m.type == T_Q4_K)
        hipLaunchKernelGGL(k_prep_a<T_Q4_K>, dim3(grid), dim3(64), 0, s, m, a);
    else if (m.type == T_Q5_K)
        hipLaunchKernelGGL(k_prep_a<T_Q5_K>, dim3(grid), dim3(64), 0, s, m, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_prep_b(const uint8_t *q8, int n_tokens, int nb, uint8_t *b, hipStream_t s) {
    hipLaunchKernelGGL(k_prep_b, dim3(cdiv(n_tokens, 32) * nb), dim3(64), 0, s, q8, n_tokens, nb, b);
    return hipGetLastError();
}

template <int NT>
static hipError_t gemm_split(const GemmArgs &g, hipStream_t s) {
    const int grid = cdiv(g.rows, 16) * cdiv(cdiv(g.n_tokens, 16), NT);
    hipLaunchKernelGGL((k_kq_gemm_split<NT>), dim3(grid), dim3(64 * GS_WAVES), 0, s, g);
    return hipGetLastError();
}

static hipError_t gemm_2x2(const GemmArgs &g, hipStream_t s) {
    const int lds = (int)sizeof(GemmLDS);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_kq_gemm_2x2), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    const int grid = cdiv(cdiv(g.rows, 32), RG) * cdiv(cdiv(g.n_tokens, 32), TG);
    hipLaunchKernelGGL(k_kq_gemm_2x2, dim3(grid), dim3(64 * NW), lds, s, g);
    return hipGetLastError();
}

// The forms' times on rows of 4096 beyond about 7.6 us that all share, in ns; they
// go with K (256 .. 16384 measured).  Row operands in the 256 MB cache between L2
// and HBM, as in a call repeated on one matrix (1024 .. 16384 rows, 16 .. 512
// tokens):
//   split, NT = 1, 2, 3, 4: 19, 22, 30, 35 per workgroup from 256 on (4096 rows,
//     48 / 64 / 96 / 128 tokens with the best NT: 18.9 / 19.6 / 22.2 / 25.2 us in
//     all); with NT = 4 (190 VGPRs) workgroups come in rounds of 512 (512: 25.2
//     us, 768: 38.8, 1024: 42).
//   2 x 2: 24400 per round of 256 workgroups, one per CU (192: 33 us, 384: 57).
//   LDS: 33000 for the first 256 workgroups, 26000 for each 256 more (256: 41 us,
//     384: 61, 768: 103).
// Beyond that cache the split form, whose waves load their own operands, loses
// most: 24, 35, 43, 52 per workgroup, 2 x 2 28700 per round, LDS 48000 and 28000
// for each 256 more (48 tokens, 12288 rows of 16384, 440 MB: 141 / 122 / 183 us;
// 32 tokens, 16384 rows of 12288: 111 / 96 / 143; 48 tokens, 65536 rows of 4096:
// 178 / 141 / 115).  The line: of matrices read from HBM one after the other, 147
// MB (4096 rows of 16384) still has the cached times' order at every token count
// and 110 MB (12288 of 4096) misses by 8% at 33 to 48 tokens only, 220 MB (12288
// of 8192) by 12% there.
struct FormTimes {
    int split[4], round_2x2, lds0, lds;
};
static constexpr FormTimes KQ_CACHED = {{19, 22, 30, 35}, 24400, 7000, 26000};
static constexpr FormTimes KQ_BEYOND = {{24, 35, 43, 52}, 28700, 20000, 28000};
static constexpr size_t KQ_CACHED_BYTES = 192u << 20;

static long long split_ns(const FormTimes &f, int rows, int n_tokens, int nt) {
    long long w = (long long)cdiv(rows, 16) * cdiv(cdiv(n_tokens, 16), nt);
    if (nt == 4) w = 512LL * cdiv(w, 512);
    return f.split[nt - 1] * (w > 256 ? w : 256);
}

// shape: 0 default, 1 the split form, 2 the 2 x 2 form, 3 the LDS form.
hipError_t launch_kq_gemm(const GemmArgs &g, hipStream_t s) {
    if (g.n_tokens < 1 || g.nb < 1 || g.nb > 64) return hipErrorInvalidValue;
    const int rows = g.rows;
    const FormTimes &f = gemm_a_bytes(rows, g.nb) > KQ_CACHED_BYTES ? KQ_BEYOND : KQ_CACHED;
    int nt = 1;
    for (int n = 2; n <= 4; ++n)
        if (split_ns(f, rows, g.n_tokens, n) < split_ns(f, rows, g.n_tokens, nt)) nt = n;
    const long long lds_wgs = (long long)cdiv(rows, 128) * cdiv(g.n_tokens, 64);
    int shape = g.shape;
    if (shape == 0) {
        const long long t1 = split_ns(f, rows, g.n_tokens, nt);
        const long long t2 = (long long)f.round_2x2 * cdiv((long long)cdiv(rows, 64) * cdiv(g.n_tokens, 64), 256);
        const long long t3 = f.lds0 + (long long)f.lds * cdiv(lds_wgs, 256);
        shape = t1 <= t2 && t1 <= t3 ? 1 : t2 <= t3 ? 2 : 3;
    }
    if (shape == 1) {
        switch (nt) {
        case 1: return gemm_split<1>(g, s);
        case 2: return gemm_split<2>(g, s);
        case 3: return gemm_split<3>(g, s);
        default: return gemm_split<4>(g, s);
        }
    }
    if (shape == 2) return gemm_2x2(g, s);
    hipLaunchKernelGGL(k_kq_gemm_lds, dim3((int)lds_wgs), dim3(64 * GL_WAVES), 0, s, g);
    return hipGetLastError();
}

}  // namespace lbh
