// Pieces shared by the attention kernels that keep a 64-key tile's V in LDS as
// fp16 V'^T rows (rq_prefill.hip, rq_attention.hip): the MFMA wrappers, the
// query rotation, the online-softmax + P V step of one tile and the epilogue.
//
// Layouts (wave64, lane l, g = l / 16, col = l % 16):
//   scores S^T (16 keys x 16 query positions per key block b): lane (g, col)
//     holds position col's scores of keys 16b + 4g + i, i = 0..3, b = 0..3;
//   O^T = V'^T P'^T on v_mfma_f32_16x16x32_f16 (A 16 x 32: lane holds row l % 16,
//     k = 8g .. 8g+7), two k-steps per tile: k-step s, element j of lane group g
//     is key 32s + 4g + j (j < 4) or 32s + 16 + 4g + j - 4 (j >= 4) -- exactly the
//     scores the lane holds, so P needs no transpose; acc[m] holds position col's
//     output dims 16m + 4g + i.
#pragma once

#include "rq_common.h"

namespace rq {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

constexpr int kAttnD = 128;  // head_dim
constexpr int kAttnKT = 64;  // keys per tile
constexpr int kAttnPQ = 16;  // query positions per wave
constexpr float kAttnLog2e = 1.4426950408889634f;

// fp16 MFMA of the P V product (fp32 accumulation).
__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

// 16-bit MFMA in the q dtype (bf16 or fp16 operands, fp32 accumulation): Q K^T
// over K rounded to the q dtype.
template <int DT>
__device__ __forceinline__ f32x4 mfma_qk(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == RQ_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return mfma_f16(a, b, c);
}

// Two fp32 values rounded to the 16-bit dtype, packed low | high << 16 (one v_cvt_pk_{bf16,f16}_f32).
template <int DT>
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    if constexpr (DT == RQ_DTYPE_BF16) {
        typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
    } else {
        typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, f16x2));
    }
}

// Two fp32 values rounded to fp16, packed low | high << 16 (one v_cvt_pk_f16_f32).
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    const f16x2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// V'^T tile: 128 dim rows of 64 fp16 keys (128 bytes), 16-byte piece c of row d
// at d * 128 + 16 * (c ^ (d & 7)) (XOR swizzle: the 16 rows an MFMA operand read
// touches fall in distinct bank groups).  Key t = 16b + 4gg + i sits in piece
// 4 (b >> 1) + gg, element 4 (b & 1) + i.
__host__ __device__ constexpr int vt_piece(int d, int c) { return d * 128 + 16 * (c ^ (d & 7)); }

// R's diagonal 4 x 4 blocks in LDS: row d holds R[d][d & ~3 .. +3] (2-wide blocks: two of them,
// with zeros off the block).  A wave reads R once per query and once per output dim; from
// memory those are 128 dependent-latency loads of a few distinct rows per lane.
constexpr int kRotBytes = kAttnD * 16;
__device__ __forceinline__ void load_rotation(float4 *rot, const float *R, int tid) {
    if (tid < kAttnD) rot[tid] = *reinterpret_cast<const float4 *>(R + tid * kAttnD + (tid & ~3));
}

// 8 consecutive head dims base .. base+7 (base a multiple of 8; raw: those dims of q) of
// q_rot = q R^T, rounded to the q dtype: R is block diagonal with RB-wide blocks (2 or 4), so
// the 8 dims need only these 8 inputs.  Each output is the fma chain over its
// block in increasing k, starting from the first product
// (fused_paged_rq_decode.py:271 computes q.f32 @ R^T, then casts).  rot: load_rotation's rows.
// PERM: packed in the order e0 e2 e4 e6 e1 e3 e5 e7 (K rows looked up by byte permutes).
template <int DT, int RB, bool PERM>
__device__ __forceinline__ u32x4 rotate_q8(u32x4 raw, int base, const float4 *rot) {
    float xin[8], qr[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) xin[k] = Elem<DT>::to_f32((raw[k >> 1] >> (16 * (k & 1))) & 0xffffu);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float4 r = rot[base + k];
        const float rc[4] = {r.x, r.y, r.z, r.w};
        const int b0 = k & ~(RB - 1);  // first dim of k's block
        float acc = __builtin_fmaf(xin[b0], rc[b0 & 3], 0.f);
#pragma unroll
        for (int i = 1; i < RB; ++i) acc = __builtin_fmaf(xin[b0 + i], rc[(b0 + i) & 3], acc);
        qr[k] = acc;
    }
    if constexpr (PERM)
        return u32x4{pack_pair<DT>(qr[0], qr[2]), pack_pair<DT>(qr[4], qr[6]), pack_pair<DT>(qr[1], qr[3]),
                     pack_pair<DT>(qr[5], qr[7])};
    else
        return u32x4{pack_pair<DT>(qr[0], qr[1]), pack_pair<DT>(qr[2], qr[3]), pack_pair<DT>(qr[4], qr[5]),
                     pack_pair<DT>(qr[6], qr[7])};
}

// Work item of a workgroup in a grid (query blocks, kv heads, sequences).
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// Each (sequence, kv head) pair's query blocks are cut into S slices (S = 8 / kv
// heads when that divides both 8 and the query blocks, else 1), and the
// (pair, slice) units are dealt to the XCDs in order: XCD j takes units j, j + 8,
// ... one after another.  So the query blocks that stream one pair's keys share
// S L2s, and each sequence's work is spread over all 8 XCDs: with whole pairs
// (S = 1) and 4 kv heads, the XCDs 0-3 would hold the even and 4-7 the odd
// sequences, whatever their lengths.  Slice c of a pair holds its query blocks
// c, c + S, ... (causal blocks grow heavier with the position), and within a slice
// the last (heaviest) query blocks go first.  When the units do not divide into 8,
// the plain order.  Both are bijections of the grid onto (query block, kv head,
// sequence).
__device__ __forceinline__ void attn_work_item(int &qblk, int &h, int64_t &seq) {
    const uint32_t nx = gridDim.x, ny = gridDim.y;
    const uint32_t lin = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    uint32_t pair = blockIdx.y + ny * blockIdx.z, xo = blockIdx.x;
    // S: 2, 4 or 8 (a power of two) for 4, 2 or 1 kv heads; 1 otherwise
    const uint32_t S = (ny == 1u || ny == 2u || ny == 4u) && nx % (8u / ny) == 0 ? 8u / ny : 1u;
    const uint32_t k = lin >> 3;  // rank of this workgroup on its XCD
    if (S == 1u) {
        if ((ny * gridDim.z) % 8u == 0) {
            pair = (lin & 7u) + 8u * (k / nx);
            xo = k % nx;
        }
    } else {  // 8 units per sequence: always a multiple of 8
        const uint32_t sh = __builtin_ctz(S);
        const uint32_t len = nx >> sh;                   // query blocks per slice
        const uint32_t u = (lin & 7u) + 8u * (k / len);  // (pair, slice) unit
        pair = u >> sh;
        xo = ((k % len) << sh) + (u & (S - 1u));  // slice c: query blocks c, c + S, ... (heavy and light mixed)
    }
    qblk = (int)(nx - 1 - xo);
    h = (int)(pair % ny);
    seq = pair / ny;
}

// Running state of one wave's 16 query positions (one per lane column).
// acc = sum P' V' and lsum = sum P' 2^-e_v carry the same factor 2^-e_run, so
// out = acc / l; m_run is in the score's base-2 units.
struct AttnState {
    f32x4 acc[8];
    f32x4 lsum;  // row 0 (lanes g = 0, element 0): the row sum of the weights
    float m_run;
    int e_run;
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int m = 0; m < 8; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
        lsum = f32x4{0.f, 0.f, 0.f, 0.f};
        m_run = -INFINITY;
        e_run = -14;
    }
};

// Row-sum operand of a tile: lanes of MFMA row 0 (col == 0) hold 2^-e_v in fp16
// (normal or denormal), the others zero.
__device__ __forceinline__ u32x4 rowsum_operand(int e_v, int col) {
    const uint32_t w = col == 0 ? pack_f16(ldexpf(1.f, -e_v), ldexpf(1.f, -e_v)) : 0u;
    return u32x4{w, w, w, w};
}

// Online softmax over one tile and O^T += V'^T P'^T.
//   s: this lane's 16 scores (masked ones -INFINITY), in base 2 once multiplied by scale;
//   e_v: the tile's V exponent, V' = V 2^-e_v in fp16 (|V'| below max|centroid|);
//   vt: the tile's V'^T rows; koff0 / koff1: this lane's pieces g and 4 + g of row
//       col (vt_piece(col, g), vt_piece(col, 4 + g));
//   ones: the tile's row-sum operand (rowsum_operand(e_v, col), col = lane % 16).
__device__ __forceinline__ void softmax_pv(AttnState &st, const float (&s)[16], float scale, int e_v,
                                           const uint8_t *vt, int koff0, int koff1, const u32x4 ones) {
    float tmax = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
    tmax = rows_max(tmax) * scale;
    // Lazy running max: rescale only when a position's max exceeds m_run by more
    // than 8 in log2 units, so p <= 2^8 in between (P' = p 2^(e_v - e_run) <= 2^8
    // stays in fp16); acc and lsum are relative to the same m_run either way.
    if (__any(tmax - st.m_run > 8.f)) {
        const float m_new = fmaxf(st.m_run, tmax);
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(st.m_run - m_new);
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) st.acc[m][i] *= alpha;
        st.lsum *= alpha;
        st.m_run = m_new;
    }
    // V exponent of the tile: acc carries 2^-e_run, and P' = p 2^(e_v - e_run) <= 2^8
    // in fp16 (the exponent's fma adds e_v - e_run).  The row sum is one more MFMA
    // row: sum P' 2^-e_v = 2^-e_run sum p, with the same rounded weights as the
    // numerator (the reference sums p in fp32 and rounds it for P V,
    // fused_paged_rq_int8_prefill.py:214-229).
    if (e_v > st.e_run) {  // uniform: one tile per workgroup
        const float f = ldexpf(1.f, st.e_run - e_v);
#pragma unroll
        for (int m = 0; m < 8; ++m) st.acc[m] *= f;
        st.lsum *= f;
        st.e_run = e_v;
    }
    const float bias = (st.m_run == -INFINITY ? 0.f : -st.m_run) + (float)(e_v - st.e_run);
    // k-step t takes the scores of key blocks 2t and 2t + 1, in the lane's order.
    u32x4 pop[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * t + e], scale, bias));
        pop[t] = u32x4{pack_f16(p[0], p[1]), pack_f16(p[2], p[3]), pack_f16(p[4], p[5]), pack_f16(p[6], p[7])};
    }
    st.lsum = mfma_f16(ones, pop[0], st.lsum);
    st.lsum = mfma_f16(ones, pop[1], st.lsum);
    // 8 blocks of 16 head dims (dim 16m + col; its swizzle term is col & 7), two k-steps
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const u32x4 v0 = *reinterpret_cast<const u32x4 *>(vt + 16 * m * 128 + koff0);
        const u32x4 v1 = *reinterpret_cast<const u32x4 *>(vt + 16 * m * 128 + koff1);
        st.acc[m] = mfma_f16(v0, pop[0], st.acc[m]);
        st.acc[m] = mfma_f16(v1, pop[1], st.acc[m]);
    }
}

// 1 / (row sum of the weights) of this lane's position (0 when nothing was seen).
__device__ __forceinline__ float attn_inv_l(const AttnState &st) {
    const float l_run = rows_sum(st.lsum[0]);  // rows 4g: only g = 0 holds row 0
    return l_run > 0.f ? 1.f / l_run : 0.f;
}

// Four dims d0 .. d0+3 (a 4-dim block of R or two 2-dim ones) of out_rot, rounded to the q
// dtype, rotated back by R and rounded again: out[d] = fma chain over the block in increasing k
// of round(o[k]) * R[k][d] (fused_paged_rq_decode.py:308 order).
template <int DT, int RB>
__device__ __forceinline__ uint2 rotate_back4(const float (&acc)[4], float inv_l, int d0, const float4 *rot) {
    const uint32_t p01 = pack_pair<DT>(acc[0] * inv_l, acc[1] * inv_l), p23 = pack_pair<DT>(acc[2] * inv_l, acc[3] * inv_l);
    const float o[4] = {Elem<DT>::to_f32(p01 & 0xffffu), Elem<DT>::to_f32(p01 >> 16), Elem<DT>::to_f32(p23 & 0xffffu),
                        Elem<DT>::to_f32(p23 >> 16)};
    float rc[4][4], w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 r = rot[d0 + i];
        rc[i][0] = r.x, rc[i][1] = r.y, rc[i][2] = r.z, rc[i][3] = r.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k0 = j & ~(RB - 1);  // first row of d0 + j's block
        w[j] = o[k0] * rc[k0][j];
#pragma unroll
        for (int i = 1; i < RB; ++i) w[j] = __builtin_fmaf(o[k0 + i], rc[k0 + i][j], w[j]);
    }
    return make_uint2(pack_pair<DT>(w[0], w[1]), pack_pair<DT>(w[2], w[3]));
}

// Epilogue of one position (lane column): out_rot = acc / l rounded to the q
// dtype, rotated back by R and rounded again.  Lane (g, col) holds dims
// 16m + 4g + i (i = 0..3): a whole 4-dim block of R (or two 2-dim ones, whose
// off-block entries are exact zeros), so the back-rotation runs in registers.  g = lane / 16.
template <int DT, int RB>
__device__ __forceinline__ void store_rotated(const AttnState &st, float inv_l, uint16_t *orow, const float4 *rot, int g) {
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const int d0 = 16 * m + 4 * g;
        const float a[4] = {st.acc[m][0], st.acc[m][1], st.acc[m][2], st.acc[m][3]};
        *reinterpret_cast<uint2 *>(orow + d0) = rotate_back4<DT, RB>(a, inv_l, d0, rot);
    }
}

// ---------------------------------------------------------------------------
// The 32-position tile step (queries longer than 16 tokens): one wave takes 32
// query positions of one head on v_mfma_f32_32x32x16_{bf16,f16} (wave64, lane l,
// hh = l / 32, col = l % 32):
//   A (32 x 16): lane holds row col, k = 8hh .. 8hh+7;  B (16 x 32): column col, same k;
//   C (32 x 32): lane holds column col, rows 8j + 4hh + i (j, i < 4) in element 4j + i.
// A tile operand read from LDS (1 KB a wave) feeds 32 positions instead of 16, a key
// block's maximum needs one cross-lane step instead of two, and lane-invariant work
// (addresses, tile scales, branches) is spent once for twice the scores.
//   S^T = K Q^T per 32-key block b: lane (hh, col) holds position col's scores of keys
//     32b + 8j + 4hh + i;
//   O^T += V'^T P'^T: k-step s (16 keys) takes elements 8 (s & 1) .. +7 of block s >> 1, so
//     lane half hh's k slot 4j + i is key 16s + 8j + 4hh + i (j < 2): P needs no transpose.
// K rows are 256 bytes, V'^T rows 128 (64 fp16 keys; piece 2s + hh holds k-step s's keys of
// lane half hh).  The XOR swizzles below give the 16 lanes that share an LDS pass of a
// ds_read_b128 (lanes 0-3, 12-15, 20-27 and their like) 16 distinct 16-byte slots.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kAttnPW = 32;  // query positions per wave
__host__ __device__ constexpr int kw_piece(int r, int c) { return r * 256 + 16 * (c ^ (r & 15)); }
__host__ __device__ constexpr int vw_piece(int d, int c) { return d * 128 + 16 * (c ^ ((d >> 1) & 7)); }
// V'^T place of key quad tq (keys 4 tq .. 4 tq + 3) of a dim row: its piece and the byte in it.
__host__ __device__ constexpr int vw_quad_piece(int tq) { return 2 * (tq >> 2) + (tq & 1); }
__host__ __device__ constexpr int vw_quad_byte(int tq) { return 8 * ((tq >> 1) & 1); }

template <int DT>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (DT == RQ_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
}

// Running state of one wave's 32 positions (one per lane column; both lane halves of a
// column agree on m_run).  acc[m][4j + i] = out_rot dim 32m + 8j + 4hh + i, times 2^-e_run;
// l_run = this lane's share of the row sum, times 2^-e_run.
struct WideState {
    f32x16 acc[4];
    float l_run, m_run;
    int e_run;
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[m] = f32x16{};
        l_run = 0.f;
        m_run = -INFINITY;
        e_run = -14;
    }
};

// The steps of one 64-key tile, in this order: scores, mask, wide_max (raises the running max
// and V exponent for the tile), wide_exp_pair x 16, wide_add_sum and the P V products.

// Operand reads from a tile's K rows kt (k-step ks, 32-key block b) and V'^T rows vt (k-step t,
// 32-dim block m).  Piece 2ks + hh of K row col sits at slot (2ks) ^ hh ^ (col & 15), so its
// address is the lane's offset ^ 32 ks, and likewise for V'^T.
struct WideOffsets {
    int k, v;
    __device__ __forceinline__ WideOffsets(int hh, int col) : k(kw_piece(col, hh)), v(vw_piece(col, hh)) {}
    // The offsets again, as values the compiler cannot hoist from: inside a loop, the 12 addresses
    // made from them are then computed at each use (one VALU) instead of held in registers.
    __device__ __forceinline__ WideOffsets fresh() const {
        WideOffsets o = *this;
        asm volatile("" : "+v"(o.k), "+v"(o.v));
        return o;
    }
};
__device__ __forceinline__ u32x4 wide_k(const uint8_t *kt, const WideOffsets &o, int ks, int b) {
    return *reinterpret_cast<const u32x4 *>(kt + (o.k ^ (32 * ks)) + b * (32 * 256));
}
__device__ __forceinline__ u32x4 wide_v(const uint8_t *vt, const WideOffsets &o, int t, int m) {
    return *reinterpret_cast<const u32x4 *>(vt + (o.v ^ (32 * t)) + m * (32 * 128));
}

// Scores of keys at or past lim become -inf (lim: the position's key limit in the tile, less
// 4hh; the lane's keys are 32b + 8j + i).
__device__ __forceinline__ void wide_mask(f32x16 (&s)[2], int lim) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[b][e] = (32 * b + 8 * (e >> 2) + (e & 3)) < lim ? s[b][e] : -INFINITY;
}

// This lane's maximum of a tile's scores.
__device__ __forceinline__ float wide_lane_max(const f32x16 (&s)[2]) {
    float m = s[0][0];
#pragma unroll
    for (int e = 1; e < 32; ++e) m = fmaxf(m, s[e >> 4][e & 15]);
    return m;
}

// Running max, V exponent and P' = p 2^(e_v - e_run) <= 2^8 as in softmax_pv; returns the
// exponent's bias.  lane_max: wide_lane_max of the (masked) scores.
__device__ __forceinline__ float wide_max(WideState &st, float lane_max, float scale, int e_v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lane_max), __float_as_uint(lane_max), false, false);
    const float tmax = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    if (__any((tmax - st.m_run) * scale > 8.f)) {
        const float m_new = fmaxf(st.m_run, tmax);
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((st.m_run - m_new) * scale);
#pragma unroll
        for (int m = 0; m < 4; ++m) st.acc[m] *= alpha;
        st.l_run *= alpha;
        st.m_run = m_new;
    }
    if (e_v > st.e_run) {  // uniform: one tile per workgroup
        const float f = ldexpf(1.f, st.e_run - e_v);
#pragma unroll
        for (int m = 0; m < 4; ++m) st.acc[m] *= f;
        st.l_run *= f;
        st.e_run = e_v;
    }
    return (st.m_run == -INFINITY ? 0.f : -st.m_run * scale) + (float)(e_v - st.e_run);
}

// One pair of P', pair i (0..15): its place in the P V operand (k-step t = i / 4: elements 8 (t & 1)
// .. +7 of block t / 2), and the row sum of the rounded weights in fp32 (v_dot2_f32_f16: exact
// products, denormals kept).
__device__ __forceinline__ void wide_exp_pair(const f32x16 (&s)[2], int i, float scale, float bias, uint32_t (&pop)[16],
                                              float &l) {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    const f16x2 one = {(_Float16)1.f, (_Float16)1.f};
    const int t = i >> 2, e = 8 * (t & 1) + 2 * (i & 3);
    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t >> 1][e], scale, bias));
    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t >> 1][e + 1], scale, bias));
    const uint32_t p = pack_f16(p0, p1);
    pop[i] = p;
    l = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p), one, l, false);
}
__device__ __forceinline__ u32x4 wide_p(const uint32_t (&pop)[16], int t) {
    return u32x4{pop[4 * t], pop[4 * t + 1], pop[4 * t + 2], pop[4 * t + 3]};
}
// The tile's weights join the row sum.
__device__ __forceinline__ void wide_add_sum(WideState &st, float l, int e_v) {
    st.l_run = __builtin_fmaf(l, ldexpf(1.f, -e_v), st.l_run);
}

// Query operand of one wave: position `pos` (lane column) of head hq, k-step s = dims 16s + 8hh
// .. +7 of q_rot.  wide_query_load reads the row (zeros unless valid), wide_query rotates it in
// place.
__device__ __forceinline__ void wide_query_load(u32x4 (&qop)[8], const uint16_t *qrow, bool valid, int hh) {
#pragma unroll
    for (int s_ = 0; s_ < 8; ++s_)
        qop[s_] = valid ? *reinterpret_cast<const u32x4 *>(qrow + 16 * s_ + 8 * hh) : u32x4{0u, 0u, 0u, 0u};
}
template <int DT, bool PERM>
__device__ __forceinline__ void wide_query(u32x4 (&qop)[8], const float4 *rot, int rot_block, int hh) {
    if (rot_block == 4) {
#pragma unroll
        for (int s = 0; s < 8; ++s) qop[s] = rotate_q8<DT, 4, PERM>(qop[s], 16 * s + 8 * hh, rot);
    } else {
#pragma unroll
        for (int s = 0; s < 8; ++s) qop[s] = rotate_q8<DT, 2, PERM>(qop[s], 16 * s + 8 * hh, rot);
    }
}

// Epilogue of a wave's 32 positions: orow = the output row of this lane's position (written
// when `valid`).  Both lane halves of a column take part in the sum.
template <int DT, int RB>
__device__ __forceinline__ void wide_store_rb(const WideState &st, float inv_l, uint16_t *orow, const float4 *rot, int hh) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d0 = 32 * m + 8 * j + 4 * hh;
            const float a[4] = {st.acc[m][4 * j], st.acc[m][4 * j + 1], st.acc[m][4 * j + 2], st.acc[m][4 * j + 3]};
            *reinterpret_cast<uint2 *>(orow + d0) = rotate_back4<DT, RB>(a, inv_l, d0, rot);
        }
    }
}
template <int DT>
__device__ __forceinline__ void wide_store(const WideState &st, bool valid, uint16_t *orow, const float4 *rot,
                                           int rot_block, int hh) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(st.l_run), __float_as_uint(st.l_run), false, false);
    const float l = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const float inv_l = l > 0.f ? 1.f / l : 0.f;  // a position that sees no key: zeros
    if (!valid) return;
    if (rot_block == 4) wide_store_rb<DT, 4>(st, inv_l, orow, rot, hh);
    else wide_store_rb<DT, 2>(st, inv_l, orow, rot, hh);
}

}  // namespace rq
