// Prefill attention over the packed RotorQuant cache on 16-bit MFMA (gfx950).
//
// Serves two reference paths with one arithmetic:
//   * fused_paged_rq_int8_prefill
//     (src/rotorquant_vllm/triton/fused_paged_rq_int8_prefill.py:247-363, kernel :43-239),
//     as rq_int8_prefill;
//   * the backend's non-fused path (src/rotorquant_vllm/vllm/rq_backend.py:937-1036), as
//     rq_paged_prefill.
// Attention in the rotated space, q_rot = q R^T rounded to the q dtype, K and V =
// dtype(centroid * norm), output rounded and rotated back by R.
//
// Q K^T runs on the q dtype's MFMA: the products of the two 16-bit operands are exact
// and summed in fp32.  The reference quantizes both to int8 for its first product; on
// gfx950 that takes three int8 passes (a hi/lo split of q and of K: one pass is 0.1 off
// where 2e-2 is allowed), 24 MFMAs and two conversions per score where the 16-bit product
// takes 16 MFMAs of the same length and none, and is exact.  8 x 4096 causal, 32 / 8
// heads: 1503 us with the int8 passes, 1326 us without; error against 64 bits 3.8e-3
// either way (the output's bf16 roundings).
// Differences from the reference, on purpose:
//   * any number of sequences per launch (cu_seqlens_q), and query i of a
//     sequence sits at position seq_len - q_len + i (chunked prefill with a
//     cached prefix is causal-correct; the reference places it at i);
//   * key tiles entirely above the causal diagonal are skipped.
//   P V runs on the fp16 MFMA, as the reference's 16-bit product (:217-227) but
//   with 11-bit operands on both sides: V' = V * 2^-e_tile in fp16, V the
//   reference's centroid * norm rounded to the q dtype (:224), 2^e_tile above the
//   64-key tile's largest v norm, and P' = p * 2^(e_tile - e_run) in fp16, e_run
//   the largest e_tile so far (acc is rescaled when it grows); the row sum is the fp32
//   sum of P', the rounded weights.
//
// Two kernels per call:
//   * prefill_pack_kernel decodes every 64-key tile of every (sequence, kv head)
//     once into a "tile image" in the caller's workspace: K rows in the q dtype,
//     fp16 V'^T rows, the tile's V exponent, laid out exactly as the attention
//     kernel keeps them in LDS;
//   * prefill_attn_kernel: a wave takes 32 query positions of one head, a workgroup
//     four consecutive (position group, query head) units of a (sequence, kv head).
//     It streams the tile images of its sequence and kv head into a double-buffered
//     LDS area with direct global -> LDS copies (the copy of tile t+1 runs while tile
//     t is computed), so the inner loop is MFMA and softmax only (the wide_* steps of
//     rq_attn_tile.h, with the MFMA layouts).
#include <algorithm>
#include <type_traits>

#include "rq_attn_tile.h"

namespace rq {

constexpr int kPD = kAttnD;   // head_dim
constexpr int kKT = kAttnKT;  // keys per tile
constexpr int kPW = kAttnPW;  // query positions per wave
constexpr int kWaves = 4;     // waves of an attention workgroup
constexpr float kLog2eP = kAttnLog2e;

struct PrefillArgs {
    const void *q;
    int64_t q_st, q_sh;
    const int32_t *cu_q;
    const uint8_t *cache;
    int64_t stride_block, stride_token;
    int block_size, bs_shift;
    int64_t num_blocks;
    int H, G;
    int dense3;         // dense 3-bit index layout of the cache
    const int32_t *bt;
    int64_t bt_ss, max_blocks;
    const int32_t *seq_lens;
    const float *kc, *vc;
    int nkc, nvc;
    const float *R;
    int rot_block;
    float score_scale;  // sm_scale * log2(e)
    int causal;         // 0: every query sees all seq_lens[b] keys
    int64_t max_tiles;  // tile images per (sequence, kv head) in the workspace
    uint8_t *ws;        // tile images [num_seqs][H][max_tiles][kImBytes]
    int nx, split;      // query blocks; workgroups per query block (key chunks), > 1: partials in `part`
    float *part;        // [(seq, kv head, query block, chunk)][wave] partials of kPartFloats
    void *out;
    int64_t o_st, o_sh;
};

// Tile image (bytes), the same in the workspace and in LDS: 64 K rows of 128 dims in the q
// dtype (kw_piece: piece c holds dims 8c .. 8c+7), 128 V'^T rows of 64 fp16 keys (vw_piece),
// then the tile's V exponent.
constexpr int kImK = 0;
constexpr int kImVt = kImK + kKT * kPD * 2;
constexpr int kImVe = kImVt + kPD * kKT * 2;                 // int: e_tile, 2^e_tile > the tile's largest v norm
constexpr int kImBytes = (kImVe + 4 + 1023) / 1024 * 1024;
constexpr int kLdsK = kImVt + 16, kLdsV = kImVe - kImVt;       // LDS buffers: K rows and V exponent; V'^T rows

// Keys of a sequence the attention may read: its length, bounded by the block
// table's capacity and by the workspace's tile images.
__device__ __forceinline__ int visible_keys(const PrefillArgs &a, int64_t seq) {
    const int64_t cap = min(a.max_blocks * a.block_size, a.max_tiles * kKT);
    return (int)min((int64_t)a.seq_lens[seq], cap);
}

// ---- pack: one workgroup (256 threads) per (tile, kv head, sequence) --------
template <int DT>
__global__ __launch_bounds__(256) void prefill_pack_kernel(PrefillArgs a) {
    const int tile = blockIdx.x, h = blockIdx.y;
    const int64_t seq = blockIdx.z;
    const int L_eff = visible_keys(a, seq);
    const int k0 = tile * kKT;
    if (k0 >= L_eff) return;
    const int nk = min(kKT, L_eff - k0);
    const int tid = threadIdx.x;
    uint8_t *img = a.ws + (((int64_t)seq * a.H + h) * a.max_tiles + tile) * kImBytes;
    const SlotLayout SL(a.H, kPD, a.dense3 != 0);
    __shared__ uint64_t toff[kKT];

    // K and V are the reference's values, dtype(centroid * norm).
    __shared__ float ktab[16], vtab[16];
    __shared__ float knorm[kKT], vnorm[kKT];
    __shared__ float vscale;  // 2^-e_v
    if (tid < 16) {
        ktab[tid] = tid < a.nkc ? a.kc[tid] : 0.f;
        vtab[tid] = tid < a.nvc ? a.vc[tid] : 0.f;
    }
    if (tid < kKT) {
        // token offset (keys past the tile's end read slot 0 and get zero norms)
        uint64_t off = 0;
        float nkv = 0.f, nvv = 0.f;
        if (tid < nk) {
            const int pos = k0 + tid;
            int lb, o;
            if (a.bs_shift >= 0) {
                lb = pos >> a.bs_shift;
                o = pos & (a.block_size - 1);
            } else {
                lb = pos / a.block_size;
                o = pos - lb * a.block_size;
            }
            int64_t phys = a.bt[seq * a.bt_ss + lb];
            phys = (phys < 0 || phys >= a.num_blocks) ? 0 : phys;
            off = (uint64_t)(phys * a.stride_block + (int64_t)o * a.stride_token);
            nkv = *reinterpret_cast<const float *>(a.cache + off + SL.k_norm + 4 * h);
            nvv = *reinterpret_cast<const float *>(a.cache + off + SL.v_norm + 4 * h);
        }
        toff[tid] = off;
        // tile scale: the power of two above the largest v norm
        float vx = fmaxf(nvv, 0.f);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) vx = fmaxf(vx, __shfl_xor(vx, o));
        // 2^e_v > vx, clamped to [-14, 24]: norms below 2^-14 keep v' at their own scale, and
        // norms above 2^24 would overflow v' in fp16.
        const int e_v = min(24, max(-14, (int)((__float_as_uint(vx) >> 23) & 0xffu) - 126));
        knorm[tid] = nkv;
        vnorm[tid] = nvv;
        if (tid == 0) {
            *reinterpret_cast<int *>(img + kImVe) = e_v;
            vscale = ldexpf(1.f, -e_v);
        }
    }
    __syncthreads();
    // This thread's index dwords -- K: (key, dword) w = tid + 256 r, r < 4; V: dword
    // tid >> 4 of the keys of quad tid & 15 -- all loaded before the first image store:
    // a load issued after a store would wait for it (the compiler cannot rule out that
    // they alias, and the memory counter completes in order), one round per loop step.
    static_assert(kKT * 16 == 4 * 256, "four K index dwords per thread");
    uint32_t xk[4], xv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int w = tid + 256 * r;
        xk[r] = idx_dword(a.cache + toff[w >> 4] + SL.k_idx + h * SL.ib, w & 15, a.dense3 != 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        xv[i] = idx_dword(a.cache + toff[4 * (tid & 15) + i] + SL.v_idx + h * SL.ib, tid >> 4, a.dense3 != 0);
    // K rows in the q dtype: dims 8 dw .. 8 dw + 7 of key tk, one 16-byte piece
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int w = tid + 256 * r;
        const int tk = w >> 4, dw = w & 15;
        const uint32_t x = xk[r];
        const float nrm = knorm[tk];
        uint32_t pr[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // byte j: dim 8 dw + 2j in the high nibble, + 1 in the low one
            const uint32_t e0 = Elem<DT>::from_f32(opaque(ktab[(x >> (8 * j + 4)) & 15u] * nrm));
            const uint32_t e1 = Elem<DT>::from_f32(opaque(ktab[(x >> (8 * j)) & 15u] * nrm));
            pr[j] = e0 | (e1 << 16);
        }
        *reinterpret_cast<u32x4 *>(img + kImK + kw_piece(tk, dw)) =
            u32x4{pr[0], pr[1], pr[2], pr[3]};
    }
    // V'^T rows: v' = dtype(centroid * norm) * 2^-e_v (exact), rounded to fp16 (exact
    // unless below fp16's normal range; |v'| < max|centroid|).  Thread (key quad, dword) writes 4 consecutive
    // keys = 8 bytes per dim.
    {
        const int tq = tid & 15, dw = tid >> 4;  // key quad (4 consecutive keys), dword position
        const uint32_t(&x)[4] = xv;
        const int t0 = 4 * tq;
        const int piece = vw_quad_piece(tq), elem_off = vw_quad_byte(tq);
        float nv[4];
        const float vs = vscale;
#pragma unroll
        for (int i = 0; i < 4; ++i) nv[i] = vnorm[t0 + i];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // byte j of the dword: dims 8 dw + 2j (high nibble), + 1 (low)
#pragma unroll
            for (int par = 0; par < 2; ++par) {
                const int d = 8 * dw + 2 * j + par;
                uint32_t e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t idx = (x[i] >> (8 * j + (par ? 0 : 4))) & 15u;
                    // V rounded to the q dtype first, as the reference (fused_paged_rq_int8_prefill.py:224)
                    const float v = Elem<DT>::to_f32(Elem<DT>::from_f32(opaque(vtab[idx] * nv[i])));
                    e[i] = f32_to_f16_bits(v * vs);
                }
                *reinterpret_cast<uint2 *>(img + kImVt + vw_piece(d, piece) + elem_off) =
                    make_uint2(e[0] | (e[1] << 16), e[2] | (e[3] << 16));
            }
        }
    }
}

// ---- key chunks ---------------------------------------------------------------
// With few query blocks (a short chunk behind a long prefix) `split` workgroups take the tiles
// of one query block, each a contiguous run of them, and prefill_merge_kernel adds up their
// partials: per position the accumulators, and (max in base 2 plus V exponent, row sum).
// What bounds a call without them: one chain of tiles per query block on a few of the CUs.  One
// sequence, 32 / 8 heads, whole call: 64 tokens behind 16000 keys 370 -> 70 us; 200 behind 2000
// 73 -> 38; one 1500-token prompt (which already fills the GPU) 61 -> 47 by the wider waves alone.
constexpr int kPartFloats = kPW * kPD + kPW * 2;
constexpr int kMinChunk = 4;  // tiles of a chunk, at least (a workgroup's fixed work is worth about 6)
__device__ __forceinline__ int chunk_tiles(const PrefillArgs &a, int n_tiles) {
    return max(kMinChunk, (n_tiles + a.split - 1) / a.split);
}
// Query block -> its first unit, unit count of the sequence and key tiles (see prefill_attn_kernel).
struct QueryBlock {
    int q0, T, L, units, f0, kv_end, n_tiles;
};
__device__ __forceinline__ QueryBlock query_block(const PrefillArgs &a, int64_t seq, int qblk) {
    QueryBlock b;
    b.q0 = a.cu_q[seq];
    b.T = a.cu_q[seq + 1] - b.q0;
    b.L = a.seq_lens[seq];
    const int L_eff = visible_keys(a, seq);
    b.units = b.T > 0 ? (b.T + kPW - 1) / kPW * a.G : 0;
    b.f0 = qblk * kWaves;
    const int last_i = min(b.T, (min(b.f0 + kWaves, b.units) - 1) / a.G * kPW + kPW) - 1;
    b.kv_end = a.causal ? min(L_eff, b.L - b.T + last_i + 1) : L_eff;  // keys [0, kv_end) may be visible
    b.n_tiles = b.kv_end > 0 ? (b.kv_end + kKT - 1) / kKT : 0;
    return b;
}

// ---- attention ----------------------------------------------------------------
// What bounds it: vector issue and the matrix cores side by side.  A wave's tile is 32 MFMAs of
// 32 cycles and about 115 vector instructions of 4 with 32 exponentials of 8 to 9; the MFMA unit
// is busy 48 % of the time at 8 x 4096.  Two waves per SIMD (two workgroups of four waves per CU:
// each has its own barriers, so one computes while the other waits): 64 accumulator, 64 score
// and 32 query registers a lane.  Steps on 8 x 4096 causal, 32 / 8 heads, whole call: 16-position
// waves at four per SIMD 1326 us; 32-position waves, one phase after the other 1337;
// interleaved (step, below; measured again in the final form there) 1375; R read from LDS instead of memory 1190; rotations without a
// branch per dim and one rounding 1173.  Without the tile copies it takes 1082, without the tile
// loop about 250 (copies of two tiles, rotations and stores).
template <int DT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attn_kernel(PrefillArgs a) {
    int qblk, h;
    int64_t seq;
    attn_work_item(qblk, h, seq);
    int chunk = 0;
    if (a.split > 1) {
        chunk = qblk % a.split;
        qblk /= a.split;
    }
    const QueryBlock qb = query_block(a, seq, qblk);
    const int q0 = qb.q0, T = qb.T, units = qb.units, f0 = qb.f0, kv_end = qb.kv_end;
    const int pos_base = qb.L - T;  // position of query 0
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int hh = lane >> 5, col = lane & 31;
    // This wave's unit: (32-position group, query head of the GQA group) of the sequence and
    // kv head, in position-group-major order; the workgroup's units span two position
    // groups at most when G >= 4 (whatever G, the four SIMDs carry one wave each).
    if (f0 >= units) return;
    const int f = f0 + wave;
    const int i0 = f < units ? f / a.G * kPW : T;  // first query index (units past the end: inactive)
    const int hq = h * a.G + f % a.G;
    const bool wave_active = i0 < T;
    const int my_i = i0 + col;              // query index of this lane's column
    const int my_pos = pos_base + my_i;
    // This workgroup's tiles [t0, t0 + n_tiles) and, of those, the first nw that this wave takes part
    // in (the causal bound of its positions); t below counts from t0.
    const bool causal = a.causal;
    int t0 = 0, n_tiles = qb.n_tiles;
    if (a.split > 1) {
        const int per = chunk_tiles(a, n_tiles);
        t0 = chunk * per;
        n_tiles = min(per, n_tiles - t0);
        if (n_tiles <= 0) return;  // (the merge does not look at this chunk)
    }
    const int wv_end = causal ? min(kv_end, pos_base + i0 + kPW) : kv_end;
    const int nw = wave_active ? max(0, min(n_tiles, (max(wv_end, 0) + kKT - 1) / kKT - t0)) : 0;

    // LDS: two K buffers (K rows and the tile's V exponent) and two V'^T buffers.
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t *const kbuf[2] = {lds, lds + kLdsK};
    uint8_t *const vbuf[2] = {lds + 2 * kLdsK, lds + 2 * kLdsK + kLdsV};
    float4 *const rot = reinterpret_cast<float4 *>(lds + 2 * (kLdsK + kLdsV));

    // Tile images of this (sequence, kv head), copied global -> LDS 1 KB per wave instruction.
    // The rotation of the query operand overlaps the first copies.
    const uint8_t *img0 = a.ws + (((int64_t)seq * a.H + h) * a.max_tiles + t0) * kImBytes;
    const uint32_t lds0 = lds_addr(lds);
    auto copy_rows = [&](int t, int from, uint32_t dst_) {
        const uint64_t s = reinterpret_cast<uint64_t>(img0 + (int64_t)t * kImBytes + from);
        // wave-uniform operands of the copies (the compiler cannot prove it here)
        const uint32_t slo = __builtin_amdgcn_readfirstlane((uint32_t)s);
        const uint32_t shi = __builtin_amdgcn_readfirstlane((uint32_t)(s >> 32));
        const uint8_t *src = reinterpret_cast<const uint8_t *>(((uint64_t)shi << 32) | slo);
        const uint32_t dst = __builtin_amdgcn_readfirstlane(dst_);
        static_assert(kImVt % (1024 * kWaves) == 0 && kImVe - kImVt == kImVt, "whole copies per wave");
#pragma unroll
        for (int u = 0; u < kImVt / (1024 * kWaves); ++u) {
            const int c = u * kWaves + wave;
            copy16(src + c * 1024, 16 * lane, dst + c * 1024);
        }
        if (from == kImK && wave == 0 && lane == 0) copy16(src + kImVe, 0, dst + kImVt);  // the tile's V exponent
    };
    auto copy_k = [&](int t) { if (t < n_tiles) copy_rows(t, kImK, lds0 + (t & 1) * kLdsK); };
    auto copy_v = [&](int t) { if (t < n_tiles) copy_rows(t, kImVt, lds0 + 2 * kLdsK + (t & 1) * kLdsV); };
    // ---- Q^T operand (columns = this wave's 32 positions): q_rot rounded to the q dtype ----
    // (the query row is loaded before the first copies go out: a wait of the compiler's for a
    // load also waits for every copy issued before it)
    u32x4 qop[8];
    {
        const bool qvalid = wave_active && my_i < T;
        const uint16_t *qrow = reinterpret_cast<const uint16_t *>(a.q) + (int64_t)(q0 + (qvalid ? my_i : 0)) * a.q_st +
                               (int64_t)hq * a.q_sh;
        wide_query_load(qop, qrow, qvalid, hh);
    }
    load_rotation(rot, a.R, tid);
    __syncthreads();
#pragma unroll
    for (int s_ = 0; s_ < 8; ++s_) asm volatile("" : "+v"(qop[s_]));  // (arrived)
    copy_k(0);
    copy_v(0);
    copy_k(1);
    copy_v(1);
    wide_query<DT, false>(qop, rot, a.rot_block, hh);

    WideState st;
    st.init();
    const WideOffsets wo(hh, col);
    const float scale = a.score_scale;
    f32x16 sa[2], sb[2];  // scores of an even and of an odd tile
    float bias = 0.f;     // of the tile whose exponentials come next
    int e_v = 0;          // its V exponent
    // Mask of tile t's scores: at the diagonal and the end.
    auto mask = [&](int t, f32x16 (&s)[2]) {
        const int k0 = (t0 + t) * kKT, nk = min(kKT, kv_end - k0);
        // every key of the tile visible to all 32 positions of this wave: no mask
        if (!(nk == kKT && (!causal || k0 + kKT - 1 <= pos_base + i0)))
            wide_mask(s, (causal ? min(k0 + nk, my_pos + 1) : k0 + nk) - (k0 + 4 * hh));
    };
    auto v_exponent = [&](const uint8_t *kt) {
        return __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int *>(kt + kImVt));
    };

    // The first two tile images landed while the query operand was built.
    wait_copies<0>();
    __syncthreads();
    if (nw > 0) {
        sa[0] = sa[1] = f32x16{};
#pragma unroll
        for (int f = 0; f < 16; ++f) sa[f & 1] = mfma32<DT>(wide_k(kbuf[0], wo, f >> 1, f & 1), qop[f >> 1], sa[f & 1]);
        mask(0, sa);
        e_v = v_exponent(kbuf[0]);
        bias = wide_max(st, wide_lane_max(sa), scale, e_v);
    }
    // Before tile t: its V'^T and tile t+1's K have landed (for every wave), and every wave is
    // done with tile t's K and tile t-1's V'^T, whose buffers are refilled.
    auto turn = [&](int t) {
        wait_copies<0>();
        __syncthreads();
        copy_k(t + 2);
        if (t > 0) copy_v(t + 1);
    };
    // Tile t (t % 2 == par): its exponentials and P V from sc, and tile t+1's scores into sn.
    auto step = [&](auto par, int t, f32x16 (&sc)[2], f32x16 (&sn)[2]) {
        constexpr int P = decltype(par)::value;
        turn(t);
        const uint8_t *kt = kbuf[P ^ 1], *vt = vbuf[P];
        uint32_t pop[16];
        float l = 0.f;
        // Tile t+1's scores run on the matrix cores under tile t's exponentials, and tile t's
        // P V under the search for tile t+1's maximum: an MFMA occupies its unit for 32 cycles
        // and leaves the wave free to issue about 7 vector instructions.  Against the same step one phase
        // after the other (equal bits): 8 x 4096 1190 -> 1180 us, one prompt of 700 28.0 -> 27.4, 3 chunks of 1500
        // behind 5000 and 40 decodes 423 -> 417.  The compiler neither interleaves them by itself nor reads
        // operands far enough ahead of an LDS read's latency, so each slot below is
        // fenced: an operand read, an MFMA, and a sixteenth of the vector work.
        constexpr int kAhead = 5;  // operand reads in flight
        constexpr int kPairsA = 10;
        static_assert(kPairsA + 12 / 2 >= 16, "every weight before its product");
        const WideOffsets o = wo.fresh();
        u32x4 kf[16], vf[16];
        int e_next = *reinterpret_cast<const int *>(kt + kImVt);
#pragma unroll
        for (int f = 0; f < kAhead; ++f) kf[f] = wide_k(kt, o, f >> 1, f & 1);
        sn[0] = sn[1] = f32x16{};
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            if (f + kAhead < 16) kf[f + kAhead] = wide_k(kt, o, (f + kAhead) >> 1, (f + kAhead) & 1);
            else vf[f + kAhead - 16] = wide_v(vt, o, (f + kAhead - 16) >> 2, (f + kAhead - 16) & 3);
            sn[f & 1] = mfma32<DT>(kf[f], qop[f >> 1], sn[f & 1]);
            // pairs 0 .. 9 of the 16; the others run under the P V products that do not need them yet
            if (kPairsA * (f + 1) / 16 > kPairsA * f / 16) {
                wide_exp_pair(sc, kPairsA * f / 16, scale, bias, pop, l);
                // (values used only after the mask's branch would be computed there)
                asm volatile("" : "+v"(l), "+v"(pop[kPairsA * f / 16]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        e_next = __builtin_amdgcn_readfirstlane(e_next);
        mask(t + 1, sn);
        float lm = -INFINITY;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            if (f + kAhead < 16) vf[f + kAhead] = wide_v(vt, o, (f + kAhead) >> 2, (f + kAhead) & 3);
            st.acc[f & 3] = mfma32<RQ_DTYPE_F16>(vf[f], wide_p(pop, f >> 2), st.acc[f & 3]);
            lm = fmaxf(fmaxf(lm, sn[f >> 3][2 * (f & 7)]), sn[f >> 3][2 * (f & 7) + 1]);
            if (f % 2 == 0 && kPairsA + f / 2 < 16) wide_exp_pair(sc, kPairsA + f / 2, scale, bias, pop, l);
            __builtin_amdgcn_sched_barrier(0);
        }
        wide_add_sum(st, l, e_v);
        e_v = e_next;
        bias = wide_max(st, lm, scale, e_v);
    };
    // This wave's last tile.
    auto last = [&](const uint8_t *vt, const f32x16 (&sc)[2]) {
        uint32_t pop[16];
        float l = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) wide_exp_pair(sc, i, scale, bias, pop, l);
        wide_add_sum(st, l, e_v);
#pragma unroll
        for (int f = 0; f < 16; ++f)
            st.acc[f & 3] = mfma32<RQ_DTYPE_F16>(wide_v(vt, wo, f >> 2, f & 3), wide_p(pop, f >> 2), st.acc[f & 3]);
    };
    int t = 0;
    while (t + 1 < nw) {
        step(std::integral_constant<int, 0>{}, t++, sa, sb);
        if (t + 1 >= nw) break;
        step(std::integral_constant<int, 1>{}, t++, sb, sa);
    }
    if (nw > 0) {
        turn(t);
        if (t & 1) last(vbuf[1], sb);
        else last(vbuf[0], sa);
        ++t;
    }
    for (; t < n_tiles; ++t) turn(t);  // tiles above this wave's diagonal: only their copies and barriers
    if (!wave_active) return;

    if (a.split > 1) {
        float *pt = a.part + ((((seq * a.H + h) * a.nx + qblk) * a.split + chunk) * kWaves + wave) * (int64_t)kPartFloats;
        auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(st.l_run), __float_as_uint(st.l_run), false, false);
        const float l = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if (hh == 0)  // m_run = -inf (no key of the chunk seen) stays -inf
            *reinterpret_cast<float2 *>(pt + kPW * kPD + 2 * col) = make_float2(st.m_run * scale + (float)st.e_run, l);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<float4 *>(pt + col * kPD + 32 * m + 8 * j + 4 * hh) =
                    make_float4(st.acc[m][4 * j], st.acc[m][4 * j + 1], st.acc[m][4 * j + 2], st.acc[m][4 * j + 3]);
        return;
    }
    // ---- epilogue: normalise, round to the q dtype, rotate back by R, round ----
    const bool ovalid = my_i < T;
    uint16_t *orow = reinterpret_cast<uint16_t *>(a.out) + (int64_t)(q0 + (ovalid ? my_i : 0)) * a.o_st + (int64_t)hq * a.o_sh;
    wide_store<DT>(st, ovalid, orow, rot, a.rot_block, hh);
}

// One workgroup per unit of a split call: thread (position p = tid / 8, part = tid % 8) adds up 16 dims
// of the chunks' partials, relative to the largest maximum, then the epilogue as above.
template <int DT>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
    const int f = blockIdx.x, h = blockIdx.y;
    const int64_t seq = blockIdx.z;
    const int qblk = f / kWaves;
    const QueryBlock qb = query_block(a, seq, qblk);
    if (f >= qb.units) return;
    __shared__ float4 rot[kPD];
    load_rotation(rot, a.R, threadIdx.x);
    __syncthreads();
    const int p = threadIdx.x >> 3, part = threadIdx.x & 7;
    const int qi = f / a.G * kPW + p;
    if (qi >= qb.T) return;
    const int per = chunk_tiles(a, qb.n_tiles), nch = (qb.n_tiles + per - 1) / per;
    const int64_t stride = (int64_t)kWaves * kPartFloats;  // between chunks
    const float *pt = a.part + ((((seq * a.H + h) * a.nx + qblk) * a.split) * kWaves + f % kWaves) * (int64_t)kPartFloats;
    float M = -INFINITY, l = 0.f, acc[16] = {};
    for (int c = 0; c < nch; ++c) {
        const float *pc = pt + c * stride;
        const float2 ml = *reinterpret_cast<const float2 *>(pc + kPW * kPD + 2 * p);
        float4 x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = *reinterpret_cast<const float4 *>(pc + p * kPD + 16 * part + 4 * k);
        const float Mn = fmaxf(M, ml.x);
        const float keep = M == Mn ? 1.f : __builtin_amdgcn_exp2f(M - Mn);          // M = -inf: 0
        const float w = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - Mn);
        M = Mn;
        l = l * keep + w * ml.y;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float xs[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[4 * k + i] = acc[4 * k + i] * keep + w * xs[i];
        }
    }
    const float inv_l = l > 0.f ? 1.f / l : 0.f;
    uint16_t *orow = reinterpret_cast<uint16_t *>(a.out) + (int64_t)(qb.q0 + qi) * a.o_st + (int64_t)(h * a.G + f % a.G) * a.o_sh;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int d0 = 16 * part + 4 * k;
        const float o[4] = {acc[4 * k], acc[4 * k + 1], acc[4 * k + 2], acc[4 * k + 3]};
        *reinterpret_cast<uint2 *>(orow + d0) =
            a.rot_block == 4 ? rotate_back4<DT, 4>(o, inv_l, d0, rot) : rotate_back4<DT, 2>(o, inv_l, d0, rot);
    }
}

template <int DT>
static void launch_pack(const PrefillArgs &a, int64_t num_seqs, hipStream_t st) {
    dim3 grid((unsigned)a.max_tiles, (unsigned)a.H, (unsigned)num_seqs);
    hipLaunchKernelGGL((prefill_pack_kernel<DT>), grid, dim3(256), 0, st, a);
}

template <int DT>
static void launch_attn(const PrefillArgs &a, int64_t num_seqs, hipStream_t st) {
    const size_t lds = 2 * (size_t)(kLdsK + kLdsV) + kRotBytes;
    dim3 grid((unsigned)(a.nx * a.split), (unsigned)a.H, (unsigned)num_seqs);
    hipLaunchKernelGGL((prefill_attn_kernel<DT>), grid, dim3(64 * kWaves), lds, st, a);
    if (a.split > 1) {
        dim3 mgrid((unsigned)(a.nx * kWaves), (unsigned)a.H, (unsigned)num_seqs);
        hipLaunchKernelGGL((prefill_merge_kernel<DT>), mgrid, dim3(256), 0, st, a);
    }
}

static int64_t prefill_tiles(int64_t max_seq_len) { return (max_seq_len + kKT - 1) / kKT; }

// Query blocks of the longest query, and the key chunks of each: as many as fit the GPU's two
// workgroups per CU, when that is at least two, of kSplitTiles tiles each by the call's bound on the
// lengths (the kernel divides each block's own tiles).
struct PrefillShape {
    int64_t nx, split;
};
constexpr int kSplitTiles = 8;
static PrefillShape prefill_shape(int64_t num_seqs, int G, int H, int64_t max_q_len, int64_t max_seq_len) {
    const int64_t nx = ((max_q_len + kPW - 1) / kPW * G + kWaves - 1) / kWaves;
    const int64_t wgs = nx * H * num_seqs, slots = 2 * (int64_t)device_cus();
    int64_t split = 1;
    if (wgs > 0 && 2 * wgs <= slots) split = std::min<int64_t>(slots / wgs, prefill_tiles(max_seq_len) / kSplitTiles);
    return {nx, std::max<int64_t>(1, split)};
}
static int64_t partial_bytes(const PrefillShape &p, int64_t num_seqs, int H) {
    return p.split > 1 ? p.nx * p.split * H * num_seqs * kWaves * (int64_t)kPartFloats * 4 : 0;
}

}  // namespace rq

using namespace rq;

extern "C" int64_t rq_int8_prefill_workspace_bytes(int64_t num_seqs, int32_t num_kv_heads, int64_t max_seq_len) {
    if (num_seqs <= 0 || num_kv_heads <= 0 || max_seq_len <= 0) return 0;
    return num_seqs * num_kv_heads * prefill_tiles(max_seq_len) * kImBytes;
}

extern "C" int64_t rq_prefill_split_workspace_bytes(int64_t num_seqs, int32_t num_q_heads, int32_t num_kv_heads,
                                                    int64_t max_q_len, int64_t max_seq_len) {
    const int64_t images = rq_int8_prefill_workspace_bytes(num_seqs, num_kv_heads, max_seq_len);
    if (images == 0 || max_q_len <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0) return images;
    return images + partial_bytes(prefill_shape(num_seqs, num_q_heads / num_kv_heads, num_kv_heads, max_q_len, max_seq_len),
                                  num_seqs, num_kv_heads);
}

namespace {

// The two entry points share the kernels.  fused: rq_int8_prefill, which takes the
// reference kernel's codebook sizes only (8 or 16 entries).
int prefill_call(bool fused, int causal, const void *q, int32_t dtype, int64_t total_q, int32_t num_q_heads,
                 int64_t q_stride_tok, int64_t q_stride_head, const int32_t *cu_seqlens_q, int64_t num_seqs,
                 int64_t max_q_len, const uint8_t *kv_cache, int64_t num_blocks, int32_t block_size,
                 int64_t stride_block, int64_t stride_token, int32_t num_kv_heads, int32_t head_dim,
                 int32_t index_layout, const int32_t *block_table, int64_t max_blocks, int64_t bt_stride_seq,
                 const int32_t *seq_lens, int64_t max_seq_len, const float *k_centroids, int32_t n_k_centroids,
                 const float *v_centroids, int32_t n_v_centroids, const float *rotation, int32_t rot_block,
                 float sm_scale, void *out, int64_t out_stride_tok, int64_t out_stride_head, void *workspace,
                 int64_t workspace_bytes, void *stream) {
    RQ_CHECK_ARG(dtype == RQ_DTYPE_BF16 || dtype == RQ_DTYPE_F16, "prefill dtype must be f16 or bf16");
    RQ_CHECK_ARG(head_dim == kPD, "head_dim %d unsupported (only %d)", head_dim, kPD);
    RQ_CHECK_ARG(num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0 && num_q_heads / num_kv_heads <= 16,
                 "num_q_heads %d / num_kv_heads %d must be an integer <= 16", num_q_heads, num_kv_heads);
    if (fused)
        RQ_CHECK_ARG((n_k_centroids == 8 || n_k_centroids == 16) && (n_v_centroids == 8 || n_v_centroids == 16),
                     "centroid counts must be 8 or 16");
    else
        RQ_CHECK_ARG(n_k_centroids >= 1 && n_k_centroids <= 16 && n_v_centroids >= 1 && n_v_centroids <= 16,
                     "centroid counts must be 1..16");
    RQ_CHECK_ARG(rot_block == 2 || rot_block == 4, "rot_block %d must be 2 or 4", rot_block);
    RQ_CHECK_ARG(num_seqs >= 0 && total_q >= 0 && max_q_len >= 0 && block_size >= 1 && max_blocks >= 0 &&
                     max_seq_len >= 0,
                 "bad sizes");
    const int lrc = check_index_layout(index_layout, head_dim, n_k_centroids, n_v_centroids);
    if (lrc) return lrc;
    RQ_CHECK_ARG(stride_token % 4 == 0 && stride_block % 4 == 0 && ((uintptr_t)kv_cache % 4) == 0,
                 "cache slots must be 4-byte aligned");
    RQ_CHECK_ARG(((uintptr_t)q % 16) == 0 && (q_stride_tok * 2) % 16 == 0 && (q_stride_head * 2) % 16 == 0,
                 "q rows must be 16-byte aligned");
    RQ_CHECK_ARG(((uintptr_t)rotation % 16) == 0, "rotation must be 16-byte aligned");
    if (num_seqs == 0 || max_q_len == 0 || num_blocks == 0 || max_seq_len == 0) return RQ_OK;
    const int64_t need = rq_int8_prefill_workspace_bytes(num_seqs, num_kv_heads, max_seq_len);
    RQ_CHECK_SPACE(workspace_bytes >= need, "workspace too small: the call needs %lld bytes (got %lld)",
                   (long long)need, (long long)workspace_bytes);
    RQ_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace % 16) == 0, "workspace must be 16-byte aligned");
    PrefillArgs a{};
    a.q = q;
    a.q_st = q_stride_tok;
    a.q_sh = q_stride_head;
    a.cu_q = cu_seqlens_q;
    a.cache = kv_cache;
    a.stride_block = stride_block;
    a.stride_token = stride_token;
    a.block_size = block_size;
    a.bs_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
    a.num_blocks = num_blocks;
    a.H = num_kv_heads;
    a.G = num_q_heads / num_kv_heads;
    a.dense3 = index_layout == RQ_INDEX_DENSE3;
    a.bt = block_table;
    a.bt_ss = bt_stride_seq;
    a.max_blocks = max_blocks;
    a.seq_lens = seq_lens;
    a.kc = k_centroids;
    a.vc = v_centroids;
    a.nkc = n_k_centroids;
    a.nvc = n_v_centroids;
    a.R = rotation;
    a.rot_block = rot_block;
    a.score_scale = sm_scale * kLog2eP;
    a.causal = causal != 0;
    a.max_tiles = prefill_tiles(max_seq_len);
    a.ws = static_cast<uint8_t *>(workspace);
    // key chunks when the workspace also holds their partials (after the tile images)
    PrefillShape shape = prefill_shape(num_seqs, a.G, a.H, max_q_len, max_seq_len);
    if (workspace_bytes < need + partial_bytes(shape, num_seqs, a.H)) shape.split = 1;
    a.nx = (int)shape.nx;
    a.split = (int)shape.split;
    a.part = reinterpret_cast<float *>(a.ws + need);
    a.out = out;
    a.o_st = out_stride_tok;
    a.o_sh = out_stride_head;
    hipStream_t st = (hipStream_t)stream;
    const bool bf = dtype == RQ_DTYPE_BF16;
    if (bf) launch_pack<RQ_DTYPE_BF16>(a, num_seqs, st);
    else launch_pack<RQ_DTYPE_F16>(a, num_seqs, st);
    int rc = check_launch("prefill_pack_kernel");
    if (rc) return rc;
    if (bf) launch_attn<RQ_DTYPE_BF16>(a, num_seqs, st);
    else launch_attn<RQ_DTYPE_F16>(a, num_seqs, st);
    return check_launch("prefill_attn_kernel");
}

}  // namespace

extern "C" int rq_int8_prefill(const void *q, int32_t dtype, int64_t total_q, int32_t num_q_heads,
                               int64_t q_stride_tok, int64_t q_stride_head, const int32_t *cu_seqlens_q,
                               int64_t num_seqs, int64_t max_q_len, const uint8_t *kv_cache, int64_t num_blocks,
                               int32_t block_size, int64_t stride_block, int64_t stride_token, int32_t num_kv_heads,
                               int32_t head_dim, int32_t index_layout, const int32_t *block_table,
                               int64_t max_blocks, int64_t bt_stride_seq, const int32_t *seq_lens,
                               int64_t max_seq_len,
                               const float *k_centroids, int32_t n_k_centroids, const float *v_centroids,
                               int32_t n_v_centroids, const float *rotation, int32_t rot_block, float sm_scale,
                               void *out, int64_t out_stride_tok, int64_t out_stride_head, void *workspace,
                               int64_t workspace_bytes, void *stream) {
    return prefill_call(true, 1, q, dtype, total_q, num_q_heads, q_stride_tok, q_stride_head, cu_seqlens_q,
                        num_seqs, max_q_len, kv_cache, num_blocks, block_size, stride_block, stride_token,
                        num_kv_heads, head_dim, index_layout, block_table, max_blocks, bt_stride_seq, seq_lens,
                        max_seq_len, k_centroids, n_k_centroids, v_centroids, n_v_centroids, rotation, rot_block,
                        sm_scale, out, out_stride_tok, out_stride_head, workspace, workspace_bytes, stream);
}

extern "C" int64_t rq_paged_prefill_workspace_bytes(int64_t num_seqs, int32_t num_kv_heads, int64_t max_seq_len) {
    return rq_int8_prefill_workspace_bytes(num_seqs, num_kv_heads, max_seq_len);
}

extern "C" int rq_paged_prefill(const void *q, int32_t dtype, int64_t total_q, int32_t num_q_heads,
                                int64_t q_stride_tok, int64_t q_stride_head, const int32_t *cu_seqlens_q,
                                int64_t num_seqs, int64_t max_q_len, int32_t causal, const uint8_t *kv_cache,
                                int64_t num_blocks, int32_t block_size, int64_t stride_block, int64_t stride_token,
                                int32_t num_kv_heads, int32_t head_dim, int32_t index_layout,
                                const int32_t *block_table, int64_t max_blocks, int64_t bt_stride_seq,
                                const int32_t *seq_lens, int64_t max_seq_len, const float *k_centroids,
                                int32_t n_k_centroids, const float *v_centroids, int32_t n_v_centroids,
                                const float *rotation, int32_t rot_block, float sm_scale, void *out,
                                int64_t out_stride_tok, int64_t out_stride_head, void *workspace,
                                int64_t workspace_bytes, void *stream) {
    return prefill_call(false, causal, q, dtype, total_q, num_q_heads, q_stride_tok, q_stride_head, cu_seqlens_q,
                        num_seqs, max_q_len, kv_cache, num_blocks, block_size, stride_block, stride_token,
                        num_kv_heads, head_dim, index_layout, block_table, max_blocks, bt_stride_seq, seq_lens,
                        max_seq_len, k_centroids, n_k_centroids, v_centroids, n_v_centroids, rotation, rot_block,
                        sm_scale, out, out_stride_tok, out_stride_head, workspace, workspace_bytes, stream);
}
