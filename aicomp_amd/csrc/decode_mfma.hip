// Paged decode attention on gfx950 matrix cores: the hot kernel of the path.
//
// Replaces  F.scaled_dot_product_attention(query, full_key, full_value,
//           attn_mask=None, is_causal=False)      opt_prime/opt_prime/kv_cache.py:397-403
// and the two .contiguous() prefix copies that feed it (kv_cache.py:391-392):
// K and V are read once, in place, through the block table.
//
// Shape covered: head_dim 128, block_size 16, bf16 or fp16 queries, pools of the query type or
// fp8-e4m3 (the kernels are written over a 16-bit element format, see common.h), up to 16 query
// heads per KV head; and head_dim 64 (up to 8 heads per KV head) by treating two consecutive
// tokens, which are contiguous in the pool, as one 128-element row: every head takes two B-operand columns, one per token
// parity, with the query in the matching half of the row and zeros in the other,
// and the two columns' partial softmaxes are merged at the end.  Same instruction
// stream per byte as head_dim 128.  Float32 queries over float32 pools, head_dim 128 and
// 64, up to 16 heads per KV head, run the same two schedules on the float32 matrix
// instruction (decode_tile_f32_quad.h up to four heads per KV head, decode_tile_f32.h beyond).  Everything else goes to the vector-ALU kernel.
//
// HBM-bound: per sequence 2 * L * Hkv * D * e_kv bytes of K/V are streamed and
// used exactly once; 4 * G flop per byte (bf16), far below the MFMA roof, so
// the design goal is bytes in flight, not flops.
//
// Work split   one workgroup per (partition, KV head, sequence), of 4 waves, or of 8 where a CU has
//              one workgroup at most and a partition more than 16 tiles.  A wave owns whole 32-token tiles (two 16-token blocks) and its
//              own online-softmax state; no workgroup barrier in the loop.
// Loads        a (block, KV head) tile is 16 rows * 256 B contiguous (bf16):
//              each global_load_dwordx4 of a wave reads 1 KB = 4 whole rows,
//              lane l -> row l/16, 16-byte chunk l%16.  One table lookup per
//              block, wave-uniform (scalar).
// K            staged through a wave-private LDS tile (unpadded 256-byte rows whose
//              16-byte chunks are permuted by a function of the row, so that the
//              operand reads run at the full LDS rate) and read back
//              as the A operand of  S^T = K Q^T  (v_mfma_f32_16x16x32_bf16 / _f16),
//              the G query heads (padded to 16 columns) sharing every K tile.
// V            never touches LDS.  Lane (c = l%16, q = l/16) of load i holds
//              dims 8c..8c+7 of token 4i+q; picking the j-th 16-bit half of
//              loads 0..7 (v_perm_b32) is exactly the A operand of
//              O^T[dim 8c+j][head] += V^T P^T  for the token order the QK
//              product was laid out in (rows of the K tile are permuted on the
//              LDS read to match), so P goes from accumulator to operand
//              without leaving its lane.
// Softmax      log2 domain, running max per head made wave-uniform with two
//              lane swaps (lanes l, l^16, l^32, l^48 hold the same head).
// Split-K      partitions write (max, sum, unnormalised output) to the
//              workspace; a second, small kernel merges them.
#include "common.h"
#include "rope_math.h"

#include <atomic>

namespace aicomp {

namespace {

#include "decode_tile16.h"

constexpr int SK_MAX_WAVES = 4096;     // balanced schedule: at most 1024 workgroups of 4 waves

struct MfmaParams {
    void* out;
    const void* query;
    void* k_pool;
    void* v_pool;
    const int32_t* block_table;
    int64_t block_table_stride;
    const int32_t* context_lens;
    int hq, hkv, group, max_blocks;
    int64_t num_blocks;
    float qk_mul;               // scale * log2(e)
    const float* k_scale;
    const float* v_scale;
    int partition_size, num_parts, part_turn;
    float* ws_acc;
    float* ws_ml;
    // fused append (optional): row b of new_key / new_value is token context_lens[b]-1
    const void* new_key;
    const void* new_value;
    int64_t new_token_stride, new_head_stride;     // elements
    // rotary embedding of the query rows and the new K row (kernels with ROPE; see rope_append.hip)
    const void* cos_tab;
    const void* sin_tab;
    int64_t tab_stride, tab_rows;
    const int64_t* positions;
    const int64_t* slots;                          // where the new row goes
    int64_t q_token_stride, q_head_stride;
};

#include "decode_tile_f32.h"
#include "decode_tile_f32_quad.h"

// query rows of (sequence, KV head) in the tensor, and its new rows
template <typename T, typename Params>
__device__ __forceinline__ const typename T::Fmt::raw* q_rows(const Params& p, int seq, int kvh) {
    return (const typename T::Fmt::raw*)p.query + ((int64_t)seq * p.hq + kvh * p.group) * T::DQ;
}
template <typename T, typename Params>
__device__ __forceinline__ const typename T::Fmt::raw* new_row(const void* rows, const Params& p, int seq, int kvh) {
    return (const typename T::Fmt::raw*)rows + (int64_t)seq * p.new_token_stride + (int64_t)kvh * p.new_head_stride;
}

// The rotary embedding of a workgroup's rows, every wave for itself: the group's query rows to q_lds, one after the
// other, and the new K row to k_lds.  Bit for bit what rope_append.hip leaves (same roundings, same order).
template <typename T>
__device__ __forceinline__ void rope_rows(const MfmaParams& p, int seq, int kvh, int64_t pos, typename T::Fmt::raw* q_lds,
                                          typename T::Fmt::raw* k_lds, int lane) {
    typedef typename T::Fmt::elem Elem;
    constexpr int CH = T::DQ / 16, HALF = T::DQ / 2, PER = 64 / CH;          // lanes per row, rows per pass
    const int c8 = 8 * (lane & (CH - 1)), G = p.group;
    const Elem* cr = (const Elem*)p.cos_tab + pos * p.tab_stride + c8;
    const Elem* sr = (const Elem*)p.sin_tab + pos * p.tab_stride + c8;
    Raw8<Elem> raw[4];
    raw[0].load(cr); raw[1].load(cr + HALF); raw[2].load(sr); raw[3].load(sr + HALF);
    for (int row = lane / CH; row <= G; row += PER) {
        const Elem* src = (row < G ? (const Elem*)p.query + seq * p.q_token_stride + (int64_t)(kvh * G + row) * p.q_head_stride
                                   : (const Elem*)new_row<T>(p.new_key, p, seq, kvh)) + c8;
        Raw8<Elem> lo, hi;
        lo.load(src);
        hi.load(src + HALF);
        float xl[8], xh[8], cl[8], ch[8], sl[8], sh[8];
        lo.unpack(xl); hi.unpack(xh);
        raw[0].unpack(cl); raw[1].unpack(ch); raw[2].unpack(sl); raw[3].unpack(sh);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float ol = rot1<Elem, true>(xl[j], xh[j], cl[j], sl[j]);
            xh[j] = rot1<Elem>(xh[j], xl[j], ch[j], sh[j]);
            xl[j] = ol;
        }
        Elem* dst = (Elem*)(row < G ? q_lds + row * T::DQ : k_lds) + c8;
        Row8<Elem>::store(dst, xl);
        Row8<Elem>::store(dst + HALF, xh);
    }
}

// A new row into its slot alone (a slot that is not where the table has the row's last token).
template <typename T>
__device__ __forceinline__ void store_new_row(const MfmaParams& p, const typename T::Fmt::raw* key,
                                              const typename T::Fmt::raw* value, int kvh, int64_t slot, int lane) {
    typedef typename T::Fmt::raw Raw;
    const int64_t row = (slot / BS * p.hkv + kvh) * BS + slot % BS;
    if constexpr (T::FP8) {
        if (lane < T::DQ / 8) {
            ((uint2*)p.k_pool)[row * (T::DQ / 8) + lane] = quant8_fp8<typename T::Fmt>(*(const uint4*)(key + 8 * lane), p.k_scale[kvh]);
            ((uint2*)p.v_pool)[row * (T::DQ / 8) + lane] = quant8_fp8<typename T::Fmt>(*(const uint4*)(value + 8 * lane), p.v_scale[kvh]);
        }
    } else {
        for (int d = lane; d < T::DQ; d += 64) {
            ((Raw*)p.k_pool)[row * T::DQ + d] = key[d];
            ((Raw*)p.v_pool)[row * T::DQ + d] = value[d];
        }
    }
}

// ROPE: the query rows come as projected, with strides of their own, and are rotated here, like the new K row: a decode
// step of a layer is then this launch alone, where the rotary + append launch before it and the rotated query's way
// through memory cost 3.3 us of device and 6 us of host time (8 rows of 900 tokens, 32 / 8 heads, D 64).
template <typename T, int NW, bool ROPE>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 2 : 1)
paged_decode_mfma_kernel(MfmaParams p) {
    // KV head fastest: the workgroups launched together read the Hkv slices of the same
    // physical blocks, i.e. one contiguous Hkv*4 KB piece of each pool
    constexpr int DQ = T::DQ, TT = T::TT, BPT = T::BPT, NPAR = T::NPAR;
    const int kvh = blockIdx.x;
    const int seq = blockIdx.z;
    const int turned = (int)blockIdx.y - (seq & p.part_turn);      // see launch_decode_mfma
    const int part = turned < 0 ? turned + p.num_parts : turned;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15;      // MFMA row / column index of this lane
    const int g4 = lane >> 4;       // MFMA k-group of this lane
    const int G = p.group;
    const int ncol = NPAR * G;      // B-operand columns in use
    const int start = part * p.partition_size;
    const int blk_base = start / BS;

    // Prologue loads, all issued before anything waits: the context length (scalar), the
    // partition's slice of the block table (one coalesced vector load: lane i holds entry
    // blk_base + i, later picked out with v_readlane, so the loop has no table loads at
    // all) and the query rows.
    const int32_t* table = p.block_table + (int64_t)seq * p.block_table_stride;
    int tab_first = 0;                       // first entry (relative to blk_base) held in `tab`
    int tab = (blk_base + lane < p.max_blocks) ? table[blk_base + lane] : 0;

    typename T::Q qf;
    if constexpr (!ROPE) T::load_q(qf, q_rows<T>(p, seq, kvh), G, lane);

    const int len = min(p.context_lens[seq], p.max_blocks * BS);   // never read past the table row
    // (a position without a row in the tables rotates by row 0 and is not stored, a slot outside the pool is a padding row's)
    const int64_t pos_in = ROPE ? p.positions[seq] : 0, slot = ROPE ? p.slots[seq] : -1;
    __shared__ __attribute__((aligned(16))) unsigned char lds[NW * KTILE_BYTES];
    const bool pos_ok = pos_in >= 0 && pos_in < p.tab_rows;
    const bool stored = ROPE && pos_ok && slot >= 0 && slot < p.num_blocks * BS;
    __shared__ __attribute__((aligned(16))) typename T::Fmt::raw k_new[ROPE ? NW : 1][ROPE ? DQ : 1];
    if (start >= len) {
        if (len <= 0 && part == 0) {   // nothing to attend to: the output row is defined as zero
            auto* o = (typename T::Fmt::raw*)p.out + ((int64_t)seq * p.hq + kvh * G) * DQ;
            for (int i = tid; i < G * DQ; i += blockDim.x) o[i] = 0;
            if constexpr (ROPE) {
                if (stored && w == 0) {
                    rope_rows<T>(p, seq, kvh, pos_in, (typename T::Fmt::raw*)lds, k_new[0], lane);
                    store_new_row<T>(p, k_new[0], new_row<T>(p.new_value, p, seq, kvh), kvh, slot, lane);
                }
            }
        }
        return;
    }
    // (ROPE: the caller's idea of the lengths sized the grid, and the last partition takes what is left of a row)
    const int end = ROPE && part + 1 == p.num_parts ? len : min(len, start + p.partition_size);
    const int ntiles = (end - start + TT - 1) / TT;

    __shared__ float sm_m[NW][16];
    __shared__ float sm_l[NW][16];
    unsigned char* kt = lds + w * KTILE_BYTES;

    const float cmul = p.qk_mul * (T::FP8 ? p.k_scale[kvh] : 1.f);

    typename T::State st;
    if constexpr (!T::QUAD) clear_state(st);

    // physical blocks of tile tt (wave-uniform); the held table slice is refilled every 64 blocks
    int64_t bb[4] = {0, 0, 0, 0};
    auto tile_blocks = [&](int tt) {
        const int i0 = BPT * tt;
        if (i0 - tab_first >= 64) {
            tab_first = i0;
            tab = (blk_base + i0 + lane < p.max_blocks) ? table[blk_base + i0 + lane] : 0;
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0) here, so the common path never waits on `tab`
        }
#pragma unroll
        for (int j = 0; j < BPT; ++j)
            bb[j] = clamp_block(__builtin_amdgcn_readlane(tab, i0 + j - tab_first), p.num_blocks);
    };

    const typename T::Offsets ko = T::offsets(lane);

    if (w < ntiles) {
        typename T::Regs kv;
        tile_blocks(w);
        T::load(kv, p, bb, kvh, lane);
        if constexpr (ROPE) {                     // through the wave's K tile, before any K is there
            rope_rows<T>(p, seq, kvh, pos_ok ? pos_in : 0, (typename T::Fmt::raw*)kt, k_new[w], lane);
            __builtin_amdgcn_wave_barrier();
            T::load_q(qf, (const typename T::Fmt::raw*)kt, G, lane);
        }
        T::q_operand(qf, qf, G, lane);
        int tt = w;
        for (; tt + NW < ntiles; tt += NW) {      // steady state: never the partition's last tile
            tile_blocks(tt + NW);
            T::template process<true, false>(st, kv, qf, kt, ko, p, bb, kvh, lane, start + tt * TT, end, cmul);
        }
        const int tile_start = start + tt * TT;
        // the sequence's newest token lives in this tile (bb still holds its blocks: the last lookup
        // above was for this wave's final tile)
        if (p.new_key != nullptr && end == len && tile_start < len && tile_start + TT >= len) {
            // Same rule as the separate one-token append: the row is stored only where the table names a
            // block of the pool and the length fits the table; otherwise the call leaves the pools alone
            // (and attends over what the clamped table entry holds, like the unfused sequence of calls).
            const int raw_blk = __builtin_amdgcn_readlane(tab, BPT * tt + ((len - 1 - tile_start) >> 4) - tab_first);
            const bool at_table = p.context_lens[seq] == len && raw_blk >= 0 && raw_blk < p.num_blocks;
            const typename T::Fmt::raw* nv = new_row<T>(p.new_value, p, seq, kvh);
            if constexpr (ROPE) {
                if (stored && at_table && (int64_t)raw_blk * BS + ((len - 1) & (BS - 1)) == slot)
                    T::inject(kv, p, k_new[w], nv, kvh, lane, tile_start, len, bb);
                else if (stored)
                    store_new_row<T>(p, k_new[w], nv, kvh, slot, lane);
            } else if (at_table) {
                T::inject(kv, p, new_row<T>(p.new_key, p, seq, kvh), nv, kvh, lane, tile_start, len, bb);
            }
        }
        if (tile_start + TT > end)
            T::template process<false, true>(st, kv, qf, kt, ko, p, bb, kvh, lane, tile_start, end, cmul);
        else
            T::template process<false, false>(st, kv, qf, kt, ko, p, bb, kvh, lane, tile_start, end, cmul);
    }
    // ---- wave result: the accumulators of column r16 into its row of the wave's own K tile region
    float* osm = (float*)kt;        // 16 columns of at most 128 floats: 8192 bytes, the whole tile
    if constexpr (T::QUAD) {
        T::finish(st, osm, sm_m[w], sm_l[w], 1, lane, G);
    } else {
        const float m = st.m;
        float lsum = st.lsum;
        lsum += __shfl_xor(lsum, 16);
        lsum += __shfl_xor(lsum, 32);
        if (r16 < ncol) {
            T::store_acc(osm + r16 * T::OROW, st, g4);
            if (g4 == 0) { sm_m[w][r16] = m; sm_l[w][r16] = lsum; }
        }
    }
    __syncthreads();

    const float vs = T::FP8 ? p.v_scale[kvh] : 1.f;
    const bool direct = p.num_parts == 1;     // unsplit call: no merge needed
    for (int idx = tid; idx < G * DQ; idx += 64 * NW) {
        const int h = idx / DQ, dd = idx % DQ;
        float mxw, num, den;
        merge_waves<T, NW>((const unsigned char*)lds, sm_m, sm_l, h, dd, mxw, num, den);
        const int head = kvh * G + h;
        if (direct) {
            ((typename T::Fmt::raw*)p.out)[((int64_t)seq * p.hq + head) * DQ + dd] =
                T::Fmt::from_f32(den == 0.f ? 0.f : vs * num / den);     // (a NaN stays one, as in the merge kernels)
        } else {
            const int64_t slot = ((int64_t)seq * p.hq + head) * p.num_parts + part;
            p.ws_acc[slot * DQ + dd] = num;
            if (dd == 0) { p.ws_ml[slot * 2] = mxw; p.ws_ml[slot * 2 + 1] = den; }
        }
    }
}


// ---------------------------------------------------------------------------------------
// Prompt chunks of a small grid (see launch_prefill_rows).  A workgroup of the prefill kernel proper walks all keys of
// its 128 query rows tile by tile, 1.3 us a step when it has a CU to itself, and a call of few chunks leaves most CUs
// without one.  Here the columns of the decode tiles are 16 query rows of a chunk (D 64: 8, two columns each), the waves
// of a workgroup split the keys like those of a decode row, and the rows' partial softmaxes are merged
// through LDS: eight (sixteen) times the workgroups, a chain of keys / (tile x waves) rounds.  Every workgroup reads its
// keys through its CU's 64 bytes per clock, which is what bounds it, and why large grids, whose CUs are busy
// anyway, share a tile between 128 rows instead.
struct PrefillRowsParams {
    void* out;
    const void* query;
    void* k_pool;
    void* v_pool;
    const int32_t* block_table;
    int64_t block_table_stride;
    const int32_t* context_lens;
    const int32_t* cu_q_lens;
    int hq, hkv, group, gpack, max_blocks;
    int64_t num_blocks;
    float qk_mul;
    const float* k_scale;
    const float* v_scale;
    const int32_t* items;       // (sequence, tile of `sub` workgroups) pairs, grid.y of them (NULL: grid.y numbers sequences)
    int num_seqs, sub;
};

template <typename T, int NW>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 2 : 1)
paged_prefill_rows_kernel(PrefillRowsParams p) {
    constexpr int DQ = T::DQ, TT = T::TT, BPT = T::BPT, NPAR = T::NPAR;
    constexpr int ROWS = 16 / NPAR;                                  // query rows per workgroup
    typedef typename T::Fmt::raw Raw;
    const int hgroup = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    const int pos_per_wg = ROWS / p.gpack;
    int seq = blockIdx.y;
    int64_t qtile = (int)(gridDim.z - 1 - blockIdx.z);              // expensive first
    if (p.items != nullptr) {
        seq = p.items[2 * blockIdx.y];
        const int q = p.items[2 * blockIdx.y + 1];
        if (seq < 0 || seq >= p.num_seqs || q < 0) return;
        qtile = (int64_t)q * p.sub + blockIdx.z;
    }
    const int q_begin = p.cu_q_lens[seq];
    const int n = p.cu_q_lens[seq + 1] - q_begin;
    const int ctx = min(p.context_lens[seq], p.max_blocks * BS);
    const int prior = ctx - n;
    if (n <= 0 || qtile * pos_per_wg >= n) return;
    const int q0 = (int)qtile * pos_per_wg;
    auto out_row = [&](int row) -> Raw* {                            // NULL: beyond the chunk
        const int pos = q0 + row / p.gpack;
        return pos < n ? (Raw*)p.out + ((int64_t)(q_begin + pos) * p.hq + hgroup * p.gpack + row % p.gpack) * DQ : nullptr;
    };
    if (prior < 0) {                   // a context shorter than the chunk itself: zero rows, as in the other kernels
        for (int i = tid; i < ROWS * DQ; i += 64 * NW)
            if (Raw* o = out_row(i / DQ)) o[i % DQ] = 0;
        return;
    }
    __shared__ __attribute__((aligned(16))) unsigned char lds[NW * KTILE_BYTES];
    __shared__ float sm_m[NW][16];
    __shared__ float sm_l[NW][16];
    unsigned char* kt = lds + w * KTILE_BYTES;

    const int kvh = (hgroup * p.gpack) / p.group;                    // workgroup-uniform
    const int32_t* table = p.block_table + (int64_t)seq * p.block_table_stride;
    int tab_first = 0;
    int tab = lane < p.max_blocks ? table[lane] : 0;

    // this lane's column: its row, and the first key the row does not see (rows beyond the chunk: computed, not stored)
    const int row = r16 / NPAR, qpos = q0 + row / p.gpack;
    const int kv_end = min(ctx, prior + q0 + pos_per_wg), kv_min = prior + q0 + 1;
    const int end = qpos < n ? prior + qpos + 1 : kv_end;
    typename T::Q qf;
    T::load_q_row(qf, (const Raw*)p.query + ((int64_t)(q_begin + min(qpos, n - 1)) * p.hq + hgroup * p.gpack + row % p.gpack) * DQ, lane);
    const float cmul = p.qk_mul * (T::FP8 ? p.k_scale[kvh] : 1.f);
    const int ntiles = (kv_end + TT - 1) / TT;
    typename T::State st;
    clear_state(st);

    int64_t bb[4] = {0, 0, 0, 0};
    auto tile_blocks = [&](int tt) {
        const int i0 = BPT * tt;
        if (i0 - tab_first >= 64) {
            tab_first = i0;
            tab = i0 + lane < p.max_blocks ? table[i0 + lane] : 0;
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0) here, so the common path never waits on `tab`
        }
#pragma unroll
        for (int j = 0; j < BPT; ++j) bb[j] = clamp_block(__builtin_amdgcn_readlane(tab, i0 + j - tab_first), p.num_blocks);
    };
    const typename T::Offsets ko = T::offsets(lane);
    if (w < ntiles) {
        typename T::Regs kv;
        tile_blocks(w);
        T::load(kv, p, bb, kvh, lane);
        T::q_operand(qf, qf, ROWS, lane);
        int tt = w;
        // (the rows of a workgroup end within 16 tokens of each other: only the last NW tiles, each its wave's last, can
        // need a mask)
        for (; tt + NW < ntiles; tt += NW) {
            tile_blocks(tt + NW);
            T::template process_rows<true, false>(st, kv, qf, kt, ko, p, bb, kvh, lane, tt * TT, end, kv_end, cmul);
        }
        if (tt * TT + TT > kv_min)
            T::template process_rows<false, true>(st, kv, qf, kt, ko, p, bb, kvh, lane, tt * TT, end, kv_end, cmul);
        else
            T::template process_rows<false, false>(st, kv, qf, kt, ko, p, bb, kvh, lane, tt * TT, end, kv_end, cmul);
    }
    float lsum = st.lsum;
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    T::store_acc((float*)kt + r16 * T::OROW, st, g4);
    if (g4 == 0) { sm_m[w][r16] = st.m; sm_l[w][r16] = lsum; }
    __syncthreads();
    const float vs = T::FP8 ? p.v_scale[kvh] : 1.f;
    for (int idx = tid; idx < ROWS * DQ; idx += 64 * NW) {
        const int h = idx / DQ, dd = idx % DQ;
        Raw* o = out_row(h);
        if (o == nullptr) continue;
        float mx, num, den;
        merge_waves<T, NW>((const unsigned char*)lds, sm_m, sm_l, h, dd, mx, num, den);
        o[dd] = T::Fmt::from_f32(den == 0.f ? 0.f : vs * num / den);
    }
}

// ---------------------------------------------------------------------------------------
// Balanced schedule.  The grid above gives the hardware dispatcher workgroups of unequal
// size and leaves a tail where few of them are still streaming.  Here the launch is
// exactly one workgroup per CU and every WAVE gets the same number of 32-token tiles.
// Waves are dealt to KV heads first (wave i: head i % Hkv, part i / Hkv of that head); the
// tiles of one head over all sequences form one sequence of N tiles and part j of W owns
// tiles [j*N/W, (j+1)*N/W).  The Hkv waves of one part walk the same tiles of the same
// sequences side by side, i.e. the Hkv adjacent head slices of the same physical blocks at
// about the same time, whatever the sequences' lengths (with KV heads inside the tile order
// instead, waves drift apart on batches of unequal lengths and read isolated 2 - 4 KB slices:
// 221 -> 211 us on the fp8 Llama-3-70B shape, bf16 shapes unchanged).  A wave crossing a
// sequence boundary flushes its partial (max, sum, unnormalised output) and starts the next
// sequence, so all waves start together, stream the same number of bytes and finish together.
// Partials of head h go to slot h * (W + S) + part + sequence - strictly increasing along a
// head's schedule, hence unique - and streamk_reduce_kernel merges the slots of each row.
// No barrier after the prologue.
constexpr int SK_MAX_SEQS = 1024;

struct StreamKParams {
    void* out;
    const void* query;
    void* k_pool;
    void* v_pool;
    const int32_t* block_table;
    int64_t block_table_stride;
    const int32_t* context_lens;
    int num_seqs, hq, hkv, group, max_blocks;
    int64_t num_blocks;
    float qk_mul;
    const float* k_scale;
    const float* v_scale;
    int num_waves;
    int waves_per_head;     // num_waves / hkv
    float* ws_acc;      // [slots][G][D]
    float* ws_ml;       // [slots][G][2]
    int* ws_rows;       // [rows][2]: first and last part (wave of the row's head) holding a partial of the row
    // fused append (optional): row b of new_key / new_value is token context_lens[b]-1
    const void* new_key;
    const void* new_value;
    int64_t new_token_stride, new_head_stride;     // elements
};

template <int TT>
__device__ __forceinline__ int sk_tiles(int len, int max_blocks) {
    len = min(max(len, 0), max_blocks * BS);
    return (len + TT - 1) / TT;
}


// Token pairs (Tile16 with PAIR): every head takes two B-operand columns, one per token parity, and a
// flush merges the two columns of a head inside the wave and writes one partial of 64 floats per head.
template <typename T>
__global__ void __launch_bounds__(256, 1)     // one workgroup per CU: a wave may use the whole register file
streamk_decode_kernel(StreamKParams p) {
    constexpr int DQ = T::DQ, TT = T::TT, BPT = T::BPT;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    const int G = p.group, B = p.num_seqs;
    const int ncol = T::NPAR * G;                // B-operand columns in use

    __shared__ __attribute__((aligned(16))) unsigned char lds[NWAVES * KTILE_BYTES];
    __shared__ int prefix[SK_MAX_SEQS + 1];     // prefix[s] = tiles of the sequences before s
    __shared__ int wave_tot[NWAVES];
    unsigned char* kt = lds + w * KTILE_BYTES;

    // ---- prologue: tiles per sequence -> exclusive prefix sums
    if (B <= 64) {
        // every wave scans for itself and reads back only what it wrote: no barrier (the
        // four waves write identical values to the same words)
        const int mine = lane < B ? sk_tiles<TT>(p.context_lens[lane], p.max_blocks) : 0;
        int inc = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(inc, o);
            if (lane >= o) inc += v;
        }
        prefix[lane] = inc - mine;
        if (lane == 63) prefix[64] = inc;
        if (B < 64 && lane == B) prefix[B] = inc - mine;      // == total: lanes >= B add nothing
    } else {
        int loc[4], sum = 0;                                  // 4 sequences per thread
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int sidx = 4 * tid + k;
            loc[k] = sidx < B ? sk_tiles<TT>(p.context_lens[sidx], p.max_blocks) : 0;
            sum += loc[k];
        }
        int inc = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(inc, o);
            if (lane >= o) inc += v;
        }
        if (lane == 63) wave_tot[w] = inc;
        __syncthreads();
        int base = inc - sum;
        for (int ww = 0; ww < w; ++ww) base += wave_tot[ww];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int sidx = 4 * tid + k;
            if (sidx <= B) prefix[sidx] = base;
            base += loc[k];
        }
        if (tid == 255 && B == SK_MAX_SEQS) prefix[SK_MAX_SEQS] = base;
        __syncthreads();
    }
    // Waves are dealt to KV heads first: wave i works on head i % Hkv, and the waves_per_head waves
    // of a head split that head's tiles of all sequences evenly.  The Hkv waves with the same
    // i / Hkv then walk the same tiles of the same sequences side by side, i.e. the Hkv adjacent
    // head slices of the same physical blocks at about the same time.
    const int64_t N = __builtin_amdgcn_readfirstlane(prefix[B]);       // tiles of one head
    const int wave_id = blockIdx.x * NWAVES + w;
    const int kvh_mine = wave_id % p.hkv, part = wave_id / p.hkv;
    const int W = (int)min((int64_t)p.waves_per_head, N);  // with fewer tiles than waves, one tile each
    if (part >= W) return;
    const int64_t g0 = (int64_t)part * N / W;
    const int64_t g1 = (int64_t)(part + 1) * N / W;

    // ---- first row of this wave: largest s with prefix[s] <= g0
    int seq;
    {
        const int x = (int)g0;
        int lo = 0, hi = B;            // invariant: prefix[lo] <= x < prefix[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (prefix[mid] <= x) lo = mid; else hi = mid;
        }
        seq = __builtin_amdgcn_readfirstlane(lo);
    }
    // everything that steers the loop is wave-uniform: keep it in scalar registers
    int row_tiles = __builtin_amdgcn_readfirstlane(prefix[seq + 1] - prefix[seq]);
    int kvh = __builtin_amdgcn_readfirstlane(kvh_mine);
    int t = __builtin_amdgcn_readfirstlane((int)(g0 - prefix[seq]));

    const typename T::Offsets ko = T::offsets(lane);

    // ---- segments.  A segment is the part of one (sequence, KV head) row that falls into this
    // wave's tile range.  The next segment's query rows and table slice are requested while the
    // current one streams, and its first K/V tile is prefetched by the current segment's last
    // tile, so the loads never drain at a row boundary.
    auto load_tab = [&](int sq, int first_block) {
        const int32_t* table = p.block_table + (int64_t)sq * p.block_table_stride;
        return (first_block + lane < p.max_blocks) ? table[first_block + lane] : 0;
    };

    int nt = (int)min((int64_t)(row_tiles - t), g1 - g0);          // tiles of the current segment (>= 1)
    typename T::Q qf, qraw;
    T::load_q(qraw, q_rows<T>(p, seq, kvh), G, lane);
    int tab = load_tab(seq, BPT * t);
    typename T::Regs kv;
    // the blocks of a tile out of a table slice held one entry per lane
    auto slice_blocks = [&](int slice, int first, int64_t (&bb)[4]) {
#pragma unroll
        for (int j = 0; j < BPT; ++j) bb[j] = clamp_block(__builtin_amdgcn_readlane(slice, first + j), p.num_blocks);
    };
    {
        __builtin_amdgcn_s_waitcnt(0x0F70);                        // Q and table have landed
        T::q_operand(qf, qraw, G, lane);
        int64_t bb[4] = {0, 0, 0, 0};
        slice_blocks(tab, 0, bb);
        T::load(kv, p, bb, kvh, lane);
    }

    for (int64_t g = g0; g < g1 && seq < B;) {
        const int len = min(p.context_lens[seq], p.max_blocks * BS);
        const int blk_base = BPT * t;
        const int32_t* table = p.block_table + (int64_t)seq * p.block_table_stride;
        int tab_first = 0;
        const float cmul = p.qk_mul * (T::FP8 ? p.k_scale[kvh] : 1.f);
        auto tile_blocks = [&](int k, int64_t (&bb)[4]) {              // k-th tile of the segment
            const int i0 = BPT * k;
            if (i0 - tab_first >= 64) {
                tab_first = i0;
                tab = (blk_base + i0 + lane < p.max_blocks) ? table[blk_base + i0 + lane] : 0;
                __builtin_amdgcn_s_waitcnt(0x0F70);
            }
            slice_blocks(tab, i0 - tab_first, bb);
        };

        // the segment after this one (same wave, same KV head): the next sequence with tokens
        int nseq = seq, nkvh = kvh, nrow_tiles = row_tiles;
        const bool more = g + nt < g1;
        if (more) {
            do { ++nseq; } while (nseq < B && __builtin_amdgcn_readfirstlane(prefix[nseq + 1] - prefix[nseq]) == 0);
            nrow_tiles = nseq < B ? __builtin_amdgcn_readfirstlane(prefix[nseq + 1] - prefix[nseq]) : 0;
        }
        const bool has_next = more && nseq < B;
        int tabn = 0;
        typename T::Q qn;
        if (has_next) {
            T::load_q(qraw, q_rows<T>(p, nseq, nkvh), G, lane);
            tabn = load_tab(nseq, 0);
        }

        typename T::State st;
        if constexpr (!T::QUAD) clear_state(st);

        int64_t bb[4] = {0, 0, 0, 0};
        int k = 0;
        for (; k + 1 < nt; ++k) {
            tile_blocks(k + 1, bb);
            T::template process<true, false>(st, kv, qf, kt, ko, p, bb, kvh, lane, (t + k) * TT, len, cmul);
        }
        const int tile_start = (t + k) * TT;
        if (p.new_key != nullptr && t + k == row_tiles - 1) {       // the row's newest token lives here
            tile_blocks(k, bb);
            // Same rule as the separate one-token append: the row is stored only where the table names a
            // block of the pool and the length fits the table; otherwise the call leaves the pools alone
            // (and attends over what the clamped table entry holds, like the unfused sequence of calls).
            const int raw_blk = __builtin_amdgcn_readlane(tab, BPT * k + ((len - 1 - tile_start) >> 4) - tab_first);
            if (p.context_lens[seq] == len && raw_blk >= 0 && raw_blk < p.num_blocks)
                T::inject(kv, p, new_row<T>(p.new_key, p, seq, kvh), new_row<T>(p.new_value, p, seq, kvh), kvh, lane,
                          tile_start, len, bb);
        }
        // The segment's last tile always runs the masked body (a full tile simply masks nothing):
        // one prefetching call site, so the prefetched registers need no merging afterwards.
        int tab_ready = 0;
        if (has_next) {
            // prefetch the first tile of the next segment
            __builtin_amdgcn_s_waitcnt(0x0F70);      // next Q rows and table slice (and this tile) have landed
            T::q_operand(qn, qraw, G, lane);
            tab_ready = tabn;
            slice_blocks(tab_ready, 0, bb);
            T::template process<true, true>(st, kv, qf, kt, ko, p, bb, nkvh, lane, tile_start, len, cmul);
        } else {
            T::template process<false, true>(st, kv, qf, kt, ko, p, bb, kvh, lane, tile_start, len, cmul);
        }

        // ---- flush
        const int64_t slot = (int64_t)kvh * (p.waves_per_head + B) + part + seq;
        float lsum = 0.f;
        if constexpr (!T::QUAD) {
            lsum = st.lsum;
            lsum += __shfl_xor(lsum, 16);
            lsum += __shfl_xor(lsum, 32);
        }
        if constexpr (T::QUAD) {
            float* ml = p.ws_ml + slot * G * 2;
            T::finish(st, p.ws_acc + slot * G * DQ, ml, ml + 1, 2, lane, G);
        } else if constexpr (T::PAIR) {
            // Column (head, parity) holds its own token's half of the pair rows: parity 0 elements 0..63 of
            // its accumulator (lanes g4 = 0, 1), parity 1 elements 64..127 (lanes g4 = 2, 3).  The two are
            // partial softmaxes over the even and the odd tokens of the same segment: merged here, inside the
            // wave, so that a flush writes ONE partial of 64 floats per head.  Lane (column 2h, g4 = a) takes
            // the matching values of lane (column 2h + 1, g4 = a + 2), 33 lanes up.
            const float m1 = __shfl_xor(st.m, 1), l1 = __shfl_xor(lsum, 1);
            const float mm = fmaxf(st.m, m1);
            const float f0 = exp2f(st.m - mm), f1 = exp2f(m1 - mm);
            float mine[8][4];
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) mine[j][i] = fmaf(f1, __shfl(st.O[j][i], lane + 33), f0 * st.O[j][i]);
            if (r16 < ncol && (r16 & 1) == 0 && g4 < 2) {
                float* dst = p.ws_acc + (slot * G + (r16 >> 1)) * DQ + 32 * g4;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    *(float4*)(dst + 8 * i) = make_float4(mine[0][i], mine[1][i], mine[2][i], mine[3][i]);
                    *(float4*)(dst + 8 * i + 4) = make_float4(mine[4][i], mine[5][i], mine[6][i], mine[7][i]);
                }
                if (g4 == 0) *(float2*)(p.ws_ml + (slot * G + (r16 >> 1)) * 2) = make_float2(mm, f0 * lsum + f1 * l1);
            }
        } else if (r16 < ncol) {
            T::store_acc(p.ws_acc + (slot * G + r16) * DQ, st, g4);
            if (g4 == 0) *(float2*)(p.ws_ml + (slot * G + r16) * 2) = make_float2(st.m, lsum);
        }
        // the waves holding a row's first and last tile tell the merge kernel where its partials are
        if (lane == 0) {
            int* rm = p.ws_rows + 2 * ((int64_t)seq * p.hkv + kvh);
            if (t == 0) rm[0] = part;
            if (t + nt == row_tiles) rm[1] = part;
        }

        // ---- next segment
        g += nt;
        if (!has_next) break;
        seq = nseq; kvh = nkvh; row_tiles = nrow_tiles; t = 0;
        nt = (int)min((int64_t)row_tiles, g1 - g);
        tab = tab_ready;
        qf = qn;
    }
}

// Merge of the balanced schedule's partials: one workgroup per (KV head, sequence), S waves per
// head of the group.  The row's partials sit in consecutive slots of its head's region,
// head_slots * head + first + sequence .. + last + sequence (first / last part recorded by the
// main kernel); their weights 2^(m_i - M) are computed once (one lane
// per partial) and parked in LDS, then each lane accumulates its output dims (two at head_dim
// 128, one at head_dim 64) with independent loads.  With S = 1 (few partials per row, the usual
// batch) reductions are shuffles and there is no barrier; with S > 1 (a handful of very long rows,
// hundreds of partials each) the waves of a head take alternate groups of eight partials and add
// up through LDS.
constexpr int RED_WGT = 256;       // weights parked in LDS per wave; rows with more partials recompute the rest
template <typename E, int DQ>
__global__ void __launch_bounds__(1024)
streamk_reduce_kernel(typename E::raw* __restrict__ out, const float* __restrict__ ws_acc,
                      const float* __restrict__ ws_ml, const int* __restrict__ ws_rows,
                      const int32_t* __restrict__ context_lens, int hq, int hkv, int group,
                      const float* __restrict__ v_scale, int head_slots) {
    constexpr int NV = DQ / 64;                            // output dims per lane
    const int kvh = blockIdx.x, seq = blockIdx.y, wv = threadIdx.x >> 6;
    const int S = (int)(blockDim.x >> 6) / group;          // waves per head
    const int h = wv / S, sub = wv % S;
    const int lane = threadIdx.x & 63;
    __shared__ float wgt_all[16][RED_WGT];
    __shared__ float part[16][DQ];
    float* wgt = wgt_all[wv];
    const int64_t row = (int64_t)seq * hkv + kvh;
    auto* o = out + ((int64_t)seq * hq + kvh * group + h) * DQ;
    // the length and the row's record are requested together (the record of an empty row was never
    // written and is not used)
    const int ctx = context_lens[seq];
    const int first = ws_rows[2 * row], last = ws_rows[2 * row + 1];
    if (ctx <= 0) {                          // no tiles, no partials: the output row is zero (whole workgroup)
        if (sub == 0) {
#pragma unroll
            for (int e = 0; e < NV; ++e) o[lane + 64 * e] = 0;
        }
        return;
    }
    const int np = last - first + 1;
    const int64_t slot0 = (int64_t)kvh * head_slots + first + seq;       // the row's partials: slots slot0 .. slot0 + np - 1
    const float* ml = ws_ml + (slot0 * group + h) * 2;                  // partial i at ml[i * group * 2]
    const float* acc = ws_acc + (slot0 * group + h) * DQ + lane;        // partial i at acc[i * group * DQ]
    const int64_t stride = (int64_t)group * DQ;
    if (S == 1 && np <= 8) {
        // The usual batch: a handful of partials per row.  Their (max, sum) pairs and this lane's
        // output dims of each are requested in one go, so the kernel is two memory latencies
        // deep (record, then partials) instead of four.
        float2 mlv[8];
        float a[8][NV];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(u, np - 1);
            mlv[u] = *(const float2*)(ml + (int64_t)i * group * 2);
#pragma unroll
            for (int e = 0; e < NV; ++e) a[u][e] = acc[i * stride + 64 * e];
        }
        float mx = NEG_BIG;
#pragma unroll
        for (int u = 0; u < 8; ++u) mx = fmaxf(mx, mlv[u].x);           // repeats of the last partial change nothing
        float den = 0.f, num[NV] = {};
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float f = u < np ? exp2f(mlv[u].x - mx) : 0.f;
            den = fmaf(f, mlv[u].y, den);
#pragma unroll
            for (int e = 0; e < NV; ++e) num[e] = fmaf(f, a[u][e], num[e]);
        }
        const float inv = den > 0.f ? (v_scale ? v_scale[kvh] : 1.f) / den : 0.f;
#pragma unroll
        for (int e = 0; e < NV; ++e) o[lane + 64 * e] = E::from_f32(num[e] * inv);
        return;
    }
    // every wave of a head computes the row's max, denominator and weights for itself (np / 64 loads per lane)
    float mx = NEG_BIG;
    for (int i = lane; i < np; i += 64) mx = fmaxf(mx, ml[(int64_t)i * group * 2]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    float den = 0.f;
    for (int i = lane; i < np; i += 64) {
        const float2 v = *(const float2*)(ml + (int64_t)i * group * 2);
        const float f = exp2f(v.x - mx);
        if (i < RED_WGT) wgt[i] = f;
        den = fmaf(f, v.y, den);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) den += __shfl_xor(den, off);
    // eight partials in flight per step: the loop is pure load latency
    float num[NV] = {};
    for (int i0 = 8 * sub; i0 < np; i0 += 8 * S) {
        float a[8][NV];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u, np - 1);
#pragma unroll
            for (int e = 0; e < NV; ++e) a[u][e] = acc[i * stride + 64 * e];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u;
            const float f = i >= np ? 0.f : (i < RED_WGT ? wgt[i] : exp2f(ml[(int64_t)i * group * 2] - mx));
#pragma unroll
            for (int e = 0; e < NV; ++e) num[e] = fmaf(f, a[u][e], num[e]);
        }
    }
    if (S > 1) {                             // workgroup-uniform
#pragma unroll
        for (int e = 0; e < NV; ++e) part[wv][lane + 64 * e] = num[e];
        __syncthreads();
        if (sub != 0) return;
        for (int k = 1; k < S; ++k)
#pragma unroll
            for (int e = 0; e < NV; ++e) num[e] += part[wv + k][lane + 64 * e];
    }
    const float inv = den > 0.f ? (v_scale ? v_scale[kvh] : 1.f) / den : 0.f;
#pragma unroll
    for (int e = 0; e < NV; ++e) o[lane + 64 * e] = E::from_f32(num[e] * inv);
}

}  // namespace

// head_dim 128, or head_dim 64 handled as rows of token pairs (two B-operand columns per head,
// hence groups up to 8 and partitions of whole 64-token tiles)
bool decode_mfma_supported(const DecodeArgs& a) {
    const int group = a.hkv > 0 ? a.hq / a.hkv : 0;
    const bool f32 = a.q_dtype == AICOMP_KV_F32 && a.kv_dtype == AICOMP_KV_F32;
    const bool half = is_16bit_float(a.q_dtype) && (a.kv_dtype == a.q_dtype || a.kv_dtype == AICOMP_KV_FP8_E4M3);
    // tokens per tile: what a partition must be a multiple of
    const int tile = f32 ? (a.d == D ? TILE / 2 : TILE) : (a.d == D ? TILE : 2 * TILE);
    const bool shape = (a.d == D || a.d == 64) && group >= 1 && group <= (half && a.d == 64 ? 8 : 16) &&
                       a.partition_size % tile == 0;
    return a.cu_q_lens == nullptr && shape && a.bs == BS && (half || f32) && a.scale > 0.f && a.rows <= 65535 &&
           a.num_parts <= 65535 && ((uintptr_t)a.query % 16 == 0) && ((uintptr_t)a.k_pool % 16 == 0) &&
           ((uintptr_t)a.v_pool % 16 == 0);
}

bool decode_streamk_supported(const DecodeArgs& a) {
    // every KV head needs at least one wave of the 4 x CUs the schedule launches
    return decode_mfma_supported(a) && a.rows <= SK_MAX_SEQS && a.hkv <= 256;
}

// per slot one partial per head: G x (head_dim + 2) floats
size_t decode_streamk_workspace_bytes(int64_t rows, int hq, int hkv, int d) {
    const int64_t slots = SK_MAX_WAVES + rows * hkv;
    const int ncol = hq / hkv;
    return (size_t)slots * ncol * (size_t)(d + 2) * sizeof(float) + (size_t)rows * hkv * 2 * sizeof(int);
}

int launch_decode_streamk(const DecodeArgs& a, void* workspace) {
    // CU count of the first device used (every GPU of a node is the same part); an atomic so that
    // callers on several threads may race here harmlessly
    static std::atomic<int> cached_cus{0};
    int num_cus = cached_cus.load(std::memory_order_relaxed);
    if (num_cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
            set_error("paged_decode_attn: cannot query the CU count");
            return AICOMP_KV_EHIP;
        }
        num_cus = n;
        cached_cus.store(n, std::memory_order_relaxed);
    }
    // one workgroup per CU measured fastest (4 waves of 16 KB in flight each already cover the
    // HBM latency; a second workgroup per CU only adds partials and start-up work)
    const int wgs = min(num_cus, SK_MAX_WAVES / NWAVES);
    const int group = a.hq / a.hkv;
    const int64_t slots = SK_MAX_WAVES + a.rows * a.hkv;
    StreamKParams p;
    p.out = a.out; p.query = a.query; p.k_pool = (void*)a.k_pool; p.v_pool = (void*)a.v_pool;
    p.block_table = a.block_table; p.block_table_stride = a.block_table_stride;
    p.context_lens = a.context_lens;
    p.num_seqs = (int)a.rows; p.hq = a.hq; p.hkv = a.hkv; p.group = group; p.max_blocks = a.max_blocks;
    p.num_blocks = a.num_blocks;
    p.qk_mul = a.scale * LOG2E;
    p.k_scale = a.k_scale; p.v_scale = a.v_scale;
    p.num_waves = wgs * NWAVES;
    p.waves_per_head = p.num_waves / a.hkv;
    const bool pair = a.d == 64;
    const int ncol = group;
    p.ws_acc = (float*)workspace;
    p.ws_ml = p.ws_acc + slots * ncol * a.d;
    p.ws_rows = (int*)(p.ws_ml + slots * ncol * 2);
    p.new_key = a.new_key; p.new_value = a.new_value;
    p.new_token_stride = a.new_token_stride; p.new_head_stride = a.new_head_stride;
    const bool fp8 = a.kv_dtype == AICOMP_KV_FP8_E4M3, f16 = a.q_dtype == AICOMP_KV_F16, f32 = a.q_dtype == AICOMP_KV_F32;
#define AICOMP_LAUNCH_SK(E, PAIR)                                                                                  \
    do {                                                                                                           \
        if (fp8) hipLaunchKernelGGL((streamk_decode_kernel<Tile16<E, true, PAIR>>), dim3(wgs), dim3(256), 0, a.stream, p);  \
        else hipLaunchKernelGGL((streamk_decode_kernel<Tile16<E, false, PAIR>>), dim3(wgs), dim3(256), 0, a.stream, p);    \
    } while (0)
    if (f32) {
#define AICOMP_LAUNCH_SK32(DQ)                                                                                                 \
    do {                                                                                                                       \
        if (group <= 4) hipLaunchKernelGGL((streamk_decode_kernel<TileF32Quad<DQ>>), dim3(wgs), dim3(256), 0, a.stream, p);    \
        else hipLaunchKernelGGL((streamk_decode_kernel<TileF32<DQ>>), dim3(wgs), dim3(256), 0, a.stream, p);                   \
    } while (0)
        if (a.d == 64) AICOMP_LAUNCH_SK32(64); else AICOMP_LAUNCH_SK32(128);
#undef AICOMP_LAUNCH_SK32
    } else if (pair) { if (f16) AICOMP_LAUNCH_SK(F16Fmt, true); else AICOMP_LAUNCH_SK(Bf16Fmt, true); }
    else { if (f16) AICOMP_LAUNCH_SK(F16Fmt, false); else AICOMP_LAUNCH_SK(Bf16Fmt, false); }
#undef AICOMP_LAUNCH_SK
    AICOMP_HIP_LAUNCH_CHECK();
    // waves per head in the merge: one, unless rows are few and long (many partials per row)
    const int64_t per_row = (int64_t)p.waves_per_head / a.rows + 2;
    const int sub = per_row > 8 ? 16 / group : 1;
#define AICOMP_LAUNCH_RED(E, DQ)                                                                                  \
    hipLaunchKernelGGL((streamk_reduce_kernel<E, DQ>), dim3(a.hkv, (unsigned)a.rows), dim3(64 * group * sub), 0,  \
                       a.stream, (E::raw*)a.out, p.ws_acc, p.ws_ml, p.ws_rows, a.context_lens, a.hq, a.hkv,     \
                       group, a.v_scale, p.waves_per_head + (int)a.rows)
    if (f32) { if (a.d == 64) AICOMP_LAUNCH_RED(F32Fmt, 64); else AICOMP_LAUNCH_RED(F32Fmt, 128); }
    else if (pair) { if (f16) AICOMP_LAUNCH_RED(F16Fmt, 64); else AICOMP_LAUNCH_RED(Bf16Fmt, 64); }
    else { if (f16) AICOMP_LAUNCH_RED(F16Fmt, 128); else AICOMP_LAUNCH_RED(Bf16Fmt, 128); }
#undef AICOMP_LAUNCH_RED
    AICOMP_HIP_LAUNCH_CHECK();
    return AICOMP_KV_OK;
}

int launch_decode_mfma(const DecodeArgs& a) {
    MfmaParams p;
    p.out = a.out; p.query = a.query; p.k_pool = (void*)a.k_pool; p.v_pool = (void*)a.v_pool;
    p.block_table = a.block_table; p.block_table_stride = a.block_table_stride;
    p.context_lens = a.context_lens;
    p.hq = a.hq; p.hkv = a.hkv; p.group = a.hq / a.hkv; p.max_blocks = a.max_blocks;
    p.num_blocks = a.num_blocks;
    p.qk_mul = a.scale * LOG2E;
    p.k_scale = a.k_scale; p.v_scale = a.v_scale;
    p.partition_size = a.partition_size; p.num_parts = a.num_parts;
    // Workgroups go round the XCDs and their CUs by index, and rows of four, eight, .. partitions come round to the same ones
    // every time: where most rows are short, their first partitions, the only ones with work, all did.  A row's partitions
    // therefore start where its number says, modulo the largest power of two among them.  One row as long as the table, the others
    // a tenth of that at most, bf16, D 128, before -> turned (balanced schedule): 16 / 2 heads, 128 rows of 2048 31.3 -> 16.6 us
    // (20.6), 64 rows 19.0 -> 13.0 (16.0), 64 of 4096 31.7 -> 14.3 (22.7); 32 / 8 heads, 24 rows of 2048 17.5 -> 13.3 (17.9).  Rows
    // alike are as fast as before, and so are other numbers of partitions, which are not turned (six of 48 rows: 16.2, turned 18.5).
    p.part_turn = a.num_parts % 4 == 0 ? (1 << (31 - __builtin_clz((unsigned)a.num_parts))) - 1 : 0;
    p.ws_acc = a.ws.acc; p.ws_ml = a.ws.ml;
    p.new_key = a.new_key; p.new_value = a.new_value;
    p.new_token_stride = a.new_token_stride; p.new_head_stride = a.new_head_stride;
    p.cos_tab = a.cos_tab; p.sin_tab = a.sin_tab; p.tab_stride = a.tab_stride; p.tab_rows = a.tab_rows;
    p.positions = a.positions; p.slots = a.slots;
    p.q_token_stride = a.q_token_stride; p.q_head_stride = a.q_head_stride;
    const bool rope = a.cos_tab != nullptr;
    dim3 grid((unsigned)a.hkv, (unsigned)a.num_parts, (unsigned)a.rows);
    const bool fp8 = a.kv_dtype == AICOMP_KV_FP8_E4M3, d64 = a.d == 64;
    // Eight waves instead of four per workgroup for partitions of more than sixteen tiles in at most one
    // workgroup per CU: each is then a chain of rounds of one tile per wave at memory latency, and half the
    // rounds outweigh the longer merge (D 128, 576 tokens, 1 to 10 rows of 8 KV heads: 7.8 -> 6.9 us, fp8 9.1 ->
    // 8.0; float32 448 tokens 16.2 -> 13.9; 500 tokens, D 64, eight tiles: 5.72 us with four waves, 5.84 with
    // eight; 16 rows of 500, D 128, sixteen: 8.70 and 8.88).  A CU that has two workgroups has eight waves anyway,
    // and the larger ones are slower: 576 tokens, 256 workgroups 12.5 and 12.4, 320 workgroups 18.2 and 20.5; 1100
    // rows of 1024 tokens of fp8 406 and 464.
    const int tile = a.q_dtype == AICOMP_KV_F32 ? (d64 ? TILE : TILE / 2) : (d64 ? 2 * TILE : TILE);
    const bool wide = a.partition_size > 16 * tile && a.rows * a.hkv * a.num_parts <= 256;
#define AICOMP_LAUNCH_GRID(...)                                                                                        \
    do {                                                                                                               \
        if (rope && wide) hipLaunchKernelGGL((paged_decode_mfma_kernel<__VA_ARGS__, 8, true>), grid, dim3(512), 0, a.stream, p); \
        else if (rope) hipLaunchKernelGGL((paged_decode_mfma_kernel<__VA_ARGS__, 4, true>), grid, dim3(256), 0, a.stream, p);    \
        else if (wide) hipLaunchKernelGGL((paged_decode_mfma_kernel<__VA_ARGS__, 8, false>), grid, dim3(512), 0, a.stream, p);   \
        else hipLaunchKernelGGL((paged_decode_mfma_kernel<__VA_ARGS__, 4, false>), grid, dim3(256), 0, a.stream, p);             \
    } while (0)
#define AICOMP_LAUNCH_GRID16(E)                                                                     \
    do {                                                                                            \
        if (d64) { if (fp8) AICOMP_LAUNCH_GRID(Tile16<E, true, true>); else AICOMP_LAUNCH_GRID(Tile16<E, false, true>); } \
        else { if (fp8) AICOMP_LAUNCH_GRID(Tile16<E, true, false>); else AICOMP_LAUNCH_GRID(Tile16<E, false, false>); }   \
    } while (0)
#define AICOMP_LAUNCH_GRID32(DQ)                                                                              \
    do { if (p.group <= 4) AICOMP_LAUNCH_GRID(TileF32Quad<DQ>); else AICOMP_LAUNCH_GRID(TileF32<DQ>); } while (0)
    if (a.q_dtype == AICOMP_KV_F32) { if (d64) AICOMP_LAUNCH_GRID32(64); else AICOMP_LAUNCH_GRID32(128); }
    else if (a.q_dtype == AICOMP_KV_F16) AICOMP_LAUNCH_GRID16(F16Fmt);
    else AICOMP_LAUNCH_GRID16(Bf16Fmt);
#undef AICOMP_LAUNCH_GRID16
#undef AICOMP_LAUNCH_GRID32
#undef AICOMP_LAUNCH_GRID
    AICOMP_HIP_LAUNCH_CHECK();
    if (a.num_parts > 1) return launch_split_reduce(a);
    return AICOMP_KV_OK;
}

// Prefill of 16-bit queries on the decode tiles: `wgs` workgroups of the prefill kernel proper, of tile_pos positions each
// (what a pair of the item list names), would be too few.
int launch_prefill_rows(const DecodeArgs& a, int max_q_len, int tile_pos, int64_t wgs) {
    PrefillRowsParams p;
    p.out = a.out; p.query = a.query; p.k_pool = (void*)a.k_pool; p.v_pool = (void*)a.v_pool;
    p.block_table = a.block_table; p.block_table_stride = a.block_table_stride;
    p.context_lens = a.context_lens; p.cu_q_lens = a.cu_q_lens;
    const bool d64 = a.d == 64, fp8 = a.kv_dtype == AICOMP_KV_FP8_E4M3;
    const int rows = d64 ? 8 : 16;
    p.hq = a.hq; p.hkv = a.hkv; p.group = a.hq / a.hkv; p.max_blocks = a.max_blocks; p.num_blocks = a.num_blocks;
    p.gpack = rows % p.group == 0 ? p.group : 1;
    p.qk_mul = a.scale * LOG2E;
    p.k_scale = a.k_scale; p.v_scale = a.v_scale;
    p.items = a.items; p.num_seqs = a.num_seqs;
    const int pos = rows / p.gpack, groups = a.hq / p.gpack;
    p.sub = (tile_pos + pos - 1) / pos;
    const int tiles = (max_q_len + pos - 1) / pos;
    AICOMP_REQUIRE(tiles <= 65535 && tile_pos % pos == 0, AICOMP_KV_EINVAL, "paged_prefill_attn: grid too large");
    dim3 grid((unsigned)groups, (unsigned)a.num_seqs, (unsigned)tiles);
    if (a.items != nullptr) grid = dim3((unsigned)groups, (unsigned)a.num_items, (unsigned)p.sub);
    const bool wide = wgs <= 32;                     // (at D 64 always)
#define AICOMP_LAUNCH_ROWS(NW, ...)                                                                                          \
    hipLaunchKernelGGL((paged_prefill_rows_kernel<__VA_ARGS__, NW>), grid, dim3(64 * NW), 0, a.stream, p)
#define AICOMP_LAUNCH_ROWS16(E)                                                                                               \
    do {                                                                                                                      \
        if (d64) { if (fp8) AICOMP_LAUNCH_ROWS(8, Tile16<E, true, true, false>); else AICOMP_LAUNCH_ROWS(8, Tile16<E, false, true, false>); }        \
        else if (wide) { if (fp8) AICOMP_LAUNCH_ROWS(8, Tile16<E, true, false, false>); else AICOMP_LAUNCH_ROWS(8, Tile16<E, false, false, false>); } \
        else { if (fp8) AICOMP_LAUNCH_ROWS(4, Tile16<E, true, false, false>); else AICOMP_LAUNCH_ROWS(4, Tile16<E, false, false, false>); }          \
    } while (0)
    if (a.q_dtype == AICOMP_KV_F16) AICOMP_LAUNCH_ROWS16(F16Fmt); else AICOMP_LAUNCH_ROWS16(Bf16Fmt);
#undef AICOMP_LAUNCH_ROWS16
#undef AICOMP_LAUNCH_ROWS
    AICOMP_HIP_LAUNCH_CHECK();
    return AICOMP_KV_OK;
}

}  // namespace aicomp
