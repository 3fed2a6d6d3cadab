// Chunked-prefill causal attention for float32 models on gfx950's float32 matrix instruction.
//
// Replaces  F.scaled_dot_product_attention(query, full_key, full_value, attn_mask=None,
//           is_causal=True)                       opt_prime/opt_prime/kv_cache.py:404-415
// when the engine runs in float32 (examples/single_gpu_inference_llama.py:98-110, --dtype
// float32): queries, pools and output are float32, and every product and sum stays float32
// (v_mfma_f32_16x16x4_f32: D[16x16] += A[16x4] B[4x16], 2048 flop in 32 cycles per SIMD).  Same mask rule as the
// 16-bit kernel: query i of a chunk with prior context P sees keys j <= P + i.
//
// What bounds it: the float32 matrix instruction runs on the vector ALU's own multipliers, so every vector
// instruction of any wave of the SIMD takes its time from it (SQ_VALU_MFMA_COEXEC_CYCLES is 0).  A tile step of a wave
// is 128 products and had 185 other vector instructions: exp2f's range handling, a row max per tile, per-lane block ids
// and addresses, selects for masks that mask nothing.  It has 36: the hardware exponential, a max that moves only when
// a row's probabilities outgrow 2^8, block ids and tile addresses in scalar registers, masks behind branches.
//   us, 32/8 heads, before -> now     D 128                     D 64
//   2048 tokens                       309 -> 270 (127 TFLOP/s)  180 -> 153
//   4096                              1184 -> 1118              680 -> 582
//   512 after 1300                    118 -> 104                68 -> 58
// Products are busy 84 % of the first one's cycles; of 64 chunks of 32 tokens over 4000, 1112 -> 1005 us, 89 %.
//
// Work split   one workgroup (8 waves) per (128 query rows, sequence); a row is a (position,
//              head) pair, the G heads of one KV head packed per position when G divides 16, so a
//              K/V tile staged in LDS serves the whole group.  A wave owns 16 rows.
// Small grids  a row of tiles is a chain of steps on one CU, 3.5 us each, and a small grid leaves the other CUs idle.
//              There KW = 4 or 2 waves share the 16 rows and split the keys of a tile, a workgroup has 128 / KW rows, and
//              the waves' partial rows are added up through LDS at the end: KW times the workgroups, steps KW
//              times shorter (launch_prefill_mfma_f32 has the lines and both sides).
// K/V tiles    32 tokens (KW = 4: 64), global -> registers (one tile ahead) -> LDS, double-buffered, one barrier per
//              tile.  K rows of head_dim floats + 16 bytes, V rows unpadded: either operand read has every four lanes in
//              one 64-byte segment of a bank line and a half-wave in all four.
// S^T = K Q^T  A = K rows from LDS, B = the wave's query rows (registers, pre-multiplied by
//              scale * log2 e).  The k index of MFMA m in lane group g is 16 (m / 4) + 4 g + m % 4:
//              one 16-byte LDS read supplies the A operands of four MFMAs, read one group of products ahead.
// softmax      online, base 2, per lane one query.
// O^T += V^T P^T  A = V^T: lane (r, g) reads dims 64 half + 4 r .. + 3 of token 4 g + e, one 16-byte LDS read per four
//              MFMAs (a 4-byte read per MFMA before: 3 % more); B = P^T is exactly what the lane already holds.
#include "common.h"

#include <algorithm>
#include <atomic>

namespace aicomp {

namespace {

constexpr int BS = 16;
constexpr int WAVES = 8;
constexpr int NT = 64 * WAVES;
constexpr int WG_ROWS = 16 * WAVES;     // query rows per workgroup, where every wave has rows of its own
constexpr float NEG_BIG = -1.0e30f;
constexpr float LAZY = 256.f;           // sum of a lane's probabilities up to which a row's reference max stays

struct PrefillF32Params {
    float* out;
    const float* query;
    const float* k_pool;
    const float* v_pool;
    const int32_t* block_table;
    int64_t block_table_stride;
    const int32_t* context_lens;
    const int32_t* cu_q_lens;
    int hq, hkv, group, gpack, max_blocks;
    int num_blocks;
    int num_cus;                        // CUs of the device (0: expensive tiles first)
    float qk_mul;
    const int32_t* items;               // (sequence, query tile) pairs; grid.y numbers them (NULL: none)
    int num_seqs;
};

// KW: waves that share 16 query rows and split the keys of a tile (1: none do).
template <int DH, int KW>
__global__ void __launch_bounds__(NT, KW <= 2 ? 4 : 2)
paged_prefill_mfma_f32_kernel(PrefillF32Params p) {
    constexpr int HB = KW == 1 ? 2 : 1;         // 16-token blocks of a tile that a wave multiplies
    constexpr int KT = 16 * HB * KW;            // tokens per LDS tile
    constexpr int RW = WAVES / KW;              // waves with rows of their own
    constexpr int ROWS = 16 * RW;               // query rows per workgroup
    constexpr int KROW = DH * 4 + 16;           // LDS row stride in bytes
    constexpr int KROWF = KROW / 4;             // ... in floats
    constexpr int KTILE_F = KT * KROWF;         // floats per K tile
    constexpr int TILES_F = KTILE_F + KT * DH;  // ... and of a K and a V tile
    constexpr int HALVES = DH / 64;
    constexpr int NQ = DH / 16;                 // 16-element chunks of a row (QK: 4 MFMAs each; PV: output tiles)
    constexpr int CPR = DH / 4;                 // float4 chunks per row
    constexpr int RPL = NT / CPR;               // rows one load of the workgroup covers (16 or 32)
    constexpr int NL = KT / RPL;                // loads per tile and pool (2 or 1)
    const int hgroup = blockIdx.x;
    int seq = blockIdx.y;
    int64_t qtile = prefill_tile_of_slice(blockIdx.z, gridDim.z, p.num_cus, gridDim.x * gridDim.y);
    if (p.items != nullptr) {           // the caller's own order: workgroup row y takes pair y
        seq = p.items[2 * blockIdx.y];
        qtile = p.items[2 * blockIdx.y + 1];
        if (seq < 0 || seq >= p.num_seqs || qtile < 0) return;
        qtile = qtile * KW + (int)blockIdx.z;       // (a pair's tile is WG_ROWS rows)
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    const int pos_per_wg = ROWS / p.gpack;
    const int rw = KW == 1 ? w : w % RW;             // which rows
    const int key0 = KW == 1 ? 0 : 16 * HB * (w / RW);  // which keys of a tile

    extern __shared__ __attribute__((aligned(16))) float lds[];     // [2][K tile | V tile]

    const int q_begin = p.cu_q_lens[seq];
    const int n = p.cu_q_lens[seq + 1] - q_begin;
    const int ctx = min(p.context_lens[seq], p.max_blocks * BS);
    const int prior = ctx - n;
    if (qtile * pos_per_wg >= n || n <= 0) return;
    const int q0 = (int)qtile * pos_per_wg;
    if (prior < 0) {
        // a context shorter than the chunk itself: the rows are defined as zero, as in the other kernels
        for (int i = tid; i < ROWS * CPR; i += NT) {
            const int zrow = i / CPR, chunk = i % CPR;
            const int pos = q0 + zrow / p.gpack, hd = hgroup * p.gpack + zrow % p.gpack;
            if (pos < n)
                *(float4*)(p.out + ((int64_t)(q_begin + pos) * p.hq + hd) * DH + 4 * chunk) = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        return;
    }

    const int kvh = (hgroup * p.gpack) / p.group;
    const int row = 16 * rw + r16;
    const int qpos = q0 + row / p.gpack;
    const int head = hgroup * p.gpack + row % p.gpack;
    const bool row_valid = qpos < n;
    const int qabs = row_valid ? prior + qpos : ctx - 1;        // padded rows: computed, never stored
    // (a wave whose rows all lie beyond the chunk's end has nothing to compute: it only takes part in
    // the tile loads and barriers)
    const int wave_kv_end = q0 + (16 * rw) / p.gpack >= n ? 0 : min(ctx, prior + q0 + (16 * rw + 15) / p.gpack + 1);
    const int wave_kv_min = prior + q0 + (16 * rw) / p.gpack;
    const int kv_end = min(ctx, prior + q0 + pos_per_wg);
    const int ntiles = (kv_end + KT - 1) / KT;

    // Q as the B operand: MFMA 4 q + e of chunk q takes element 16 q + 4 g4 + e of this lane's row
    f32x4_t qf[NQ];
    const float* qrow = p.query + ((int64_t)(q_begin + min(qpos, n - 1)) * p.hq + head) * DH + 4 * g4;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        qf[q] = *(const f32x4_t*)(qrow + 16 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[q][e] *= p.qk_mul;
    }

    float m = NEG_BIG, lsum = 0.f;
    f32x4_t O[NQ];
#pragma unroll
    for (int j = 0; j < NQ; ++j) O[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int32_t* table = p.block_table + (int64_t)seq * p.block_table_stride;
    const int last_blk = (ctx - 1) >> 4;

    // global -> registers: load i of the workgroup covers rows RPL * i .. of the tile, this thread
    // one 16-byte chunk of one row.  Rows at or beyond the context read the last valid block
    // (their K scores are masked and their V rows zeroed when the tile is written to LDS).
    // The block ids are read one tile ahead of the rows, so that neither load is waited for where it is issued.
    // (Ext-vector types: arrays of float4 went to scratch memory, and a tile's loads were waited for at once:
    // 2048 tokens, 32/8 heads, D 128 371 us, now 326; 512 after 2048 257 and 230; D 64 192 and 187.)
    f32x4_t sk[NL], sv[NL];
    int blk[NL];
    const int trow = tid / CPR, tchunk = 4 * (tid % CPR);
    const int wrow = __builtin_amdgcn_readfirstlane(trow) & ~15;      // first row of the wave's block within a load
    const uint32_t in_block = (uint32_t)((trow & 15) * DH + tchunk);  // elements
    auto fetch_ids = [&](int t) {
#pragma unroll
        for (int i = 0; i < NL; ++i) blk[i] = table[min((t * KT + RPL * i + wrow) >> 4, last_blk)];
    };
    auto fetch = [&]() {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int64_t base = ((int64_t)max(0, min(blk[i], p.num_blocks - 1)) * p.hkv + kvh) * (BS * DH);
            sk[i] = *(const f32x4_t*)(p.k_pool + base + in_block);
            sv[i] = *(const f32x4_t*)(p.v_pool + base + in_block);
        }
    };
    auto stash = [&](int t, int buf) {
        float* kb = lds + buf * TILES_F + trow * KROWF + tchunk;
        float* vb = lds + buf * TILES_F + KTILE_F + trow * DH + tchunk;
        if ((t + 1) * KT > ctx) {                                       // the context's last tile
#pragma unroll
            for (int i = 0; i < NL; ++i)
                if (t * KT + RPL * i + trow >= ctx) sv[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            *(f32x4_t*)(kb + RPL * i * KROWF) = sk[i];
            *(f32x4_t*)(vb + RPL * i * DH) = sv[i];
        }
    };

    fetch_ids(0);
    fetch();
    fetch_ids(1);
    for (int t = 0; t < ntiles; ++t) {
        const int buf = t & 1;
        stash(t, buf);
        if (t + 1 < ntiles) {
            fetch();
            fetch_ids(t + 2);         // (beyond the context: the last block's)
        }
        __syncthreads();          // tile t visible; everyone is done with the buffer tile t + 1 will use
        const int tile_start = t * KT;
        const int first = tile_start + key0;
        if (first >= wave_kv_end) continue;                            // wave-uniform: above the diagonal
        const float* kb = lds + buf * TILES_F + key0 * KROWF;
        const float* vb = lds + buf * TILES_F + KTILE_F + key0 * DH;

        // ---- S^T = K Q^T for the wave's 16-token blocks of the tile
        f32x4_t sa[HB];
#pragma unroll
        for (int h = 0; h < HB; ++h) sa[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        f32x4_t ka[2][HB];
        auto read_k = [&](int q, f32x4_t (&x)[HB]) {
#pragma unroll
            for (int h = 0; h < HB; ++h) x[h] = *(const f32x4_t*)(kb + (16 * h + r16) * KROWF + 16 * q + 4 * g4);
        };
        read_k(0, ka[0]);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (q + 1 < NQ) read_k(q + 1, ka[(q + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < HB; ++h)
                    sa[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[q & 1][h][e], qf[q][e], sa[h], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }

        // ---- online softmax: lane (query r16, g4) holds tokens first + 16 h + 4 g4 + i.  The reference max m moves only
        // when a lane's probabilities of this tile add up to more than LAZY (always on a row's first tile), for all
        // rows of the wave together: a lane's sum over a tile stays at most 2^8.  (Not the same floats as under the true
        // max, which is further from m by some real number, but of the same relative error.)
        if (first + 16 * HB - 1 > wave_kv_min) {                       // wave-uniform
#pragma unroll
            for (int k = 0; k < 4 * HB; ++k)
                if (first + 16 * (k >> 2) + 4 * g4 + (k & 3) > qabs) sa[k >> 2][k & 3] = -INFINITY;
        }
        float pr[4 * HB], psum = 0.f;
#pragma unroll
        for (int k = 0; k < 4 * HB; ++k) {
            pr[k] = __builtin_amdgcn_exp2f(sa[k >> 2][k & 3] - m);
            psum += pr[k];
        }
        if (__any(!(psum <= LAZY))) {
            float mx = sa[0][0];
#pragma unroll
            for (int k = 1; k < 4 * HB; ++k) mx = fmaxf(mx, sa[k >> 2][k & 3]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = fmaxf(m, mx);
            const float alpha = __builtin_amdgcn_exp2f(m - m_new);
            psum = 0.f;
#pragma unroll
            for (int k = 0; k < 4 * HB; ++k) {
                pr[k] = __builtin_amdgcn_exp2f(sa[k >> 2][k & 3] - m_new);
                psum += pr[k];
            }
            lsum *= alpha;
            m = m_new;
#pragma unroll
            for (int j = 0; j < NQ; ++j) O[j] *= alpha;
        }
        lsum += psum;

        // ---- O^T += V^T P^T: A = V[token 16 h + 4 g4 + e][dims 64 half + 4 r16 + x], B = this lane's own P values
        f32x4_t va[2][HALVES];
        auto read_v = [&](int t8, f32x4_t (&x)[HALVES]) {
#pragma unroll
            for (int f = 0; f < HALVES; ++f)
                x[f] = *(const f32x4_t*)(vb + (16 * (t8 >> 2) + 4 * g4 + (t8 & 3)) * DH + 64 * f + 4 * r16);
        };
        read_v(0, va[0]);
#pragma unroll
        for (int t8 = 0; t8 < 4 * HB; ++t8) {
            if (t8 + 1 < 4 * HB) read_v(t8 + 1, va[(t8 + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < HALVES; ++f)
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    O[4 * f + x] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[t8 & 1][f][x], pr[t8], O[4 * f + x], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // lane (query r16, g4) holds O^T[dim 64 half + 16 g4 + 4 i + x][query] in O[4 half + x][i]
    float l = lsum;
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if constexpr (KW > 1) {
        // the waves of a row add up through LDS: row r of wave w at part + (16 w + r) * OROW, its (max, sum) behind the rows
        constexpr int OROW = DH + 4;
        float* part = lds;
        float* ml = lds + WAVES * 16 * OROW;
        __syncthreads();                                               // everyone is done with the tiles
#pragma unroll
        for (int f = 0; f < HALVES; ++f)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(float4*)(part + (16 * w + r16) * OROW + 64 * f + 16 * g4 + 4 * i) =
                    make_float4(O[4 * f][i], O[4 * f + 1][i], O[4 * f + 2][i], O[4 * f + 3][i]);
        if (g4 == 0) { ml[2 * (16 * w + r16)] = m; ml[2 * (16 * w + r16) + 1] = l; }
        __syncthreads();
        for (int i = tid; i < ROWS * CPR; i += NT) {
            const int orow = i / CPR, chunk = 4 * (i % CPR);
            const int pos = q0 + orow / p.gpack, hd = hgroup * p.gpack + orow % p.gpack;
            if (pos >= n) continue;
            float mx = NEG_BIG, den = 0.f;
#pragma unroll
            for (int k = 0; k < KW; ++k) mx = fmaxf(mx, ml[2 * (k * ROWS + orow)]);
            f32x4_t num = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KW; ++k) {
                const int r = k * ROWS + orow;                         // 16 w + row within the wave, w = k RW + its row wave
                const float f = __builtin_amdgcn_exp2f(ml[2 * r] - mx);
                den = fmaf(f, ml[2 * r + 1], den);
                num += f * *(const f32x4_t*)(part + r * OROW + chunk);
            }
            const float inv = den > 0.f ? 1.f / den : 0.f;
            *(f32x4_t*)(p.out + ((int64_t)(q_begin + pos) * p.hq + hd) * DH + chunk) = num * inv;
        }
        return;
    }
    // As they lie, the four lanes of a row would each write 16 bytes of four 64-byte segments.  Transposed over them (lane
    // group and i change places: swaps of the halves of the wave, then of its odd and even rows) they write one segment.
    // Of short fresh chunks the output is most of the bytes: 13 of 46, D 128 18.2 -> 17.0 us, D 64 11.2 -> 10.3;
    // 32 of 24, 64/8 heads, D 128 25.8 -> 24.1.
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(O[j][0]), __float_as_uint(O[j][2]), false, false);
        const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(O[j][1]), __float_as_uint(O[j][3]), false, false);
        const auto a = __builtin_amdgcn_permlane16_swap(u[0], v[0], false, false);
        const auto b = __builtin_amdgcn_permlane16_swap(u[1], v[1], false, false);
        O[j] = f32x4_t{__uint_as_float(a[0]), __uint_as_float(a[1]), __uint_as_float(b[0]), __uint_as_float(b[1])};
    }
    if (row_valid) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        float* o = p.out + ((int64_t)(q_begin + qpos) * p.hq + head) * DH + 4 * g4;
#pragma unroll
        for (int f = 0; f < HALVES; ++f)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(float4*)(o + 64 * f + 16 * i) =
                    make_float4(O[4 * f][i] * inv, O[4 * f + 1][i] * inv, O[4 * f + 2][i] * inv, O[4 * f + 3][i] * inv);
    }
}

template <int DH, int KW>
hipError_t launch_f32_variant(const PrefillF32Params& p, dim3 grid, hipStream_t stream) {
    // two buffers of a K and a V tile, where the waves of a row then leave their partial rows and (max, sum)
    constexpr size_t tiles = (size_t)2 * (KW <= 2 ? 32 : 16 * KW) * (2 * DH * 4 + 16);
    constexpr size_t rows = KW == 1 ? 0 : (size_t)WAVES * 16 * (DH + 4 + 2) * 4;
    constexpr size_t lds_bytes = tiles > rows ? tiles : rows;
    if (lds_bytes > 64 * 1024) {
        // above the 64 KB a kernel may use without asking: a per-device function attribute, set once
        static std::atomic<unsigned long long> done{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (!(dev < 64 && ((done.load(std::memory_order_acquire) >> dev) & 1ull))) {
            e = hipFuncSetAttribute((const void*)paged_prefill_mfma_f32_kernel<DH, KW>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
            if (e != hipSuccess) return e;
            if (dev < 64) done.fetch_or(1ull << dev, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL((paged_prefill_mfma_f32_kernel<DH, KW>), grid, dim3(NT), lds_bytes, stream, p);
    return hipSuccess;
}

}  // namespace

bool prefill_mfma_f32_supported(const DecodeArgs& a, int max_q_len) {
    return a.cu_q_lens != nullptr && max_q_len > 0 && a.q_dtype == AICOMP_KV_F32 && a.kv_dtype == AICOMP_KV_F32 &&
           (a.d == 128 || a.d == 64) && a.bs == BS && a.hkv > 0 && a.hq % a.hkv == 0 && a.scale > 0.f &&
           a.num_seqs <= 65535 && a.num_blocks <= INT32_MAX && ((uintptr_t)a.query % 16 == 0) &&
           ((uintptr_t)a.out % 16 == 0) && ((uintptr_t)a.k_pool % 16 == 0) && ((uintptr_t)a.v_pool % 16 == 0);
}

int prefill_mfma_f32_tile_positions(int hq, int hkv) {
    const int group = hq / hkv;
    return WG_ROWS / ((16 % group == 0) ? group : 1);
}

int launch_prefill_mfma_f32(const DecodeArgs& a, int max_q_len) {
    PrefillF32Params p;
    p.out = (float*)a.out; p.query = (const float*)a.query;
    p.k_pool = (const float*)a.k_pool; p.v_pool = (const float*)a.v_pool;
    p.block_table = a.block_table; p.block_table_stride = a.block_table_stride;
    p.context_lens = a.context_lens; p.cu_q_lens = a.cu_q_lens;
    p.hq = a.hq; p.hkv = a.hkv; p.group = a.hq / a.hkv; p.max_blocks = a.max_blocks;
    p.num_blocks = (int)a.num_blocks;
    p.gpack = (16 % p.group == 0) ? p.group : 1;
    p.qk_mul = a.scale * LOG2E;
    // CU count of the first device used (every GPU of a node is the same part); 0 if unknown
    static std::atomic<int> cached_cus{-1};
    int num_cus = cached_cus.load(std::memory_order_relaxed);
    if (num_cus < 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 0)
            n = 0;
        num_cus = n;
        cached_cus.store(n, std::memory_order_relaxed);
    }
    p.num_cus = num_cus;
    p.items = a.items; p.num_seqs = a.num_seqs;
    const int groups = a.hq / p.gpack, pos_per_wg = WG_ROWS / p.gpack;
    // workgroups of `share` waves per row, from what the host knows (all rows, the longest chunk): the same with and
    // without a list of items, whose pairs name tiles of 128 rows
    const auto workgroups = [&](int share) {
        const int64_t pos = pos_per_wg / share, tiles = (max_q_len + pos - 1) / pos;
        return groups * std::min(tiles * a.num_seqs, a.rows / pos + a.num_seqs);
    };
    // Waves that share rows (us, 32/8 heads, D 128, with 1 / 2 / 4 of them; in brackets the workgroups of 128 rows):
    //   8 chunks of 32 over 2000 (64)    262 /     /  94    one of 400 over 1024 (104)   188 / 110 / 113
    //   one prompt of 512 (128)           73 /     /  31    one of 1024 (256)           143 /  88 / 110
    //   48 of 32 over 1000 (384)         269 / 232 /        one of 1600 (400)           223 / 201 /
    //   32 of 32 over 1000 (256)         152 / 154 / 188    one of 2048 (512)           280 / 318 /
    //   11 of 9 to 38 over up to 431 (176) 72 / 40 /
    // Two of them also even out what CUs get in a causal prompt; beyond 400 the larger K/V traffic and a second round
    // cost more.  Many chunks have tiles alike, with nothing to even out: there workgroups beyond one per CU only wait
    // for each other, whatever the prior contexts (in brackets the workgroups with 1 / 2 / 4):
    //   8 of 46   (128 / 192 / 384)  14.6 / 13.7 / 18.4   over 1024  145 / 87 / 100
    //   16 of 24  (128 / 256 / 384)  13.9 / 12.2 / 17.5   over 1024  143 / 85 / 102
    //   13 of 46  (208 / 312 / 624)  17.0 / 19.1 / 25.6   over 256    51 / 53 / 58
    //   8 of 70   (192 / 320 / 576)  20.1 / 22.6 / 23.9   over 64     29 / 31 / 33
    const int64_t wgs = workgroups(1);
    int kw = wgs <= 128 ? 4 : wgs <= 400 ? 2 : 1;
    if (a.num_seqs >= 8) {
        if (kw == 4 && workgroups(4) > 256) kw = 2;
        else if (kw == 2 && wgs <= 256 && workgroups(2) > 256) kw = 1;
    }
    const int pos = pos_per_wg / kw;
    const int qtiles = (max_q_len + pos - 1) / pos;
    AICOMP_REQUIRE(qtiles <= 65535, AICOMP_KV_EINVAL, "paged_prefill_attn: grid too large");
    dim3 grid((unsigned)groups, (unsigned)a.num_seqs, (unsigned)qtiles);
    if (a.items != nullptr) grid = dim3((unsigned)groups, (unsigned)a.num_items, (unsigned)kw);
    const bool d64 = a.d == 64;
    const hipError_t e = kw == 4   ? (d64 ? launch_f32_variant<64, 4>(p, grid, a.stream) : launch_f32_variant<128, 4>(p, grid, a.stream))
                         : kw == 2 ? (d64 ? launch_f32_variant<64, 2>(p, grid, a.stream) : launch_f32_variant<128, 2>(p, grid, a.stream))
                                   : (d64 ? launch_f32_variant<64, 1>(p, grid, a.stream) : launch_f32_variant<128, 1>(p, grid, a.stream));
    AICOMP_REQUIRE(e == hipSuccess, AICOMP_KV_EHIP, "paged_prefill_attn: %s", hipGetErrorString(e));
    AICOMP_HIP_LAUNCH_CHECK();
    return AICOMP_KV_OK;
}

}  // namespace aicomp
