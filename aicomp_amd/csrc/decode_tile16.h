// Decode tiles of 16-bit queries: 32 rows of 128 elements that one wave loads, scores and sums up by itself.  Included, in
// the kernels' own namespace, by the decode kernels and by the prefill kernel (whose one-token rows stream through them).
#pragma once

constexpr int D = 128;
constexpr int BS = 16;
constexpr int TILE = 32;               // tokens per wave iteration (two blocks)
constexpr int NWAVES = 4;
constexpr int KROW = 256;              // LDS row stride in bytes: unpadded, 16-byte chunks swizzled (below)
constexpr int KTILE_BYTES = TILE * KROW;   // 8192 per wave
constexpr float NEG_BIG = -1.0e30f;
template <bool FP8> struct TileRegs;
template <> struct TileRegs<false> { uint4 r[8]; };
template <> struct TileRegs<true> { uint2 r[8]; };

// Issue the 8 loads of one 32-token tile of one pool.  blk0/blk1 are the two
// physical blocks (wave-uniform); lane l reads row l/16, chunk l%16 of each
// 4-row group.
// K/V rows are read exactly once per call: non-temporal loads keep them from displacing
// everything else in L2 (measured: 114 -> 101 us on the Llama-3-8B decode shape).
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
// (ONCE; prefill's workgroups share their rows and keep them in L2)
template <bool ONCE = true>
__device__ __forceinline__ uint4 tile_ld(const uint4* p) {
    u32x4_t v;
    if constexpr (ONCE) v = __builtin_nontemporal_load((const u32x4_t*)p); else v = *(const u32x4_t*)p;
    return make_uint4(v[0], v[1], v[2], v[3]);
}
template <bool ONCE = true>
__device__ __forceinline__ uint2 tile_ld(const uint2* p) {
    u32x2_t v;
    if constexpr (ONCE) v = __builtin_nontemporal_load((const u32x2_t*)p); else v = *(const u32x2_t*)p;
    return make_uint2(v[0], v[1]);
}
#define TILE_LD(ptr) tile_ld<ONCE>(ptr)
template <bool FP8, bool ONCE>
__device__ __forceinline__ void load_tile(TileRegs<FP8>& t, const void* pool, int64_t blk0,
                                          int64_t blk1, int hkv, int kvh, int lane) {
    if constexpr (FP8) {
        const uint2* p0 = (const uint2*)pool + (blk0 * hkv + kvh) * (BS * D / 8) + lane;
        const uint2* p1 = (const uint2*)pool + (blk1 * hkv + kvh) * (BS * D / 8) + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            t.r[i] = TILE_LD(p0 + i * 64);
            t.r[4 + i] = TILE_LD(p1 + i * 64);
        }
    } else {
        const uint4* p0 = (const uint4*)pool + (blk0 * hkv + kvh) * (BS * D / 8) + lane;
        const uint4* p1 = (const uint4*)pool + (blk1 * hkv + kvh) * (BS * D / 8) + lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            t.r[i] = TILE_LD(p0 + i * 64);
            t.r[4 + i] = TILE_LD(p1 + i * 64);
        }
    }
}

// head_dim 64: a 32-row tile of 128-element rows is 64 tokens, each row a PAIR of consecutive
// tokens (token 2r in elements 0..63, token 2r+1 in 64..127; contiguous in the pool).  Four
// blocks of 8 such rows.
template <bool FP8, bool ONCE>
__device__ __forceinline__ void load_tile_pair(TileRegs<FP8>& t, const void* pool, int64_t blk0, int64_t blk1,
                                               int64_t blk2, int64_t blk3, int hkv, int kvh, int lane) {
    const int64_t blk[4] = {blk0, blk1, blk2, blk3};
    if constexpr (FP8) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint2* p = (const uint2*)pool + (blk[b] * hkv + kvh) * (BS * 64 / 8) + lane;
            t.r[2 * b] = TILE_LD(p);
            t.r[2 * b + 1] = TILE_LD(p + 64);
        }
    } else {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint4* p = (const uint4*)pool + (blk[b] * hkv + kvh) * (BS * 64 / 8) + lane;
            t.r[2 * b] = TILE_LD(p);
            t.r[2 * b + 1] = TILE_LD(p + 64);
        }
    }
}

// load i of a tile as eight elements of the query's 16-bit format E (fp8 pools are widened, exactly)
template <typename E, bool FP8>
__device__ __forceinline__ uint4 tile_elems(const TileRegs<FP8>& t, int i) {
    if constexpr (FP8) return E::from_fp8(t.r[i]);
    else return t.r[i];
}

__device__ __forceinline__ int64_t clamp_block(int b, int64_t num_blocks) {
    return b < 0 ? 0 : (b >= num_blocks ? num_blocks - 1 : (int64_t)b);
}

// Where a lane writes and reads the wave's K tile.  Chunk slot s of tile row r holds the row's
// chunk s ^ swz(r), swz(r) = ((r / 4) % 4) | ((r % 4) * 4): the operand read below then has every
// four consecutive lanes in one aligned 64-byte segment and each half-wave spread evenly over the
// four segments of a 256-byte bank line, which is what the LDS needs to deliver 256 bytes per
// clock (rows padded to 272 bytes are free of bank collisions among the sixteen lanes of an MFMA
// row group, yet run at half that rate: a quarter of the LDS cycles were conflict cycles).
//   write  load i of lane (q = lane / 16, c = lane % 16) is row 4 i + q, chunk c:
//          swz = (i % 4) | (q * 4), so four distinct offsets, picked by i % 4
//   read   sub-tile a, k-step s, lane (r16, g4): row 16 a + 4 (r16 % 4) + r16 / 4, chunk 4 s + g4:
//          swz of that row is r16 itself, so the slot is (4 s + g4) ^ r16
struct KTileOffsets {
    int wr[4];
    int rd[4];
};
__device__ __forceinline__ KTileOffsets k_tile_offsets(int lane) {
    const int r16 = lane & 15, g4 = lane >> 4;
    KTileOffsets o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        o.wr[k] = g4 * KROW + ((r16 ^ (k | (g4 << 2))) << 4);
        o.rd[k] = (4 * (r16 & 3) + (r16 >> 2)) * KROW + (((4 * k + g4) ^ r16) << 4);
    }
    return o;
}

// Per-wave running state of the online softmax and the output accumulators.
template <int NO>
struct WaveStateT {
    float m, lsum;
    f32x4_t O[NO];
};
typedef WaveStateT<8> WaveState;
template <int NO>
__device__ __forceinline__ void clear_state(WaveStateT<NO>& st) {
    st.m = NEG_BIG; st.lsum = 0.f;
#pragma unroll
    for (int j = 0; j < NO; ++j) st.O[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// One 32-token tile: K registers -> LDS -> S^T = K Q^T -> online softmax -> O^T += V^T P^T.
// NEXT: prefetch the wave's next tile (blocks nb0/nb1) into the same registers.
// MASK: the tile crosses `end` (of this lane's column) or `v_end` (of all); scores beyond the one are dropped, V rows
// beyond the other zeroed.
// PAIR: rows are token pairs (head_dim 64): row r of the tile holds tokens tile_start + 2r and
// + 2r + 1, the B-operand columns are (head, parity) pairs, column c scoring token 2r + (c & 1).
// ONCE (a decode row, which sees both tokens of a pair): the two share every dot product, the query column being zero
// over the other token's half.  Rows of a chunk need not see the second token, and 0 times its key is NaN where that is
// not finite: there each half of a row is summed by itself and a column takes its own (as many products).
// LEAN (one-token rows in the prefill kernel): fewer registers; and a key of -inf has no weight, as in that kernel's other
// rows, where in a shared product it would leave NaN in the other token's score.
template <typename E, bool FP8, bool NEXT, bool MASK, bool PAIR, bool ONCE, bool LEAN>
__device__ __forceinline__ void process_tile(WaveState& st, TileRegs<FP8>& kr, TileRegs<FP8>& vr,
                                             const uint4 (&qf)[4], unsigned char* kt, const KTileOffsets& ko,
                                             const void* k_pool, const void* v_pool,
                                             int64_t nb0, int64_t nb1, int hkv, int kvh_next, int lane,
                                             int g4, int tile_start, int end, int v_end, float cmul,
                                             int64_t nb2 = 0, int64_t nb3 = 0) {
    constexpr bool HALVES = PAIR && (!ONCE || LEAN);     // a row's score summed over either half by itself
    // ---- K tile -> LDS, then prefetch the next K tile into the same registers
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint4 kk = tile_elems<E, FP8>(kr, i);
        // PAIR, one dot product for a row's two tokens: a token beyond the context must not leave non-finite
        // values in the row
        if (PAIR && !HALVES && MASK && tile_start + 2 * (4 * i + g4) + ((lane & 15) >> 3) >= v_end) kk = make_uint4(0, 0, 0, 0);
        *(uint4*)(kt + ko.wr[i & 3] + i * 4 * KROW) = kk;
    }
    if (NEXT) {
        if constexpr (PAIR) load_tile_pair<FP8, ONCE>(kr, k_pool, nb0, nb1, nb2, nb3, hkv, kvh_next, lane);
        else load_tile<FP8, ONCE>(kr, k_pool, nb0, nb1, hkv, kvh_next, lane);
    }

    // ---- S^T = K Q^T for the two 16-token sub-tiles
    constexpr int NH = HALVES ? 2 : 1;                   // sums of a row's score: its halves, or one
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f}, t0 = s0, t1 = s1;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint4 a0 = *(const uint4*)(kt + ko.rd[s]);
        const uint4 a1 = *(const uint4*)(kt + ko.rd[s] + 16 * KROW);
        f32x4_t &x0 = NH == 2 && s >= 2 ? t0 : s0, &x1 = NH == 2 && s >= 2 ? t1 : s1;
        x0 = E::mfma(a0, qf[s], x0);
        x1 = E::mfma(a1, qf[s], x1);
    }
    if constexpr (NH == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s0[i] = lane & 1 ? t0[i] : s0[i];
            s1[i] = lane & 1 ? t1[i] : s1[i];
        }
    }
    // lane (head r16, g4) now holds tokens tile_start + 16a + 4i + g4 in s_a[i]
    float sc[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) { sc[i] = s0[i] * cmul; sc[4 + i] = s1[i] * cmul; }
    if (MASK) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = 16 * (k >> 2) + 4 * (k & 3) + g4;
            const int tok = PAIR ? tile_start + 2 * r + (lane & 1) : tile_start + r;
            if (tok >= end) sc[k] = NEG_BIG;
        }
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])),
                     fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
    // A tile of a short row is a chain of latencies, of which two shuffles through LDS and the range handling of exp2f were a
    // tenth: one row of 500 tokens, D 64 5.82 -> 5.62 us, D 128 6.86 -> 6.40, 16 rows of 700, 16 / 2 heads 11.4 -> 10.9;
    // rows that stream as before.  (exp2f and the bare instruction differ below 2^-126 alone, which leaves it as 0.)
    mx = xor32_max(xor16_max(mx));
    const float m_new = fmaxf(st.m, mx);
    const float alpha = __builtin_amdgcn_exp2f(st.m - m_new);
    float pr[8], psum = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        pr[k] = __builtin_amdgcn_exp2f(sc[k] - m_new);
        // (by its bits: a comparison of floats may take a NaN for anything where they are compiled not to occur)
        if (MASK && __builtin_bit_cast(uint32_t, sc[k]) == __builtin_bit_cast(uint32_t, NEG_BIG)) pr[k] = 0.f;
        psum += pr[k];
    }
    st.lsum = st.lsum * alpha + psum;
    st.m = m_new;
    if (__any(alpha != 1.f)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) st.O[j] *= alpha;
    }
    // P^T as the B operand: k-slot 4a + i <-> token 16a + 4i + g4, this lane's own values
    uint4 pw;
    pw.x = E::pack(pr[0], pr[1]); pw.y = E::pack(pr[2], pr[3]);
    pw.z = E::pack(pr[4], pr[5]); pw.w = E::pack(pr[6], pr[7]);

    // ---- V: registers -> A operand of O^T += V^T P^T.  Load i of lane (c, q) is token 4i + q.
    uint4 vv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        vv[i] = tile_elems<E, FP8>(vr, i);
        // PAIR: chunks 8..15 of a row belong to the pair's second token
        const int vtok = PAIR ? tile_start + 2 * (4 * i + g4) + ((lane & 15) >> 3) : tile_start + 4 * i + g4;
        if (MASK && vtok >= v_end) vv[i] = make_uint4(0, 0, 0, 0);
    }
    auto operand = [&](int j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        const uint32_t* v0 = (const uint32_t*)&vv[0];
        return make_uint4(__builtin_amdgcn_perm(v0[4 * 1 + (j >> 1)], v0[4 * 0 + (j >> 1)], sel),
                          __builtin_amdgcn_perm(v0[4 * 3 + (j >> 1)], v0[4 * 2 + (j >> 1)], sel),
                          __builtin_amdgcn_perm(v0[4 * 5 + (j >> 1)], v0[4 * 4 + (j >> 1)], sel),
                          __builtin_amdgcn_perm(v0[4 * 7 + (j >> 1)], v0[4 * 6 + (j >> 1)], sel));
    };
    uint4 af[8];
    if constexpr (LEAN) {
        // half of the operands are used up before the other half is made: sixteen registers fewer while the next V tile is on
        // its way, for a kernel whose other path holds three waves per SIMD
#pragma unroll
        for (int j = 0; j < 4; ++j) af[j] = operand(j);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) st.O[j] = E::mfma(af[j], pw, st.O[j]);
    }
#pragma unroll
    for (int j = LEAN ? 4 : 0; j < 8; ++j) af[j] = operand(j);
    if constexpr (LEAN) __builtin_amdgcn_sched_barrier(0);
    if (NEXT) {
        if constexpr (PAIR) load_tile_pair<FP8, ONCE>(vr, v_pool, nb0, nb1, nb2, nb3, hkv, kvh_next, lane);
        else load_tile<FP8, ONCE>(vr, v_pool, nb0, nb1, hkv, kvh_next, lane);
    }
#pragma unroll
    for (int j = LEAN ? 4 : 0; j < 8; ++j) st.O[j] = E::mfma(af[j], pw, st.O[j]);
}

// 8 elements of format E -> 8 e4m3 codes: clamp(x / scale, +-448), round to nearest even
template <typename E>
__device__ __forceinline__ uint2 quant8_fp8(const uint4& x, float scale) {
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = fminf(fmaxf(E::to_f32((uint16_t)(w[i] & 0xffffu)) / scale, -448.f), 448.f);
        f[2 * i + 1] = fminf(fmaxf(E::to_f32((uint16_t)(w[i] >> 16)) / scale, -448.f), 448.f);
    }
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
    return make_uint2((uint32_t)lo, (uint32_t)hi);
}

// Fused append: the tile that holds the sequence's newest token (context_lens - 1) takes its K/V
// row from new_key / new_value instead of what was loaded from the pool, and writes it to the pool
// (the append itself).  No other wave of the launch reads that token, so no cross-wave ordering is
// needed.  A tile row is one token (16 lanes of 8 elements), or with PAIR half a row (8 lanes).
template <typename E, bool FP8, bool PAIR, typename Params>
__device__ __forceinline__ void inject_new_row(TileRegs<FP8>& kr, TileRegs<FP8>& vr, const Params& p,
                                               const uint16_t* key, const uint16_t* value, int kvh, int lane,
                                               int tile_start, int len, const int64_t (&bb)[4]) {
    constexpr int DQ = PAIR ? 64 : D;
    const int tau = len - 1 - tile_start;              // token within the tile, wave-uniform
    const int blk_i = tau >> 4, tb = tau & 15;         // block of the tile, token within the block
    const int c = PAIR ? (lane & 7) : (lane & 15);     // 8-element chunk of the new row this lane holds
    // register slot and lanes of that token: load i of lane l is row 4i + l/16 (chunk l%16) of the tile
    const int row = PAIR ? (tau >> 1) : tau;
    const bool mine = (lane >> 4) == (row & 3) && (!PAIR || ((lane >> 3) & 1) == (tau & 1));
    const int slot = row >> 2;
    const uint4 nk = *(const uint4*)(key + 8 * c);
    const uint4 nv = *(const uint4*)(value + 8 * c);
    const int64_t blk = bb[blk_i];
    const int64_t dst = ((blk * p.hkv + kvh) * BS + tb) * (DQ / 8) + c;        // 8-element chunks
    if constexpr (FP8) {
        const uint2 ck = quant8_fp8<E>(nk, p.k_scale[kvh]);
        const uint2 cv = quant8_fp8<E>(nv, p.v_scale[kvh]);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (mine && i == slot) { kr.r[i] = ck; vr.r[i] = cv; }
        if (mine) { ((uint2*)p.k_pool)[dst] = ck; ((uint2*)p.v_pool)[dst] = cv; }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (mine && i == slot) { kr.r[i] = nk; vr.r[i] = nv; }
        if (mine) { ((uint4*)p.k_pool)[dst] = nk; ((uint4*)p.v_pool)[dst] = nv; }
    }
}

// ---------------------------------------------------------------------------------------
// What a schedule needs to know about the tiles it walks: the two kernels below are written over
// one of these.  A tile is TT tokens of one KV head, BPT blocks, 8 KB of K and 8 KB of V per wave
// (half of that for fp8), loaded with eight loads of each.
// Tile16: 16-bit queries E over pools of E or fp8, head_dim 128, or 64 as rows of token pairs.
template <typename E, bool FP8_, bool PAIR_, bool ONCE = true, bool LEAN = false>
struct Tile16 {
    typedef E Fmt;
    static constexpr bool FP8 = FP8_, PAIR = PAIR_, QUAD = false;
    static constexpr int DQ = PAIR ? 64 : D;             // head_dim of the tensors
    static constexpr int TT = PAIR ? 2 * TILE : TILE;    // tokens per tile
    static constexpr int BPT = TT / BS;                  // blocks per tile
    static constexpr int OROW = D;                       // floats per B column of the accumulators
    static constexpr int NPAR = PAIR ? 2 : 1;            // B columns per query head
    typedef WaveState State;
    typedef KTileOffsets Offsets;
    struct Q { uint4 r[4]; };
    struct Regs { TileRegs<FP8> k, v; };
    __device__ __forceinline__ static Offsets offsets(int lane) { return k_tile_offsets(lane); }

    // raw query rows of a (sequence, KV head), one after the other; columns beyond the group are zeroed by q_operand only
    // when the rows are used, so that issuing the loads never waits for them.
    // PAIR: column c = (head c / 2, parity c % 2): k-slot s covers row elements 32s + 8 g4 .., which are
    // the query's elements (32s + 8 g4) % 64 when the slot lies in the column's own half of the row.
    __device__ __forceinline__ static void load_q(Q& q, const uint16_t* rows, int group, int lane) {
        const int r16 = lane & 15, h = PAIR ? (r16 >> 1) : r16;
        load_q_row(q, rows + min(h, group - 1) * DQ, lane);
    }
    __device__ __forceinline__ static void load_q_row(Q& q, const uint16_t* row, int lane) {      // the row of the lane's column
        const int g4 = lane >> 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) q.r[s] = *(const uint4*)(row + (PAIR ? ((32 * s + 8 * g4) & 63) : 32 * s + 8 * g4));
    }
    __device__ __forceinline__ static void q_operand(Q& q, const Q& raw, int group, int lane) {
        const int r16 = lane & 15, g4 = lane >> 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            bool use = r16 < NPAR * group;
            if constexpr (PAIR) use = use && ((32 * s + 8 * g4 >= 64) == ((r16 & 1) != 0));
            q.r[s] = use ? raw.r[s] : make_uint4(0, 0, 0, 0);
        }
    }
    template <typename Params>
    __device__ __forceinline__ static void load(Regs& t, const Params& p, const int64_t (&bb)[4], int kvh, int lane) {
        if constexpr (PAIR) {
            load_tile_pair<FP8, ONCE>(t.k, p.k_pool, bb[0], bb[1], bb[2], bb[3], p.hkv, kvh, lane);
            load_tile_pair<FP8, ONCE>(t.v, p.v_pool, bb[0], bb[1], bb[2], bb[3], p.hkv, kvh, lane);
        } else {
            load_tile<FP8, ONCE>(t.k, p.k_pool, bb[0], bb[1], p.hkv, kvh, lane);
            load_tile<FP8, ONCE>(t.v, p.v_pool, bb[0], bb[1], p.hkv, kvh, lane);
        }
    }
    template <bool NEXT, bool MASK, typename Params>
    __device__ __forceinline__ static void process(State& st, Regs& t, const Q& q, unsigned char* kt, const Offsets& ko,
                                                   const Params& p, const int64_t (&nb)[4], int kvh_next, int lane,
                                                   int tile_start, int end, float cmul) {
        process_rows<NEXT, MASK>(st, t, q, kt, ko, p, nb, kvh_next, lane, tile_start, end, end, cmul);
    }
    // columns with ends of their own (rows of a chunk)
    template <bool NEXT, bool MASK, typename Params>
    __device__ __forceinline__ static void process_rows(State& st, Regs& t, const Q& q, unsigned char* kt, const Offsets& ko,
                                                        const Params& p, const int64_t (&nb)[4], int kvh_next, int lane,
                                                        int tile_start, int end, int v_end, float cmul) {
        process_tile<E, FP8, NEXT, MASK, PAIR, ONCE, LEAN>(st, t.k, t.v, q.r, kt, ko, p.k_pool, p.v_pool, nb[0], nb[1], p.hkv,
                                               kvh_next, lane, lane >> 4, tile_start, end, v_end, cmul, nb[2], nb[3]);
    }
    template <typename Params>
    __device__ __forceinline__ static void inject(Regs& t, const Params& p, const uint16_t* key, const uint16_t* value,
                                                  int kvh, int lane, int tile_start, int len, const int64_t (&bb)[4]) {
        inject_new_row<E, FP8, PAIR>(t.k, t.v, p, key, value, kvh, lane, tile_start, len, bb);
    }
    // this lane's accumulators into the row of its column: elements 32 g4 + 8 i + j from O[j][i]
    __device__ __forceinline__ static void store_acc(float* row, const State& st, int g4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float* dst = row + 32 * g4 + 8 * i;
            *(float4*)dst = make_float4(st.O[0][i], st.O[1][i], st.O[2][i], st.O[3][i]);
            *(float4*)(dst + 4) = make_float4(st.O[4][i], st.O[5][i], st.O[6][i], st.O[7][i]);
        }
    }
};

// Where wave w left its accumulator rows: the waves' tiles one after the other, or a function of w.
__device__ __forceinline__ const float* wave_rows(const unsigned char* lds, int w) { return (const float*)(lds + w * KTILE_BYTES); }
template <typename F>
__device__ __forceinline__ const float* wave_rows(const F& kt_of, int w) { return (const float*)kt_of(w); }

// Dim dd of row h over a workgroup's waves: its max, weighted sum and weight (PAIR: over the two parity columns of the
// row too, whose useful halves are elements 0..63 and 64..127 of their accumulators).
template <typename T, int NW, typename Acc>
__device__ __forceinline__ void merge_waves(Acc acc, const float (&sm_m)[NW][16], const float (&sm_l)[NW][16], int h, int dd,
                                            float& mx, float& num, float& den) {
    constexpr int NPAR = T::NPAR;
    mx = NEG_BIG;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int par = 0; par < NPAR; ++par) mx = fmaxf(mx, sm_m[w][NPAR * h + par]);
    num = den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int par = 0; par < NPAR; ++par) {
            const int c = NPAR * h + par;
            const float f = exp2f(sm_m[w][c] - mx);
            num = fmaf(f, wave_rows(acc, w)[c * T::OROW + dd + 64 * par], num);
            den = fmaf(f, sm_l[w][c], den);
        }
}
