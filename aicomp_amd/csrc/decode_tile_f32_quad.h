// TileF32Quad: float32 queries and pools, head_dim 128 (tiles of 16 tokens) or 64 (32 tokens), up to four query heads
// per KV head, on v_mfma_f32_4x4x1_16b_f32.  Included by decode_mfma.hip, inside its namespace.
//
// TileF32 multiplies sixteen columns whatever the group is; a decode group is often one or four heads, and the float32 matrix
// instruction runs on the vector ALU's multipliers, so a tile cost a wave 2048 cycles of which three quarters
// were zeros.  A row of a small call is a chain of such tiles on one CU: four rows of 512 tokens, D 64, 32 / 8 heads
// spent 3.5 of their 10.2 us in them.  The 4x4 form multiplies sixteen independent 4 x 4 blocks at the same
// rate: 512 cycles per tile.  (Two sets of blocks for groups of eight halve the products too, but need 64 registers of
// queries and spill 33: one row of 500 tokens, 64 / 8 heads, 22 us against 11.)
//   QK  a block's rows are four tokens, its columns four heads, and the blocks are the tile's tokens times KQ parts of
//       head_dim (32 elements each); a lane holds its token's K chunks (A) and its head's elements (B).  The KQ partial
//       scores are added up by lane swaps that leave every lane 2 (D 64) or 1 (128) whole scores: its own.
//   PV  a block's rows are the four heads, its columns four dims: V (B) goes from the load to the multiplier, 1 KB of
//       consecutive rows per load, and P (A) is broadcast from the block that holds the load's token to the
//       blocks of that token's dims (cbsz / abid), so it never leaves its register.
// us per call, before -> now, 32 / 8 heads: D 64, one row of 100 tokens 5.1 -> 4.9, 500 10.1 -> 7.0, four rows of 64..512
// 10.2 -> 7.0; D 128, one row of 500 14.6 -> 11.5, 4 of 2000 (split) 17.6 -> 16.2; where the call streams, 64 rows of
// 256..2048, D 64 57.4 -> 56.0 and D 128 102.7 -> 102.3.  Now a CU's 64 bytes per clock bound a row (500 tokens, D 64: 256 KB).
// Which token a lane scores follows from that; K goes through the wave's LDS tile, its 16-byte chunks permuted
// (swz) so that every four lanes of the operand read lie in one aligned 64-byte segment of the bank line and a
// half-wave in all four.
//   lane l = 4 b + j: block b, column (head) or row (token) j
//   D 64   KQ 2: part l / 32; token 8 a + 4 (j & 1) + 2 (j >> 1) + t, a = (l / 4) % 4, t = (l / 16) % 2
//          after the swap: tokens 8 a + 4 r + l / 16, r = 0, 1;  V load i: token 4 i + l / 16
//   D 128  KQ 4: part l / 16; token 2 a + (j >> 1) + 8 (j & 1)
//          after the swaps: token 2 a + l / 32 + 8 ((l / 16) % 2);  V load i: token 2 i + l / 32
template <int DQ_>
struct TileF32Quad {
    typedef F32Fmt Fmt;
    static constexpr bool FP8 = false, PAIR = false, QUAD = true;
    static constexpr int DQ = DQ_;
    static constexpr int TT = DQ == 128 ? 16 : 32;       // tokens per tile
    static constexpr int BPT = TT / BS;
    static constexpr int OROW = DQ;
    static constexpr int NPAR = 1;
    static constexpr int KQ = DQ / 32;
    static constexpr int NR = 4 / KQ;                    // scores of a lane
    static constexpr int ROWB = DQ * 4;
    static constexpr int RPL = 1024 / ROWB;              // rows of a load
    struct State {
        float m = NEG_BIG, lsum = 0.f;
        f32x4_t O[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    };
    struct Q { f32x4_t r[8]; };
    struct Regs { uint4 k[8], v[8]; };
    struct Offsets { int wr, cb, rd; };

    __device__ __forceinline__ static Offsets offsets(int lane) {
        const int a = (lane >> 2) & 3, j = lane & 3;
        Offsets o;
        o.wr = (lane >> (DQ == 64 ? 4 : 5)) * ROWB + (DQ == 64 ? 0 : ((lane >> 4) & 1) * 256);
        o.cb = ((lane & 15) ^ (lane >> 5)) << 4;
        if constexpr (DQ == 64) {
            const int tok = 8 * a + 4 * (j & 1) + 2 * (j >> 1) + ((lane >> 4) & 1);
            o.rd = tok * ROWB + (((8 * (lane >> 5)) ^ (tok >> 1)) << 4);
        } else {
            const int tok = 2 * a + (j >> 1) + 8 * (j & 1);
            const int swz = (tok & 1) | ((tok >> 3) << 1) | (((tok >> 1) & 3) << 2);
            o.rd = tok * ROWB + ((lane >> 5) << 8) + (((8 * ((lane >> 4) & 1)) ^ swz) << 4);
        }
        return o;
    }
    // load i of lane l is tile row RPL i + l / (64 / RPL), with the lane's chunk
    __device__ __forceinline__ static int write_at(const Offsets& o, int i) {
        const int swz = DQ == 64 ? 2 * i : ((i >> 2) << 1) | ((i & 3) << 2);       // (the lane's part is in cb)
        return i * 1024 + o.wr + (o.cb ^ (swz << 4));
    }

    __device__ __forceinline__ static void load_q(Q& q, const float* rows, int group, int lane) {
        const int part = DQ == 64 ? lane >> 5 : lane >> 4;
        const float* row = rows + min(lane & 3, group - 1) * DQ + 32 * part;
#pragma unroll
        for (int c = 0; c < 8; ++c) q.r[c] = *(const f32x4_t*)(row + 4 * c);
    }
    __device__ __forceinline__ static void q_operand(Q& q, const Q& raw, int group, int lane) {
        const bool use = (lane & 3) < group;
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) q.r[c][e] = use ? raw.r[c][e] : 0.f;
    }

    template <typename Params>
    __device__ __forceinline__ static void load_rows(uint4 (&r)[8], const void* pool, const Params& p, const int64_t (&bb)[4],
                                                     int kvh, int lane) {
        constexpr int LPB = 8 / BPT;                     // loads per block
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const uint4* src = (const uint4*)pool + (bb[b] * p.hkv + kvh) * (BS * DQ / 4) + lane;
#pragma unroll
            for (int i = 0; i < LPB; ++i) r[LPB * b + i] = tile_ld(src + 64 * i);
        }
    }
    template <typename Params>
    __device__ __forceinline__ static void load(Regs& t, const Params& p, const int64_t (&bb)[4], int kvh, int lane) {
        load_rows(t.k, p.k_pool, p, bb, kvh, lane);
        load_rows(t.v, p.v_pool, p, bb, kvh, lane);
    }

    // a + b of the two halves (of the 16-lane rows) of the wave: the lower half (even rows) gets a's sum, the other b's
    __device__ __forceinline__ static float swap_add32(float a, float b) {
        const u32x2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    __device__ __forceinline__ static float swap_add16(float a, float b) {
        const u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    template <int CTRL>
    __device__ __forceinline__ static float quad(float x) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
    }

    // NEXT: prefetch the wave's next tile (blocks nb) into the same registers; MASK: the tile crosses `end`
    template <bool NEXT, bool MASK, typename Params>
    __device__ __forceinline__ static void process(State& st, Regs& t, const Q& q, unsigned char* kt, const Offsets& ko,
                                                   const Params& p, const int64_t (&nb)[4], int kvh_next, int lane,
                                                   int tile_start, int end, float cmul) {
#pragma unroll
        for (int i = 0; i < 8; ++i) *(uint4*)(kt + write_at(ko, i)) = t.k[i];
        if (NEXT) load_rows(t.k, p.k_pool, p, nb, kvh_next, lane);

        // ---- partial scores of the lane's part, two accumulation chains
        f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const f32x4_t k4 = *(const f32x4_t*)(kt + (ko.rd ^ (c << 4)));
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e & 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(k4[e], q.r[c][e], acc[e & 1], 0, 0, 0);
        }
        const f32x4_t part = acc[0] + acc[1];
        const float s02 = swap_add32(part[0], part[2]), s13 = swap_add32(part[1], part[3]);
        float sc[NR], e[NR], sum = 0.f;
        if constexpr (NR == 2) { sc[0] = s02; sc[1] = s13; }
        else sc[0] = swap_add16(s02, s13);
        // online softmax: the head's reference max moves only when a lane's probabilities of a tile outgrow 2^8
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            if (MASK && tile_start + token(lane, r) >= end) sc[r] = -INFINITY;
            e[r] = __builtin_amdgcn_exp2f(fmaf(sc[r], cmul, -st.m));
            sum += e[r];
        }
        if (__any(!(sum <= 256.f))) {
            float mx = sc[0] * cmul;
            if constexpr (NR == 2) mx = fmaxf(mx, sc[1] * cmul);
#pragma unroll
            for (int o = 4; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
            const float m_new = fmaxf(st.m, mx);
            const float alpha = __builtin_amdgcn_exp2f(st.m - m_new);
            st.m = m_new;
            sum = 0.f;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                e[r] = __builtin_amdgcn_exp2f(fmaf(sc[r], cmul, -m_new));
                sum += e[r];
            }
            st.lsum *= alpha;
            // an accumulator's elements are the heads, one lane of a quad each
            const f32x4_t al = {quad<0x00>(alpha), quad<0x55>(alpha), quad<0xaa>(alpha), quad<0xff>(alpha)};
#pragma unroll
            for (int x = 0; x < 4; ++x) st.O[x] *= al;
        }
        st.lsum += sum;
        // ---- O += P V
        uint4 vv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            vv[i] = t.v[i];
            if (MASK && tile_start + RPL * i + (lane >> (DQ == 64 ? 4 : 5)) >= end) vv[i] = make_uint4(0, 0, 0, 0);
        }
        if (NEXT) load_rows(t.v, p.v_pool, p, nb, kvh_next, lane);
        pv<0>(st, vv, e);
    }
    // load i: P of its tokens from block i / 2 of every four (D 128: i of every eight)
    template <int I>
    __device__ __forceinline__ static void pv(State& st, const uint4 (&vv)[8], const float (&e)[NR]) {
        constexpr int CB = DQ == 64 ? 2 : 3, AB = DQ == 64 ? I >> 1 : I, R = DQ == 64 ? I & 1 : 0;
        const float v[4] = {__uint_as_float(vv[I].x), __uint_as_float(vv[I].y), __uint_as_float(vv[I].z), __uint_as_float(vv[I].w)};
#pragma unroll
        for (int x = 0; x < 4; ++x) st.O[x] = __builtin_amdgcn_mfma_f32_4x4x1f32(e[R], v[x], st.O[x], CB, AB, 0);
        if constexpr (I < 7) pv<I + 1>(st, vv, e);
    }
    __device__ __forceinline__ static int token(int lane, int r) {
        const int a = (lane >> 2) & 3;
        return DQ == 64 ? 8 * a + 4 * r + (lane >> 4) : 2 * a + (lane >> 5) + 8 * ((lane >> 4) & 1);
    }

    // fused append (see inject_new_row): the lanes that loaded the newest token's chunks take the new
    // row's instead and write them to the pools
    template <typename Params>
    __device__ __forceinline__ static void inject(Regs& t, const Params& p, const float* key, const float* value, int kvh,
                                                  int lane, int tile_start, int len, const int64_t (&bb)[4]) {
        const int tau = len - 1 - tile_start;                            // wave-uniform
        const int64_t dst = ((bb[tau >> 4] * p.hkv + kvh) * BS + (tau & 15)) * (DQ / 4);
        const int chunk = lane & (DQ / 4 - 1);
        const bool mine = lane / (DQ / 4) == tau % RPL;
        const uint4 k4 = ((const uint4*)key)[chunk], v4 = ((const uint4*)value)[chunk];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (mine && i == tau / RPL) { t.k[i] = k4; t.v[i] = v4; }
        if (mine) { ((uint4*)p.k_pool)[dst + chunk] = k4; ((uint4*)p.v_pool)[dst + chunk] = v4; }
    }

    // the wave's result: head h's unnormalised row at rows + h DQ, its max and sum at m_out / l_out [h * ml_stride]
    __device__ __forceinline__ static void finish(const State& st, float* rows, float* m_out, float* l_out, int ml_stride,
                                                  int lane, int group) {
        float l = st.lsum;
#pragma unroll
        for (int o = 4; o < 64; o <<= 1) l += __shfl_xor(l, o);
        if (lane < group) { m_out[lane * ml_stride] = st.m; l_out[lane * ml_stride] = l; }
        // lanes of one l / 16 (D 128: l / 32) hold sums over every fourth (second) token, all four heads each: the
        // swaps leave a lane one head's (two heads') sum over all
        f32x4_t even, odd;                                               // heads 0 | 2 and 1 | 3 in the lower | upper half
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            even[x] = swap_add32(st.O[x][0], st.O[x][2]);
            odd[x] = swap_add32(st.O[x][1], st.O[x][3]);
        }
        if constexpr (DQ == 64) {
            f32x4_t one;
#pragma unroll
            for (int x = 0; x < 4; ++x) one[x] = swap_add16(even[x], odd[x]);
            const int h = lane >> 4;
            if (h < group) *(f32x4_t*)(rows + h * DQ + 4 * (lane & 15)) = one;
        } else {
            const int h = 2 * (lane >> 5);
            if (h < group) *(f32x4_t*)(rows + h * DQ + 4 * (lane & 31)) = even;
            if (h + 1 < group) *(f32x4_t*)(rows + (h + 1) * DQ + 4 * (lane & 31)) = odd;
        }
    }
};
