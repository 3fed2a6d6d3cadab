// TileF32: float32 queries and pools, head_dim 128 (tiles of 16 tokens) or 64 (32 tokens), on the
// float32 matrix instruction v_mfma_f32_16x16x4_f32, for groups of more than four query heads per KV head (smaller
// ones: decode_tile_f32_quad.h).  Included by decode_mfma.hip, inside its namespace.
//
// A tile (8 KB of K, 8 KB of V) costs a wave 64 MFMAs of 32 cycles, 2048 cycles: 19 TB/s with all 1024 SIMDs
// at work, so a batch that fills the chip is bound by HBM like the 16-bit tiles.  The rows of a small call
// are on few CUs, and a row is then a chain of such tiles on its CU's four SIMDs (640 tokens of D 128, one
// workgroup: ten tiles each, 17.6 us).  What it replaced is the vector-ALU kernel, bound by the lane
// reductions of its dot products, with the append as a launch of its own and always a merge launch:
//   64 rows of 256..2048 tokens, 32 / 8 heads     D 128  170.5 -> 100.6 us per call (6.0 TB/s)
//                                                 D 64    90.0 ->  56.8 us
//   8 rows of 1000..4096, 64 / 8 heads, D 128     95.6 -> 37.1 us;  one row of 16384  60.4 -> 30.5 us
//   4 rows of 64..512, D 64                       three launches, 15.2 us -> one
//
// Everything stays float32: products and sums are those of the vector ALU, sixteen times fewer
// instructions.  A tile is 8 KB of K and 8 KB of V, the same loads as a 16-bit tile of twice the tokens.
//   K   through the wave's LDS tile: rows of 4 DQ bytes, chunk slot c ^ (row % 16) in the low four
//       bits of the 16-byte chunk index, so that every four consecutive lanes of the operand read
//       address one aligned 64-byte segment of the bank line and a half-wave all four.  One 16-byte
//       read feeds four MFMAs: MFMA e of chunk read q takes element 16 q + 4 g4 + e in lane group g4.
//   V   never touches LDS: lane (r16, g4) loads chunks r16 (and r16 + 16) of token 16 a + 4 g4 + e, and
//       component x of such a chunk is the A operand of output tile (half, x) for k index g4, whose
//       row m is dim 64 half + 4 m + x.  The probability the same lane computed for that token is the
//       B operand: P stays in its lane.
template <int DQ_>
struct TileF32 {
    typedef F32Fmt Fmt;
    static constexpr bool FP8 = false, PAIR = false, QUAD = false;
    static constexpr int DQ = DQ_;
    static constexpr int TT = DQ == 128 ? 16 : 32;       // tokens per tile
    static constexpr int BPT = TT / BS;
    static constexpr int OROW = DQ;
    static constexpr int NPAR = 1;
    static constexpr int NSUB = TT / 16;                 // 16-token sub-tiles
    static constexpr int HALVES = DQ / 64;               // 64-element halves of a row
    static constexpr int ROWB = DQ * 4;                  // bytes per row
    typedef WaveStateT<4 * HALVES> State;
    struct Q { float4 r[DQ / 16]; };
    struct Regs { uint4 k[8], v[8]; };                   // v[(4 a + e) * HALVES + half]
    struct Offsets { int wr, cb, rd[4]; };

    __device__ __forceinline__ static Offsets offsets(int lane) {
        const int r16 = lane & 15, g4 = lane >> 4;
        Offsets o;
        const int row0 = DQ == 128 ? lane >> 5 : lane >> 4, chunk = DQ == 128 ? lane & 31 : lane & 15;
        o.wr = row0 * ROWB;
        o.cb = (chunk ^ row0) << 4;
#pragma unroll
        for (int k = 0; k < 4; ++k) o.rd[k] = r16 * ROWB + (((4 * k + g4) ^ r16) << 4);
        return o;
    }
    // load i of lane l is tile row (1024 / ROWB) i + row0, with the lane's chunk
    __device__ __forceinline__ static int write_at(const Offsets& o, int i) {
        constexpr int RPL = 1024 / ROWB;
        return i * 1024 + o.wr + (o.cb ^ (((RPL * i) & 15) << 4));
    }

    __device__ __forceinline__ static void load_q(Q& q, const float* rows, int group, int lane) {
        const int r16 = lane & 15, g4 = lane >> 4;
        const float* row = rows + min(r16, group - 1) * DQ + 4 * g4;
#pragma unroll
        for (int s = 0; s < DQ / 16; ++s) q.r[s] = *(const float4*)(row + 16 * s);
    }
    __device__ __forceinline__ static void q_operand(Q& q, const Q& raw, int group, int lane) {
        const bool use = (lane & 15) < group;
#pragma unroll
        for (int s = 0; s < DQ / 16; ++s) q.r[s] = use ? raw.r[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    }

    template <typename Params>
    __device__ __forceinline__ static void load_k(Regs& t, const Params& p, const int64_t (&bb)[4], int kvh, int lane) {
        constexpr int LPB = 8 / BPT;                     // loads per block
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const uint4* src = (const uint4*)p.k_pool + (bb[b] * p.hkv + kvh) * (BS * DQ / 4) + lane;
#pragma unroll
            for (int i = 0; i < LPB; ++i) t.k[LPB * b + i] = tile_ld(src + 64 * i);
        }
    }
    template <typename Params>
    __device__ __forceinline__ static void load_v(Regs& t, const Params& p, const int64_t (&bb)[4], int kvh, int lane) {
        const int r16 = lane & 15, g4 = lane >> 4;
#pragma unroll
        for (int a = 0; a < NSUB; ++a) {
            const uint4* src = (const uint4*)p.v_pool + (bb[a] * p.hkv + kvh) * (BS * DQ / 4) + (4 * g4) * (DQ / 4) + r16;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < HALVES; ++h) t.v[(4 * a + e) * HALVES + h] = tile_ld(src + e * (DQ / 4) + 16 * h);
        }
    }
    template <typename Params>
    __device__ __forceinline__ static void load(Regs& t, const Params& p, const int64_t (&bb)[4], int kvh, int lane) {
        load_k(t, p, bb, kvh, lane);
        load_v(t, p, bb, kvh, lane);
    }

    // NEXT: prefetch the wave's next tile (blocks nb) into the same registers; MASK: the tile crosses `end`
    template <bool NEXT, bool MASK, typename Params>
    __device__ __forceinline__ static void process(State& st, Regs& t, const Q& q, unsigned char* kt, const Offsets& ko,
                                                   const Params& p, const int64_t (&nb)[4], int kvh_next, int lane,
                                                   int tile_start, int end, float cmul) {
        const int g4 = lane >> 4;
#pragma unroll
        for (int i = 0; i < 8; ++i) *(uint4*)(kt + write_at(ko, i)) = t.k[i];
        if (NEXT) load_k(t, p, nb, kvh_next, lane);

        // ---- S^T = K Q^T, two accumulation chains per sub-tile
        f32x4_t s[NSUB][2];
#pragma unroll
        for (int a = 0; a < NSUB; ++a) s[a][0] = s[a][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DQ / 16; ++c)
#pragma unroll
            for (int a = 0; a < NSUB; ++a) {
                const float4 k4 = *(const float4*)(kt + 16 * a * ROWB + ko.rd[c & 3] + (c >> 2) * 256);
                f32x4_t& x = s[a][c & 1];
                x = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.x, q.r[c].x, x, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.y, q.r[c].y, x, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.z, q.r[c].z, x, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_16x16x4f32(k4.w, q.r[c].w, x, 0, 0, 0);
            }
        // ---- online softmax: lane (head r16, g4) holds tokens tile_start + 16 a + 4 g4 + i
        constexpr int NS = 4 * NSUB;
        float sc[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            sc[k] = (s[k >> 2][0][k & 3] + s[k >> 2][1][k & 3]) * cmul;
            if (MASK && tile_start + 16 * (k >> 2) + 4 * g4 + (k & 3) >= end) sc[k] = NEG_BIG;
        }
        float mx = sc[0];
#pragma unroll
        for (int k = 1; k < NS; ++k) mx = fmaxf(mx, sc[k]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(st.m, mx);
        const float alpha = exp2f(st.m - m_new);
        float pr[NS], psum = 0.f;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            pr[k] = exp2f(sc[k] - m_new);
            if (MASK && sc[k] == NEG_BIG) pr[k] = 0.f;
            psum += pr[k];
        }
        st.lsum = st.lsum * alpha + psum;
        st.m = m_new;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int j = 0; j < 4 * HALVES; ++j) st.O[j] *= alpha;
        }
        // ---- O^T += V^T P^T
        uint4 vv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            vv[i] = t.v[i];
            const int tok = tile_start + 16 * (i / (4 * HALVES)) + 4 * g4 + (i / HALVES) % 4;
            if (MASK && tok >= end) vv[i] = make_uint4(0, 0, 0, 0);
        }
        if (NEXT) load_v(t, p, nb, kvh_next, lane);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float b = pr[i / HALVES];                              // token (a, e): i / HALVES = 4 a + e
            f32x4_t* o = &st.O[4 * (i % HALVES)];
            o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vv[i].x), b, o[0], 0, 0, 0);
            o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vv[i].y), b, o[1], 0, 0, 0);
            o[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vv[i].z), b, o[2], 0, 0, 0);
            o[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vv[i].w), b, o[3], 0, 0, 0);
        }
    }

    // fused append (see inject_new_row): the lanes that loaded the newest token's chunks take the new
    // row's instead and write them to the pools
    template <typename Params>
    __device__ __forceinline__ static void inject(Regs& t, const Params& p, const float* key, const float* value, int kvh,
                                                  int lane, int tile_start, int len, const int64_t (&bb)[4]) {
        const int tau = len - 1 - tile_start;                            // wave-uniform
        const uint4 *nk = (const uint4*)key, *nv = (const uint4*)value;
        const int64_t dst = ((bb[tau >> 4] * p.hkv + kvh) * BS + (tau & 15)) * (DQ / 4);
        constexpr int RPL = 1024 / ROWB;                                 // tile rows per load
        const int row0 = DQ == 128 ? lane >> 5 : lane >> 4, chunk = DQ == 128 ? lane & 31 : lane & 15;
        const bool mine_k = row0 == tau % RPL;
        const uint4 k4 = nk[chunk];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (mine_k && i == tau / RPL) t.k[i] = k4;
        if (mine_k) ((uint4*)p.k_pool)[dst + chunk] = k4;
        const int r16 = lane & 15, g4 = lane >> 4;
        const bool mine_v = g4 == ((tau >> 2) & 3);
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
            const uint4 v4 = nv[r16 + 16 * h];
#pragma unroll
            for (int ae = 0; ae < 4 * NSUB; ++ae)
                if (mine_v && ae == 4 * (tau >> 4) + (tau & 3)) t.v[ae * HALVES + h] = v4;
            if (mine_v) ((uint4*)p.v_pool)[dst + r16 + 16 * h] = v4;
        }
    }

    // this lane's accumulators into the row of its column: dims 64 half + 16 g4 + 4 i + x from O[4 half + x][i]
    __device__ __forceinline__ static void store_acc(float* row, const State& st, int g4) {
#pragma unroll
        for (int h = 0; h < HALVES; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(float4*)(row + 64 * h + 16 * g4 + 4 * i) = make_float4(st.O[4 * h][i], st.O[4 * h + 1][i],
                                                                        st.O[4 * h + 2][i], st.O[4 * h + 3][i]);
    }
};
