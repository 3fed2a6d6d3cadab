// Token sampling: temperature -> top-k -> top-p (nucleus) -> multinomial, one launch, or two to four when the
// rows are cut into parts.
//
// Replaces the step after the attention path,
//   opt_prime/opt_prime/inference.py:786-843 (_sample_token):
//     logits / temperature; remove logits < k-th largest; sort descending, cumulative
//     softmax, remove entries whose preceding cumulative mass exceeds top_p (the first
//     entry always stays); softmax of what is left; torch.multinomial
// which in PyTorch is a full-vocabulary sort plus about ten elementwise / scan launches
// per token.  Greedy decoding (do_sample == False, :806-808) is the argmax.
//
// One workgroup of 1024 lanes per row (or part of a row); nothing is sorted.
//   1  row maximum and argmax on the raw logits (a positive temperature keeps the order)
//   2  top-k (k <= 1024, the usual case): the k-th largest of the 1024 per-lane maxima bounds the
//      row's k-th largest value from below, so a second pass over the row collects the
//      candidates (about k) into LDS; selection of the k-th value, the nucleus threshold and the
//      draw then run on that list.  Two passes over the row in total, neither dividing nor
//      exponentiating more than the candidates.
//   2' without top-k, or when the candidates do not fit (masses of equal logits): radix select
//      over the whole row on order-preserving integer keys (digits of 11, 11 and 10 bits, count
//      histograms in LDS), nucleus threshold by the same walk over MASS histograms, and a draw
//      located by wave segment, lane chunk and element.
// Probability mass is carried as 2^-40 fixed point in 64-bit integers, so every sum is
// exact, order independent and reproducible; ties at the nucleus threshold are kept in
// index order (what a stable descending sort would do).
//
// A row (128 K logits = 512 KB in fp32) on one CU is bound by what that CU can load and compare, two
// passes of it, with three quarters of the chip idle at 64 rows; the full-row histogram passes are
// LDS-atomic bound when many logits share the leading key bits.  A caller with scratch memory therefore
// has greedy and top-k calls cut into parts of a row first (sample_parts_kernel), and draws from the whole row or
// a nucleus of it too (sample_max_kernel and what follows it).
#include "common.h"

#include <type_traits>

namespace aicomp {

namespace {

constexpr int NT = 1024;                 // lanes per workgroup
constexpr int NW = NT / 64;              // waves
constexpr int BINS = 2048;
constexpr int LIST_CAP = 4096;          // candidate list of the top-k fast path (64 KB of LDS with weights)
constexpr uint32_t LIST_SLACK = 64;      // raw values below the bound that may still tie with it after the division
constexpr float LIST_MAX_TEMPERATURE = 32.f;   // at most ~T+1 raw values share a quotient: 64 covers this
constexpr float W_ONE = 1099511627776.f; // 2^40: weight of the row maximum

struct SampleParams {
    int64_t* out;                        // [B] token ids
    const void* logits;                  // [B, V]
    int64_t row_stride;                  // elements
    float* probs_out;                    // optional [B, V]: the distribution drawn from
    const float* uniforms;               // [B] in [0, 1)
    int vocab;
    float temperature;
    int top_k;                           // <= 0 or >= V: off
    float top_p;                         // >= 1: off
    int greedy;
    // rows cut into parts (NULL / 0: not): what sample_parts_kernel leaves for sample_kernel
    unsigned int* part_count;            // [B, parts] candidates of a part, PART_WHOLE: take the whole row instead
    uint2* part_list;                    // [B, parts, part_cap] (order key of the scaled logit, index)
    int parts, part_size;                // part_size: a multiple of 4 and at most PART_MAX
    int part_cap;                        // candidates of a part: part_capacity()
    // a draw from the whole row, cut into parts: what sample_max_kernel and sample_mass_kernel leave
    unsigned long long* seg_mass;        // [B, parts, NW] mass of each segment
    float* part_max;                     // [B, parts] raw maximum
    // ... and for a nucleus of it (NULL: top_p >= 1), with part_list and part_count
    unsigned long long* part_hist;       // [B, parts, NBINS] mass of each slice of logits
    unsigned long long* part_group;      // [B, parts, GROUPS] and of each 32 of them
    unsigned long long* kept_mass;       // [B, parts, NW] of the segments' logits above the slice that holds the threshold
    unsigned long long* cut;             // [B, 2] that slice (NBINS: not found), what is left of the mass limit at it
};

constexpr int PART_SLOTS = 16;                      // logits a lane of a part holds in registers
constexpr int PART_MAX = NT * PART_SLOTS;           // 16384
constexpr int GREEDY_CAP = 256;                     // room per part of a greedy call, which keeps one: 2 KB apart
constexpr int RAW_CAP = 4096;                       // candidates of a part before the exact test
constexpr int MAX_PARTS = 16;
constexpr int MERGE_SLOTS = 16;                     // candidates a lane of the merge takes: 16 lists of 1024 per row
constexpr int PART_MAX_K = 256;
constexpr int PART_MAX_BATCH = 1024;
constexpr unsigned int PART_WHOLE = 0xffffffffu;

// float -> key with the same order (larger float, larger key).  -0.0 gets the key of +0.0: the
// reference compares floats (`logits < kth`), for which the two zeros are one value.
__device__ __forceinline__ uint32_t order_key(float x) {
    uint32_t b = __float_as_uint(x);
    if (b == 0x80000000u) b = 0u;
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    const uint32_t b = (k & 0x80000000u) ? (k ^ 0x80000000u) : ~k;
    return __uint_as_float(b);
}

template <typename T>
__device__ __forceinline__ float scaled_logit(const T* row, int i, float temperature);
template <>
__device__ __forceinline__ float scaled_logit<float>(const float* row, int i, float temperature) {
    return temperature == 1.f ? row[i] : row[i] / temperature;
}
template <>
__device__ __forceinline__ float scaled_logit<bf16_t>(const bf16_t* row, int i, float temperature) {
    const float x = bf16_to_f32(row[i].bits);
    // the division of a bf16 tensor is rounded back to bf16, as the eager division is
    return temperature == 1.f ? x : (float)(__bf16)(x / temperature);
}

template <>
__device__ __forceinline__ float scaled_logit<f16_t>(const f16_t* row, int i, float temperature) {
    const float x = f16_to_f32(row[i].bits);
    return temperature == 1.f ? x : (float)(_Float16)(x / temperature);
}

// four consecutive logits in one load (16 bytes of fp32, 8 bytes of bf16 / fp16)
template <typename T> struct Load4;
template <> struct Load4<float> {
    __device__ __forceinline__ static void get(const float* p, float* x) {
        const float4 v = *(const float4*)p;
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    }
};
template <> struct Load4<bf16_t> {
    __device__ __forceinline__ static void get(const bf16_t* p, float* x) {
        const uint2 v = *(const uint2*)p;
        x[0] = __uint_as_float(v.x << 16); x[1] = __uint_as_float(v.x & 0xffff0000u);
        x[2] = __uint_as_float(v.y << 16); x[3] = __uint_as_float(v.y & 0xffff0000u);
    }
};
template <> struct Load4<f16_t> {
    __device__ __forceinline__ static void get(const f16_t* p, float* x) {
        const uint2 v = *(const uint2*)p;
        x[0] = f16_to_f32((uint16_t)(v.x & 0xffffu)); x[1] = f16_to_f32((uint16_t)(v.x >> 16));
        x[2] = f16_to_f32((uint16_t)(v.y & 0xffffu)); x[3] = f16_to_f32((uint16_t)(v.y >> 16));
    }
};
// For fp16 rows: a raw value below which the scaled, rounded logit is certainly below `q_scaled`.
// A quotient rounds up by at most half a unit in the last place of the result, 2^-25 in fp16's
// subnormal range, so everything from q - max(2^-24, |q| 2^-10) up may still reach q; the
// float division adds a relative 2^-24.  Other types: +inf (no extra lowering).
template <typename T> __device__ __forceinline__ float f16_raw_bound(float q_scaled, float temperature) {
    if constexpr (std::is_same<T, f16_t>::value) {
        const float y = (q_scaled - fmaxf(5.9604645e-8f, fabsf(q_scaled) * 9.765625e-4f)) * temperature;
        return y - fabsf(y) * 9.5367431640625e-7f;
    } else {
        (void)q_scaled; (void)temperature;
        return 0.f;                                    // not used for the other types
    }
}
template <typename T> __device__ __forceinline__ float apply_temperature(float x, float temperature);
template <> __device__ __forceinline__ float apply_temperature<float>(float x, float temperature) {
    return temperature == 1.f ? x : x / temperature;
}
template <> __device__ __forceinline__ float apply_temperature<bf16_t>(float x, float temperature) {
    return temperature == 1.f ? x : (float)(__bf16)(x / temperature);
}
template <> __device__ __forceinline__ float apply_temperature<f16_t>(float x, float temperature) {
    return temperature == 1.f ? x : (float)(_Float16)(x / temperature);
}

// f(index, scaled logit) over the elements [begin, end) owned by `rank` of `nranks` lanes.
// With 16-byte aligned rows a lane takes four consecutive elements per load and keeps U
// loads in flight (the passes are latency bound); each lane visits its elements in ascending index order.
template <typename T, int U = 16, typename F>
__device__ __forceinline__ void for_each_logit(const T* row, int begin, int end, float temperature,
                                               int rank, int nranks, bool vec_ok, F f) {
    int tail = begin;
    if (vec_ok) {
        const int n4 = (end - begin) / 4;              // begin is a multiple of 4 for every caller
        for (int j0 = rank; j0 < n4; j0 += U * nranks) {
            float a[U][4];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = j0 + u * nranks;
                Load4<T>::get(row + begin + 4 * (j < n4 ? j : j0), a[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = j0 + u * nranks;
                if (j < n4) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) f(begin + 4 * j + e, apply_temperature<T>(a[u][e], temperature));
                }
            }
        }
        tail = begin + 4 * n4;
    }
    for (int i = tail + rank; i < end; i += nranks) f(i, scaled_logit<T>(row, i, temperature));
}

// 2^-40 fixed-point weight exp(x - m) of a logit (x <= m, so the weight is in [0, 1]): the hardware
// exponential, then the two 32-bit halves of w * 2^40 from two float -> uint32 conversions (a
// float -> uint64 conversion is a long instruction sequence, and this runs once per logit in the
// full-row passes).  A NaN logit gets weight 0.
__device__ __forceinline__ uint64_t weight_of(float x, float m) {
    const float w = __builtin_amdgcn_exp2f((x - m) * LOG2E);
    const float s8 = w * 256.f;                                  // exact scaling, [0, 256]
    const float hi_f = floorf(s8);
    const uint32_t hi = (uint32_t)hi_f;                          // w * 2^8, integer part
    const uint32_t lo = (uint32_t)((s8 - hi_f) * 4294967296.f);  // fraction * 2^32 (the difference is exact)
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src) {
    const uint32_t lo = __shfl((uint32_t)v, src), hi = __shfl((uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t wave_sum64(uint64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)v, o), hi = __shfl_xor((uint32_t)(v >> 32), o);
        v += ((uint64_t)hi << 32) | lo;
    }
    return v;
}
// Sum over the lanes up to and including this one, in the vector ALU (every lane active): four shifts within a
// row of sixteen lanes, then the rows' last lanes broadcast onwards.
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_add64(unsigned long long v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS, 0xf, false);
    return v + ((unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ unsigned long long wave_scan_dpp64(unsigned long long v) {
    v = dpp_add64<0x111, 0xf>(v);            // row_shr 1, 2, 4, 8
    v = dpp_add64<0x112, 0xf>(v);
    v = dpp_add64<0x114, 0xf>(v);
    v = dpp_add64<0x118, 0xf>(v);
    v = dpp_add64<0x142, 0xa>(v);            // row_bcast 15: into rows 1 and 3
    return dpp_add64<0x143, 0xc>(v);         // row_bcast 31: into rows 2 and 3
}
__device__ __forceinline__ unsigned long long readlane64(unsigned long long v, int lane) {
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return (unsigned long long)hi << 32 | lo;
}

// The largest key with its low ten bits clear that at least r lanes of the wave reach (0: fewer do).
// Bit by bit with a ballot: 22 compares, no LDS and no barrier.
__device__ __forceinline__ uint32_t wave_rth_bound(uint32_t key, int r) {
    uint32_t t = 0;
#pragma unroll
    for (int bit = 31; bit >= 10; --bit) {
        const uint32_t cand = t | (1u << bit);
        if (__popcll(__ballot(key >= cand)) >= r) t = cand;
    }
    return t;
}

// The largest over the lanes of a row of sixteen.
__device__ __forceinline__ uint32_t largest_of_16(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));   // row_ror 8, 4, 2, 1
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false));
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false));
}

// A bound of the top_k-th largest of all lanes' entries, N each (0: none), from below: each wave's r-th largest entry, r =
// ceil(top_k / 16), and of these the largest one that top_k entries reach (0: none does).  Any lane may hold any number of
// the top; the waves' shares of it should be alike.  reach[0 .. NW) is zero before the first of two barriers.
template <int N>
__device__ __forceinline__ uint32_t bound_of_entries(const uint32_t (&key)[N], int top_k, uint32_t* bounds, unsigned int* reach, int lane,
                                                     int wave) {
    const int r = (top_k + NW - 1) / NW;
    uint32_t mine = 0;
#pragma unroll 1
    for (int bit = 31; bit >= 10; --bit) {
        const uint32_t cand = mine | (1u << bit);
        int n = 0;
#pragma unroll
        for (int u = 0; u < N; ++u) n += __popcll(__ballot(key[u] >= cand));
        if (n >= r) mine = cand;
    }
    if (lane == 0) bounds[wave] = mine;
    __syncthreads();
    const uint32_t t = bounds[lane & 15];
    unsigned int entries = 0;
#pragma unroll 1
    for (int w = 0; w < NW; ++w) {
        const uint32_t cand = (uint32_t)__builtin_amdgcn_readlane((int)t, w);
        unsigned int n = 0;
#pragma unroll
        for (int u = 0; u < N; ++u) n += (unsigned int)__popcll(__ballot(key[u] >= cand));
        entries = lane == w ? n : entries;
    }
    if (lane < NW) atomicAdd(&reach[lane], entries);
    __syncthreads();
    return largest_of_16(reach[lane & 15] >= (unsigned int)top_k ? t : 0u);
}

// What a raw logit has to reach so that its scaled key can be key_ls = the scaled key of key_l: a
// prefilter of one compare per element (it lets through whatever the key order would, -0.0 next to +0.0,
// and everything when the bound lies below -inf, whose key decodes to a NaN).
template <typename T> __device__ __forceinline__ float raw_bound(uint32_t key_l, uint32_t key_ls, float temperature) {
    // quotients of neighbouring raw values are more than half a unit in the last place apart where they
    // are normal, so at most three round to one value; LIST_SLACK covers the subnormal ones
    const uint32_t steps = fabsf(key_value(key_ls)) >= 2.4e-38f ? 4u : LIST_SLACK;
    const uint32_t slack = steps * (sizeof(T) == 2 ? 0x10000u : 1u);              // bf16 values are 2^16 keys apart
    float lo = key_value(key_l > slack ? key_l - slack : 0u);
    if constexpr (std::is_same<T, f16_t>::value) {
        const float b = f16_raw_bound<T>(key_value(key_ls), temperature);
        if (b < lo) lo = b;
    }
    return lo;
}

// Shared state of the radix walks (one row)
struct Shared {
    alignas(16) unsigned long long mass[BINS];
    alignas(16) unsigned int cnt[BINS];
    unsigned long long seg_mass[NW];
    unsigned int seg_tied[NW];
    float red_f[NW];
    int red_i[NW];
    // results broadcast by wave 0
    unsigned int sel_digit;
    unsigned long long sel_above_mass;
    unsigned int sel_above_cnt;
    // candidates of the top-k fast path
    unsigned int n_list;
    alignas(16) unsigned int list_key[LIST_CAP];
    alignas(16) unsigned int list_idx[LIST_CAP];
    alignas(16) unsigned long long list_w[LIST_CAP];
};

// Wave 0: walking the bins from the top, find the bin that holds the k-th element
// (by count).  Returns digit and the count strictly above it.
__device__ __forceinline__ void pick_by_count(Shared& s, int nbins, unsigned int k, int lane) {
    // lane owns bins [hi - 32*lane - 31, hi - 32*lane], i.e. lane 0 the top 32 bins: read as eight
    // 16-byte vectors (independent loads; a dependent chain of 32 LDS reads costs microseconds)
    constexpr int per = BINS / 64;
    const int top = nbins - 1 - lane * per;            // highest bin of this lane; nbins is a multiple of per
    unsigned int c[per];                               // c[j] = count of bin top - j
    if (top >= per - 1) {
        const uint4* v = (const uint4*)&s.cnt[top - (per - 1)];
#pragma unroll
        for (int q = 0; q < per / 4; ++q) {
            const uint4 x = v[q];
            c[per - 1 - 4 * q] = x.x; c[per - 2 - 4 * q] = x.y; c[per - 3 - 4 * q] = x.z; c[per - 4 - 4 * q] = x.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < per; ++j) c[j] = 0;
    }
    unsigned int local = 0;
#pragma unroll
    for (int j = 0; j < per; ++j) local += c[j];
    unsigned int incl = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned int o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
    }
    const unsigned int excl = incl - local;
    // first lane (from the top) whose inclusive count reaches k
    const unsigned long long hit = __ballot(incl >= k);
    const int owner = hit ? __ffsll((long long)hit) - 1 : 63;
    if (lane == owner) {
        unsigned int run = excl;
        int chosen = 0;
        unsigned int above = excl;
        bool done = false;
#pragma unroll
        for (int j = 0; j < per; ++j) {
            if (!done && top - j >= 0) {
                chosen = top - j;
                above = run;
                run += c[j];
                done = run >= k;
            }
        }
        s.sel_digit = (unsigned int)chosen;
        s.sel_above_cnt = above;
    }
}

// Wave 0: lowest bin d with mass(bins > d) <= limit.  Returns digit and that mass.
__device__ __forceinline__ void pick_by_mass(Shared& s, int nbins, unsigned long long limit, int lane) {
    const int per = BINS / 64;
    unsigned long long local = 0;
    for (int j = 0; j < per; ++j) {
        const int b = nbins - 1 - (lane * per + j);
        if (b >= 0) local += s.mass[b];
    }
    const unsigned long long incl = wave_scan_dpp64(local);
    const unsigned long long excl = incl - local;
    // mass above the LAST bin of a lane's range is incl - mass[last]; the walk continues past a
    // lane while even the mass above the first bin of the next lane (= incl) is <= limit
    const unsigned long long cont = __ballot(incl <= limit);
    // owner: first lane from the top for which incl > limit (the walk stops inside it); if none, the last lane
    const unsigned long long stop = ~cont;
    const int last_lane = nbins / per - 1;        // lanes beyond it own no bins
    int owner = stop ? __ffsll((long long)stop) - 1 : 63;
    if (owner > last_lane) owner = last_lane;
    if (lane == owner) {
        unsigned long long above = excl;          // mass above the current bin
        int chosen = nbins - 1 - lane * per;
        for (int j = 0; j < per; ++j) {
            const int b = nbins - 1 - (lane * per + j);
            if (b < 0) break;
            if (above > limit) break;             // cannot happen at j == 0 (excl <= limit for the owner)
            chosen = b;
            s.sel_above_mass = above;
            above += s.mass[b];
        }
        s.sel_digit = (unsigned int)chosen;
    }
}

constexpr int SHIFTS[3] = {21, 10, 0};
constexpr int WIDTHS[3] = {11, 11, 10};

// Key of the k-th largest element of a source (all lanes call; `src(f)` runs f(index, value) over
// the lane's share of the elements).  Three histogram rounds over digits of 11, 11 and 10 bits.
// With fewer than three levels the result is the lower edge of the bin that holds the k-th largest
// element at that resolution: a lower bound of its key.
template <typename Src>
__device__ __forceinline__ uint32_t select_kth(Shared& s, Src src, unsigned int k, int tid, int lane, int wave,
                                               int levels = 3) {
    uint32_t prefix = 0, pmask = 0;
    for (int lvl = 0; lvl < levels; ++lvl) {
        const int nb = 1 << WIDTHS[lvl];
        const int sh = SHIFTS[lvl];
        __syncthreads();
        for (int b = tid; b < BINS; b += NT) s.cnt[b] = 0;
        __syncthreads();
        src([&](int, float x) {
            const uint32_t key = order_key(x);
            if ((key & pmask) == prefix) atomicAdd(&s.cnt[(key >> sh) & (nb - 1)], 1u);
        });
        __syncthreads();
        if (wave == 0) pick_by_count(s, nb, k, lane);
        __syncthreads();
        k -= s.sel_above_cnt;
        prefix |= s.sel_digit << sh;
        pmask |= (uint32_t)(nb - 1) << sh;
    }
    return prefix;
}

struct Nucleus {
    uint32_t key_t;              // keep key > key_t ...
    unsigned int tie_keep;       // ... plus the first tie_keep elements (index order) with key == key_t
    bool tie_rule;               // false: keep every key >= key_t
};

// Nucleus threshold over the elements with key >= key_k: the same radix walk on mass histograms.
template <typename Src>
__device__ __forceinline__ Nucleus nucleus_threshold(Shared& s, Src src, uint32_t key_k, float m, float top_p,
                                                     int tid, int lane, int wave, int first_level = 0,
                                                     uint32_t prefix0 = 0, uint32_t pmask0 = 0,
                                                     unsigned long long limit0 = 0) {
    // first_level > 0: the caller has already walked the upper digit levels (prefix, mask and what is
    // left of the mass limit below the bins above the chosen one)
    uint32_t prefix = prefix0, pmask = pmask0;
    unsigned long long limit = limit0;
    for (int lvl = first_level; lvl < 3; ++lvl) {
        const int nb = 1 << WIDTHS[lvl];
        const int sh = SHIFTS[lvl];
        __syncthreads();
        for (int b = tid; b < BINS; b += NT) { s.mass[b] = 0; s.cnt[b] = 0; }
        __syncthreads();
        src([&](int, float x) {
            const uint32_t key = order_key(x);
            if (key >= key_k && (key & pmask) == prefix) {
                const int b = (key >> sh) & (nb - 1);
                atomicAdd(&s.mass[b], (unsigned long long)weight_of(x, m));
                atomicAdd(&s.cnt[b], 1u);
            }
        });
        __syncthreads();
        if (lvl == 0) {
            // total mass after top-k: sum of the first-level bins (every kept element is in one)
            unsigned long long z = 0;
            for (int b = tid; b < BINS; b += NT) z += s.mass[b];
            z = wave_sum64(z);
            if (lane == 0) s.seg_mass[wave] = z;
            __syncthreads();
            z = 0;
            for (int w = 0; w < NW; ++w) z += s.seg_mass[w];
            limit = (unsigned long long)((double)fmaxf(top_p, 0.f) * (double)z);
            __syncthreads();
        }
        if (wave == 0) pick_by_mass(s, nb, limit, lane);
        __syncthreads();
        limit -= s.sel_above_mass;
        prefix |= s.sel_digit << sh;
        pmask |= (uint32_t)(nb - 1) << sh;
    }
    // the last chosen bin holds exactly the elements with key == prefix
    const unsigned int n_t = s.cnt[s.sel_digit];
    const unsigned long long m_t = s.mass[s.sel_digit];
    Nucleus r;
    r.key_t = prefix;
    r.tie_rule = true;
    if (n_t == 0) r.tie_keep = 0;
    else {
        const unsigned long long w_t = m_t / n_t;              // identical keys, identical weights
        const unsigned long long c = w_t ? limit / w_t + 1 : (unsigned long long)n_t;
        r.tie_keep = (unsigned int)(c < n_t ? c : n_t);
    }
    if (r.key_t < key_k) { r.key_t = key_k; r.tie_rule = false; r.tie_keep = 0xffffffffu; }   // nucleus wider than top-k
    __syncthreads();
    return r;
}

// One part of a row per workgroup: the part is read once, into registers, and what may be among the
// row's top k leaves it.  Each wave finds the r-th largest of its 64 lane maxima, r = ceil(k / 16); at
// least 16 r >= k elements of the part reach the smallest of the sixteen, so whatever lies below it (in
// scaled order, ties stay) is not among the part's top k, nor the row's.  About 2.6 k of 16384 pass at
// k = 50.  Where likely tokens are neighbours, and so in few waves, more pass than there is room for: then the tight bound of
// bound_of_entries, from what passed (64 rows of 128256, logits of deviation 1 less ln(1 + index), k 50 38.9 -> 27.2 us, k 256
// 50.0 -> 32.7; 2000 neighbours 20 above all others, k 50 39.4 -> 25.1, which with room for 2048 that pass went the whole way).  At
// once it would leave a usual row's merge too few lanes with entries, k 50 12.3 -> 24.6.  A logit of -inf has no mass and is
// left out; a part with a NaN, or with more than RAW_CAP that pass, or with more than part_cap candidates all the same (masses of
// equal logits: sorted bf16 rows, 64 of 128256, k 50 40 -> 47), sends its row the whole way.  Greedy: the part's
// argmax is its one candidate.
//
// Bound by latency: one round of loads, 22 ballots, three barriers, a few dozen appends.  64 rows of 128256
// float32, k = 50: 8.8 us here and 5.2 us in sample_merge_kernel as traced, where one launch took 25.5 us.
template <typename T, bool GREEDY>
__global__ void __launch_bounds__(NT)
sample_parts_kernel(SampleParams p) {
    __shared__ uint32_t red_key[NW];
    __shared__ unsigned int red_idx[NW];
    __shared__ unsigned int n_list, n_raw, whole;
    __shared__ float raw_x[RAW_CAP];
    __shared__ unsigned int raw_i[RAW_CAP];
    const int row_idx = blockIdx.x, part = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const int begin = part * p.part_size;
    const int n = min(p.vocab - begin, p.part_size);              // at least 1
    if (tid == 0) { n_list = 0; n_raw = 0; whole = 0; }

    // slot 4 u + e: element 4 (tid + NT u) + e of a row with 16-byte alignment, tid + NT (4 u + e) of another
    const bool vec = ((uintptr_t)row % 16) == 0;
    const int n4 = vec ? n / 4 : 0;
    float x[PART_SLOTS], xt = -INFINITY;
    if (n4 > 0) {
#pragma unroll
        for (int u = 0; u < PART_SLOTS / 4; ++u) Load4<T>::get(row + begin + 4 * min(tid + NT * u, n4 - 1), x + 4 * u);
        if (tid < n - 4 * n4) xt = scaled_logit<T>(row, begin + 4 * n4 + tid, 1.f);
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i)
            if (tid + NT * (i / 4) >= n4) x[i] = -INFINITY;
    } else {
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i) x[i] = scaled_logit<T>(row, begin + min(tid + NT * i, n - 1), 1.f);
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i)
            if (tid + NT * i >= n) x[i] = -INFINITY;
    }
    auto index_of = [&](int i) -> unsigned int {
        return (unsigned int)(begin + (n4 > 0 ? 4 * (tid + NT * (i / 4)) + (i & 3) : tid + NT * i));
    };
    const unsigned int tail_idx = (unsigned int)(begin + 4 * n4 + tid);
    const int64_t slot = (int64_t)row_idx * p.parts + part;
    uint2* list = p.part_list + slot * (GREEDY ? GREEDY_CAP : p.part_cap);

    if constexpr (GREEDY) {
        // ascending indices within a lane (the tail's lie above all others), the lowest one wins a tie
        float best = -INFINITY;
        unsigned int best_i = 0x7fffffffu;
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i)
            if (x[i] > best) { best = x[i]; best_i = index_of(i); }
        if (xt > best) { best = xt; best_i = tail_idx; }
        uint32_t key = order_key(best);
        auto take = [&](uint32_t k2, unsigned int i2) {
            if (k2 > key || (k2 == key && i2 < best_i)) { key = k2; best_i = i2; }
        };
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t k2 = __shfl_xor(key, o);
            const unsigned int i2 = __shfl_xor(best_i, o);
            take(k2, i2);
        }
        if (lane == 0) { red_key[wave] = key; red_idx[wave] = best_i; }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < NW; ++w) take(red_key[w], red_idx[w]);
            list[0] = make_uint2(key, best_i);
            p.part_count[slot] = 1u;
        }
        return;
    }

    float best = xt;
    bool nan = xt != xt;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) { best = fmaxf(best, x[i]); nan |= x[i] != x[i]; }
    const uint32_t bound = wave_rth_bound(order_key(best), (p.top_k + NW - 1) / NW);
    if (lane == 0) red_key[wave] = bound;
    __syncthreads();
    if (nan) whole = 1u;
    uint32_t key_l = red_key[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) key_l = min(key_l, red_key[w]);
    const uint32_t key_ls = order_key(apply_temperature<T>(key_value(key_l), p.temperature));
    const float raw_lo = raw_bound<T>(key_l, key_ls, p.temperature);
    // what passes the prefilter goes through LDS, so that the exact test is made once per candidate
    unsigned int pass = 0;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) pass |= !(x[i] < raw_lo) && x[i] > -INFINITY ? 1u << i : 0u;
    pass |= !(xt < raw_lo) && xt > -INFINITY ? 1u << PART_SLOTS : 0u;
    if (pass) {
        unsigned int j = atomicAdd(&n_raw, (unsigned int)__popc(pass));
#pragma unroll
        for (int i = 0; i <= PART_SLOTS; ++i)
            if (pass >> i & 1u) {
                if (j < RAW_CAP) {
                    raw_x[j] = i < PART_SLOTS ? x[i < PART_SLOTS ? i : 0] : xt;
                    raw_i[j] = i < PART_SLOTS ? index_of(i) : tail_idx;
                }
                ++j;
            }
    }
    __syncthreads();
    const unsigned int nr = n_raw;
    for (unsigned int i = tid; i < min(nr, (unsigned int)RAW_CAP); i += NT) {
        const uint32_t key = order_key(apply_temperature<T>(raw_x[i], p.temperature));
        if (key >= key_ls) {
            const unsigned int j = atomicAdd(&n_list, 1u);
            if (j < (unsigned int)p.part_cap) list[j] = make_uint2(key, raw_i[i]);
        }
    }
    __syncthreads();
    if (__builtin_expect(nr > (unsigned int)p.part_cap, 0) && nr <= RAW_CAP && n_list > (unsigned int)p.part_cap && !whole) {
        // some waves have next to nothing of the top, and the smallest of the bounds is theirs
        uint32_t key[RAW_CAP / NT];
#pragma unroll
        for (int j = 0; j < RAW_CAP / NT; ++j) {
            const unsigned int i = lane * NW + wave + NT * j;
            key[j] = i < nr ? order_key(apply_temperature<T>(raw_x[i], p.temperature)) : 0u;
        }
        if (tid < NW) red_idx[tid] = 0;
        __syncthreads();                                          // (n_list is read above by all)
        if (tid == 0) n_list = 0;
        const uint32_t least = max(max(key_ls, 1u), bound_of_entries(key, p.top_k, red_key, red_idx, lane, wave));
#pragma unroll
        for (int j = 0; j < RAW_CAP / NT; ++j)
            if (key[j] >= least) {
                const unsigned int at = atomicAdd(&n_list, 1u);
                if (at < (unsigned int)p.part_cap) list[at] = make_uint2(key[j], raw_i[lane * NW + wave + NT * j]);
            }
        __syncthreads();
    }
    if (tid == 0) p.part_count[slot] = whole || nr > RAW_CAP || n_list > (unsigned int)p.part_cap ? PART_WHOLE : n_list;
}

// Index of the row's maximum, the lowest one among equals (0: nothing above -inf).
template <typename T, int U, typename S>
__device__ __forceinline__ int block_argmax(S& s, const T* row, int V, bool vec_ok) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    for_each_logit<T, U>(row, 0, V, 1.f, tid, NT, vec_ok, [&](int i, float x) {
        if (x > best) { best = x; best_i = i; }       // lowest index wins ties within a lane (ascending i)
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o);
        const int oi = __shfl_xor(best_i, o);
        if (ob > best || (ob == best && oi < best_i)) { best = ob; best_i = oi; }
    }
    __syncthreads();
    if (lane == 0) { s.red_f[wave] = best; s.red_i[wave] = best_i; }
    __syncthreads();
    best = s.red_f[0]; best_i = s.red_i[0];
    for (int w = 1; w < NW; ++w) {
        const float ob = s.red_f[w];
        const int oi = s.red_i[w];
        if (ob > best || (ob == best && oi < best_i)) { best = ob; best_i = oi; }
    }
    return best_i == 0x7fffffff ? 0 : best_i;
}

// A row without finite mass (all -inf, NaN): the argmax, and an all-zero distribution.
template <typename T, int U, typename S>
__device__ __forceinline__ void no_mass(S& s, const SampleParams& p, int row_idx, const T* row, bool vec_ok) {
    const int best_i = block_argmax<T, U>(s, row, p.vocab, vec_ok);
    if (threadIdx.x == 0) p.out[row_idx] = best_i;
    if (p.probs_out)
        for (int i = threadIdx.x; i < p.vocab; i += NT) p.probs_out[(int64_t)row_idx * p.vocab + i] = 0.f;
}

// Sum of v over the lanes before this one, and over all.
__device__ __forceinline__ unsigned long long block_scan(Shared& s, unsigned long long v, unsigned long long& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long incl = wave_scan_dpp64(v);            // -> sum before this lane
    if (lane == 63) s.seg_mass[wave] = incl;
    __syncthreads();
    unsigned long long before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const unsigned long long x = s.seg_mass[w];
        before += w < wave ? x : 0ull;
        total += x;
    }
    return before + incl - v;
}

// Ranks of the entries wave + NW l (mine, lane l) of a list of n among the 64 G at list_w: those above it, by (key, ~index) and, << 16, by
// ~index alone.  The entries are in registers, 64 to a compare: a ballot and a scalar count per 64 pairs, where reading
// them from LDS for every pair was bound by those reads.  The zeros behind the list are above nothing.
template <int G>
__device__ __forceinline__ uint32_t list_ranks(const unsigned long long* list_w, int n, unsigned long long mine, int lane, int wave) {
    unsigned long long x[G];
#pragma unroll
    for (int g = 0; g < G; ++g) x[g] = list_w[64 * g + lane];
    uint32_t ranks = 0;
    for (int l = 0; NW * l + wave < n; ++l) {
        const unsigned long long me = readlane64(mine, l);
        int by_key = 0, by_index = 0;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            by_key += __popcll(__ballot(x[g] > me));
            by_index += __popcll(__ballot((uint32_t)x[g] > (uint32_t)me));
        }
        ranks = lane == l ? (uint32_t)(by_key | by_index << 16) : ranks;
    }
    return ranks;
}

// At most one candidate per lane, in list_key and list_idx.
// No histograms: every candidate is ranked in the descending order a stable sort would give (key, then
// index) and in index order, by counting; with top-k the one of rank k-1 holds the k-th largest key;
// the mass before a candidate in the first order decides the nucleus, a scan in the second
// order the draw.  Exact 64-bit sums.  Without top-k the list is everything above a cut of the
// whole row and z_row the mass of the whole row.
// A chain of short steps between barriers: four of them, five with top_p.  One launch over 64 rows of 32000 float32: k 65 16.5
// -> 15.4 us, k 256 23.0 -> 21.9, k 600 58.0 -> 53.9 (eight barriers before, ranks by LDS reads, scans by LDS permutes).
template <typename T, int U>
__device__ __forceinline__ void draw_from_small_list(Shared& s, const SampleParams& p, int row_idx, const T* row, bool vec_ok,
                                                     float m, bool has_topk, unsigned long long z_row) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), V = p.vocab;
    const int n = __builtin_amdgcn_readfirstlane((int)s.n_list);    // 1..NT
    // (key, ~index) as one number: one compare per pair
    s.list_w[tid] = tid < n ? (unsigned long long)s.list_key[tid] << 32 | ~s.list_idx[tid] : 0ull;
    __syncthreads();
    unsigned long long* sorted = s.mass;                            // descending; s.cnt: the ranks by index in this order
    const unsigned long long mine = s.list_w[NW * lane + wave];
    uint32_t ranks;
    if (n <= 128) ranks = list_ranks<2>(s.list_w, n, mine, lane, wave);
    else if (n <= 256) ranks = list_ranks<4>(s.list_w, n, mine, lane, wave);
    else if (n <= 384) ranks = list_ranks<6>(s.list_w, n, mine, lane, wave);
    else {                                                          // (1024 at a time: 32 registers)
        ranks = list_ranks<8>(s.list_w, n, mine, lane, wave);
        if (n > 512) ranks += list_ranks<8>(s.list_w + 512, n, mine, lane, wave);
    }
    if (NW * lane + wave < n) {
        sorted[ranks & 0xffffu] = mine;
        s.cnt[ranks & 0xffffu] = ranks >> 16;
    }
    __syncthreads();
    // lane t takes the t-th entry of the sorted order
    const uint32_t kth = has_topk && n >= p.top_k ? (uint32_t)(sorted[p.top_k - 1] >> 32) : 0u;   // fewer than k: all of them stay
    unsigned int by_index = 0, idx = 0;
    uint64_t w = 0;
    if (tid < n) {
        const unsigned long long e = sorted[tid];
        by_index = s.cnt[tid];
        idx = ~(uint32_t)e;
        if ((uint32_t)(e >> 32) >= kth) w = weight_of(key_value((uint32_t)(e >> 32)), m);        // ties at the k-th value all stay
    }
    unsigned long long z = 0;
    if (p.top_p < 1.f) {
        const unsigned long long before = block_scan(s, w, z);
        // an entry stays while the mass before it is at most top_p of the total (of the row's total
        // when the list is a cut of the whole row rather than its top k)
        const unsigned long long limit = (unsigned long long)((double)fmaxf(p.top_p, 0.f) * (double)(has_topk ? z : z_row));
        if (before > limit) w = 0;
    }
    if (tid < n) { s.list_w[by_index] = w; s.list_idx[by_index] = idx; }    // (both last read before the ranks were written)
    __syncthreads();
    w = 0;
    if (tid < n) { w = s.list_w[tid]; idx = s.list_idx[tid]; }
    const unsigned long long before = block_scan(s, w, z);              // kept mass at lower indices
    if (z == 0) {                                  // non-finite logits: fall back to the argmax
        no_mass<T, U>(s, p, row_idx, row, vec_ok);
        return;
    }
    unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z);
    if (target >= z) target = z - 1;
    if (before <= target && target < before + w) p.out[row_idx] = idx;
    if (p.probs_out) {
        for (int i = tid; i < V; i += NT) p.probs_out[(int64_t)row_idx * V + i] = 0.f;
        __syncthreads();
        const double inv_z = 1.0 / (double)z;
        if (w) p.probs_out[(int64_t)row_idx * V + idx] = (float)((double)w * inv_z);
    }
}
// The whole of a row by one workgroup.  U: loads in flight per lane.
template <typename T, int U>
__device__ __forceinline__ void sample_row(const SampleParams& p, Shared& s, int row_idx) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const int V = p.vocab;
    const float temp = p.temperature;

    // ---------------------------------------------------------------- 1. maximum
    // On the raw logits: dividing by a positive temperature keeps the order, so the maximum of
    // the scaled row is the scaled maximum and no division is needed in this pass (one v_max per
    // element).
    const bool vec_ok = ((uintptr_t)row % 16) == 0;
    float lane_best = -INFINITY;                      // raw maximum of this lane's share of the row
    for_each_logit<T, U>(row, 0, V, 1.f, tid, NT, vec_ok, [&](int, float x) { lane_best = fmaxf(lane_best, x); });
    float best = lane_best;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = fmaxf(best, __shfl_xor(best, o));
    if (lane == 0) s.red_f[wave] = best;
    __syncthreads();
    best = s.red_f[0];
    for (int w = 1; w < NW; ++w) best = fmaxf(best, s.red_f[w]);
    const float m = apply_temperature<T>(best, temp);

    auto over_row = [&](auto f) { for_each_logit<T, U>(row, 0, V, temp, tid, NT, vec_ok, f); };
    auto over_list = [&](auto f) {
        const int n = (int)s.n_list;
        for (int j = tid; j < n; j += NT) f((int)s.list_idx[j], key_value(s.list_key[j]));
    };

    // ---------------------------------------------------------------- 2. top-k: key of the k-th largest
    // With k <= 1024 the k-th largest of the 1024 per-lane maxima is a lower bound of the row's k-th
    // largest value (the maxima are elements of the row), so one more pass collects every
    // candidate (about k of them) into LDS, and selection, nucleus walk and draw run on that
    // list.  The pass compares raw keys against the bound lowered by LIST_SLACK representable
    // values (several raw values can divide to the same scaled value, and ties at the k-th
    // scaled value all stay) and divides only what passes.  A row whose candidates do not fit
    // (masses of equal values) takes the full-row walk.
    uint32_t key_k = 0;                          // keep keys >= key_k
    bool use_list = false;
    int nuc_first = 0;                           // nucleus walk already done down to this digit level (no top-k) ...
    uint32_t nuc_prefix = 0, nuc_pmask = 0;      // ... with this key prefix ...
    unsigned long long nuc_limit = 0;            // ... and this much of the mass limit left
    const bool topk_on = p.top_k > 0 && p.top_k < V;
    if (topk_on && p.top_k <= NT && temp <= LIST_MAX_TEMPERATURE) {
        auto over_lane_max = [&](auto f) { f(tid, lane_best); };
        // two digit levels (22 of 32 key bits): a bound 2^-13 relative below the k-th largest maximum
        // lets in a few more candidates and saves a histogram round
        const uint32_t key_l = select_kth(s, over_lane_max, (unsigned int)p.top_k, tid, lane, wave, 2);
        const uint32_t key_ls = order_key(apply_temperature<T>(key_value(key_l), temp));
        if (tid == 0) s.n_list = 0;
        __syncthreads();
        // the exact test on the scaled key follows the prefilter
        const float raw_lo = raw_bound<T>(key_l, key_ls, temp);
        for_each_logit<T, U>(row, 0, V, 1.f, tid, NT, vec_ok, [&](int i, float x) {
            if (!(x < raw_lo)) {
                const uint32_t key = order_key(apply_temperature<T>(x, temp));
                if (key >= key_ls) {
                    const unsigned int j = atomicAdd(&s.n_list, 1u);
                    if (j < LIST_CAP) { s.list_key[j] = key; s.list_idx[j] = (unsigned int)i; }
                }
            }
        });
        __syncthreads();
        use_list = s.n_list <= LIST_CAP;
    }
    if (use_list && s.n_list <= NT && s.n_list >= (unsigned int)p.top_k) {
        draw_from_small_list<T, U>(s, p, row_idx, row, vec_ok, m, true, 0ull);
        return;
    }

    // ---------------------------------------------------------------- 2b. nucleus without top-k
    // One pass gives the exact mass of the row and, for the logits within NUCLEUS_SPAN of the
    // maximum only (the rest cannot hold the threshold unless the row is very flat, and would cost
    // an LDS atomic each), a first-level mass histogram.  If the walk finds the threshold bin inside
    // that region, everything from that bin up is collected and, when it fits one candidate per
    // lane, handled like a top-k list.  Otherwise the full-row walk below runs.
    if (!topk_on && p.top_p < 1.f) {
        constexpr float NUCLEUS_SPAN = 12.f;
        const float cut_f = m - NUCLEUS_SPAN;
        const int nb0 = 1 << WIDTHS[0];
        for (int b2 = tid; b2 < BINS; b2 += NT) { s.mass[b2] = 0; s.cnt[b2] = 0; }
        if (tid == 0) s.n_list = 0;
        __syncthreads();
        unsigned long long zacc = 0;
        over_row([&](int, float x) {
            const uint64_t w = weight_of(x, m);
            zacc += w;
            if (x >= cut_f) {
                const int b2 = (int)(order_key(x) >> SHIFTS[0]) & (nb0 - 1);
                atomicAdd(&s.mass[b2], (unsigned long long)w);
                atomicAdd(&s.cnt[b2], 1u);
            }
        });
        zacc = wave_sum64(zacc);
        if (lane == 0) s.seg_mass[wave] = zacc;
        __syncthreads();
        unsigned long long z_row = 0;
        for (int wv = 0; wv < NW; ++wv) z_row += s.seg_mass[wv];
        if (z_row == 0) {
            no_mass<T, U>(s, p, row_idx, row, vec_ok);
            return;
        }
        const unsigned long long limit = (unsigned long long)((double)fmaxf(p.top_p, 0.f) * (double)z_row);
        if (wave == 0) pick_by_mass(s, nb0, limit, lane);
        __syncthreads();
        const uint32_t d0 = s.sel_digit;
        if (d0 > (order_key(cut_f) >> SHIFTS[0])) {               // the whole bin lies inside the histogrammed region
            // candidates from that bin up
            unsigned int c = (tid >= (int)d0 ? s.cnt[tid] : 0u) + (tid + NT >= (int)d0 ? s.cnt[tid + NT] : 0u);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
            if (lane == 0) s.seg_tied[wave] = c;
            __syncthreads();
            unsigned int n_est = 0;
            for (int wv = 0; wv < NW; ++wv) n_est += s.seg_tied[wv];
            const uint32_t key_lo_s = d0 << SHIFTS[0];
            if (n_est <= (unsigned int)NT) {
                // raw prefilter: the scaled bound times the temperature, lowered by more than the division
                // (and, for bf16 rows, the rounding of the quotient) can move a value
                const float t_raw = key_value(key_lo_s) * temp;
                float raw_lo = temp == 1.f ? key_value(key_lo_s)
                                           : t_raw - fabsf(t_raw) * (sizeof(T) == 2 ? 0.0078125f : 9.5367431640625e-7f);
                if constexpr (std::is_same<T, f16_t>::value) {
                    const float b = f16_raw_bound<T>(key_value(key_lo_s), temp);
                    if (b < raw_lo) raw_lo = b;
                }
                for_each_logit<T, U>(row, 0, V, 1.f, tid, NT, vec_ok, [&](int i, float x) {
                    if (!(x < raw_lo)) {
                        const uint32_t key = order_key(apply_temperature<T>(x, temp));
                        if (key >= key_lo_s) {
                            const unsigned int j = atomicAdd(&s.n_list, 1u);
                            if (j < LIST_CAP) { s.list_key[j] = key; s.list_idx[j] = (unsigned int)i; }
                        }
                    }
                });
                __syncthreads();
                if (s.n_list <= NT) {
                    draw_from_small_list<T, U>(s, p, row_idx, row, vec_ok, m, false, z_row);
                    return;
                }
            }
            // too many for a list: the full-row walk continues below from the second digit level
            nuc_first = 1;
            nuc_prefix = key_lo_s;
            nuc_pmask = (uint32_t)(nb0 - 1) << SHIFTS[0];
            nuc_limit = limit - s.sel_above_mass;
        }
        __syncthreads();
    }
    if (topk_on)
        key_k = use_list ? select_kth(s, over_list, (unsigned int)p.top_k, tid, lane, wave)
                         : select_kth(s, over_row, (unsigned int)p.top_k, tid, lane, wave);

    // ---------------------------------------------------------------- 3. nucleus threshold
    Nucleus nu;
    nu.key_t = key_k; nu.tie_keep = 0xffffffffu; nu.tie_rule = false;
    if (p.top_p < 1.f)
        nu = use_list ? nucleus_threshold(s, over_list, key_k, m, p.top_p, tid, lane, wave)
                      : nucleus_threshold(s, over_row, key_k, m, p.top_p, tid, lane, wave, nuc_first, nuc_prefix,
                                          nuc_pmask, nuc_limit);
    const uint32_t key_t = nu.key_t;
    const unsigned int tie_keep = nu.tie_keep;
    const bool tie_rule = nu.tie_rule;
    __syncthreads();

    if (use_list) {
        // ------------------------------------------------------------ 4a. draw from the candidate list
        // Every kept element is on the list.  Weights first (a tied element needs its rank among
        // the tied ones in index order), then each entry's mass-before in index order; both by
        // plain loops over the list, which holds about k entries.
        const int n = (int)s.n_list;
        const uint64_t w_tie = tie_rule ? weight_of(key_value(key_t), m) : 0;
        for (int j = tid; j < n; j += NT) {
            const uint32_t key = s.list_key[j];
            const unsigned int idx = s.list_idx[j];
            uint64_t w = 0;
            if (tie_rule ? key > key_t : key >= key_t) w = weight_of(key_value(key), m);
            else if (tie_rule && key == key_t) {
                unsigned int rank = 0;
                for (int i0 = 0; i0 < n; i0 += 8) {
                    uint32_t kk[8], ii[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) { kk[u] = s.list_key[min(i0 + u, n - 1)]; ii[u] = s.list_idx[min(i0 + u, n - 1)]; }
#pragma unroll
                    for (int u = 0; u < 8; ++u) rank += i0 + u < n && kk[u] == key_t && ii[u] < idx;
                }
                if (rank < tie_keep) w = w_tie;
            }
            s.list_w[j] = w;
        }
        __syncthreads();
        unsigned long long part = 0;
        for (int j = tid; j < n; j += NT) part += s.list_w[j];
        part = wave_sum64(part);
        if (lane == 0) s.seg_mass[wave] = part;
        __syncthreads();
        unsigned long long z2 = 0;
        for (int w = 0; w < NW; ++w) z2 += s.seg_mass[w];
        if (z2 == 0) {                                 // non-finite logits: fall back to the argmax
            no_mass<T, U>(s, p, row_idx, row, vec_ok);
            return;
        }
        unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z2);
        if (target >= z2) target = z2 - 1;
        if (p.probs_out) {
            for (int i = tid; i < V; i += NT) p.probs_out[(int64_t)row_idx * V + i] = 0.f;
            __syncthreads();
        }
        const double inv_z = 1.0 / (double)z2;
        if (p.probs_out)
            for (int j = tid; j < n; j += NT) {
                const uint64_t w = s.list_w[j];
                if (w) p.probs_out[(int64_t)row_idx * V + s.list_idx[j]] = (float)((double)w * inv_z);
            }
        // The draw in index order without comparing every pair of entries: kept mass per bucket of
        // consecutive indices (one bucket per lane), a scan over the buckets to find the one that
        // holds the target, then the few entries of that bucket among themselves.
        int sh = 0;
        while (((V - 1) >> sh) >= NT) ++sh;
        __syncthreads();
        s.mass[tid] = 0;                               // NT <= BINS buckets
        if (tid == 0) s.sel_above_cnt = 0;
        __syncthreads();
        for (int j = tid; j < n; j += NT) {
            const uint64_t w = s.list_w[j];
            if (w) atomicAdd(&s.mass[s.list_idx[j] >> sh], (unsigned long long)w);
        }
        __syncthreads();
        const unsigned long long mine_b = s.mass[tid];
        unsigned long long incl = wave_scan_dpp64(mine_b);
        if (lane == 63) s.seg_mass[wave] = incl;
        __syncthreads();
        unsigned long long base = 0;
        for (int w = 0; w < wave; ++w) base += s.seg_mass[w];
        incl += base;
        if (mine_b && incl - mine_b <= target && target < incl) {      // exactly one bucket
            s.sel_digit = (unsigned int)tid;
            s.sel_above_mass = incl - mine_b;
        }
        __syncthreads();
        const unsigned int bucket = s.sel_digit;
        const unsigned long long bucket_base = s.sel_above_mass;
        // the list positions of that bucket's entries go to the key array (the keys are no longer needed)
        for (int j = tid; j < n; j += NT)
            if (s.list_w[j] && (s.list_idx[j] >> sh) == bucket) s.list_key[atomicAdd(&s.sel_above_cnt, 1u)] = (unsigned int)j;
        __syncthreads();
        const int nb = (int)s.sel_above_cnt;           // at most n
        for (int a = tid; a < nb; a += NT) {
            const int j = (int)s.list_key[a];
            const unsigned int idx = s.list_idx[j];
            const unsigned long long w = s.list_w[j];
            unsigned long long before = bucket_base;
            for (int b = 0; b < nb; ++b) {
                const int i = (int)s.list_key[b];
                before += s.list_idx[i] < idx ? s.list_w[i] : 0ull;
            }
            if (before <= target && target < before + w) p.out[row_idx] = idx;
        }
        return;
    }

    // ---------------------------------------------------------------- 4. draw in index order
    // wave w owns the contiguous segment [w*seg, (w+1)*seg)
    const int seg = ((V + NW - 1) / NW + 63) / 64 * 64;
    const int s0 = wave * seg, s1 = min(V, s0 + seg);
    unsigned long long mass_gt = 0;
    unsigned int n_tied = 0;
    uint64_t w_t_val = 0;
    for_each_logit<T, U>(row, s0, max(s0, s1), temp, lane, 64, vec_ok, [&](int, float x) {
        const uint32_t key = order_key(x);
        if (tie_rule ? key > key_t : key >= key_t) mass_gt += weight_of(x, m);
        else if (tie_rule && key == key_t) ++n_tied;
    });
    if (tie_rule) w_t_val = weight_of(key_value(key_t), m);
    mass_gt = wave_sum64(mass_gt);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n_tied += __shfl_xor(n_tied, o);
    if (lane == 0) { s.seg_mass[wave] = mass_gt; s.seg_tied[wave] = n_tied; }
    __syncthreads();
    unsigned long long z2 = 0, my_base = 0, my_total = 0;
    unsigned int tied_base = 0, my_tied_base = 0;
    for (int w = 0; w < NW; ++w) {
        const unsigned int nt = s.seg_tied[w];
        const unsigned int kept = tie_rule ? (tied_base >= tie_keep ? 0u : min(nt, tie_keep - tied_base)) : 0u;
        const unsigned long long tot = s.seg_mass[w] + (unsigned long long)kept * w_t_val;
        if (w == wave) { my_base = z2; my_tied_base = tied_base; my_total = tot; }
        z2 += tot;
        tied_base += nt;
    }
    if (z2 == 0) {                                 // no mass at all (non-finite logits): fall back to the argmax
        no_mass<T, U>(s, p, row_idx, row, vec_ok);
        return;
    }
    unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z2);
    if (target >= z2) target = z2 - 1;
    const float inv_z = (float)(1.0 / (double)z2);
    auto weight_or_tie = [&](float x, bool& tied) -> uint64_t {
        const uint32_t key = order_key(x);
        tied = false;
        if (tie_rule ? key > key_t : key >= key_t) return weight_of(x, m);
        tied = tie_rule && key == key_t;
        return 0;
    };

    if (p.probs_out) {
        // the distribution itself, on request: every wave walks its segment in steps of 64 with a
        // running count of the tied elements seen so far
        unsigned int tied_seen = my_tied_base;
        for (int i0 = s0; i0 < s1; i0 += 64) {
            const int i = i0 + lane;
            uint64_t w = 0;
            bool tied = false;
            if (i < s1) w = weight_or_tie(scaled_logit<T>(row, i, temp), tied);
            const unsigned long long tb = __ballot(tied);
            if (tied && tied_seen + __popcll(tb & ((1ull << lane) - 1ull)) < tie_keep) w = w_t_val;
            tied_seen += __popcll(tb);
            if (i < s1) p.probs_out[(int64_t)row_idx * V + i] = (float)((double)w * (double)inv_z);
        }
    }

    // only the wave whose segment holds the target goes on
    if (!(my_base <= target && target < my_base + my_total)) return;

    // lane chunks of the segment: totals per lane, scans over the wave, then the owning lane's chunk
    // is walked by the whole wave
    const int chunk = ((s1 - s0 + 63) / 64 + 3) / 4 * 4;
    const int c0 = min(s1, s0 + lane * chunk), c1 = min(s1, c0 + chunk);
    unsigned long long lane_mass = 0;
    unsigned int lane_tied = 0;
    for_each_logit<T, U>(row, c0, c1, temp, 0, 1, vec_ok, [&](int, float x) {
        bool tied;
        lane_mass += weight_or_tie(x, tied);
        lane_tied += tied;
    });
    unsigned int tied_incl = lane_tied;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned int o = __shfl_up(tied_incl, d);
        if (lane >= d) tied_incl += o;
    }
    const unsigned int lane_tied_base = my_tied_base + tied_incl - lane_tied;
    if (tie_rule && lane_tied_base < tie_keep)
        lane_mass += (unsigned long long)min(lane_tied, tie_keep - lane_tied_base) * w_t_val;
    const unsigned long long incl = my_base + wave_scan_dpp64(lane_mass);
    const unsigned long long hit = __ballot(lane_mass != 0 && incl > target);
    if (!hit) return;                                          // cannot happen: the segment holds the target
    const int owner = __ffsll((long long)hit) - 1;
    unsigned long long running = shfl64(incl, owner) - shfl64(lane_mass, owner);
    unsigned int tied_seen = __shfl(lane_tied_base, owner);
    const int w0 = __shfl(c0, owner), w1 = __shfl(c1, owner);
    for (int i0 = w0; i0 < w1; i0 += 64) {
        const int i = i0 + lane;
        uint64_t w = 0;
        bool tied = false;
        if (i < w1) w = weight_or_tie(scaled_logit<T>(row, i, temp), tied);
        const unsigned long long tb = __ballot(tied);
        if (tied && tied_seen + __popcll(tb & ((1ull << lane) - 1ull)) < tie_keep) w = w_t_val;
        tied_seen += __popcll(tb);
        const unsigned long long sc = wave_scan_dpp64(w);
        const unsigned long long h2 = __ballot(w != 0 && running + sc > target);
        if (h2) {
            if (lane == __ffsll((long long)h2) - 1) p.out[row_idx] = i;
            return;
        }
        running += shfl64(sc, 63);
    }
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));      // as in wave_scan_dpp64
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// SLOTS entries per lane of the lists of a row's parts, read while their lengths are still on the way.
// Lane -> part lane >> lp of 2^(6 - lp) >= parts; a list goes round the waves in pieces of at most eight entries
// (64 bytes), so that their shares of it are alike.  TURN: each slot goes to the lanes of the next part, so that a list longer
// than its lanes has the other parts' too: the row's top may be in one part.
template <int SLOTS, bool TURN>
struct Lists {
    uint2 e[SLOTS];
    unsigned int count;                                      // entries of the list of the lane's part
    int at, stride;

    __device__ __forceinline__ void load(const SampleParams& p, int row_idx, int lane, int wave) {
        const int lp = __clz(p.parts - 1) - 26, piece = min(lp, 3);
        const int q = lane >> lp, l = lane & ((1 << lp) - 1);
        stride = NW << lp;
        at = ((((l >> piece) * NW) + wave) << piece) + (l & ((1 << piece) - 1));
        const unsigned int* counts = p.part_count + (int64_t)row_idx * p.parts;
        const uint2* lists = p.part_list + (int64_t)row_idx * p.parts * p.part_cap;
        auto part = [&](int u) { return TURN ? (q + u) & ((64 >> lp) - 1) : q; };
#pragma unroll
        for (int u = 0; u < SLOTS; ++u) {
            e[u] = make_uint2(0u, 0u);
            if (SLOTS <= 4 || u * stride < p.part_cap)
                e[u] = lists[(part(u) < p.parts ? part(u) : 0) * p.part_cap + min(at + u * stride, p.part_cap - 1)];
        }
        count = q < p.parts ? counts[q] : 0u;
    }
    // a list is longer than its lanes' SLOTS, or than its room
    __device__ __forceinline__ bool too_long(const SampleParams& p) const {
        return __any(count > (unsigned int)min(p.part_cap, SLOTS * stride));
    }
    __device__ __forceinline__ bool empty() const { return !__any(count != 0u); }
    // whether any lane of the wave has an entry in slot u
    __device__ __forceinline__ bool used(int u) const { return SLOTS <= 4 || __any((unsigned int)(u * stride) < count); }
    // key 0 (no candidate has it) beyond a list's end; the lane's largest key
    __device__ __forceinline__ uint32_t trim(int lane) {
        uint32_t top = 0;
#pragma unroll
        for (int u = 0; u < SLOTS; ++u) {
            if (!used(u)) break;
            const unsigned int c = TURN && u ? __shfl(count, (lane + u * (stride / NW)) & 63) : count;
            if ((unsigned int)(at + u * stride) >= c) e[u].x = 0u;
            top = max(top, e[u].x);
        }
        return top;
    }
};

// A bound of the row's top_k-th largest key from below, 1 at least, out of the lanes' largest ones: the largest of the waves'
// bounds that top_k lanes of all waves reach (the smallest of the sixteen always is such a one, but lets several times as
// many pass).  s.cnt[0 .. NW) is zero before; two barriers.
__device__ __forceinline__ uint32_t bound_of_lanes(const SampleParams& p, Shared& s, uint32_t top, int lane, int wave) {
    const uint32_t bound = wave_rth_bound(top, (p.top_k + NW - 1) / NW);
    if (lane == 0) s.seg_tied[wave] = bound;
    __syncthreads();
    const uint32_t t = s.seg_tied[lane & 15];
    unsigned int reach = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const unsigned int r = (unsigned int)__popcll(__ballot(top >= (uint32_t)__builtin_amdgcn_readlane((int)t, w)));
        reach = lane == w ? r : reach;
    }
    if (lane < NW) atomicAdd(&s.cnt[lane], reach);
    __syncthreads();
    return max(largest_of_16(s.cnt[lane & 15] >= (unsigned int)p.top_k ? t : 0u), 1u);
}

// The usual draw from the candidates of a row's parts, top_k <= FewK: false (for the whole workgroup, nothing written)
// where a list is longer than its lanes' FEW_SLOTS, more than FEW candidates pass the bound or, with the ties of the k-th,
// more than 64 stay.
//
// Latency bound, one workgroup per row: what it takes is a chain of memory and LDS latencies and barriers, so it has
// three of the latter.  The lists are read while their lengths are still on the way; a candidate's rank is counted with
// one 64-bit compare and a ballot per 64 others, a wave for the candidates of four lanes; and once they are in order
// at most 64 are left, which the first wave finishes in registers.  64 rows of eight parts, k = 50: 11.5 -> 5.2 us as traced (about ten barriers before, the mass
// before an entry by two scans over all waves).
constexpr int FEW = 256, FEW_K = 64;
// 16-bit logits lie close enough for ties (bf16 a sixteenth apart between 8 and 16), so with k near 64 those of the k-th are
// often a lane too many, and one such row holds up the launch.  64 rows of 32000, one launch, then parts: bf16 k 56 15.1 and
// 13.2 us, k 60 15.2 and 16.8, k 64 15.4 and 17.6; fp16 k 60 15.3 and 13.4, k 64 15.4 and 17.5; 256 rows, k 64 15.5 and 20.2.
template <typename T> struct FewK { static constexpr int value = FEW_K; };
template <> struct FewK<bf16_t> { static constexpr int value = 56; };
template <> struct FewK<f16_t> { static constexpr int value = 60; };
constexpr int FEW_SLOTS = 4;               // 512 entries of a list of eight parts; at k = 50 one in 60 rows has a longer one than 256
template <typename T>
__device__ __forceinline__ bool merge_few(const SampleParams& p, Shared& s, int row_idx) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    Lists<FEW_SLOTS, false> lists;
    lists.load(p, row_idx, lane, wave);
    if (tid < FEW) s.list_w[tid] = 0;
    if (tid < NW) s.cnt[tid] = 0;
    if (tid == 0) s.n_list = 0;
    if (lists.too_long(p) || lists.empty()) return false;
    const uint32_t top = lists.trim(lane);
    const uint2 (&e)[FEW_SLOTS] = lists.e;
    const uint32_t key_l = bound_of_lanes(p, s, top, lane, wave);
    unsigned long long pass[FEW_SLOTS];
    unsigned int mine_n = 0;
#pragma unroll
    for (int u = 0; u < FEW_SLOTS; ++u) {
        pass[u] = __ballot(e[u].x >= key_l);
        mine_n += (unsigned int)__popcll(pass[u]);
    }
    unsigned int j = 0;
    if (lane == 0 && mine_n) j = atomicAdd(&s.n_list, mine_n);
    j = __builtin_amdgcn_readfirstlane(j);
#pragma unroll
    for (int u = 0; u < FEW_SLOTS; ++u) {
        const unsigned int at_u = j + __popcll(pass[u] & ((1ull << lane) - 1ull));
        if (e[u].x >= key_l && at_u < FEW) s.list_w[at_u] = (unsigned long long)e[u].x << 32 | ~e[u].y;
        j += (unsigned int)__popcll(pass[u]);
    }
    __syncthreads();
    const int n = (int)s.n_list;
    if (n > FEW) return false;
    // ranks by (key, then index): entry 64 g + l in lane l, this wave counts for the entries of lanes 4 wave ..
    unsigned long long x[FEW / 64];
#pragma unroll
    for (int g = 0; g < FEW / 64; ++g) x[g] = s.list_w[64 * g + lane];
    unsigned long long* sorted = s.mass;
#pragma unroll
    for (int g = 0; g < FEW / 64; ++g) {
        if (64 * g >= n) break;
        int rank = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned long long me = readlane64(x[g], 4 * wave + i);
            int r = 0;
#pragma unroll
            for (int h = 0; h < FEW / 64; ++h) r += __popcll(__ballot(x[h] > me));       // (zeros are above nothing)
            rank = lane == 4 * wave + i ? r : rank;
        }
        if (lane >> 2 == wave && x[g] != 0) sorted[rank] = x[g];
    }
    __syncthreads();
    const uint32_t kth = n >= p.top_k ? (uint32_t)(sorted[p.top_k - 1] >> 32) : 1u;        // fewer than k: all of them stay
    const uint32_t key_m = (uint32_t)(sorted[0] >> 32);
    const bool ties = n > FEW_K && (uint32_t)(sorted[FEW_K] >> 32) >= kth;           // more than a lane each
    if (ties || !(key_value(key_m) < INFINITY)) return false;
    if (wave != 0) return true;
    // lane t: the t-th largest.  Nucleus: an entry stays while the mass before it is at most top_p of the total.
    const unsigned long long mine = lane < n ? sorted[lane] : 0;
    const uint32_t key = (uint32_t)(mine >> 32);
    const bool stays = key >= kth;
    unsigned int idx = ~(uint32_t)mine;
    unsigned long long w = stays ? weight_of(key_value(key), key_value(key_m)) : 0;
    int left = __popcll(__ballot(stays));                                     // lanes 0 .. left - 1
    if (p.top_p < 1.f) {
        const unsigned long long incl = wave_scan_dpp64(w), z = readlane64(incl, 63);
        const unsigned long long limit = (unsigned long long)((double)fmaxf(p.top_p, 0.f) * (double)z);
        if (incl - w > limit) w = 0;
        left = __popcll(__ballot(stays && incl - w <= limit));
    }
    // into index order: a lane's place is the number of lower indices
    int place = 0;
    for (int u = 0; u < left; ++u) place += (unsigned int)__builtin_amdgcn_readlane((int)idx, u) < idx ? 1 : 0;
    if (lane >= left) { place = lane; w = 0; }
    idx = (unsigned int)__builtin_amdgcn_ds_permute(4 * place, (int)idx);
    const uint32_t w_lo = (uint32_t)__builtin_amdgcn_ds_permute(4 * place, (int)(uint32_t)w);
    const uint32_t w_hi = (uint32_t)__builtin_amdgcn_ds_permute(4 * place, (int)(uint32_t)(w >> 32));
    w = (unsigned long long)w_hi << 32 | w_lo;
    const unsigned long long incl = wave_scan_dpp64(w), z = readlane64(incl, 63);
    unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z);
    if (target >= z) target = z - 1;
    if (incl - w <= target && target < incl) p.out[row_idx] = idx;
    return true;
}

// The draw from the candidates of a row's parts: those of all parts hold the row's top k, with ties (all finite
// logits if there are fewer).  Beyond merge_few's the lists are read and bounded as there, but turned, which leaves little more than
// k candidates (230 at k = 200) for draw_from_small_list.  A row that its parts gave up, or with more than a lane's each, is done
// whole.  16 rows of 128256, parts and merge, by replayed graphs: k 100 21.2 -> 18.4 us, k 200 27.1 -> 21.0, k 256 32.5 -> 23.6 (before, a
// list's entry was found by comparisons with all lists' ends, and the smallest of the waves' bounds let in twice as many; slots
// that no lane has an entry for took 1.1).  A language model's rows have their top in few parts: logits of deviation 2.5 less
// ln(1 + index), 64 rows of 128256, k 200 30.2 -> 27.2, k 256 33.1 -> 30.6; with lists that keep to their part's lanes, fewer than k of
// them then, such rows were done whole, 33.5 and 51.2.
template <typename T>
__global__ void __launch_bounds__(NT)
sample_merge_kernel(SampleParams p) {
    __shared__ Shared s;
    const int row_idx = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const bool vec_ok = ((uintptr_t)row % 16) == 0;
    if (p.top_k <= FewK<T>::value && p.probs_out == nullptr) {
        if (merge_few<T>(p, s, row_idx)) return;
        __syncthreads();
    }
    Lists<MERGE_SLOTS, true> lists;
    lists.load(p, row_idx, lane, wave);
    if (tid < NW) s.cnt[tid] = 0;
    if (tid == 0) s.n_list = 0;
    if (!lists.too_long(p)) {
        if (lists.empty()) {                 // nothing above -inf
            no_mass<T, 4>(s, p, row_idx, row, vec_ok);
            return;
        }
        const uint32_t top = lists.trim(lane);
        const uint2 (&e)[MERGE_SLOTS] = lists.e;
        const uint32_t largest = wave_max(top);
        if (lane == 0) s.red_i[wave] = (int)largest;
        const uint32_t key_l = bound_of_lanes(p, s, top, lane, wave);
        const uint32_t key_m = wave_max((uint32_t)s.red_i[lane & 15]);
        unsigned int mine_n = 0;
#pragma unroll
        for (int u = 0; u < MERGE_SLOTS; ++u) {
            if (!lists.used(u)) break;
            mine_n += (unsigned int)__popcll(__ballot(e[u].x >= key_l));
        }
        unsigned int j = 0;
        if (lane == 0 && mine_n) j = atomicAdd(&s.n_list, mine_n);
        j = __builtin_amdgcn_readfirstlane(j);
#pragma unroll
        for (int u = 0; u < MERGE_SLOTS; ++u) {
            if (!lists.used(u)) break;
            const unsigned long long pass = __ballot(e[u].x >= key_l);
            const unsigned int at = j + __popcll(pass & ((1ull << lane) - 1ull));
            if (e[u].x >= key_l && at < NT) { s.list_key[at] = e[u].x; s.list_idx[at] = e[u].y; }
            j += (unsigned int)__popcll(pass);
        }
        __syncthreads();
        if (s.n_list <= NT) {
            draw_from_small_list<T, 4>(s, p, row_idx, row, vec_ok, key_value(key_m), true, 0ull);
            return;
        }
    }
    __syncthreads();
    sample_row<T, 4>(p, s, row_idx);
}

// A draw from the whole row (neither top-k nor top-p), the row cut into parts of sixteen segments: the parts' maxima, the
// segments' masses under the row's maximum (whole numbers, so any order of the sum gives the same one), and the
// element within the segment that holds the target.
//
// One CU reads a row of 128256 float32 twice in 40 us, at its 64 bytes per clock and with an exponential per logit; three
// launches of a few latencies each have the whole chip for it.  64 rows of 128256 float32: 54.9 -> 16.0 us.
//
// A nucleus (top_p alone) goes the same way with one launch more: the masses of 2048 slices of logits below the
// maximum give the slice that holds the threshold (a few dozen logits of a usual row), and what lies above it is summed by
// segment.  64 rows: 45.7 -> 34.5 us (38.4 while every part read its row's 2048 slices of all parts, 128 KB, where it now reads
// the sums of 64 groups of them and one group); 8 rows 42.2 -> 23.8.
// Rows of unit variance at temperature 1, whose nucleus is half the row: 64 rows 154 -> 60 us.  Nearly flat rows, whose
// threshold slice holds more logits than the lists, are done whole after the three launches, see sample_parts().
constexpr int SEG = PART_MAX / NW;                  // logits of a segment, one wave's: 16 per lane
// The lane's sixteen logits of the segment [begin, begin + n), -inf beyond it: four groups of four, 256 apart (IN_ORDER:
// next to each other).
template <typename T, bool IN_ORDER>
__device__ __forceinline__ void load_segment(const T* row, int begin, int n, bool vec_ok, int lane, float (&x)[PART_SLOTS]) {
    if (vec_ok && n == SEG) {
#pragma unroll
        for (int u = 0; u < PART_SLOTS / 4; ++u)
            Load4<T>::get(row + begin + (IN_ORDER ? PART_SLOTS * lane + 4 * u : 4 * (lane + 64 * u)), x + 4 * u);
    } else {
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i)
            x[i] = scaled_logit<T>(row, begin + max(0, min(IN_ORDER ? PART_SLOTS * lane + i : lane + 64 * i, n - 1)), 1.f);
#pragma unroll
        for (int i = 0; i < PART_SLOTS; ++i)
            if ((IN_ORDER ? PART_SLOTS * lane + i : lane + 64 * i) >= n) x[i] = -INFINITY;
    }
}
// Segment `seg` (part NW + wave) of a row: where it begins, how many logits it has (0 or less: none).
__device__ __forceinline__ int segment_begin(const SampleParams& p, int seg, int& n) {
    const int part = seg / NW, begin = part * p.part_size + seg % NW * SEG;
    n = min(SEG, min(p.vocab, (part + 1) * p.part_size) - begin);
    return n > 0 ? begin : 0;
}

template <typename T>
__global__ void __launch_bounds__(NT)
sample_max_kernel(SampleParams p) {
    __shared__ float red[NW];
    const int row_idx = blockIdx.x, part = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    int n;
    const int begin = segment_begin(p, part * NW + wave, n);
    float x[PART_SLOTS];
    load_segment<T, false>(row, begin, n, ((uintptr_t)row % 16) == 0, lane, x);
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) best = fmaxf(best, x[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = fmaxf(best, __shfl_xor(best, o));
    if (lane == 0) red[wave] = best;
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int w = 0; w < NW; ++w) best = fmaxf(best, red[w]);
        p.part_max[(int64_t)row_idx * p.parts + part] = best;
    }
}

// (the loads of a loop over the parts would be waited for one by one)
__device__ __forceinline__ float row_max_of_parts(const SampleParams& p, int row_idx, int lane) {
    float best = p.part_max[(int64_t)row_idx * p.parts + min(lane, p.parts - 1)];
#pragma unroll
    for (int o = MAX_PARTS / 2; o > 0; o >>= 1) best = fmaxf(best, __shfl_xor(best, o));
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(best)));
}

// Slices of the logits below the row's maximum, for the nucleus threshold: 160 to a unit, 12.8 units in all.
constexpr int NBINS = 2048;
constexpr float BINS_PER_UNIT = 160.f;
constexpr int GROUPS = 64, GROUP = NBINS / GROUPS;
constexpr int NUCLEUS_CAP = 512;                    // logits of a part in one slice
__device__ __forceinline__ int slice_of(float x, float m) {          // never falls as x does; NBINS: below all of them, or NaN
    const float d = (m - x) * BINS_PER_UNIT;
    return d < (float)NBINS ? (int)d : NBINS;
}

// NUCLEUS: the masses of the slices too, by LDS atomics.
template <typename T, bool NUCLEUS>
__global__ void __launch_bounds__(NT)
sample_mass_kernel(SampleParams p) {
    __shared__ alignas(16) unsigned long long hist[NUCLEUS ? NBINS : 2];
    const int row_idx = blockIdx.x, part = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const int64_t slot = (int64_t)row_idx * p.parts + part;
    int n;
    const int begin = segment_begin(p, part * NW + wave, n);
    float x[PART_SLOTS];
    load_segment<T, false>(row, begin, n, ((uintptr_t)row % 16) == 0, lane, x);
    const float m = apply_temperature<T>(row_max_of_parts(p, row_idx, lane), p.temperature);
    if constexpr (NUCLEUS) {
        for (int b = tid; b < NBINS; b += NT) hist[b] = 0;
        __syncthreads();
    }
    unsigned long long mass = 0;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) {
        const float v = apply_temperature<T>(x[i], p.temperature);
        const unsigned long long w = weight_of(v, m);
        mass += w;
        if constexpr (NUCLEUS) {
            const int b = slice_of(v, m);
            if (b < NBINS) atomicAdd(&hist[b], w);
        }
    }
    mass = readlane64(wave_scan_dpp64(mass), 63);
    if (lane == 0) p.seg_mass[slot * NW + wave] = mass;
    if constexpr (NUCLEUS) {
        __syncthreads();
        static_assert(NBINS == 2 * NT && GROUP == 32, "two slices per lane, a group per sixteen lanes");
        const ulonglong2 h = *(const ulonglong2*)(hist + 2 * tid);
        *(ulonglong2*)(p.part_hist + slot * NBINS + 2 * tid) = h;
        unsigned long long g = h.x + h.y;
        g = dpp_add64<0x111, 0xf>(g);            // row_shr 1, 2, 4, 8: the last of sixteen lanes has their sum
        g = dpp_add64<0x112, 0xf>(g);
        g = dpp_add64<0x114, 0xf>(g);
        g = dpp_add64<0x118, 0xf>(g);
        if ((lane & 15) == 15) p.part_group[slot * GROUPS + tid / 16] = g;
    }
}

// A lane's segments of a row, in index order, and their masses
constexpr int SEGS = MAX_PARTS * NW, SEGS_PER_LANE = SEGS / 64;
__device__ __forceinline__ unsigned long long lane_segments(const unsigned long long* segs, int nsegs, int lane,
                                                            unsigned long long (&w)[SEGS_PER_LANE]) {
    unsigned long long mine = 0;
#pragma unroll
    for (int j = 0; j < SEGS_PER_LANE; ++j) {
        const unsigned long long v = segs[min(SEGS_PER_LANE * lane + j, nsegs - 1)];
        w[j] = SEGS_PER_LANE * lane + j < nsegs ? v : 0;
        mine += w[j];
    }
    return mine;
}
// The segment that holds `target` and the mass before it (the whole wave; `incl`: of the segments up to this lane's).
__device__ __forceinline__ int find_segment(const unsigned long long (&w)[SEGS_PER_LANE], unsigned long long mine,
                                            unsigned long long incl, unsigned long long target, int lane,
                                            unsigned long long& base) {
    int seg = 0;
    unsigned long long before = incl - mine;
    bool found = false;
    base = 0;
#pragma unroll
    for (int j = 0; j < SEGS_PER_LANE; ++j) {
        if (w[j] && before <= target && target < before + w[j]) { seg = SEGS_PER_LANE * lane + j; base = before; found = true; }
        before += w[j];
    }
    const unsigned long long hit = __ballot(found);                 // one lane: the target is below the sum
    const int owner = hit ? __ffsll((long long)hit) - 1 : 0;
    base = readlane64(base, owner);
    return __builtin_amdgcn_readlane(seg, owner);
}
// The draw within a segment: the element whose share of the mass, after `at` before this lane's first, holds `target`.
__device__ __forceinline__ void draw_in_lane(const SampleParams& p, int row_idx, int first, const unsigned long long (&w)[PART_SLOTS],
                                             unsigned long long at, unsigned long long target) {
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) {
        if (w[i] && at <= target && target < at + w[i]) p.out[row_idx] = first + i;
        at += w[i];
    }
}

template <typename T>
__global__ void __launch_bounds__(NT)
sample_locate_kernel(SampleParams p) {
    __shared__ struct { float red_f[NW]; int red_i[NW]; } s;
    const int row_idx = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const bool vec_ok = ((uintptr_t)row % 16) == 0;
    unsigned long long w[SEGS_PER_LANE];
    const unsigned long long mine = lane_segments(p.seg_mass + (int64_t)row_idx * p.parts * NW, p.parts * NW, lane, w);
    const unsigned long long incl = wave_scan_dpp64(mine), z = readlane64(incl, 63);
    if (z == 0) {                                   // the same in every wave
        no_mass<T, 4>(s, p, row_idx, row, vec_ok);
        return;
    }
    if (wave != 0) return;
    unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z), base;
    if (target >= z) target = z - 1;
    int n;
    const int begin = segment_begin(p, find_segment(w, mine, incl, target, lane, base), n);
    float x[PART_SLOTS];
    load_segment<T, true>(row, begin, n, vec_ok, lane, x);
    const float m = apply_temperature<T>(row_max_of_parts(p, row_idx, lane), p.temperature);
    unsigned long long we[PART_SLOTS], sum = 0;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) {
        we[i] = weight_of(apply_temperature<T>(x[i], p.temperature), m);
        sum += we[i];
    }
    draw_in_lane(p, row_idx, begin + PART_SLOTS * lane, we, base + wave_scan_dpp64(sum) - sum, target);
}

// Sum over the parts of a row of the lane's element of `at` (n of them per part)
__device__ __forceinline__ unsigned long long sum_of_parts(const unsigned long long* at, int n, int parts, int i) {
    unsigned long long sum = 0;
    for (int q0 = 0; q0 < parts; q0 += 8) {
        unsigned long long h[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) h[q] = at[(int64_t)min(q0 + q, parts - 1) * n + i];
#pragma unroll
        for (int q = 0; q < 8; ++q) sum += q0 + q < parts ? h[q] : 0ull;
    }
    return sum;
}
// The first of the wave's entries at which the running sum passes `left` (64: none); `left` less what lies before it.
__device__ __forceinline__ int pass_point(unsigned long long mine, unsigned long long& left) {
    const unsigned long long incl = wave_scan_dpp64(mine);
    const unsigned long long over = __ballot(incl > left);
    if (!over) return 64;
    const int at = __ffsll((long long)over) - 1;
    left -= readlane64(incl - mine, at);
    return at;
}

// The slice that holds the nucleus threshold, from the parts' slices: what lies above it is summed by segment, its own
// logits leave the part as a list.
template <typename T>
__global__ void __launch_bounds__(NT)
sample_slice_kernel(SampleParams p) {
    __shared__ unsigned int n_list;
    const int row_idx = blockIdx.x, part = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const int64_t slot = (int64_t)row_idx * p.parts + part;
    int n;
    const int begin = segment_begin(p, part * NW + wave, n);
    const bool vec = ((uintptr_t)row % 16) == 0 && n == SEG;
    float x[PART_SLOTS];
    load_segment<T, false>(row, begin, n, ((uintptr_t)row % 16) == 0, lane, x);
    if (tid == 0) n_list = 0;
    unsigned long long w[SEGS_PER_LANE];
    const unsigned long long mine = lane_segments(p.seg_mass + (int64_t)row_idx * p.parts * NW, p.parts * NW, lane, w);
    // every wave for itself: the group of slices, then the slice, at which the sum passes the limit
    const unsigned long long groups = sum_of_parts(p.part_group + (int64_t)row_idx * p.parts * GROUPS, GROUPS, p.parts, lane);
    const unsigned long long z = readlane64(wave_scan_dpp64(mine), 63);
    unsigned long long left = (unsigned long long)((double)fmaxf(p.top_p, 0.f) * (double)z);
    const int group = pass_point(groups, left);
    int slice = NBINS;                               // the slices do not reach it (or there is no mass)
    if (group < GROUPS) {
        const int64_t at = (int64_t)row_idx * p.parts * NBINS + group * GROUP;
        const unsigned long long h = sum_of_parts(p.part_hist + at, NBINS, p.parts, lane % GROUP);
        slice = group * GROUP + pass_point(lane < GROUP ? h : 0, left);
    }
    __syncthreads();
    if (part == 0 && tid == 0) { p.cut[2 * row_idx] = slice; p.cut[2 * row_idx + 1] = left; }
    if (slice == NBINS) return;
    const float m = apply_temperature<T>(row_max_of_parts(p, row_idx, lane), p.temperature);
    uint2* list = p.part_list + slot * NUCLEUS_CAP;
    unsigned long long mass = 0;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) {
        const float v = apply_temperature<T>(x[i], p.temperature);
        const int b = slice_of(v, m);
        if (b < slice) mass += weight_of(v, m);
        if (b == slice) {
            const unsigned int j = atomicAdd(&n_list, 1u);
            const int at = vec ? 4 * (lane + 64 * (i / 4)) + (i & 3) : lane + 64 * i;
            if (j < NUCLEUS_CAP) list[j] = make_uint2(order_key(v), (unsigned int)(begin + at));
        }
    }
    mass = readlane64(wave_scan_dpp64(mass), 63);
    if (lane == 0) p.kept_mass[slot * NW + wave] = mass;
    __syncthreads();
    if (tid == 0) p.part_count[slot] = n_list;
}

// The draw from the nucleus.  Of the slice's logits those stay whose mass before them, by falling value and then by
// index, is at most what is left of the limit; with them added to their segments the draw goes as from the whole row.
// A row whose slice was not found, or holds more logits than the lanes, is done whole.
template <typename T>
__global__ void __launch_bounds__(NT)
sample_nucleus_kernel(SampleParams p) {
    __shared__ Shared s;
    __shared__ unsigned int stays[SEG / 32];
    const int row_idx = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    const int nsegs = p.parts * NW, slice = (int)p.cut[2 * row_idx];
    const unsigned long long left = p.cut[2 * row_idx + 1];
    int total = 0, mine_at = -1;                    // this lane's entry of the parts' lists
    if (slice < NBINS) {
        const int counts = lane < p.parts ? (int)p.part_count[(int64_t)row_idx * p.parts + lane] : 0;
        const bool fits = !__any(counts > NUCLEUS_CAP);
        for (int q = 0; q < p.parts; ++q) {
            const int c = __builtin_amdgcn_readlane(counts, q);
            if (tid >= total && tid < total + c) mine_at = q * NUCLEUS_CAP + tid - total;
            total += c;
        }
        if (!fits) total = NT + 1;
    }
    if (slice == NBINS || total > NT) {             // the same in every lane
        sample_row<T, 4>(p, s, row_idx);
        return;
    }
    const float m = apply_temperature<T>(row_max_of_parts(p, row_idx, lane), p.temperature);
    unsigned long long* segs = s.mass;              // [SEGS]
    if (tid < SEGS) segs[tid] = tid < nsegs ? p.kept_mass[(int64_t)row_idx * nsegs + tid] : 0;
    if (tid < SEG / 32) stays[tid] = 0;
    // entries with a larger order come first; zeros are no entries
    unsigned long long me = 0, w = 0;
    if (mine_at >= 0) {
        const uint2 e = p.part_list[(int64_t)row_idx * p.parts * NUCLEUS_CAP + mine_at];
        me = (unsigned long long)e.x << 32 | ~e.y;
        w = weight_of(key_value(e.x), m);
    }
    unsigned long long* order = s.list_w;
    unsigned long long* weight = s.list_w + NT;
    order[tid] = me;
    weight[tid] = w;
    __syncthreads();
    unsigned long long before = 0;
    for (int j0 = 0; j0 < total; j0 += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) before += order[j0 + j] > me ? weight[j0 + j] : 0ull;       // (NT is a multiple of 8)
    }
    const bool stay = me != 0 && before <= left;
    const int idx = (int)~(unsigned int)me, part = stay ? idx / p.part_size : 0, in_part = idx - part * p.part_size;
    const int seg = part * NW + in_part / SEG;
    if (stay) atomicAdd(&segs[seg], w);
    __syncthreads();
    unsigned long long ws[SEGS_PER_LANE];
    const unsigned long long mine = lane_segments(segs, SEGS, lane, ws);
    const unsigned long long incl = wave_scan_dpp64(mine), z = readlane64(incl, 63);
    unsigned long long target = (unsigned long long)((double)p.uniforms[row_idx] * (double)z), base;
    if (target >= z) target = z - 1;
    const int at_seg = find_segment(ws, mine, incl, target, lane, base);     // in every wave alike
    if (stay && seg == at_seg) atomicOr(&stays[in_part % SEG / 32], 1u << (in_part & 31));
    __syncthreads();
    if (wave != 0) return;
    int n;
    const int begin = segment_begin(p, at_seg, n);
    float x[PART_SLOTS];
    load_segment<T, true>(row, begin, n, ((uintptr_t)row % 16) == 0, lane, x);
    const unsigned int mask = stays[lane / 2] >> PART_SLOTS * (lane & 1);
    unsigned long long we[PART_SLOTS], sum = 0;
#pragma unroll
    for (int i = 0; i < PART_SLOTS; ++i) {
        const float v = apply_temperature<T>(x[i], p.temperature);
        const int b = slice_of(v, m);
        we[i] = b < slice || (b == slice && (mask >> i & 1u)) ? weight_of(v, m) : 0ull;
        sum += we[i];
    }
    draw_in_lane(p, row_idx, begin + PART_SLOTS * lane, we, base + wave_scan_dpp64(sum) - sum, target);
}

template <typename T>
__global__ void __launch_bounds__(NT)
sample_kernel(SampleParams p) {
    __shared__ Shared s;
    sample_row<T, 16>(p, s, blockIdx.x);
}

// Greedy: the argmax, from the parts' candidates if there are any.
template <typename T>
__global__ void __launch_bounds__(NT)
greedy_kernel(SampleParams p) {
    __shared__ Shared s;
    const int row_idx = blockIdx.x, tid = threadIdx.x, V = p.vocab;
    const T* row = (const T*)p.logits + (int64_t)row_idx * p.row_stride;
    int best_i;
    if (p.parts) {
        uint2 c = p.part_list[(int64_t)row_idx * p.parts * GREEDY_CAP];
        for (int q = 1; q < p.parts; ++q) {
            const uint2 o = p.part_list[((int64_t)row_idx * p.parts + q) * GREEDY_CAP];
            if (o.x > c.x || (o.x == c.x && o.y < c.y)) c = o;
        }
        best_i = c.y == 0x7fffffffu ? 0 : (int)c.y;
    } else {
        best_i = block_argmax<T, 16>(s, row, V, ((uintptr_t)row % 16) == 0);
    }
    if (tid == 0) p.out[row_idx] = best_i;
    if (p.probs_out)
        for (int i = tid; i < V; i += NT) p.probs_out[(int64_t)row_idx * V + i] = i == best_i ? 1.f : 0.f;
}

}  // namespace

// How many parts the rows of a call are cut into (1: none).  A second launch and the merge cost about 5 us for top_k <= FewK
// (merge_few) and 7 to 10 us beyond, so it has to save more.  us per call, one launch -> parts:
//   few (k 50)          float32  20000, 2 parts: 1 row 14.4 -> 10.0, 64 15.8 -> 11.3, 1024 61.3 -> 44.3
//                                50256, 4 parts: 1 row 16.0 -> 10.9, 64 16.7 -> 11.7, 128 17.2 -> 13.9, 1024 86.7 -> 66.5
//                                128256, 8 parts: 1 row 20 -> 10.7, 64 23 -> 14.4, 512 88 -> 61;  262144: 16 rows 29 -> 11.3
//                       16-bit   32000: 64 rows 16.6 -> 11.6, 1024 63.4 -> 45.6;  81920: 64 20.7 -> 13.9, 1024 90.4 -> 78.8
//                                128256: 64 rows 22.3 -> 13.9, 128 22.5 -> 20.3, 1024 109 -> 115;  262144: 64 31.7 -> 25.8,
//                                128 34.2 -> 37.9 (half the bytes to save on): six parts and more up to 1024 parts
//                                up to 256 rows of one launch are under way together, parts 512 at a time (k 20, of 40000, 65536
//                                and 81920): 160 rows 14.4 -> 13.7, 128 15.3 -> 13.9, 128 18.1 -> 16.3;  256 rows 14.6 -> 16.7,
//                                15.5 -> 19.6, 224 18.8 -> 21.9;  288 rows 26.8 -> 22.9, 28.9 -> 26.5, 39.2 -> 29.2.  512 of
//                                65536: k 50 35.7 -> 39.1, with top_p 0.9 39.4 -> 36.8 (which the line does not know)
//                       float32, k 64  32768, 2 parts: 128 rows 14.7 -> 13.8, 256 14.9 -> 17.2, 288 27.9 -> 26.3;  65536, 4: 128
//                                15.8 -> 17.3, 192 26.1 -> 21.9
//   rows whose loads cannot be vectors (a stride that is no multiple of 16 bytes): at once
//     bf16, k 50        50257: 64 rows 24.4 -> 17.3;  greedy float32 50257: 64 rows 11.4 -> 7.6
//   the whole row       float32  20000, 2 parts: 1 row 14.8 -> 10.9, 1024 62.9 -> 49.3;  50256: 64 rows 26.3 -> 11.7
//   (top_p off)         128256: 1 row 50.9 -> 11.3, 64 54.9 -> 16.0, 1024 281 -> 203;  262144: 64 rows 106 -> 31.5
//                       bf16     20000: 64 rows 17.5 -> 12.1, 1024 66.2 -> 42.7;  128256: 64 61.0 -> 16.0, 1024 258 -> 146
//   k to 256            float32  40000, 3 parts: k 65 1 row 15.4 -> 13.3, 64 15.7 -> 14.4, 96 15.8 -> 16.5;  k 200 18.9 -> 16.4, 19.5 -> 17.6,
//   from three parts on          19.6 -> 20.4;  50256, 4: k 200 64 rows 20.0 -> 17.6, 96 20.0 -> 20.2, 128 20.9 -> 21.2
//                                81920, 5: 96 rows k 65 20.0 -> 17.5, k 200 24.0 -> 23.4, 128 24.2 -> 22.1, 27.7 -> 28.2
//                                128256, 8: k 200 64 rows 26.0 -> 23.0, 128 34.5 -> 31.9, 256 50.7 -> 47, 512 92 -> 87, k 65 86 -> 70
//                                262144, 16: k 200 16 rows 32.9 -> 19.3, 256 96 -> 79;  4096 parts: 34 MB of lists
//                       bf16     40000: k 200 64 rows 20.3 -> 17.9, 128 20.7 -> 21.1;  50256: 64 21.0 -> 17.9, 128 21.1 -> 21.0
//                                128256: 64 rows k 65 21.6 -> 17.5, k 200 26.2 -> 22.2, 128 22.1 -> 24.3, 27.2 -> 30.8
//                                262144: 64 rows k 200 35.9 -> 31.3, 128 38.0 -> 47.3
//                       (32000, 2 parts, whose calls ask for no scratch: 64 rows k 65 15.6 -> 14.6, k 200 19.2 -> 17.1)
//   greedy, from six parts on
//                       128256: 16 rows 9.1 -> 7.2, 64 10.8 -> 9.8, 128 14.1 -> 17.2: up to 512 parts
// A nucleus of the whole row takes four launches, about 22 us of them where a row is short, so it pays from four parts on and
// while the rows leave CUs idle.  us per call, temperature 0.8, top_p 0.9, one launch -> parts:
//   float32  32000, 2 parts: 1 row 21.0 -> 22.4;  50256, 4: 1 row 24.3 -> 22.4, 64 25.7 -> 24.8, 128 26.1 -> 34.2;  50257: 64 35.3 -> 25.7
//            81920, 5: 64 rows 35.9 -> 31.7, 128 38.4 -> 48.1;  128256, 8: 1 row 41.5 -> 23.3, 32 45.5 -> 25.1, 64 45.7 -> 34.5,
//            128 55.1 -> 65.5;  262144, 16: 1 row 74.4 -> 25.0, 64 92.5 -> 67.7, 128 101 -> 114
//   bf16     128256: 1 row 44.7 -> 23.8, 64 48.1 -> 34.1, 128 49.1 -> 53.8
// Rows so flat that a slice of 1/160 holds more than 512 logits of a part or 1024 in all lose the three launches: top_p 0.9,
// temperature 1, 128256 float32, standard deviation 0.1: 1 row 151 -> 170, 64 157 -> 190;  0.001: 64 158 -> 211;  equal
// logits: 64 714 -> 766.  50257, standard deviation 0.1: 64 92 -> 69, 0.001: 94 -> 123.  What a row is like is not known
// before its slices are, and a language model's rows are none of these (unit variance: 155 -> 60 and 93 -> 36).
constexpr int NUCLEUS_MIN_PARTS = 4, NUCLEUS_MAX_BATCH = 64;
static bool whole_row(int vocab, int top_k, int greedy) { return !greedy && (top_k <= 0 || top_k >= vocab); }
static int sample_parts(int batch, int vocab, int64_t row_stride, float temperature, int top_k, int greedy, int dtype) {
    const int parts = (int)(((int64_t)vocab + PART_MAX - 1) / PART_MAX);
    if (parts < 2 || parts > MAX_PARTS || batch > PART_MAX_BATCH) return 1;
    if (whole_row(vocab, top_k, greedy)) return parts;
    if (!greedy && (top_k > PART_MAX_K || !(temperature <= LIST_MAX_TEMPERATURE))) return 1;
    const int per_16 = dtype == AICOMP_KV_F32 ? 4 : 8;
    if (batch > 1 && row_stride % per_16 != 0) return parts;
    const int all = batch * parts;
    const bool f32 = dtype == AICOMP_KV_F32, together = batch <= 256;
    const int few = f32 ? FewK<float>::value : dtype == AICOMP_KV_F16 ? FewK<f16_t>::value : FewK<bf16_t>::value;
    if (!greedy && top_k <= few) {
        if (f32) return top_k <= 50 || parts >= 4 || batch <= 128 || !together ? parts : 1;
        if (parts >= 6) return all <= 1024 ? parts : 1;
        return !together || all <= (parts == 5 ? 640 : 512) ? parts : 1;
    }
    if (greedy) return parts >= 6 && all <= 512 ? parts : 1;
    if (parts < 3) return 1;
    return f32 && parts >= 8 ? (all <= 4096 ? parts : 1) : batch <= 64 ? parts : 1;
}

// Candidates a part has room for.  Of 16384 normally distributed logits about 2.7 k pass the bound of sixteen waves
// (55 for k <= 16), the most seen in 12000 parts 335 at k = 50 and 825 at k = 256; a part with more (masses
// of equal logits) sends its row the whole way.  At k = 50 a row of 128256 has 42 KB, 43 MB for 1024 rows.
// Greedy, 64 rows of eight parts: 9.75 us with the parts 2 KB or 8 KB apart, 9.9 with 1 KB, 10.1 with 128 bytes
// and the distance an argument.
static int part_capacity(int top_k, int greedy) { return greedy ? GREEDY_CAP : 256 + 8 * top_k < 1024 ? 256 + 8 * top_k : 1024; }

// Scratch of a draw from the whole row: the nucleus' share only where such a call is cut
struct WholeRowSpace {
    unsigned long long *seg_mass, *kept_mass, *part_hist, *part_group, *cut;
    uint2* list;
    unsigned int* count;
    float* part_max;
    size_t bytes;
    WholeRowSpace(int batch, int parts, void* at) {
        char* p = (char*)at;
        auto take = [&](size_t bytes_each, size_t n) { char* q = p; p += bytes_each * n; return q; };
        const size_t all = (size_t)batch * parts;
        const bool nucleus = parts >= NUCLEUS_MIN_PARTS && batch <= NUCLEUS_MAX_BATCH;
        part_hist = (unsigned long long*)take(8 * NBINS, nucleus ? all : 0);         // first: 16-byte loads
        seg_mass = (unsigned long long*)take(8 * NW, all);
        part_group = (unsigned long long*)take(8 * GROUPS, nucleus ? all : 0);
        kept_mass = (unsigned long long*)take(8 * NW, nucleus ? all : 0);
        list = (uint2*)take(8 * NUCLEUS_CAP, nucleus ? all : 0);
        cut = (unsigned long long*)take(16, nucleus ? batch : 0);
        count = (unsigned int*)take(4, nucleus ? all : 0);
        part_max = (float*)take(4, all);
        bytes = p - (char*)at;
        if (!nucleus) part_hist = nullptr;
    }
};

size_t sample_workspace_bytes(int batch, int vocab, int64_t row_stride, float temperature, int top_k, int greedy, int dtype) {
    const int parts = sample_parts(batch, vocab, row_stride, temperature, top_k, greedy, dtype);
    if (parts < 2) return 0;
    if (whole_row(vocab, top_k, greedy)) return WholeRowSpace(batch, parts, nullptr).bytes;
    return (size_t)batch * parts * (part_capacity(top_k, greedy) * sizeof(uint2) + sizeof(unsigned int));
}

template <typename T>
static void launch_rows(const SampleParams& p, int batch, hipStream_t stream) {
    if (p.greedy) {
        if (p.parts) hipLaunchKernelGGL((sample_parts_kernel<T, true>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
        hipLaunchKernelGGL((greedy_kernel<T>), dim3(batch), dim3(NT), 0, stream, p);
    } else if (p.parts && p.seg_mass) {
        hipLaunchKernelGGL((sample_max_kernel<T>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
        if (p.part_hist) {
            hipLaunchKernelGGL((sample_mass_kernel<T, true>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
            hipLaunchKernelGGL((sample_slice_kernel<T>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
            hipLaunchKernelGGL((sample_nucleus_kernel<T>), dim3(batch), dim3(NT), 0, stream, p);
        } else {
            hipLaunchKernelGGL((sample_mass_kernel<T, false>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
            hipLaunchKernelGGL((sample_locate_kernel<T>), dim3(batch), dim3(NT), 0, stream, p);
        }
    } else if (p.parts) {
        hipLaunchKernelGGL((sample_parts_kernel<T, false>), dim3(batch, p.parts), dim3(NT), 0, stream, p);
        hipLaunchKernelGGL((sample_merge_kernel<T>), dim3(batch), dim3(NT), 0, stream, p);
    } else {
        hipLaunchKernelGGL((sample_kernel<T>), dim3(batch), dim3(NT), 0, stream, p);
    }
}

int launch_sample(int64_t* out, const void* logits, int64_t row_stride, float* probs_out,
                  const float* uniforms, int batch, int vocab, float temperature, int top_k, float top_p,
                  int greedy, int dtype, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    SampleParams p;
    p.out = out; p.logits = logits; p.row_stride = row_stride; p.probs_out = probs_out;
    p.uniforms = uniforms; p.vocab = vocab; p.temperature = temperature; p.top_k = top_k;
    p.top_p = top_p; p.greedy = greedy;
    p.part_count = nullptr; p.part_list = nullptr; p.parts = 0; p.part_size = 0; p.part_cap = 0;
    p.seg_mass = nullptr; p.part_max = nullptr;
    p.part_hist = nullptr; p.part_group = nullptr; p.kept_mass = nullptr; p.cut = nullptr;
    const size_t need = sample_workspace_bytes(batch, vocab, row_stride, temperature, top_k, greedy, dtype);
    if (need && workspace && workspace_bytes >= need) {
        const int parts = sample_parts(batch, vocab, row_stride, temperature, top_k, greedy, dtype);
        p.part_size = ((vocab + parts - 1) / parts + 3) / 4 * 4;       // parts * part_size < vocab + 4 parts
        p.parts = (vocab + p.part_size - 1) / p.part_size;             // none is empty
        if (whole_row(vocab, top_k, greedy)) {
            const WholeRowSpace at(batch, parts, workspace);
            const bool nucleus = top_p < 1.f;
            // the distribution itself is written by one workgroup per row
            if (probs_out || (nucleus && (!at.part_hist || (uintptr_t)workspace % 16))) p.parts = 0;
            else {
                p.seg_mass = at.seg_mass; p.part_max = at.part_max;
                if (nucleus) {
                    p.part_hist = at.part_hist; p.part_group = at.part_group; p.kept_mass = at.kept_mass; p.cut = at.cut;
                    p.part_list = at.list; p.part_count = at.count;
                }
            }
        } else {
            p.part_cap = part_capacity(top_k, greedy);
            p.part_list = (uint2*)workspace;
            p.part_count = (unsigned int*)(p.part_list + (size_t)batch * p.parts * p.part_cap);
        }
    }
    if (dtype == AICOMP_KV_F32) launch_rows<float>(p, batch, stream);
    else if (dtype == AICOMP_KV_F16) launch_rows<f16_t>(p, batch, stream);
    else launch_rows<bf16_t>(p, batch, stream);
    AICOMP_HIP_LAUNCH_CHECK();
    return AICOMP_KV_OK;
}

}  // namespace aicomp
