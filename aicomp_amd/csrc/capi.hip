// extern "C" entry points: argument validation and kernel dispatch.
// The declarations, with the reference interfaces they replace, are in
// include/aicomp_kv.h.
#include "common.h"

#include <algorithm>
#include <stdlib.h>
#include <string.h>

#include <atomic>

// Split-K scratch of aicomp_paged_decode_attn_append_static: device memory that belongs to the
// loaded library, one copy per GPU, held until the process ends.  In host code this name is only
// a handle for hipGetSymbolAddress: the address a kernel may use is what that call returns.
static __device__ __align__(256) unsigned char scratch[AICOMP_KV_STATIC_SCRATCH_BYTES];

namespace aicomp {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int launch_kv_append(const void* key, const void* value, int64_t token_stride, int64_t head_stride,
                     void* k_pool, void* v_pool, const int64_t* slot_mapping, int64_t T, int hkv,
                     int d, int bs, int64_t num_blocks, int in_dtype, int pool_dtype,
                     const float* k_scale, const float* v_scale, hipStream_t stream);

bool prefill_mfma_supported(const DecodeArgs& a, int max_q_len);
int launch_prefill_mfma(const DecodeArgs& a, int max_q_len);
int prefill_mfma_tile_positions(int hq, int hkv, int max_q_len);
int prefill_mfma_f32_tile_positions(int hq, int hkv);
bool prefill_mfma_f32_supported(const DecodeArgs& a, int max_q_len);
int launch_prefill_mfma_f32(const DecodeArgs& a, int max_q_len);
bool prefill_tiled_supported(const DecodeArgs& a, int max_q_len);
int launch_prefill_tiled(const DecodeArgs& a, int max_q_len);

static int check_common(int hq, int hkv, int d, int bs, int max_blocks, int64_t num_blocks,
                        int q_dtype, int kv_dtype, const float* k_scale, const float* v_scale,
                        const char* who) {
    AICOMP_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0, AICOMP_KV_EINVAL,
                   "%s: %d query heads are not a multiple of %d KV heads", who, hq, hkv);
    AICOMP_REQUIRE(d > 0 && bs > 0 && max_blocks >= 0 && num_blocks > 0, AICOMP_KV_EINVAL,
                   "%s: bad sizes (head_dim %d, block_size %d, max_blocks %d, num_blocks %lld)",
                   who, d, bs, max_blocks, (long long)num_blocks);
    AICOMP_REQUIRE(dtype_size(q_dtype) && dtype_size(kv_dtype), AICOMP_KV_EINVAL,
                   "%s: unknown element type (query %d, pool %d)", who, q_dtype, kv_dtype);
    if (kv_dtype == AICOMP_KV_FP8_E4M3)
        AICOMP_REQUIRE(k_scale && v_scale, AICOMP_KV_EINVAL,
                       "%s: an fp8 pool needs k_scale and v_scale", who);
    return AICOMP_KV_OK;
}

// shapes the balanced schedule and the matrix-core grid schedule both take
static bool streamk_shape(int batch, int hq, int hkv, int d, int bs, int q_dtype, int kv_dtype) {
    const bool half = is_16bit_float(q_dtype) && (kv_dtype == q_dtype || kv_dtype == AICOMP_KV_FP8_E4M3);
    const bool f32 = q_dtype == AICOMP_KV_F32 && kv_dtype == AICOMP_KV_F32;
    return (d == 128 || d == 64) && hq / hkv <= (half && d == 64 ? 8 : 16) && bs == 16 && (half || f32) && batch <= 1024;
}

// A decode call over few, short rows is a chain of launch and memory latencies, not a stream: the
// balanced schedule (set up for 256 CUs of work, always followed by its merge kernel) then loses to
// one workgroup per (row, KV head, partition) on the grid schedule, without any merge kernel when
// no row can be longer than whole_row_tokens (measured on 1 to 16 rows of 512 and 2048 tokens: 5.4-8.5 against 9-13 us, 8-15 against
// 11-17 us).  "Small" is rows x (table width x block size) at or
// below a process-wide threshold: 32768 by default, or the value of the environment variable
// AICOMP_KV_SMALL_DECODE_TOKENS when the library first needs it (read once, never again), or what
// aicomp_kv_set_small_decode_tokens() stored last (0 keeps every automatic call of a supported
// shape on the balanced schedule).  Larger calls may take it too: see grid_call.  The sizing helpers and the decode calls read the same word.
static std::atomic<long long>& small_decode_tokens() {
    static std::atomic<long long> limit{[] {
        const char* e = getenv("AICOMP_KV_SMALL_DECODE_TOKENS");
        return e ? atoll(e) : 32768LL;
    }()};
    return limit;
}

static bool small_call(int64_t rows, int bs, int max_blocks) {
    return rows * (int64_t)max_blocks * bs <= small_decode_tokens().load(std::memory_order_relaxed);
}

// Tokens up to which a row of the matrix-core grid schedule is whole in `wgs` (row, KV head) workgroups.
// Few workgroups: the line lies where the merge's launch (about 3 us of device and 3 us of host time) costs what the longer
// chain of one workgroup does: 1000 and 1200 tokens at D 64 whole 7.2 and 7.4 us, split 8.0 us, 2000 tokens 9.7 and 7.9;
// D 128: 760 tokens 7.7 and 8.8, 1000 tokens 9.2 and 8.2 us.  Other pools: 640.  Float32 at D 64: 640 tokens of
// one row whole 10.1 us, split 9.4 (and 3 us of host time), 768 tokens 11.3 and 9.9.  A float32 row at D 128
// is as many bytes as two bf16 rows on its CU: whole up to 448 tokens where the split has a CU for each of its
// workgroups (one row of 448 12.2 whole, 11.5 split; 512 tokens 13.1 and 12.1, 640 15.3
// and 11.9), otherwise up to 640 (16 rows of 8 KV heads, 640 tokens 19.1 and 21.5, 768 tokens 21.8 and 23.2).
// At the two float32 lines themselves the split is 0.7 us faster on the device, which is less than the host
// time that its second launch takes.
// More workgroups share the memory's bandwidth, a longer row is then hidden behind the others and neither a split nor the
// balanced schedule has its start and merge to show for it.  Whole / the better of the two, us, 8 KV heads:
//   bf16 D 128   128 workgroups 768 tokens 11.5 / 13.0, 1168 16.6 / 14.6;  256  1168 19.2 / 22.1, 1536 23.3 / 25.6 (of unlike
//                lengths 1616 19.5 / 16.7);  512  1200 36.5 / 39.0, 1600 46.4 / 46.0;  1024  1200 64.1 / 68.6, 1600 84.1 / 91.1
//   bf16 D 64    128  1536 12.7 / 12.6;  256  1600 16.0 / 20.7, 2100 18.1 / 22.0;  512  1168 20.4 / 24.7, 2600 0.94, 3600 0.98
//   fp8 D 128    128  1168 0.98;  256  1536 0.81, 2100 0.83;  512  1600 0.93, 2672 0.96;  of D 64  256  2672 0.78;  512  3600 0.89
//   float32 D 64 256  1168 0.87;  384  1200 1.02;  512  1200 0.94, 1600 1.03;  16 / 2 heads, bf16: 128 800 0.86, 256 1200 0.82
// One head per KV head merges little: 8 / 8 heads, D 128, 384 workgroups 1200 tokens 30.6 / 28.8.  More than 512 workgroups come
// in rounds: 768 of D 64, 2112 tokens 51.2 / 49.0, of fp8 54.4 / 53.0.
// Between 256 and 512 workgroups some CUs have two, and two long rows on one of them wait for each other's loads while others idle: the
// limit grows half as fast there, and at 512, two on every CU, is whole again.  384 workgroups, lengths lognormal (median an eighth of the table; of five draws the mean and the worst) /
// spread evenly / alike, whole to balanced: bf16 D 128 1216 tokens 0.97, 1.19 / 1.06 / 0.95, 1344 1.06, 1.38 / 1.04 / 0.94;  D 64 1920 0.89, 0.96 /
// 1.06 / 0.91, 2560 1.07, 1.33 / 1.07 / 0.98;  fp8 1920 0.99, 1.10 / 1.05 / 0.96, 2240 1.07, 1.13 / 1.03 / 1.01;  512: bf16 D 128 1472 0.95, 1.15 /
// 0.92 / 0.90, D 64 2560 0.96, 1.17 / 0.93 / 0.90, 3072 1.03, 1.10 / 1.02 / 0.91, fp8 1920 0.95, 1.13 / 0.90 / 0.88, 2880 1.10, 1.19 / 0.97 / 0.94.
// The table's width is all that is known here.  One row as long as it among rows a tenth of that, and rows alike, at the ends of the lines:
// bf16 D 128 64 rows of 1648 22.8 / 19.3, 70.0 / 76.4;  D 64 64 of 3072 20.9 / 17.8, 67.3 / 72.1;  fp8 D 128 64 of 2560 23.7 / 20.9, 60.3 / 64.6.
static int64_t whole_row_tokens(int64_t wgs, int group, int d, int64_t max_ctx, int kv_dtype) {
    const int64_t uneven = wgs > 256 && wgs < 512 ? (wgs - 256) / 2 : 0;
    const int64_t more = std::min<int64_t>(std::max<int64_t>(wgs - uneven - 64, 0), 448), rounds = wgs > 512 ? 2048 : 4096;
    if (is_16bit_float(kv_dtype)) return d == 64 ? std::min(1280 + 4 * more, rounds) : 768 + (group > 1 ? 2 : 1) * more;
    if (kv_dtype == AICOMP_KV_FP8_E4M3) return d == 64 ? std::min<int64_t>(640 + 10 * more, 4096) : std::min(640 + 5 * more, rounds);
    if (d == 64) return std::min<int64_t>(640 + 3 * more / 2, 1100);
    return wgs * ((max_ctx + 255) / 256) <= 256 ? 448 : 640;
}

// Whether an automatic call takes the grid schedule.  Beyond the threshold (one that is at least the default; a lower
// one pins the schedule) it still does where its rows are whole, and where few (row, KV head) pairs are long: each of the
// balanced schedule's waves then has so few tiles that its start and flush outweigh them.  Split in 256 tokens / balanced, us,
// 8 KV heads, by tokens x KV heads:  24 rows of 2096 (402 k) 27.3 / 29.2, 2672 (513 k) 30.3 / 31.6, of unlike lengths 15.9 /
// 19.0 and 21.2 / 23.3;  32 of 2096 (537 k) 34.3 / 34.7, 48 of 1600 (614 k) 34.9 / 35.8, 2096 (805 k) 45.8 / 45.9;  16 / 2 heads:
// 64 of 2112 (270 k) 0.95, 3600 (461 k) 1.00, 16 of 3584 (115 k) 0.76;  fp8 pools cross earlier: 16 of 2672 (342 k) 0.94,
// 24 of 2096 (402 k) 1.02, 2672 (513 k) 1.05;  float32 rows of D 128 at once (48 of 800 46.5 / 37.8).  A raised threshold does
// not move that line: the split would need more scratch than the balanced schedule (64 rows of 4096, 64 / 8 heads 34 MB, 19).
// With pools that take turns (every call reads cold rows), partitions turned, one long row / lengths spread evenly / rows alike, split to
// balanced: 16 / 2 heads 128 rows of 2048 0.81 / 1.01 / 1.04, 1648 0.72 / 1.03 / 1.09;  32 / 8 24 of 2048 0.74 / 1.00 / 0.99;  fp8 24 of
// 2048 0.73 / 1.07 / 1.06, 16 of 2560 0.82 / 0.95 / 1.08, D 64 0.87 / 0.93 / 1.10.
static bool grid_call(int64_t rows, int hq, int hkv, int d, int bs, int max_blocks, int kv_dtype) {
    if (small_call(rows, bs, max_blocks)) return true;
    const int64_t limit = small_decode_tokens().load(std::memory_order_relaxed), max_ctx = (int64_t)max_blocks * bs;
    if (limit < 32768 || rows * hkv > 2048) return false;               // (measured up to there)
    return max_ctx <= whole_row_tokens(rows * hkv, hq / hkv, d, max_ctx, kv_dtype) ||
           (max_ctx <= 4096 && !(kv_dtype == AICOMP_KV_F32 && d == 128) &&
            rows * hkv * max_ctx <= (kv_dtype == AICOMP_KV_FP8_E4M3 ? 393216 : 524288));
}

static int auto_partition(int64_t rows, int hq, int hkv, int d, int bs, int max_blocks, int kv_dtype, bool matrix_shape) {
    // Longer partitions amortise a workgroup's start-up and merge; shorter ones give the
    // 256 CUs enough workgroups when there are few (sequence, KV head) rows.
    const int64_t max_ctx = (int64_t)max_blocks * bs;
    int ps;
    if (matrix_shape && grid_call(rows, hq, hkv, d, bs, max_blocks, kv_dtype)) {
        // matrix-core grid schedule: whole rows (a whole number of its 64-token tiles) and no merge launch, or partitions of
        // 256 tokens
        ps = max_ctx <= whole_row_tokens(rows * hkv, hq / hkv, d, max_ctx, kv_dtype) ? (int)((max_ctx + 63) / 64 * 64) : 256;
    } else {
        ps = 64;       // vector-ALU kernel on few short rows: spread the call wide
        for (int cand : {1024, 512, 256, 128}) {
            if (rows * hkv * ((max_ctx + cand - 1) / cand) >= 1024) { ps = cand; break; }
        }
    }
    ps = (ps + bs - 1) / bs * bs;
    return ps;
}

}  // namespace aicomp

using namespace aicomp;

extern "C" {

int aicomp_kv_version(void) { return 302; }

const char* aicomp_kv_last_error(void) { return g_err; }

long long aicomp_kv_set_small_decode_tokens(long long tokens) {
    std::atomic<long long>& limit = small_decode_tokens();
    return tokens < 0 ? limit.load(std::memory_order_relaxed) : limit.exchange(tokens, std::memory_order_relaxed);
}

int aicomp_kv_append(const void* key, const void* value, int64_t kv_token_stride,
                     int64_t kv_head_stride, void* k_pool, void* v_pool,
                     const int64_t* slot_mapping, int64_t num_tokens, int num_kv_heads,
                     int head_dim, int block_size, int64_t num_blocks, int in_dtype,
                     int pool_dtype, const float* k_scale, const float* v_scale, void* stream) {
    AICOMP_REQUIRE(num_tokens >= 0, AICOMP_KV_EINVAL, "kv_append: negative token count");
    if (num_tokens == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE(key && value && k_pool && v_pool && slot_mapping, AICOMP_KV_EINVAL,
                   "kv_append: null pointer");
    AICOMP_REQUIRE(num_kv_heads > 0 && head_dim > 0 && block_size > 0 && num_blocks > 0,
                   AICOMP_KV_EINVAL, "kv_append: bad sizes (Hkv %d, D %d, BS %d, blocks %lld)",
                   num_kv_heads, head_dim, block_size, (long long)num_blocks);
    AICOMP_REQUIRE(dtype_size(in_dtype) && dtype_size(pool_dtype), AICOMP_KV_EINVAL,
                   "kv_append: unknown element type (in %d, pool %d)", in_dtype, pool_dtype);
    AICOMP_REQUIRE(kv_head_stride >= head_dim && kv_token_stride >= 0, AICOMP_KV_EINVAL,
                   "kv_append: strides (%lld, %lld) overlap rows of %d elements",
                   (long long)kv_token_stride, (long long)kv_head_stride, head_dim);
    return launch_kv_append(key, value, kv_token_stride, kv_head_stride, k_pool, v_pool,
                            slot_mapping, num_tokens, num_kv_heads, head_dim, block_size,
                            num_blocks, in_dtype, pool_dtype, k_scale, v_scale,
                            (hipStream_t)stream);
}

int aicomp_rope_kv_append(const void* q_in, void* q_out, int64_t q_token_stride,
                          int64_t q_head_stride, int64_t qo_token_stride, int64_t qo_head_stride,
                          const void* key, const void* value, int64_t kv_token_stride,
                          int64_t kv_head_stride, const void* cos, const void* sin,
                          int64_t table_stride, int64_t table_rows, const int64_t* positions,
                          void* k_pool, void* v_pool, const int64_t* slot_mapping,
                          int64_t num_tokens, int num_q_heads, int num_kv_heads, int head_dim,
                          int block_size, int64_t num_blocks, int in_dtype, int pool_dtype,
                          const float* k_scale, const float* v_scale, void* stream) {
    AICOMP_REQUIRE(num_tokens >= 0, AICOMP_KV_EINVAL, "rope_kv_append: negative token count");
    if (num_tokens == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE(q_in && q_out && key && value && cos && sin && k_pool && v_pool && slot_mapping,
                   AICOMP_KV_EINVAL, "rope_kv_append: null pointer");
    AICOMP_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && head_dim > 0 && block_size > 0 &&
                   num_blocks > 0 && table_rows > 0, AICOMP_KV_EINVAL,
                   "rope_kv_append: bad sizes (Hq %d, Hkv %d, D %d, BS %d, blocks %lld, table rows %lld)",
                   num_q_heads, num_kv_heads, head_dim, block_size, (long long)num_blocks,
                   (long long)table_rows);
    AICOMP_REQUIRE(in_dtype == AICOMP_KV_F32 || is_16bit_float(in_dtype), AICOMP_KV_EUNSUPPORTED,
                   "rope_kv_append: inputs must be float32, bfloat16 or float16 (got %d)", in_dtype);
    AICOMP_REQUIRE(pool_dtype == in_dtype || pool_dtype == AICOMP_KV_FP8_E4M3, AICOMP_KV_EUNSUPPORTED,
                   "rope_kv_append: pool type %d must be the input type %d or fp8-e4m3", pool_dtype,
                   in_dtype);
    AICOMP_REQUIRE(pool_dtype != AICOMP_KV_FP8_E4M3 || (k_scale && v_scale), AICOMP_KV_EINVAL,
                   "rope_kv_append: an fp8 pool needs k_scale and v_scale");
    AICOMP_REQUIRE(head_dim % 16 == 0, AICOMP_KV_EUNSUPPORTED,
                   "rope_kv_append: head_dim %d is not a multiple of 16", head_dim);
    const int64_t v = 16 / dtype_size(in_dtype);       // elements per 16 bytes
    AICOMP_REQUIRE(q_head_stride >= head_dim && qo_head_stride >= head_dim &&
                   kv_head_stride >= head_dim && table_stride >= head_dim && q_token_stride >= 0 &&
                   qo_token_stride >= 0 && kv_token_stride >= 0, AICOMP_KV_EINVAL,
                   "rope_kv_append: strides overlap rows of %d elements", head_dim);
    AICOMP_REQUIRE(q_token_stride % v == 0 && q_head_stride % v == 0 && qo_token_stride % v == 0 &&
                   qo_head_stride % v == 0 && kv_token_stride % v == 0 && kv_head_stride % v == 0 &&
                   table_stride % v == 0, AICOMP_KV_EUNSUPPORTED,
                   "rope_kv_append: strides must be multiples of %lld elements (16 bytes)", (long long)v);
    AICOMP_REQUIRE(((uintptr_t)q_in | (uintptr_t)q_out | (uintptr_t)key | (uintptr_t)value |
                    (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)k_pool | (uintptr_t)v_pool) % 16 == 0,
                   AICOMP_KV_EUNSUPPORTED, "rope_kv_append: pointers must be 16-byte aligned");
    return launch_rope_kv_append(q_in, q_out, q_token_stride, q_head_stride, qo_token_stride,
                                 qo_head_stride, key, value, kv_token_stride, kv_head_stride, cos, sin,
                                 table_stride, table_rows, positions, k_pool, v_pool, slot_mapping,
                                 num_tokens, num_q_heads, num_kv_heads, head_dim, block_size, num_blocks,
                                 in_dtype, pool_dtype, k_scale, v_scale, (hipStream_t)stream);
}

int aicomp_sample_tokens_split(int64_t* out, const void* logits, int64_t row_stride, float* probs_out,
                               const float* uniforms, int batch, int vocab, float temperature, int top_k,
                               float top_p, int greedy, int logits_dtype, void* workspace,
                               size_t workspace_bytes, void* stream) {
    AICOMP_REQUIRE(batch >= 0, AICOMP_KV_EINVAL, "sample_tokens: negative batch");
    if (batch == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE((uintptr_t)workspace % 8 == 0, AICOMP_KV_EINVAL, "sample_tokens: workspace must be 8-byte aligned");
    AICOMP_REQUIRE(out && logits, AICOMP_KV_EINVAL, "sample_tokens: null pointer");
    AICOMP_REQUIRE(vocab > 0 && row_stride >= vocab, AICOMP_KV_EINVAL,
                   "sample_tokens: bad sizes (vocab %d, row stride %lld)", vocab, (long long)row_stride);
    AICOMP_REQUIRE(logits_dtype == AICOMP_KV_F32 || is_16bit_float(logits_dtype), AICOMP_KV_EUNSUPPORTED,
                   "sample_tokens: logits must be float32, bfloat16 or float16 (got %d)", logits_dtype);
    if (!greedy) {
        AICOMP_REQUIRE(uniforms, AICOMP_KV_EINVAL, "sample_tokens: sampling needs uniforms");
        AICOMP_REQUIRE(temperature > 0.f, AICOMP_KV_EINVAL,
                       "sample_tokens: temperature must be positive (got %g)", (double)temperature);
        AICOMP_REQUIRE(top_p == top_p, AICOMP_KV_EINVAL, "sample_tokens: top_p is NaN");
    }
    return launch_sample(out, logits, row_stride, probs_out, uniforms, batch, vocab, temperature, top_k,
                         top_p, greedy ? 1 : 0, logits_dtype, workspace, workspace_bytes, (hipStream_t)stream);
}

int aicomp_sample_tokens(int64_t* out, const void* logits, int64_t row_stride, float* probs_out,
                         const float* uniforms, int batch, int vocab, float temperature, int top_k,
                         float top_p, int greedy, int logits_dtype, void* stream) {
    return aicomp_sample_tokens_split(out, logits, row_stride, probs_out, uniforms, batch, vocab, temperature, top_k,
                                      top_p, greedy, logits_dtype, nullptr, 0, stream);
}

size_t aicomp_sample_workspace_bytes(int batch, int vocab, int64_t row_stride, float temperature, int top_k, int greedy,
                                     int logits_dtype) {
    if (batch <= 0 || vocab <= 0) return 0;
    return sample_workspace_bytes(batch, vocab, row_stride, temperature, top_k, greedy ? 1 : 0, logits_dtype);
}

int aicomp_paged_decode_partition_size(int batch, int num_q_heads, int num_kv_heads, int head_dim,
                                       int block_size, int max_blocks_per_seq, int q_dtype,
                                       int kv_dtype) {
    if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || block_size <= 0 || max_blocks_per_seq <= 0) return 0;
    return auto_partition(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype,
                          streamk_shape(batch, num_q_heads, num_kv_heads, head_dim, block_size, q_dtype, kv_dtype));
}

static int resolve_parts(int64_t rows, int hq, int hkv, int d, int bs, int max_blocks, int kv_dtype, bool matrix_shape,
                         int& partition_size) {
    if (partition_size <= 0) partition_size = auto_partition(rows, hq, hkv, d, bs, max_blocks, kv_dtype, matrix_shape);
    const int64_t max_ctx = (int64_t)max_blocks * bs;
    int64_t parts = (max_ctx + partition_size - 1) / partition_size;
    return (int)(parts < 1 ? 1 : parts);
}

size_t aicomp_paged_decode_workspace_bytes(int batch, int num_q_heads, int num_kv_heads,
                                           int head_dim, int block_size, int max_blocks_per_seq,
                                           int q_dtype, int kv_dtype, int partition_size) {
    if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
        max_blocks_per_seq <= 0 || num_q_heads % num_kv_heads)
        return 0;
    const bool automatic = partition_size <= 0;
    const bool matrix_shape = streamk_shape(batch, num_q_heads, num_kv_heads, head_dim, block_size, q_dtype, kv_dtype);
    const int parts = resolve_parts(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype, matrix_shape, partition_size);
    size_t need = parts <= 1 ? 0 : split_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, parts);
    if (automatic && matrix_shape &&
        !grid_call(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype)) {
        const size_t sk = decode_streamk_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim);
        if (sk > need) need = sk;
    }
    return need;
}

static int decode_impl(void* out, const void* query, const void* new_key, const void* new_value,
                       int64_t kv_token_stride, int64_t kv_head_stride, void* k_pool, void* v_pool,
                       const int32_t* block_table, int64_t block_table_stride,
                       const int32_t* context_lens, int batch, int num_q_heads, int num_kv_heads,
                       int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                       float scale, int q_dtype, int kv_dtype, const float* k_scale,
                       const float* v_scale, int partition_size, void* workspace,
                       size_t workspace_bytes, void* stream, const char* who) {
    AICOMP_REQUIRE(batch >= 0, AICOMP_KV_EINVAL, "%s: negative batch", who);
    if (batch == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE(out && query && k_pool && v_pool && block_table && context_lens,
                   AICOMP_KV_EINVAL, "%s: null pointer", who);
    int rc = check_common(num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq,
                          num_blocks, q_dtype, kv_dtype, k_scale, v_scale, who);
    if (rc) return rc;
    AICOMP_REQUIRE(max_blocks_per_seq > 0 && block_table_stride >= max_blocks_per_seq,
                   AICOMP_KV_EINVAL, "%s: block table stride %lld < width %d", who,
                   (long long)block_table_stride, max_blocks_per_seq);
    AICOMP_REQUIRE(partition_size >= 0 && partition_size % block_size == 0, AICOMP_KV_EINVAL,
                   "%s: partition_size %d is not a multiple of block_size %d", who, partition_size,
                   block_size);
    const bool fused = new_key != nullptr;
    if (fused)
        AICOMP_REQUIRE(new_value && kv_head_stride >= head_dim && kv_token_stride >= 0, AICOMP_KV_EINVAL,
                       "%s: bad new_key / new_value arguments", who);
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    a.out = out; a.query = query; a.k_pool = k_pool; a.v_pool = v_pool;
    a.block_table = block_table; a.block_table_stride = block_table_stride;
    a.context_lens = context_lens; a.cu_q_lens = nullptr;
    a.num_seqs = batch; a.rows = batch;
    a.hq = num_q_heads; a.hkv = num_kv_heads; a.d = head_dim; a.bs = block_size;
    a.max_blocks = max_blocks_per_seq; a.num_blocks = num_blocks;
    a.scale = scale; a.q_dtype = q_dtype; a.kv_dtype = kv_dtype;
    a.k_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? k_scale : nullptr;
    a.v_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? v_scale : nullptr;
    a.partition_size = partition_size;
    const bool matrix_shape = streamk_shape(batch, num_q_heads, num_kv_heads, head_dim, block_size, q_dtype, kv_dtype);
    a.num_parts = resolve_parts(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype, matrix_shape, a.partition_size);
    a.stream = (hipStream_t)stream;
    // the matrix-core kernels append the new rows themselves when they can read them 16 bytes at a time
    const int64_t vec = 16 / dtype_size(q_dtype);
    const bool injectable = fused && kv_token_stride % vec == 0 && kv_head_stride % vec == 0 && (uintptr_t)new_key % 16 == 0 &&
                            (uintptr_t)new_value % 16 == 0;
    if (partition_size == 0 && decode_streamk_supported(a) &&
        !grid_call(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype)) {
        // balanced schedule: equal tile counts per wave, merged by a second kernel
        const size_t need = decode_streamk_workspace_bytes(a.rows, a.hq, a.hkv, a.d);
        AICOMP_REQUIRE(workspace && workspace_bytes >= need, AICOMP_KV_EWORKSPACE,
                       "%s: workspace of %zu bytes needed, %zu given", who, need,
                       workspace ? workspace_bytes : (size_t)0);
        AICOMP_REQUIRE((uintptr_t)workspace % 16 == 0, AICOMP_KV_EINVAL,
                       "%s: workspace must be 16-byte aligned", who);
        const bool in_kernel = injectable;
        if (fused && !in_kernel) {
            rc = launch_kv_append_last(new_key, new_value, kv_token_stride, kv_head_stride, k_pool, v_pool,
                                       block_table, block_table_stride, context_lens, batch,
                                       num_kv_heads, head_dim, block_size, max_blocks_per_seq,
                                       num_blocks, q_dtype, kv_dtype, k_scale, v_scale, a.stream);
            if (rc) return rc;
        }
        if (in_kernel) {
            a.new_key = new_key; a.new_value = new_value;
            a.new_token_stride = kv_token_stride; a.new_head_stride = kv_head_stride;
        }
        return launch_decode_streamk(a, workspace);
    }
    const bool mfma = decode_mfma_supported(a);
    const bool in_kernel = injectable && mfma;
    if (in_kernel) {
        a.new_key = new_key; a.new_value = new_value;
        a.new_token_stride = kv_token_stride; a.new_head_stride = kv_head_stride;
    } else if (fused) {
        rc = launch_kv_append_last(new_key, new_value, kv_token_stride, kv_head_stride, k_pool, v_pool,
                                   block_table, block_table_stride, context_lens, batch, num_kv_heads,
                                   head_dim, block_size, max_blocks_per_seq, num_blocks, q_dtype,
                                   kv_dtype, k_scale, v_scale, a.stream);
        if (rc) return rc;
    }
    if (a.num_parts > 1) {
        const size_t need = split_workspace_bytes(a.rows, a.hq, a.hkv, a.d, a.num_parts);
        AICOMP_REQUIRE(workspace && workspace_bytes >= need, AICOMP_KV_EWORKSPACE,
                       "%s: workspace of %zu bytes needed, %zu given", who, need,
                       workspace ? workspace_bytes : (size_t)0);
        AICOMP_REQUIRE((uintptr_t)workspace % 16 == 0, AICOMP_KV_EINVAL,
                       "%s: workspace must be 16-byte aligned", who);
        a.ws = split_workspace_view(workspace, a.rows, a.hq, a.hkv, a.d, a.num_parts);
    }
    if (mfma) return launch_decode_mfma(a);
    return launch_decode_generic(a);
}

int aicomp_paged_decode_attn(void* out, const void* query, const void* k_pool, const void* v_pool,
                             const int32_t* block_table, int64_t block_table_stride,
                             const int32_t* context_lens, int batch, int num_q_heads,
                             int num_kv_heads, int head_dim, int block_size,
                             int max_blocks_per_seq, int64_t num_blocks, float scale, int q_dtype,
                             int kv_dtype, const float* k_scale, const float* v_scale,
                             int partition_size, void* workspace, size_t workspace_bytes,
                             void* stream) {
    return decode_impl(out, query, nullptr, nullptr, 0, 0, (void*)k_pool, (void*)v_pool, block_table,
                       block_table_stride, context_lens, batch, num_q_heads, num_kv_heads, head_dim,
                       block_size, max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale,
                       v_scale, partition_size, workspace, workspace_bytes, stream,
                       "paged_decode_attn");
}

int aicomp_paged_decode_attn_append(void* out, const void* query, const void* new_key,
                                    const void* new_value, int64_t kv_token_stride,
                                    int64_t kv_head_stride, void* k_pool, void* v_pool,
                                    const int32_t* block_table, int64_t block_table_stride,
                                    const int32_t* context_lens, int batch, int num_q_heads,
                                    int num_kv_heads, int head_dim, int block_size,
                                    int max_blocks_per_seq, int64_t num_blocks, float scale,
                                    int q_dtype, int kv_dtype, const float* k_scale,
                                    const float* v_scale, int partition_size, void* workspace,
                                    size_t workspace_bytes, void* stream) {
    AICOMP_REQUIRE(batch <= 0 || (new_key && new_value), AICOMP_KV_EINVAL,
                   "paged_decode_attn_append: null new_key / new_value");
    return decode_impl(out, query, new_key, new_value, kv_token_stride, kv_head_stride, k_pool, v_pool,
                       block_table, block_table_stride, context_lens, batch, num_q_heads, num_kv_heads,
                       head_dim, block_size, max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype,
                       k_scale, v_scale, partition_size, workspace, workspace_bytes, stream,
                       "paged_decode_attn_append");
}

static int rope_decode_impl(void* out, const void* query, int64_t q_token_stride, int64_t q_head_stride,
                            const void* new_key, const void* new_value, int64_t kv_token_stride,
                            int64_t kv_head_stride, const void* cos, const void* sin, int64_t table_stride,
                            int64_t table_rows, const int64_t* positions, const int64_t* slot_mapping, void* k_pool,
                            void* v_pool, const int32_t* block_table, int64_t block_table_stride,
                            const int32_t* context_lens, int batch, int num_q_heads, int num_kv_heads, int head_dim,
                            int block_size, int max_blocks_per_seq, int64_t num_blocks, float scale, int q_dtype,
                            int kv_dtype, const float* k_scale, const float* v_scale, int longest_context, void* workspace,
                            size_t workspace_bytes, void* stream) {
    const char* who = "rope_paged_decode_attn";
    AICOMP_REQUIRE(batch >= 0, AICOMP_KV_EINVAL, "%s: negative batch", who);
    if (batch == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE(out && query && new_key && new_value && cos && sin && positions && slot_mapping && k_pool && v_pool &&
                   block_table && context_lens, AICOMP_KV_EINVAL, "%s: null pointer", who);
    int rc = check_common(num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, num_blocks, q_dtype,
                          kv_dtype, k_scale, v_scale, who);
    if (rc) return rc;
    AICOMP_REQUIRE(max_blocks_per_seq > 0 && block_table_stride >= max_blocks_per_seq, AICOMP_KV_EINVAL,
                   "%s: block table stride %lld < width %d", who, (long long)block_table_stride, max_blocks_per_seq);
    AICOMP_REQUIRE(q_head_stride >= head_dim && kv_head_stride >= head_dim && table_stride >= head_dim && table_rows > 0 &&
                   q_token_stride >= 0 && kv_token_stride >= 0, AICOMP_KV_EINVAL,
                   "%s: strides overlap rows of %d elements", who, head_dim);
    AICOMP_REQUIRE(longest_context >= 0, AICOMP_KV_EINVAL, "%s: negative longest context", who);
    // table columns to size the call for; the kernel's last partition takes a row that is longer after all
    const int columns = longest_context == 0 ? max_blocks_per_seq
                                             : std::min(max_blocks_per_seq, (int)(((int64_t)longest_context + block_size - 1) / block_size));
    const int64_t v = 16 / dtype_size(q_dtype);
    const bool vectors = (q_token_stride | q_head_stride | kv_token_stride | kv_head_stride | table_stride) % v == 0 &&
                         ((uintptr_t)new_key | (uintptr_t)new_value | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)query) % 16 == 0;
    const bool shape = streamk_shape(batch, num_q_heads, num_kv_heads, head_dim, block_size, q_dtype, kv_dtype);
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    a.out = out; a.query = query; a.k_pool = k_pool; a.v_pool = v_pool;
    a.block_table = block_table; a.block_table_stride = block_table_stride; a.context_lens = context_lens;
    a.num_seqs = batch; a.rows = batch;
    a.hq = num_q_heads; a.hkv = num_kv_heads; a.d = head_dim; a.bs = block_size;
    a.max_blocks = max_blocks_per_seq; a.num_blocks = num_blocks;
    a.scale = scale; a.q_dtype = q_dtype; a.kv_dtype = kv_dtype;
    a.k_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? k_scale : nullptr;
    a.v_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? v_scale : nullptr;
    a.num_parts = resolve_parts(batch, num_q_heads, num_kv_heads, head_dim, block_size, columns, kv_dtype, shape, a.partition_size);
    a.stream = (hipStream_t)stream;
    // A batch for the balanced schedule streams for tens of microseconds: the launch saved is lost in it.  So it is in split
    // rows of more than 512 workgroups (two calls, which the table's width sends to the balanced schedule, / this one, us:
    // 32 rows of 700, fp8 pool, 32/8 heads, D 128 18.1 / 21.1, D 64 17.2 / 18.7, 64/8 19.4 / 23.6), but for float32 groups
    // of up to four heads (32 rows of 700, D 128 37.8 / 33.4, D 64 24.4 / 20.2).
    // (counted by the lines of few workgroups, whatever the call's own partitions are)
    const int64_t max_ctx = (int64_t)columns * block_size, wgs = (int64_t)batch * num_kv_heads;
    const int64_t whole = whole_row_tokens(kv_dtype == AICOMP_KV_F32 && head_dim == 128 ? wgs : std::min<int64_t>(wgs, 64),
                                           num_q_heads / num_kv_heads, head_dim, max_ctx, kv_dtype);
    const bool few = max_ctx <= whole || wgs * ((max_ctx + 255) / 256) <= 512 ||
                     (q_dtype == AICOMP_KV_F32 && num_q_heads <= 4 * num_kv_heads);
    AICOMP_REQUIRE(vectors && shape && few && small_call(batch, block_size, columns) && decode_mfma_supported(a),
                   AICOMP_KV_EUNSUPPORTED, "%s: not a call of the matrix-core grid schedule", who);
    a.new_key = new_key; a.new_value = new_value;
    a.new_token_stride = kv_token_stride; a.new_head_stride = kv_head_stride;
    a.cos_tab = cos; a.sin_tab = sin; a.tab_stride = table_stride; a.tab_rows = table_rows;
    a.positions = positions; a.slots = slot_mapping;
    a.q_token_stride = q_token_stride; a.q_head_stride = q_head_stride;
    if (a.num_parts > 1) {
        const size_t need = split_workspace_bytes(a.rows, a.hq, a.hkv, a.d, a.num_parts);
        AICOMP_REQUIRE(workspace && workspace_bytes >= need, AICOMP_KV_EWORKSPACE,
                       "%s: workspace of %zu bytes needed, %zu given", who, need, workspace ? workspace_bytes : (size_t)0);
        AICOMP_REQUIRE((uintptr_t)workspace % 16 == 0, AICOMP_KV_EINVAL, "%s: workspace must be 16-byte aligned", who);
        a.ws = split_workspace_view(workspace, a.rows, a.hq, a.hkv, a.d, a.num_parts);
    }
    return launch_decode_mfma(a);
}

int aicomp_rope_paged_decode_attn(void* out, const void* query, int64_t q_token_stride, int64_t q_head_stride,
                                  const void* new_key, const void* new_value, int64_t kv_token_stride,
                                  int64_t kv_head_stride, const void* cos, const void* sin, int64_t table_stride,
                                  int64_t table_rows, const int64_t* positions, const int64_t* slot_mapping, void* k_pool,
                                  void* v_pool, const int32_t* block_table, int64_t block_table_stride,
                                  const int32_t* context_lens, int batch, int num_q_heads, int num_kv_heads, int head_dim,
                                  int block_size, int max_blocks_per_seq, int64_t num_blocks, float scale, int q_dtype,
                                  int kv_dtype, const float* k_scale, const float* v_scale, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    return rope_decode_impl(out, query, q_token_stride, q_head_stride, new_key, new_value, kv_token_stride,
                            kv_head_stride, cos, sin, table_stride, table_rows, positions, slot_mapping, k_pool, v_pool,
                            block_table, block_table_stride, context_lens, batch, num_q_heads, num_kv_heads, head_dim,
                            block_size, max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale, v_scale, 0,
                            workspace, workspace_bytes, stream);
}

int aicomp_rope_paged_decode_attn_sized(void* out, const void* query, int64_t q_token_stride, int64_t q_head_stride,
                                        const void* new_key, const void* new_value, int64_t kv_token_stride,
                                        int64_t kv_head_stride, const void* cos, const void* sin, int64_t table_stride,
                                        int64_t table_rows, const int64_t* positions, const int64_t* slot_mapping, void* k_pool,
                                        void* v_pool, const int32_t* block_table, int64_t block_table_stride,
                                        const int32_t* context_lens, int batch, int num_q_heads, int num_kv_heads, int head_dim,
                                        int block_size, int max_blocks_per_seq, int64_t num_blocks, float scale, int q_dtype,
                                        int kv_dtype, const float* k_scale, const float* v_scale, int longest_context, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    return rope_decode_impl(out, query, q_token_stride, q_head_stride, new_key, new_value, kv_token_stride,
                            kv_head_stride, cos, sin, table_stride, table_rows, positions, slot_mapping, k_pool, v_pool,
                            block_table, block_table_stride, context_lens, batch, num_q_heads, num_kv_heads, head_dim,
                            block_size, max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale, v_scale,
                            longest_context, workspace, workspace_bytes, stream);
}

// Device address of `scratch` on the current device, looked up once per device.
static int static_scratch(void** ptr, const char* who) {
    constexpr int MAX_DEVICES = 64;
    static std::atomic<void*> per_device[MAX_DEVICES];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        set_error("%s: cannot identify the current device (%d)", who, dev);
        return AICOMP_KV_EHIP;
    }
    void* p = per_device[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev,
                      hipGetErrorString(e));
            return AICOMP_KV_EHIP;
        }
        per_device[dev].store(p, std::memory_order_release);     // racing threads store the same address
    }
    *ptr = p;
    return AICOMP_KV_OK;
}

int aicomp_paged_decode_attn_append_static(void* out, const void* query, const void* new_key,
                                           const void* new_value, int64_t kv_token_stride,
                                           int64_t kv_head_stride, void* k_pool, void* v_pool,
                                           const int32_t* block_table, int64_t block_table_stride,
                                           const int32_t* context_lens, int batch, int num_q_heads,
                                           int num_kv_heads, int head_dim, int block_size,
                                           int max_blocks_per_seq, int64_t num_blocks, float scale,
                                           int q_dtype, int kv_dtype, const float* k_scale,
                                           const float* v_scale, int partition_size, void* stream) {
    const char* who = "paged_decode_attn_append_static";
    AICOMP_REQUIRE(batch <= 0 || (new_key && new_value), AICOMP_KV_EINVAL, "%s: null new_key / new_value", who);
    auto scratch_bytes = [&](int ps) {
        return aicomp_paged_decode_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, block_size,
                                                   max_blocks_per_seq, q_dtype, kv_dtype, ps);
    };
    // Which shapes are too large follows from the threshold alone: one above it counts as the balanced schedule would take
    // it, also where the call keeps to the grid schedule and needs less.
    const bool balanced = partition_size == 0 && num_kv_heads > 0 && batch > 0 && num_q_heads % num_kv_heads == 0 &&
                          streamk_shape(batch, num_q_heads, num_kv_heads, head_dim, block_size, q_dtype, kv_dtype) &&
                          !small_call(batch, block_size, max_blocks_per_seq);
    size_t need = std::max(scratch_bytes(partition_size),
                           balanced ? decode_streamk_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim) : (size_t)0);
    if (partition_size == 0 && need > (size_t)AICOMP_KV_STATIC_SCRATCH_BYTES && q_dtype == AICOMP_KV_F32 &&
        kv_dtype == AICOMP_KV_F32) {
        // The balanced schedule's partials have a fixed part of 4096 slots, 34 MB for sixteen heads of 128 per KV
        // head whatever the batch.  The grid schedule over partitions chosen by the number of workgroups needs
        // less: 32 rows of 2048 tokens, 16 / 1 heads, 8.5 MB.
        partition_size = auto_partition(batch, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, kv_dtype, false);
        need = scratch_bytes(partition_size);
    }
    AICOMP_REQUIRE(need <= (size_t)AICOMP_KV_STATIC_SCRATCH_BYTES, AICOMP_KV_EWORKSPACE,
                   "%s: this shape needs %zu bytes of split-K scratch, the built-in scratch holds %zu; "
                   "use aicomp_paged_decode_attn_append with a workspace of the caller's", who, need,
                   (size_t)AICOMP_KV_STATIC_SCRATCH_BYTES);
    void* ws = nullptr;
    if (need > 0) {
        const int rc = static_scratch(&ws, who);
        if (rc) return rc;
    }
    return decode_impl(out, query, new_key, new_value, kv_token_stride, kv_head_stride, k_pool, v_pool,
                       block_table, block_table_stride, context_lens, batch, num_q_heads, num_kv_heads,
                       head_dim, block_size, max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype,
                       k_scale, v_scale, partition_size, ws, need, stream, who);
}

static int prefill_impl(void* out, const void* query, const void* k_pool, const void* v_pool,
                        const int32_t* block_table, int64_t block_table_stride,
                        const int32_t* context_lens, const int32_t* cu_q_lens, int num_seqs,
                        int64_t total_q, int max_q_len, int num_q_heads, int num_kv_heads,
                        int head_dim, int block_size, int max_blocks_per_seq,
                        int64_t num_blocks, float scale, int q_dtype, int kv_dtype,
                        const float* k_scale, const float* v_scale, const int32_t* items, int num_items,
                        bool chunks, int longest_context, void* stream) {
    AICOMP_REQUIRE(num_seqs >= 0 && total_q >= 0, AICOMP_KV_EINVAL,
                   "paged_prefill_attn: negative sizes");
    if (num_seqs == 0 || total_q == 0) return AICOMP_KV_OK;
    AICOMP_REQUIRE(out && query && k_pool && v_pool && block_table && context_lens && cu_q_lens,
                   AICOMP_KV_EINVAL, "paged_prefill_attn: null pointer");
    int rc = check_common(num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq,
                          num_blocks, q_dtype, kv_dtype, k_scale, v_scale, "paged_prefill_attn");
    if (rc) return rc;
    AICOMP_REQUIRE(max_q_len > 0 && max_q_len <= total_q, AICOMP_KV_EINVAL,
                   "paged_prefill_attn: max_q_len %d out of range (total %lld)", max_q_len,
                   (long long)total_q);
    AICOMP_REQUIRE(max_blocks_per_seq > 0 && block_table_stride >= max_blocks_per_seq,
                   AICOMP_KV_EINVAL, "paged_prefill_attn: block table stride %lld < width %d",
                   (long long)block_table_stride, max_blocks_per_seq);
    AICOMP_REQUIRE(items == nullptr || num_items > 0, AICOMP_KV_EINVAL,
                   "paged_prefill_attn: an item list needs at least one item");
    DecodeArgs a;
    memset(&a, 0, sizeof(a));
    a.out = out; a.query = query; a.k_pool = k_pool; a.v_pool = v_pool;
    a.block_table = block_table; a.block_table_stride = block_table_stride;
    a.context_lens = context_lens; a.cu_q_lens = cu_q_lens;
    a.num_seqs = num_seqs; a.rows = total_q;
    a.hq = num_q_heads; a.hkv = num_kv_heads; a.d = head_dim; a.bs = block_size;
    a.max_blocks = max_blocks_per_seq; a.num_blocks = num_blocks;
    a.scale = scale; a.q_dtype = q_dtype; a.kv_dtype = kv_dtype;
    a.k_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? k_scale : nullptr;
    a.v_scale = kv_dtype == AICOMP_KV_FP8_E4M3 ? v_scale : nullptr;
    a.stream = (hipStream_t)stream;
    // an item list is taken by the two matrix-instruction kernels (and only while its length fits a
    // grid dimension); the other kernels walk the whole grid, which covers the same tiles
    if (items != nullptr && num_items <= 65535) { a.items = items; a.num_items = num_items; }
    a.chunks = chunks; a.longest_context = longest_context;
    if (prefill_mfma_supported(a, max_q_len)) return launch_prefill_mfma(a, max_q_len);
    // float32 models at head_dim 64 / 128: the float32 matrix instruction
    if (prefill_mfma_f32_supported(a, max_q_len)) return launch_prefill_mfma_f32(a, max_q_len);
    // head_dim 256, other block sizes: the tiled vector-ALU kernel (K/V staged in LDS once per 32
    // query rows)
    if (prefill_tiled_supported(a, max_q_len)) return launch_prefill_tiled(a, max_q_len);
    // what is left (pools that cannot be read 16 bytes at a time): every query row as its own
    // unsplit attention problem over its causal prefix
    a.partition_size = (int)(((int64_t)max_blocks_per_seq * block_size + block_size - 1) /
                             block_size * block_size);
    a.num_parts = 1;
    return launch_decode_generic(a);
}

int aicomp_paged_prefill_attn(void* out, const void* query, const void* k_pool, const void* v_pool,
                              const int32_t* block_table, int64_t block_table_stride,
                              const int32_t* context_lens, const int32_t* cu_q_lens, int num_seqs,
                              int64_t total_q, int max_q_len, int num_q_heads, int num_kv_heads,
                              int head_dim, int block_size, int max_blocks_per_seq,
                              int64_t num_blocks, float scale, int q_dtype, int kv_dtype,
                              const float* k_scale, const float* v_scale, void* stream) {
    return prefill_impl(out, query, k_pool, v_pool, block_table, block_table_stride, context_lens, cu_q_lens,
                        num_seqs, total_q, max_q_len, num_q_heads, num_kv_heads, head_dim, block_size,
                        max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale, v_scale, nullptr, 0,
                        false, 0, stream);
}

int aicomp_paged_prefill_attn_items(void* out, const void* query, const void* k_pool, const void* v_pool,
                                    const int32_t* block_table, int64_t block_table_stride,
                                    const int32_t* context_lens, const int32_t* cu_q_lens, int num_seqs,
                                    int64_t total_q, int max_q_len, int num_q_heads, int num_kv_heads,
                                    int head_dim, int block_size, int max_blocks_per_seq,
                                    int64_t num_blocks, float scale, int q_dtype, int kv_dtype,
                                    const float* k_scale, const float* v_scale, const int32_t* items,
                                    int num_items, void* stream) {
    AICOMP_REQUIRE(num_items >= 0 && (items != nullptr || num_items == 0), AICOMP_KV_EINVAL,
                   "paged_prefill_attn_items: %d items without a list", num_items);
    return prefill_impl(out, query, k_pool, v_pool, block_table, block_table_stride, context_lens, cu_q_lens,
                        num_seqs, total_q, max_q_len, num_q_heads, num_kv_heads, head_dim, block_size,
                        max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale, v_scale,
                        num_items > 0 ? items : nullptr, num_items, false, 0, stream);
}

static int append_prefill_impl(void* out, const void* query, const void* key, const void* value, int64_t kv_token_stride,
                               int64_t kv_head_stride, void* k_pool, void* v_pool, const int64_t* slot_mapping,
                               const int32_t* block_table, int64_t block_table_stride, const int32_t* context_lens,
                               const int32_t* cu_q_lens, int num_seqs, int64_t total_q, int max_q_len, int num_q_heads,
                               int num_kv_heads, int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                               float scale, int q_dtype, int kv_dtype, const float* k_scale, const float* v_scale,
                               const int32_t* items, int num_items, int longest_context, void* stream) {
    AICOMP_REQUIRE(longest_context >= 0, AICOMP_KV_EINVAL, "kv_append_prefill_attn: negative longest context");
    AICOMP_REQUIRE(num_items >= 0 && (items != nullptr || num_items == 0), AICOMP_KV_EINVAL,
                   "kv_append_prefill_attn: %d items without a list", num_items);
    if (key != nullptr) {
        const int rc = aicomp_kv_append(key, value, kv_token_stride, kv_head_stride, k_pool, v_pool, slot_mapping, total_q,
                                        num_kv_heads, head_dim, block_size, num_blocks, q_dtype, kv_dtype, k_scale, v_scale,
                                        stream);
        if (rc) return rc;
    }
    return prefill_impl(out, query, k_pool, v_pool, block_table, block_table_stride, context_lens, cu_q_lens,
                        num_seqs, total_q, max_q_len, num_q_heads, num_kv_heads, head_dim, block_size,
                        max_blocks_per_seq, num_blocks, scale, q_dtype, kv_dtype, k_scale, v_scale,
                        num_items > 0 ? items : nullptr, num_items, true, longest_context, stream);
}

int aicomp_kv_append_prefill_attn(void* out, const void* query, const void* key, const void* value, int64_t kv_token_stride,
                                  int64_t kv_head_stride, void* k_pool, void* v_pool, const int64_t* slot_mapping,
                                  const int32_t* block_table, int64_t block_table_stride, const int32_t* context_lens,
                                  const int32_t* cu_q_lens, int num_seqs, int64_t total_q, int max_q_len, int num_q_heads,
                                  int num_kv_heads, int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                                  float scale, int q_dtype, int kv_dtype, const float* k_scale, const float* v_scale,
                                  const int32_t* items, int num_items, void* stream) {
    return append_prefill_impl(out, query, key, value, kv_token_stride, kv_head_stride, k_pool, v_pool, slot_mapping,
                               block_table, block_table_stride, context_lens, cu_q_lens, num_seqs, total_q, max_q_len,
                               num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, num_blocks, scale,
                               q_dtype, kv_dtype, k_scale, v_scale, items, num_items, 0, stream);
}

int aicomp_kv_append_prefill_attn_sized(void* out, const void* query, const void* key, const void* value, int64_t kv_token_stride,
                                        int64_t kv_head_stride, void* k_pool, void* v_pool, const int64_t* slot_mapping,
                                        const int32_t* block_table, int64_t block_table_stride, const int32_t* context_lens,
                                        const int32_t* cu_q_lens, int num_seqs, int64_t total_q, int max_q_len, int num_q_heads,
                                        int num_kv_heads, int head_dim, int block_size, int max_blocks_per_seq, int64_t num_blocks,
                                        float scale, int q_dtype, int kv_dtype, const float* k_scale, const float* v_scale,
                                        const int32_t* items, int num_items, int longest_context, void* stream) {
    return append_prefill_impl(out, query, key, value, kv_token_stride, kv_head_stride, k_pool, v_pool, slot_mapping,
                               block_table, block_table_stride, context_lens, cu_q_lens, num_seqs, total_q, max_q_len,
                               num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq, num_blocks, scale,
                               q_dtype, kv_dtype, k_scale, v_scale, items, num_items, longest_context, stream);
}

int aicomp_paged_prefill_tile_positions(int num_q_heads, int num_kv_heads, int head_dim, int block_size,
                                        int q_dtype, int kv_dtype, int max_q_len) {
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads || max_q_len <= 0 || block_size != 16 ||
        (head_dim != 64 && head_dim != 128))
        return 0;
    if (is_16bit_float(q_dtype) && (kv_dtype == q_dtype || kv_dtype == AICOMP_KV_FP8_E4M3))
        return prefill_mfma_tile_positions(num_q_heads, num_kv_heads, max_q_len);
    if (q_dtype == AICOMP_KV_F32 && kv_dtype == AICOMP_KV_F32)
        return prefill_mfma_f32_tile_positions(num_q_heads, num_kv_heads);
    return 0;
}

}  // extern "C"
