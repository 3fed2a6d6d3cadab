// Rotary embedding of eight columns and their partners: loads, roundings and the rotation, shared by the fused
// append (rope_append.hip) and the decode kernels that rotate their own rows (decode_mfma.hip).
#pragma once

#include "common.h"

namespace aicomp {

namespace {

template <typename T> struct Row8;
template <> struct Row8<bf16_t> {
    __device__ __forceinline__ static void load(const bf16_t* p, float* f) {
        Vec16<bf16_t>::unpack(*(const uint4*)p, f);
    }
    // gfx950 converts in hardware (v_cvt_pk_bf16_f32, round to nearest even)
    __device__ __forceinline__ static uint32_t pack2(float a, float b) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 v = {(__bf16)a, (__bf16)b};
        return __builtin_bit_cast(uint32_t, v);
    }
    __device__ __forceinline__ static void store(bf16_t* p, const float* f) {
        *(uint4*)p = make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7]));
    }
    // value as the tensor type holds it
    __device__ __forceinline__ static float round(float v) { return (float)(__bf16)v; }
};
template <> struct Row8<f16_t> {
    __device__ __forceinline__ static void load(const f16_t* p, float* f) {
        Vec16<f16_t>::unpack(*(const uint4*)p, f);
    }
    __device__ __forceinline__ static void store(f16_t* p, const float* f) {
        *(uint4*)p = make_uint4(F16Fmt::pack(f[0], f[1]), F16Fmt::pack(f[2], f[3]), F16Fmt::pack(f[4], f[5]),
                                F16Fmt::pack(f[6], f[7]));
    }
    __device__ __forceinline__ static float round(float v) { return (float)(_Float16)v; }
};
template <> struct Row8<float> {
    __device__ __forceinline__ static void load(const float* p, float* f) {
        const float4 a = ((const float4*)p)[0], b = ((const float4*)p)[1];
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
    __device__ __forceinline__ static void store(float* p, const float* f) {
        ((float4*)p)[0] = make_float4(f[0], f[1], f[2], f[3]);
        ((float4*)p)[1] = make_float4(f[4], f[5], f[6], f[7]);
    }
    __device__ __forceinline__ static float round(float v) { return v; }
};

// out = round(round(x * c) + round(r * s)), products and sum as separate roundings; NEG: -r in r's place
// (rounding is symmetric, so the sign moves to the sum)
template <typename T, bool NEG = false>
__device__ __forceinline__ float rot1(float x, float r, float c, float s) {
#pragma clang fp contract(off)
    const float p1 = Row8<T>::round(x * c);
    const float p2 = Row8<T>::round(r * s);
    return Row8<T>::round(NEG ? p1 - p2 : p1 + p2);
}

// 8 elements as they lie in memory
template <typename T> struct Raw8 {
    static constexpr int V16 = 8 * sizeof(T) / 16;
    uint4 v[V16];
    __device__ __forceinline__ void load(const T* p) {
#pragma unroll
        for (int k = 0; k < V16; ++k) v[k] = ((const uint4*)p)[k];
    }
    __device__ __forceinline__ void store(T* p) const {
#pragma unroll
        for (int k = 0; k < V16; ++k) ((uint4*)p)[k] = v[k];
    }
    __device__ __forceinline__ void unpack(float* f) const { Row8<T>::load((const T*)v, f); }
};

}  // namespace

}  // namespace aicomp
