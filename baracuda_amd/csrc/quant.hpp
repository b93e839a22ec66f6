// quant.hpp -- per-token symmetric int8 quantization of a row held as 8-value
// chunks: loads, running max, scale and codes.
#pragma once

#include "bk_common.hpp"

namespace bk {

struct Bf16In { uint16_t bits; };   // element type: pointer steps of 2 bytes

// clamp(round_half_even(v * inv), qmin, qmax), the clamp in float before the
// conversion (rne_clamp: NaN -> 0, no out-of-range conversion).
__device__ __forceinline__ int8_t quant1(float v, float inv, float qmin, float qmax) {
    return (int8_t)(int)rne_clamp(v * inv, qmin, qmax);
}

// scale = max|x| / qmax (1 for an all-zero row) and its reciprocal.
__device__ __forceinline__ void quant_scale(float max_abs, float qmax, float &s, float &inv) {
    s = max_abs > 0.0f ? max_abs / qmax : 1.0f;
    inv = s != 0.0f ? 1.0f / s : 0.0f;
}

// Eight consecutive values of a row: one (bf16) or two (f32) 16-byte
// non-temporal loads.
template <typename T> struct QChunk;
template <> struct QChunk<Bf16In> {
    v4i w;
    __device__ __forceinline__ void load(const Bf16In *row, int c) {
        w = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(row) + c);
    }
    __device__ __forceinline__ void clear() { w = v4i{0, 0, 0, 0}; }
    __device__ __forceinline__ float get(int i) const {
        const uint32_t u = (uint32_t)w[i >> 1];
        return __uint_as_float((i & 1) ? (u & 0xffff0000u) : (u << 16));
    }
};
template <> struct QChunk<float> {
    v4i w[2];
    __device__ __forceinline__ void load(const float *row, int c) {
        w[0] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(row) + 2 * c);
        w[1] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(row) + 2 * c + 1);
    }
    __device__ __forceinline__ void clear() { w[0] = w[1] = v4i{0, 0, 0, 0}; }
    __device__ __forceinline__ float get(int i) const { return __int_as_float(w[i >> 2][i & 3]); }
};

template <typename T>
__device__ __forceinline__ float chunk_max(const QChunk<T> &q, float m) {
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(q.get(i)));
    return m;
}

// The chunk's 8 codes, in order.
template <typename T>
__device__ __forceinline__ v2i chunk_codes(const QChunk<T> &q, float inv, float qmin, float qmax) {
    v2i o;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t u = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) u |= (uint32_t)(uint8_t)quant1(q.get(4 * h + i), inv, qmin, qmax) << (8 * i);
        o[h] = (int)u;
    }
    return o;
}

// Max of a workgroup of WAVES waves (`red`: WAVES floats); contains a barrier.
template <int WAVES>
__device__ __forceinline__ float block_max(float v, float *red) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float m = red[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = fmaxf(m, red[w]);
    return m;
}

}  // namespace bk
