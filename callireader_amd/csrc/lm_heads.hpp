// The norm and rotation of eight columns of a row of the fused input projection, as a lane of the row kernel (lm_heads.hip) or of the decode mixer (lm_mix.hip) holds them.
#pragma once
#include "lm.hpp"

template <typename T> __device__ __forceinline__ void ld8(const T* p, float (&v)[8]);
template <> __device__ __forceinline__ void ld8<bf16>(const bf16* p, float (&v)[8]) {
    const bf16x8 x = *(const bf16x8*)p;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (float)x[e];
}
template <> __device__ __forceinline__ void ld8<float>(const float* p, float (&v)[8]) {
    const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) { v[e] = a[e]; v[4 + e] = b[e]; }
}
__device__ __forceinline__ void st8(bf16* p, const float (&v)[8]) {
    bf16x8 x;
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = (bf16)v[e];
    *(bf16x8*)p = x;
}
__device__ __forceinline__ void st8(float* p, const float (&v)[8]) {
    *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4*)(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// Eight entries e0 .. e0 + 7 of a head of P padded entries, whose P / 8 lanes sit side by side in one wave from a multiple of P / 8 on, with the constants they meet: gain (norm over `dim`
// entries where there is one), cos and sin of their pairs (a rotation of 2 * half entries: i and i + half are a pair).
struct HeadLane {
    float g[8], c[8], s[8];
    int e0, half;
    bool normed;
    __device__ __forceinline__ void ask(int first, const float* gain, int half_, const float* cos, const float* sin) {
        e0 = first; half = half_; normed = gain != nullptr;
        if (normed) ld8<float>(gain + e0, g);
        if (e0 >= 2 * half) return;
        if (half % 8 == 0) {
            const int i = e0 < half ? e0 : e0 - half;
            ld8<float>(cos + i, c);
            ld8<float>(sin + i, s);
        } else if (half % 4 == 0) {
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const int q = e0 + e, i = q < half ? q : q < 2 * half ? q - half : 0;
                const f32x4 cos4 = *(const f32x4*)(cos + i), sin4 = *(const f32x4*)(sin + i);
#pragma unroll
                for (int j = 0; j < 4; j++) { c[e + j] = cos4[j]; s[e + j] = sin4[j]; }
            }
        } else
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int q = e0 + e, i = q < half ? q : q < 2 * half ? q - half : 0;
                c[e] = cos[i]; s[e] = sin[i];
            }
    }
    // sx: the lane's eight places in the wave's own 512 floats of LDS, through which partners are read.  Every lane of the wave calls it.
    __device__ __forceinline__ void apply(int P, int dim, float eps, float* sx, float (&v)[8]) const {
        if (__builtin_amdgcn_ballot_w64(normed)) {              // (a head's lanes agree)
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) ss += v[e] * v[e];
            ss += dpp<0xB1>(ss); ss += dpp<0x4E>(ss); ss += dpp<0x141>(ss);      // lanes of eight; sixteen; half the wave; the wave
            if (P > 64) { const float o = dpp<0x128>(ss); ss += o; }
            if (P > 128) { const float o = __shfl_xor(ss, 16, 64); ss += o; }
            if (P > 256) { const float o = __shfl_xor(ss, 32, 64); ss += o; }
            if (normed) {
                const float rs = 1.0f / sqrtf(ss / (float)dim + eps);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= rs * g[e];
            }
        }
        if (!__builtin_amdgcn_ballot_w64(e0 < 2 * half)) return;
        st8(sx, v);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // (which product is rounded alone is spelled out: left to the compiler, entry 0 of every eight had the other one where entries went one by one)
        if (e0 < 2 * half) {
            if (half % 8 == 0) {
                const bool first = e0 < half;
                float u[8];
                ld8<float>(sx + (first ? half : -half), u);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = fmaf(v[e], c[e], first ? -(u[e] * s[e]) : u[e] * s[e]);
            } else if (half % 4 == 0) {                        // four entries side by side have their partners side by side
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    const int q = e0 + e;
                    const bool first = q < half;
                    if (q >= 2 * half) continue;
                    const f32x4 u = *(const f32x4*)(sx + e + (first ? half : -half));
#pragma unroll
                    for (int j = 0; j < 4; j++) v[e + j] = fmaf(v[e + j], c[e + j], first ? -(u[j] * s[e + j]) : u[j] * s[e + j]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int q = e0 + e;
                    if (q < half) v[e] = fmaf(v[e], c[e], -(sx[e + half] * s[e]));
                    else if (q < 2 * half) v[e] = fmaf(v[e], c[e], sx[e - half] * s[e]);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();                        // (the next columns overwrite sx)
    }
};
