// The residual update and norm of a few rows as a workgroup does it for itself: shared by the products that begin with it (lm_ahead.hip) and the router (moe.hip).
#pragma once
#include "lm.hpp"

constexpr int AHEAD_SEGS = 8;                                 // 256-column segments of all rows, a wave each

__device__ __forceinline__ f32x4 row4(const float* p) { return *(const f32x4*)p; }
__device__ __forceinline__ f32x4 row4(const bf16* p) { const bf16x4 v = *(const bf16x4*)p; return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
__device__ __forceinline__ void put4(float* p, f32x4 v) { *(f32x4*)p = v; }
__device__ __forceinline__ void put4(bf16* p, f32x4 v) { *(bf16x4*)p = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]}; }

// What a workgroup of 512 threads does ahead of its product: of rows row0 .. row0 + rows - 1 the sublayer sums y, x' = x + (gain_b ? rms(y) gain_b : y) (x' = y with `replace`), h = gain ? rms(x') gain : x'.
// h rows go to hs, ld apart; x' to memory by the workgroup that `writes`.  A row's squares are added segment by segment, as lm_post_kernel's waves do.  sums: AHEAD_SEGS floats
template <typename T>
__device__ __forceinline__ void update_rows(const LmAhead& p, int row0, int rows, T* hs, int ld, float* sums, bool writes) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), per = (p.Wp + 255) / 256;
    const int row = wave / per, col = (wave - row * per) * 256 + lane * 4;
    const int64_t at = (int64_t)(row0 + row) * p.Wp + col;
    const bool in = row < rows && col < p.Wp;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
    if (in) {
        if (!p.replace) x = row4(p.x + at);
        if (!p.slices) y = row4((const T*)p.Y + at);
        for (int k = 0; k < p.slices; k += 8) {                // K-slices in slice order, eight asked for together
            f32x4 v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = k + q < p.slices ? row4((const float*)p.Y + (int64_t)(k + q) * p.M * p.Wp + at) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 8; q++) y += v[q];
        }
    }
    auto norm = [&](f32x4 v) -> float {
        const float ss = wave_sum_s(v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]);
        if (lane == 0) sums[wave] = ss;
        __syncthreads();
        const int first = min(row * per, AHEAD_SEGS - per);   // (waves past the rows)
        float s = sums[first];
        for (int k = 1; k < per; k++) s += sums[first + k];
        __syncthreads();
        return 1.0f / sqrtf(s / (float)p.W + p.eps);
    };
    float rs = 1.f;
    if (p.gain_b) rs = norm(y);
    if (in) x += p.gain_b ? y * rs * row4(p.gain_b + col) : y;      // (lm_post_kernel's form: the compiler fuses the same operations)
    if (writes && in) put4(p.x_out + at, x);
    if (p.gain) rs = norm(x);
    if (in) put4(hs + row * ld + col, p.gain ? x * rs * row4(p.gain + col) : x);
    __syncthreads();
}
