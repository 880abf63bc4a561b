// One decoded token through the state of one (row, head): shared by the decode kernel (retention.hip) and the decode mixer (lm_mix.hip).
#pragma once
#include "lm.hpp"

// the sixteen dk groups of a wave sit four lanes apart
__device__ __forceinline__ f32x4 sum_groups(f32x4 o) {
    // lane ^ 4, ^ 8, ^ 16, ^ 32 on the vector pipe (LDS shuffles made a chain of four round trips of every token): the bank masks of two row shifts make the first
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int x = __float_as_int(o[e]);
        o[e] += __int_as_float(__builtin_amdgcn_update_dpp(__builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0x5, false), x, 0x114, 0xf, 0xa, false));
        o[e] += dpp<0x128>(o[e]);
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(o[e]), __float_as_uint(o[e]), false, false);
        o[e] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[e]), __float_as_uint(o[e]), false, false);
        o[e] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    }
    return o;
}
__device__ __forceinline__ float silu32(float x) { return x / (1.0f + expf(-x)); }

struct RetHead { float* state; const float* pw; int H, Kp, Vp, vdim; float eps, out_scale; };      // RetParams' fields of one layer
// A wave takes blocks of 16 value columns in turn (lm.hpp: the state's layout), the first of them asked for ahead of the token's own operands.
template <int NR> struct RetStep {
    const RetHead& p;
    float *st, decay;
    f32x4 s[NR];
    int lane, wave, nw, blocks;
    __device__ __forceinline__ RetStep(const RetHead& p, int seq, int h) : p(p) {
        lane = threadIdx.x & 63; wave = threadIdx.x >> 6; nw = blockDim.x >> 6; blocks = p.Vp >> 4;
        st = p.state + ((int64_t)seq * p.H + h) * p.Vp * p.Kp + lane * 4;
        decay = p.pw[h * (RET_CHUNK + 1) + 1];
    }
    __device__ __forceinline__ void load(int b) {
#pragma unroll
        for (int r = 0; r < NR; r++) s[r] = __builtin_nontemporal_load((const f32x4*)(st + ((int64_t)b * NR + r) * 256));
    }
    __device__ __forceinline__ void ask() { if (wave < blocks) load(wave); }
    // q, k: the head's rotated query and key; value(column): four values.  so: outputs [Vp], red: a block's squares
    template <typename F> __device__ __forceinline__ void run(bool fresh, const float* q, const float* k, F value, float* so, float* red) {
        const int g = lane >> 2, c4 = (lane & 3) * 4;
        for (int b = wave; b < blocks; b += nw) {
            if (b != wave) load(b);
            const f32x4 v = value(b * 16 + c4);
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < NR; r += 4) {
                const f32x4 qv = *(const f32x4*)(q + g * NR + r), kv = *(const f32x4*)(k + g * NR + r);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (fresh) s[r + e] = f32x4{0.f, 0.f, 0.f, 0.f};              // a state starts at zero, whatever the slot held before
                    // the fused product is spelled out: states of 64 keys as a prompt's recurrence has it (ret_recurrent_kernel), larger ones the other way round, so that neither moves with
                    // what the compiler finds around it
                    if (NR == 4) s[r + e] = __builtin_elementwise_fma(f32x4{kv[e], kv[e], kv[e], kv[e]}, v, s[r + e] * decay);
                    else s[r + e] = __builtin_elementwise_fma(s[r + e], f32x4{decay, decay, decay, decay}, kv[e] * v);
                    o += s[r + e] * qv[e];
                    __builtin_nontemporal_store(s[r + e], (f32x4*)(st + ((int64_t)b * NR + r + e) * 256));
                }
            }
            o = sum_groups(o);
            if (lane < 4) *(f32x4*)&so[b * 16 + c4] = o;
            float ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
            ss += __shfl_xor(ss, 1, 64);
            ss += __shfl_xor(ss, 2, 64);
            if (lane == 0) red[b] = ss;
        }
    }
    // after a barrier: put(column, output over the head's root mean square)
    template <typename F> __device__ __forceinline__ void finish(const float* so, const float* red, F put) {
        float ss = 0.f;
        for (int b = 0; b < blocks; b++) ss += red[b];
        const float rs = p.out_scale / sqrtf(ss / (float)p.vdim + p.eps);
        for (int c = threadIdx.x; c < p.vdim; c += blockDim.x) put(c, so[c] * rs);
    }
};
