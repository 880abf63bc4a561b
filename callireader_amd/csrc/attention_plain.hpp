// One query row against n keys in fp32 arithmetic, any element type and size: what the described decoders' attention falls back to (true fp32, sizes past the matrix-core forms).
//
// Bound by the latency of its loads when rows are few (16 workgroups for two rows of eight heads), so the loads are wide, many and coalesced: sixteen lanes share a key in q . k (64
// elements a load round), a column quad per thread in P . V with the keys dealt over the thread groups that are left, four keys' loads in flight in both.  With one key per thread and
// one column per thread instead, a row of 213 keys of 128 columns took 29 us; now 9.2 (1024 threads, decode), and 402 prompt
// rows 27 us for 37 (256 threads: the chip is full of workgroups).
#pragma once
#include "common.hpp"

template <typename T> __device__ __forceinline__ f32x4 plain_ld4(const T* p);
template <> __device__ __forceinline__ f32x4 plain_ld4<float>(const float* p) { return *(const f32x4*)p; }
template <> __device__ __forceinline__ f32x4 plain_ld4<bf16>(const bf16* p) {
    const bf16x4 v = *(const bf16x4*)p;
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

constexpr int PLAIN_MAX_COLS = 2048;
// floats of dynamic LDS for rows of `cols` columns under TPB threads
constexpr int plain_lds_floats(int cols, int tpb) { return cols + tpb + 4 * tpb; }

// Q, K, V rows of `cols` columns (a multiple of 64, at most PLAIN_MAX_COLS; keys k_rs, values v_rs apart; 4-element aligned); put(column, value) for every column below `out`.
template <typename T, int TPB, typename F>
__device__ __forceinline__ void plain_attend(const T* Q, const T* K, int64_t k_rs, const T* V, int64_t v_rs, int n, int cols, int out, float scale, float softcap, float* sm, float* red, F put) {
    constexpr int NWV = TPB / 64, ACC = PLAIN_MAX_COLS / 4 > TPB ? PLAIN_MAX_COLS / 4 / TPB : 1;
    float *q = sm, *w = sm + cols;                              // [cols], [TPB]
    f32x4* part = (f32x4*)(w + TPB);                            // [TPB]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sub = lane & 15, kq = lane >> 4;
    for (int i = tid; i < cols; i += TPB) q[i] = (float)Q[i];
    int quads = 16;                                             // threads that share a value row: a power of two >= cols / 4, at most all
    while (quads < cols / 4 && quads < TPB) quads *= 2;
    const int group = tid / quads, groups = TPB / quads, c0 = tid % quads;
    f32x4 acc[ACC];
#pragma unroll
    for (int j = 0; j < ACC; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (int k0 = 0; k0 < n; k0 += TPB) {
        const int nk = min(TPB, n - k0);
        __syncthreads();                                        // (q is there; the last block's w has been read)
        for (int b = wave * 4; b < nk; b += NWV * 16) {         // keys b + kq and three more, NWV * 4 apart
            float d[4] = {0.f, 0.f, 0.f, 0.f};
            for (int i = sub * 4; i < cols; i += 64) {
                const f32x4 qv = *(const f32x4*)(q + i);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const f32x4 kv = plain_ld4<T>(K + (int64_t)(k0 + min(b + kq + u * NWV * 4, nk - 1)) * k_rs + i);
#pragma unroll
                    for (int e = 0; e < 4; e++) d[u] += qv[e] * kv[e];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                d[u] += dpp<0xB1>(d[u]); d[u] += dpp<0x4E>(d[u]); d[u] += dpp<0x141>(d[u]); d[u] += dpp<0x128>(d[u]);      // over the sixteen lanes
                const int key = b + kq + u * NWV * 4;
                if (sub == 0 && key < nk) {
                    const float s = d[u] * scale;
                    w[key] = softcap > 0.f ? softcap * tanhf(s / softcap) : s;
                }
            }
        }
        __syncthreads();
        const float s = tid < nk ? w[tid] : -INFINITY;
        const float mx = wave_max(s);
        if (lane == 0) red[wave] = mx;
        __syncthreads();
        float m_new = m_run;
#pragma unroll
        for (int i = 0; i < NWV; i++) m_new = fmaxf(m_new, red[i]);
        const float e = tid < nk ? expf(s - m_new) : 0.f;
        w[tid] = e;
        const float sum = wave_sum(e);
        if (lane == 0) red[NWV + wave] = sum;
        __syncthreads();
        const float alpha = expf(m_run - m_new);
        float l = 0.f;
#pragma unroll
        for (int i = 0; i < NWV; i++) l += red[NWV + i];
        l_run = l_run * alpha + l;
        m_run = m_new;
#pragma unroll
        for (int j = 0; j < ACC; j++) {
            const int c = 4 * (c0 + quads * j);
            acc[j] *= alpha;
            if (c >= cols) continue;
            const T* v = V + (int64_t)k0 * v_rs + c;
            for (int k = group; k < nk; k += 4 * groups) {
                f32x4 x[4];
                float p[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int kk = k + u * groups;
                    x[u] = plain_ld4<T>(v + (int64_t)min(kk, nk - 1) * v_rs);
                    p[u] = kk < nk ? w[kk] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (k + u * groups < nk) acc[j] += p[u] * x[u];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < ACC; j++) {
        __syncthreads();
        part[tid] = acc[j];
        __syncthreads();
        const int c = 4 * (c0 + quads * j);
        if (group == 0 && c < cols) {
            f32x4 a = part[c0];
            for (int g = 1; g < groups; g++) a += part[g * quads + c0];
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (c + e < out) put(c + e, a[e] / l_run);
        }
    }
}
