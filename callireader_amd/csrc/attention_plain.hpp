// One query row against n keys in fp32 arithmetic, any element type and size: what the described decoders' attention falls back to (true fp32, sizes past the matrix-core forms).
//
// Bound by the latency of its loads when rows are few (16 workgroups for two rows of eight heads), so the loads are wide, many and coalesced: sixteen lanes share a key in q . k (64
// elements a load round), a column quad per thread in P . V with the keys dealt over the thread groups that are left, four keys' loads in flight in both.  With one key per thread and
// one column per thread instead, a row of 213 keys of 128 columns took 29 us; now 9.7 (1024 threads, decode), and 402 prompt rows 30 us for 37 (256 threads: the chip is full of
// workgroups; 27 with an order of sums of their own, which decode does not share).
#pragma once
#include "common.hpp"

template <typename T> __device__ __forceinline__ f32x4 plain_ld4(const T* p);
template <> __device__ __forceinline__ f32x4 plain_ld4<float>(const float* p) { return *(const f32x4*)p; }
template <> __device__ __forceinline__ f32x4 plain_ld4<bf16>(const bf16* p) {
    const bf16x4 v = *(const bf16x4*)p;
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

constexpr int PLAIN_MAX_COLS = 2048;
// The order of every sum is that of 1024 threads, whatever TPB is, so that a row's bits are the same decoded and in a prompt: key blocks of PLAIN_SPAN, a block's weights added over runs
// of 64 and then in run order, value sums over PLAIN_SPAN / quads interleaved shares of the block, every fourth part of the shares added first (what one of 256 threads holds), then those
// sums.  With fewer threads each takes the places of several.
constexpr int PLAIN_SPAN = 1024;
// floats of dynamic LDS for rows of `cols` columns under tpb threads; of static LDS (`red`)
constexpr int plain_lds_floats(int cols, int tpb) { return cols + PLAIN_SPAN + 4 * tpb; }
constexpr int PLAIN_RED = 2 * PLAIN_SPAN / 64;

// Q, K, V rows of `cols` columns (a multiple of 64, at most PLAIN_MAX_COLS; keys k_rs, values v_rs apart; 4-element aligned); put(column, value) for every column below `out`.
template <typename T, int TPB, typename F>
__device__ __forceinline__ void plain_attend(const T* Q, const T* K, int64_t k_rs, const T* V, int64_t v_rs, int n, int cols, int out, float scale, float softcap, float* sm, float* red, F put) {
    static_assert((TPB == PLAIN_SPAN || 4 * TPB == PLAIN_SPAN) && PLAIN_MAX_COLS / 4 <= PLAIN_SPAN / 2, "a thread takes one place or four; a place holds one column quad, a row at most half the places");
    constexpr int NWV = TPB / 64, VT = PLAIN_SPAN / TPB, RUNS = PLAIN_SPAN / 64;
    float *q = sm, *w = sm + cols;                              // [cols], [PLAIN_SPAN]
    f32x4* part = (f32x4*)(w + PLAIN_SPAN);                     // [TPB]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sub = lane & 15, kq = lane >> 4;
    for (int i = tid; i < cols; i += TPB) q[i] = (float)Q[i];
    int lq = 4;                                                 // quads places share a value row: a power of two >= cols / 4
    while (1 << lq < cols / 4) lq++;
    const int quads = 1 << lq, groups = PLAIN_SPAN >> lq;
    f32x4 acc[VT];                                              // of place tid + TPB v: column quad place % quads, share place / quads
#pragma unroll
    for (int v = 0; v < VT; v++) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (int k0 = 0; k0 < n; k0 += PLAIN_SPAN) {
        const int nk = min(PLAIN_SPAN, n - k0);
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
        float s[VT], mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < VT; v++) {
            s[v] = tid + TPB * v < nk ? w[tid + TPB * v] : -INFINITY;
            mx = fmaxf(mx, s[v]);
        }
        mx = wave_max(mx);
        if (lane == 0) red[wave] = mx;
        __syncthreads();
        float m_new = m_run;
#pragma unroll
        for (int i = 0; i < NWV; i++) m_new = fmaxf(m_new, red[i]);
#pragma unroll
        for (int v = 0; v < VT; v++) {
            float sum = 0.f;
            if (TPB * v < nk) {                                 // (uniform)
                const float e = tid + TPB * v < nk ? expf(s[v] - m_new) : 0.f;
                w[tid + TPB * v] = e;
                sum = wave_sum(e);
            }
            if (lane == 0) red[RUNS + wave + NWV * v] = sum;
        }
        __syncthreads();
        const float alpha = expf(m_run - m_new);
        float l = 0.f;
#pragma unroll
        for (int i = 0; i < RUNS; i++) l += red[RUNS + i];
        l_run = l_run * alpha + l;
        m_run = m_new;
#pragma unroll
        for (int v = 0; v < VT; v++) acc[v] *= alpha;
        constexpr int U = VT == 1 ? 4 : 1;                      // keys of a place whose loads are issued together, beside the other places'
        for (int kb = 0; kb < nk; kb += U * groups) {
            f32x4 x[VT][U];
            float p[VT][U];
#pragma unroll
            for (int v = 0; v < VT; v++) {
                const int place = tid + TPB * v, c = min(4 * (place & (quads - 1)), cols - 4);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k = kb + (place >> lq) + u * groups;
                    x[v][u] = plain_ld4<T>(V + (int64_t)(k0 + min(k, nk - 1)) * v_rs + c);
                    p[v][u] = w[min(k, nk - 1)];
                }
            }
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (kb + ((tid + TPB * v) >> lq) + u * groups < nk) acc[v] += p[v][u] * x[v][u];
        }
    }
    const int rest = max(1, groups / 4);                        // sums left when every fourth part of the shares has been added
    auto store = [&](int quad, f32x4 a) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (4 * quad + e < out) put(4 * quad + e, a[e] / l_run);
    };
    if constexpr (VT == 4) {
        if (quads > TPB) {                                      // two shares, both of them this thread's
            store(tid, acc[0] + acc[2]);
            store(tid + TPB, acc[1] + acc[3]);
            return;
        }
        part[tid] = acc[0] + acc[1] + acc[2] + acc[3];
    } else {
        part[tid] = acc[0];
        __syncthreads();
        if (tid < rest * quads) {
            f32x4 a = part[tid];
            for (int g = rest; g < groups; g += rest) a += part[g * quads + tid];
            part[tid] = a;                                      // (no other thread reads it here)
        }
    }
    __syncthreads();
    if (tid >= quads) return;
    f32x4 a = part[tid];
    for (int r = 1; r < rest; r++) a += part[r * quads + tid];
    store(tid, a);
}
