// Expert routing: scores, grouped choice, and the assignments sorted by expert for the grouped products.
#include "lm.hpp"

namespace {

constexpr int MAX_E = 1024;

// order of a wave's own LDS accesses (each wave below works in LDS of its own: no workgroup barrier)
#define WAVE_LDS_FENCE()                                      \
    do {                                                      \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    \
        __builtin_amdgcn_wave_barrier();                      \
    } while (0)

// One wave routes one token; expert e = lane + 64 j sits in register j of its lane.  s = softmax(z) over all experts; choice scores s + correction; groups of neighbouring experts ranked
// by their best choice score, the best `keep` stay open; the `top` best open choice scores win (lowest index on a tie); the weights are the winners' s, not renormalised.
// z [E]: LDS or global; ch [E], gs [groups]: LDS of the wave.
template <int EPL>
__device__ __forceinline__ void route_row(const float* z, float* ch, float* gs, const float* __restrict__ corr, int E, int top, int groups, int keep, int lane, bool live, int32_t* idx, float* wt) {
    float s[EPL], c[EPL];
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < EPL; j++) {
        const int e = lane + 64 * j;
        s[j] = e < E ? z[e] : -INFINITY;
        c[j] = e < E ? corr[e] : 0.f;
        mx = fmaxf(mx, s[j]);
    }
    mx = wave_max_s(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < EPL; j++) { s[j] = expf(s[j] - mx); sum += s[j]; }      // (exp(-inf) = 0 past E)
    sum = wave_sum_s(sum);
#pragma unroll
    for (int j = 0; j < EPL; j++) {
        s[j] /= sum;
        c[j] = lane + 64 * j < E ? s[j] + c[j] : -INFINITY;
    }
    if (keep < groups) {
        const int per = E / groups;
        WAVE_LDS_FENCE();                                      // (ch may overlay what z was read from)
#pragma unroll
        for (int j = 0; j < EPL; j++)
            if (lane + 64 * j < E) ch[lane + 64 * j] = c[j];
        WAVE_LDS_FENCE();
        for (int g = lane; g < groups; g += 64) {
            float b = -INFINITY;
            for (int e = 0; e < per; e++) b = fmaxf(b, ch[g * per + e]);
            gs[g] = b;
        }
        WAVE_LDS_FENCE();
        // a group stays open when fewer than `keep` groups beat it (a tie goes to the lower index)
#pragma unroll
        for (int j = 0; j < EPL; j++) {
            const int e = lane + 64 * j;
            if (e >= E) continue;
            const int g = e / per;
            const float b = gs[g];
            int better = 0;
            for (int o = 0; o < groups; o++) better += (gs[o] > b || (gs[o] == b && o < g)) ? 1 : 0;
            if (better >= keep) c[j] = -INFINITY;
        }
    }
    int my_e = 0;
    float my_w = 0.f;
    for (int k0 = 0; k0 < top; k0 += 64) {
        for (int k = k0; k < min(top, k0 + 64); k++) {
            float b = c[0];
#pragma unroll
            for (int j = 1; j < EPL; j++) b = fmaxf(b, c[j]);
            b = wave_max_s(b);
            int e = 0;                                         // (NaN scores match nothing: expert 0, every index stays in range)
            float w = 0.f;
            bool found = false;
#pragma unroll
            for (int j = 0; j < EPL; j++) {
                const unsigned long long hit = __ballot(c[j] == b && lane + 64 * j < E);
                if (found || hit == 0) continue;               // (wave-uniform)
                const int l = __ffsll((unsigned long long)hit) - 1;
                found = true;
                e = l + 64 * j;
                w = lane_value(s[j], l);
                if (lane == l) c[j] = -INFINITY;
            }
            if (lane == k - k0) { my_e = e; my_w = w; }
        }
        if (live && k0 + lane < top) { idx[k0 + lane] = my_e; wt[k0 + lane] = my_w; }
    }
}

template <int EPL>
__global__ __launch_bounds__(256) void lm_route_kernel(const float* __restrict__ z, int64_t ldz, int slices, const float* __restrict__ corr, int M, int E, int top, int groups, int keep,
                                                       int32_t* __restrict__ idx, float* __restrict__ wt) {
    extern __shared__ float sm[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = blockIdx.x * 4 + wave;
    float* s = sm + wave * (2 * E + groups);
    const bool live = row < M;
    const int64_t r = live ? row : M - 1;
    for (int e = lane; e < E; e += 64) {
        float v = 0.f;
        for (int k = 0; k < slices; k += 8) {
            float t[8];
#pragma unroll
            for (int q = 0; q < 8; q++) t[q] = k + q < slices ? z[((int64_t)(k + q) * M + r) * ldz + e] : 0.f;
#pragma unroll
            for (int q = 0; q < 8; q++) v += t[q];
        }
        s[e] = v;
    }
    WAVE_LDS_FENCE();
    route_row<EPL>(s, s + E, s + 2 * E, corr, E, top, groups, keep, lane, live, idx + r * top, wt + r * top);
}

// bf16 models: the router product and the routing of 16 tokens in one workgroup of 16 waves.  Wave = a quarter of K x a quarter of the experts (EB blocks of 16); the four K-slices
// meet in LDS in slice order, then wave w routes token w.
template <int EB>
__global__ __launch_bounds__(1024) void lm_router_kernel(const bf16* __restrict__ h, int64_t ldh, const bf16* __restrict__ Wr, int K, const float* __restrict__ corr, int M, int E, int top,
                                                         int groups, int keep, int32_t* __restrict__ idx, float* __restrict__ wt) {
    extern __shared__ float sm[];
    constexpr int ELD = EB * 64 + 4;
    float* part = sm;                                  // [4][16][ELD]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
    const int kq = wave >> 2, eq = wave & 3, m0 = blockIdx.x * 16;
    const int steps = K / 32, per = (steps + 3) / 4, k_lo = min(kq * per, steps), k_hi = min(k_lo + per, steps);
    const bf16* x = h + (int64_t)min(m0 + li, M - 1) * ldh + g * 8;
    const bf16* w[EB];
#pragma unroll
    for (int b = 0; b < EB; b++) w[b] = Wr + (int64_t)min((eq * EB + b) * 16 + li, E - 1) * K + g * 8;
    f32x4 acc[EB];
#pragma unroll
    for (int b = 0; b < EB; b++) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = EB > 2 ? 2 : 8 / EB;
    int ks = k_lo;
    for (; ks + U <= k_hi; ks += U) {
        bf16x8 xf[U], wf[EB][U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            xf[u] = *(const bf16x8*)(x + (ks + u) * 32);
#pragma unroll
            for (int b = 0; b < EB; b++) wf[b][u] = *(const bf16x8*)(w[b] + (ks + u) * 32);
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int b = 0; b < EB; b++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[b][u], xf[u], acc[b], 0, 0, 0);
    }
    for (; ks < k_hi; ks++)
#pragma unroll
        for (int b = 0; b < EB; b++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(w[b] + ks * 32), *(const bf16x8*)(x + ks * 32), acc[b], 0, 0, 0);
#pragma unroll
    for (int b = 0; b < EB; b++) *(f32x4*)(part + (kq * 16 + li) * ELD + (eq * EB + b) * 16 + 4 * g) = acc[b];      // experts 4 g + 0..3 of the block, token li
    __syncthreads();
    float* z = part + wave * ELD;                      // slice 0 of token `wave` becomes its sum
    for (int e = lane; e < E; e += 64) z[e] = ((z[e] + part[(16 + wave) * ELD + e]) + part[(32 + wave) * ELD + e]) + part[(48 + wave) * ELD + e];
    WAVE_LDS_FENCE();
    float* ch = part + (16 + wave) * ELD;              // slices 1 and 2 of the token are free now
    float* gs = part + (32 + wave) * ELD;
    const bool live = m0 + wave < M;
    const int64_t r = live ? m0 + wave : M - 1;
    route_row<EB>(z, ch, gs, corr, E, top, groups, keep, lane, live, idx + r * top, wt + r * top);
}

// Few rows: one workgroup per 16 tokens would pull the whole router through one CU, so K goes over LM_ROUTER_SLICES workgroups; lm_route_kernel adds the slices.
// Waves split the experts in blocks of 16.
__global__ __launch_bounds__(256) void lm_router_slice_kernel(const bf16* __restrict__ h, int64_t ldh, const bf16* __restrict__ Wr, int K, int M, int E, float* __restrict__ part, int64_t ldp) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, li = lane & 15, m0 = blockIdx.x * 16;
    const int steps = K / 32, per = (steps + (int)gridDim.y - 1) / (int)gridDim.y, k_lo = min((int)blockIdx.y * per, steps), k_hi = min(k_lo + per, steps);
    const bf16* x = h + (int64_t)min(m0 + li, M - 1) * ldh + g * 8;
    for (int b = wave; b * 16 < E; b += 4) {
        const bf16* w = Wr + (int64_t)min(b * 16 + li, E - 1) * K + g * 8;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int ks = k_lo; ks < k_hi; ks += 8) {              // eight k-steps of loads in flight; steps past the slice repeat its last one against zeros
            bf16x8 wf[8], xf[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int k = min(ks + u, k_hi - 1) * 32;
                wf[u] = *(const bf16x8*)(w + k);
                xf[u] = *(const bf16x8*)(x + k);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                if (ks + u >= k_hi) xf[u] = bf16x8{};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf[u], acc, 0, 0, 0);
            }
        }
        if (m0 + li < M) *(f32x4*)(part + ((int64_t)blockIdx.y * M + m0 + li) * ldp + b * 16 + 4 * g) = acc;
    }
}

template <int EB>
int launch_router_t(const Lm& lm, const LmLayer& L, int M, const void* h, int32_t* idx, float* wt, hipStream_t st) {
    constexpr int LDS = 4 * 16 * (EB * 64 + 4) * 4;
    static std::atomic<uint64_t> done{0};
    if (!cr_dyn_lds_once(done, (const void*)lm_router_kernel<EB>, LDS)) return CR_ERR_HIP;
    hipLaunchKernelGGL(lm_router_kernel<EB>, dim3((M + 15) / 16), dim3(1024), LDS, st, (const bf16*)h, (int64_t)lm.Wp, (const bf16*)L.router, lm.Wp, L.corr, M, L.s.experts, L.s.top, L.s.groups,
                       L.s.keep, idx, wt);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

// One workgroup: counts per expert, their prefix sums, the tile table, then every assignment's place.  The order of an expert's rows is the order its wave-sized chunks of
// assignments reach the cursor; a row's result does not depend on its place in a tile.
__global__ __launch_bounds__(1024) void lm_plan_kernel(const int32_t* __restrict__ idx, int n, int E, int tile_m, int32_t* __restrict__ perm, int4* __restrict__ tiles,
                                                       int32_t* __restrict__ n_tiles, int max_tiles) {
    __shared__ int cnt[MAX_E], cur[MAX_E], tl[MAX_E];
    const int tid = threadIdx.x;
    for (int e = tid; e < MAX_E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int i0 = tid; i0 < n; i0 += 8192) {
        int e[8];
#pragma unroll
        for (int q = 0; q < 8; q++) e[q] = i0 + 1024 * q < n ? idx[i0 + 1024 * q] : -1;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (e[q] >= 0) atomicAdd(&cnt[e[q]], 1);
    }
    __syncthreads();
    // inclusive scans over MAX_E slots (positions and tiles)
    const int c = cnt[tid], t = (c + tile_m - 1) / tile_m;
    cur[tid] = c; tl[tid] = t;
    __syncthreads();
    for (int o = 1; o < MAX_E; o <<= 1) {
        const int a = tid >= o ? cur[tid - o] : 0, b = tid >= o ? tl[tid - o] : 0;
        __syncthreads();
        cur[tid] += a; tl[tid] += b;
        __syncthreads();
    }
    const int off = cur[tid] - c, t0 = tl[tid] - t;
    if (tid == MAX_E - 1) *n_tiles = min(tl[tid], max_tiles);
    __syncthreads();
    cur[tid] = off;
    for (int k = 0; k < t; k++)
        if (t0 + k < max_tiles) tiles[t0 + k] = make_int4(tid, off + k * tile_m, min(tile_m, c - k * tile_m), (k & 7) | min(8, t - (k & ~7)) << 4);
    __syncthreads();
    for (int i0 = tid; i0 < n; i0 += 8192) {
        int e[8], at[8];
#pragma unroll
        for (int q = 0; q < 8; q++) e[q] = i0 + 1024 * q < n ? idx[i0 + 1024 * q] : -1;
#pragma unroll
        for (int q = 0; q < 8; q++) at[q] = e[q] >= 0 ? atomicAdd(&cur[e[q]], 1) : 0;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (e[q] >= 0) perm[at[q]] = i0 + 1024 * q;
    }
}

}  // namespace

bool lm_router_supported(const LmLayer& L) { return L.s.experts <= 256; }

int launch_lm_router(const Lm& lm, const LmLayer& L, int M, const void* h, int32_t* idx, float* wt, float* part, hipStream_t st) {
    if (M <= 128 && part) {
        hipLaunchKernelGGL(lm_router_slice_kernel, dim3((M + 15) / 16, LM_ROUTER_SLICES), dim3(256), 0, st, (const bf16*)h, (int64_t)lm.Wp, (const bf16*)L.router, lm.Wp, M, L.s.experts, part,
                           (int64_t)L.Ep);
        CR_HIP(hipGetLastError());
        return launch_lm_route(L, M, part, L.Ep, LM_ROUTER_SLICES, idx, wt, st);
    }
    if (L.s.experts <= 64) return launch_router_t<1>(lm, L, M, h, idx, wt, st);
    if (L.s.experts <= 128) return launch_router_t<2>(lm, L, M, h, idx, wt, st);
    if (L.s.experts <= 256) return launch_router_t<4>(lm, L, M, h, idx, wt, st);
    return cr_fail(CR_ERR_ARG, "router: %d experts", L.s.experts);
}

int launch_lm_route(const LmLayer& L, int M, const float* z, int64_t ldz, int slices, int32_t* idx, float* wt, hipStream_t st) {
    const int E = L.s.experts, G = L.s.groups;
    const dim3 grid((M + 3) / 4);
    const size_t lds = (size_t)4 * (2 * E + G) * 4;
#define ROUTE(EPL) hipLaunchKernelGGL(lm_route_kernel<EPL>, grid, dim3(256), lds, st, z, ldz, slices, L.corr, M, E, L.s.top, G, L.s.keep, idx, wt)
    if (E <= 64) ROUTE(1);
    else if (E <= 128) ROUTE(2);
    else if (E <= 256) ROUTE(4);
    else ROUTE(16);
#undef ROUTE
    CR_HIP(hipGetLastError());
    return CR_OK;
}

int launch_lm_plan(const LmLayer& L, int M, int tile_m, const int32_t* idx, int32_t* perm, int4* tiles, int32_t* n_tiles, hipStream_t st) {
    if (L.s.experts > MAX_E) return cr_fail(CR_ERR_ARG, "routing: %d experts (at most %d)", L.s.experts, MAX_E);
    const int n = M * L.s.top;
    hipLaunchKernelGGL(lm_plan_kernel, dim3(1), dim3(1024), 0, st, idx, n, L.s.experts, tile_m, perm, tiles, n_tiles, lm_max_tiles(n, L.s.experts, tile_m));
    CR_HIP(hipGetLastError());
    return CR_OK;
}
