// Expert routing: scores, grouped choice, and the assignments sorted by expert for the grouped products.
#include "diag.hpp"
#include "lm_ahead.hpp"

namespace {

constexpr int MAX_E = 1024;
constexpr int LM_PLAN_ONE = 8192;      // assignments one workgroup places by itself

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
// meet in LDS in slice order, then wave w routes token w.  Bound by the CU's load path: loaded straight as operands, a fragment is 16 rows x 64 bytes and takes four times its bytes' time,
// and four waves fetched the same tokens.  So the tokens come once, by LDS-DMA, a contiguous KiB an instruction (16 k-steps of a row and slice; the 16-byte chunks of rows in fours XORed for
// the reads), the weights from their fragment-ordered copy (wsw; without it row by row as before), and waves past the experts stay idle.  6124 tokens, 2048 x 32: 28 -> 15.8 us.
template <int EB>
__global__ __launch_bounds__(1024) void lm_router_kernel(const bf16* __restrict__ h, int64_t ldh, const bf16* __restrict__ Wr, int wsw, int K, const float* __restrict__ corr, int M, int E, int top,
                                                         int groups, int keep, int32_t* __restrict__ idx, float* __restrict__ wt) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    constexpr int ELD = EB * 64 + 4, STEPS = 16;
    float* part = sm;                                  // [4][16][ELD]
    char* xs = (char*)sm;                              // [slice][token][KiB], until the products are done: two workgroups a CU
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, li = lane & 15;
    const int kq = wave >> 2, eq = wave & 3, m0 = blockIdx.x * 16;
    const int steps = K / 32, per = (steps + 3) / 4, k_lo = min(kq * per, steps), k_hi = min(k_lo + per, steps);
    const bf16* row = h + (int64_t)min(m0 + wave, M - 1) * ldh;
    const int own = (lane ^ ((wave & 3) << 2)) * 8;    // the lane's column of a KiB of row `wave`
    const char* x = xs + (kq * 16 + li) * 1024;
    const bf16* w[EB];
    const int wstep = wsw ? 512 : 32;
#pragma unroll
    for (int b = 0; b < EB; b++) {
        const int blk = min(eq * EB + b, (E + 15) / 16 - 1);
        w[b] = wsw ? Wr + (int64_t)blk * (K / 32) * 512 + lane * 8 : Wr + (int64_t)min(blk * 16 + li, E - 1) * K + g * 8;
    }
    f32x4 acc[EB];
#pragma unroll
    for (int b = 0; b < EB; b++) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = EB > 2 ? 2 : 8 / EB;
    const bool mine = eq * EB * 16 < E;
    for (int c = 0; c < per; c += STEPS) {
        if (c) __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; s++) {
            CR_DIAG_POISON(xs + (s * 16 + wave) * 1024)
            __builtin_amdgcn_global_load_lds(CR_GLB(row + min((min(s * per, steps) + c) * 32 + own, K - 8)), CR_LDS(xs + (s * 16 + wave) * 1024), 16, 0, 0);
        }
        const int n = min(STEPS, k_hi - k_lo - c), k0 = k_lo + c;
        bf16x8 wf[EB][U];
        auto load = [&](int ks) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int b = 0; b < EB; b++)
                    if (ks + u < n) wf[b][u] = *(const bf16x8*)(w[b] + (int64_t)(k0 + ks + u) * wstep);
        };
        if (mine) load(0);
        __syncthreads();
        if (!mine) continue;
        for (int ks = 0; ks < n; ks += U) {
            if (ks) load(ks);
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (ks + u >= n) break;                // (uniform)
                const bf16x8 xf = *(const bf16x8*)(x + ((((ks + u) * 4 + g) ^ ((li & 3) << 2)) << 4));
#pragma unroll
                for (int b = 0; b < EB; b++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[b][u], xf, acc[b], 0, 0, 0);
            }
        }
    }
    __syncthreads();
    if (mine)
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

// Decode: a row's residual update, its router scores and its choice in one workgroup of eight waves, where those were three launches (24 rows, 2048 x 32: 4.6 + 3.4 + 4.8 us and two gaps -> 8.9).  Scores are
// the ones lm_router_slice_kernel and lm_route_kernel form, bit for bit -- the same K-slices on the matrix cores, added in slice order: a choice between close experts must not hang on the
// path.  A wave takes every eighth slice of all experts; the weights of its first 32 experts (fragment-ordered with wsw) are asked for ahead of the update.
constexpr int POST_COLS = 2048, POST_E = 64, POST_BATCH = 32, POST_COLS_TWO = 1536;      // columns and experts at most; experts of a batch of weights, columns at most with two batches
__global__ __launch_bounds__(512) void lm_post_route_kernel(const LmAhead a, bf16* __restrict__ h, const bf16* __restrict__ Wr, int wsw, const float* __restrict__ corr, int E, int top, int groups,
                                                            int keep, int32_t* __restrict__ idx, float* __restrict__ wt) {
    touch_args<(int)(sizeof(LmAhead) + 64)>();
    constexpr int SL = LM_ROUTER_SLICES / 8, MAX_PER = POST_COLS / 32 / LM_ROUTER_SLICES, PAIR = POST_BATCH / 16;      // slices a wave, k-steps a slice, blocks of 16 experts a batch
    __shared__ __attribute__((aligned(16))) bf16 hs[POST_COLS];
    __shared__ __attribute__((aligned(16))) float part[LM_ROUTER_SLICES][POST_E];
    __shared__ float sums[AHEAD_SEGS], z[POST_E], ch[POST_E], gs[POST_E];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), row = blockIdx.x, K = a.Wp, g = lane >> 4, li = lane & 15;
    const int steps = K / 32, per = (steps + LM_ROUTER_SLICES - 1) / LM_ROUTER_SLICES, blocks = (E + 15) / 16;
    bf16x8 w[PAIR][SL][MAX_PER];
    auto load = [&](int b0) {
#pragma unroll
        for (int j = 0; j < PAIR; j++) {
            const int b = min(b0 + j, blocks - 1);
            const bf16* p = wsw ? Wr + (int64_t)b * steps * 512 + lane * 8 : Wr + (int64_t)min(b * 16 + li, E - 1) * K + g * 8;
#pragma unroll
            for (int s = 0; s < SL; s++)
#pragma unroll
                for (int u = 0; u < MAX_PER; u++)
                    if (u < per) w[j][s][u] = *(const bf16x8*)(p + (int64_t)min((wave + 8 * s) * per + u, steps - 1) * (wsw ? 512 : 32));
        }
    };
    load(0);
    __builtin_amdgcn_sched_barrier(0);
    update_rows<bf16>(a, row, 1, hs, K, sums, true);
    if (wave * 512 + lane * 8 < K) *(bf16x8*)(h + (int64_t)row * K + wave * 512 + lane * 8) = *(const bf16x8*)(hs + wave * 512 + lane * 8);
    for (int b0 = 0; b0 < blocks; b0 += PAIR) {
        if (b0) load(b0);
#pragma unroll
        for (int j = 0; j < PAIR; j++)
#pragma unroll
            for (int s = 0; s < SL; s++) {
                const int k_lo = min((wave + 8 * s) * per, steps), k_hi = min(k_lo + per, steps);
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < MAX_PER; u++) {
                    if (k_lo + u >= k_hi) break;               // (uniform)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j][s][u], *(const bf16x8*)(hs + (k_lo + u) * 32 + g * 8), acc, 0, 0, 0);
                }
                if (li == 0 && b0 + j < blocks) *(f32x4*)(&part[wave + 8 * s][(b0 + j) * 16 + 4 * g]) = acc;      // (every column is the row)
            }
    }
    __syncthreads();
    if (wave) return;
    if (lane < E) {
        float v = 0.f;
#pragma unroll
        for (int s = 0; s < LM_ROUTER_SLICES; s++) v += part[s][lane];
        z[lane] = v;
    }
    WAVE_LDS_FENCE();
    route_row<1>(z, ch, gs, corr, E, top, groups, keep, lane, true, idx + (int64_t)row * top, wt + (int64_t)row * top);
}

template <int EB>
int launch_router_t(const Lm& lm, const LmLayer& L, int M, const void* h, int32_t* idx, float* wt, hipStream_t st) {
    constexpr int PART = 4 * 16 * (EB * 64 + 4) * 4, LDS = PART > 64 * 1024 ? PART : 64 * 1024;
    static std::atomic<uint64_t> done{0};
    if (!cr_dyn_lds_once(done, (const void*)lm_router_kernel<EB>, LDS)) return CR_ERR_HIP;
    hipLaunchKernelGGL(lm_router_kernel<EB>, dim3((M + 15) / 16), dim3(1024), LDS, st, (const bf16*)h, (int64_t)lm.Wp, L.router_dl ? L.router_dl : (const bf16*)L.router, L.router_dl != nullptr,
                       lm.Wp, L.corr, M, L.s.experts, L.s.top, L.s.groups, L.s.keep, idx, wt);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

// Assignments sorted by expert.  The order of an expert's rows is the order its wave-sized chunks of assignments reach the cursor; a row's result does not depend on its place in a tile.
// offsets of the experts (exclusive scans of counts and tiles over MAX_E slots) for thread e's expert of c rows; the tile table by the workgroup that `writes`
__device__ __forceinline__ int plan_offsets(int c, int tile_m, int* cur, int* tl, int4* tiles, int32_t* n_tiles, int max_tiles, bool writes) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, t = (c + tile_m - 1) / tile_m;
    int sc = c, st = t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(sc, o, 64), b = __shfl_up(st, o, 64);
        if (lane >= o) { sc += a; st += b; }
    }
    if (lane == 63) { cur[wave] = sc; tl[wave] = st; }
    __syncthreads();
    int off = sc - c, t0 = st - t;
    for (int w = 0; w < wave; w++) { off += cur[w]; t0 += tl[w]; }
    if (writes) {
        if (tid == MAX_E - 1) *n_tiles = min(t0 + t, max_tiles);
        for (int k = 0; k < t; k++)
            if (t0 + k < max_tiles) tiles[t0 + k] = make_int4(tid, off + k * tile_m, min(tile_m, c - k * tile_m), (k & 7) | min(8, t - (k & ~7)) << 4);
    }
    __syncthreads();
    return off;
}
// LDS counters of an expert each, over assignments [lo, hi): f(assignment, what the counter held)
template <typename F> __device__ __forceinline__ void plan_count(const int32_t* idx, int lo, int hi, int* cnt, F f) {
    for (int i0 = lo + threadIdx.x; i0 < hi; i0 += 8192) {
        int e[8], at[8];
#pragma unroll
        for (int q = 0; q < 8; q++) e[q] = i0 + 1024 * q < hi ? idx[i0 + 1024 * q] : -1;
#pragma unroll
        for (int q = 0; q < 8; q++) at[q] = e[q] >= 0 ? atomicAdd(&cnt[e[q]], 1) : 0;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (e[q] >= 0) f(i0 + 1024 * q, at[q]);
    }
}

// One workgroup for all assignments, as long as they are few
__global__ __launch_bounds__(1024) void lm_plan_kernel(const int32_t* __restrict__ idx, int n, int E, int tile_m, int32_t* __restrict__ perm, int4* __restrict__ tiles,
                                                       int32_t* __restrict__ n_tiles, int max_tiles) {
    __shared__ int cnt[MAX_E], cur[16], tl[16];
    const int tid = threadIdx.x;
    cnt[tid] = 0;
    __syncthreads();
    plan_count(idx, 0, n, cnt, [](int, int) {});
    __syncthreads();
    const int off = plan_offsets(cnt[tid], tile_m, cur, tl, tiles, n_tiles, max_tiles, true);
    cnt[tid] = off;
    __syncthreads();
    plan_count(idx, 0, n, cnt, [&](int i, int at) { perm[at] = i; });
}

// Many assignments: counting and placing them is bound by one CU's LDS atomics, so PLAN_PARTS workgroups count a part each, and as many place it behind what the parts ahead of it hold.
// One workgroup / parts, us: 32 experts 4096 6.4 / 6.8, 8192 9.4 / 9.0, 12 288 12.5 / 10.4, 24 576 19.7 / 11.5; 256 experts 4096 5.9 / 8.8, 8192 8.1 / 9.6, 12 288 10.7 / 10.6, 24 576 17.0 / 10.6.
constexpr int PLAN_PARTS = 32;
__global__ __launch_bounds__(1024) void lm_plan_count_kernel(const int32_t* __restrict__ idx, int n, int E, int32_t* __restrict__ hist) {
    __shared__ int cnt[MAX_E];
    const int tid = threadIdx.x, per = (n + PLAN_PARTS - 1) / PLAN_PARTS, lo = min((int)blockIdx.x * per, n);
    cnt[tid] = 0;
    __syncthreads();
    plan_count(idx, lo, min(lo + per, n), cnt, [](int, int) {});
    __syncthreads();
    if (tid < E) hist[blockIdx.x * E + tid] = cnt[tid];
}
__global__ __launch_bounds__(1024) void lm_plan_place_kernel(const int32_t* __restrict__ idx, int n, int E, int tile_m, const int32_t* __restrict__ hist, int32_t* __restrict__ perm,
                                                             int4* __restrict__ tiles, int32_t* __restrict__ n_tiles, int max_tiles) {
    __shared__ int cnt[MAX_E], cur[16], tl[16];
    const int tid = threadIdx.x, per = (n + PLAN_PARTS - 1) / PLAN_PARTS, lo = min((int)blockIdx.x * per, n);
    int c = 0, ahead = 0;
    if (tid < E)
#pragma unroll 8
        for (int p = 0; p < PLAN_PARTS; p++) {
            const int v = hist[p * E + tid];
            c += v;
            ahead += p < (int)blockIdx.x ? v : 0;
        }
    cnt[tid] = plan_offsets(c, tile_m, cur, tl, tiles, n_tiles, max_tiles, blockIdx.x == 0) + ahead;
    __syncthreads();
    plan_count(idx, lo, min(lo + per, n), cnt, [&](int i, int at) { perm[at] = i; });
}

}  // namespace

// A row's workgroup reads the whole router from L2.  One batch of weights travels under the update; a second one is a round trip and its bytes behind it, which pays up to 1536 columns.  A layer's
// step, us saved against the separate kernels at 9 / 24 / 64 rows: 2048 x 32 3.3 / 3.1 / 3.3, 1024 x 64 3.0 / 2.9 / 1.8, 1536 x 64 0.7 / 0.9 / 0.4; 2048 x 36 -0.4 / -0.7 / -0.8, 2048 x 64
// -2.2 / -1.9 / -1.6.
bool lm_post_route_supported(const Lm& lm, const LmLayer& L) {
    return !lm.f32 && lm.Wp <= (L.s.experts <= POST_BATCH ? POST_COLS : POST_COLS_TWO) && lm.Wp % 64 == 0 && L.s.experts <= POST_E;
}

int launch_lm_post_route(const Lm& lm, const LmLayer& L, const LmAhead& a, void* h, int32_t* idx, float* wt, hipStream_t st) {
    if (a.M <= 0 || !a.Y || !a.x || !a.x_out || !h || !idx || !wt || a.Wp != lm.Wp || !lm_post_route_supported(lm, L)) return cr_fail(CR_ERR_ARG, "update and routing: %d rows, %d experts", a.M, L.s.experts);
    hipLaunchKernelGGL(lm_post_route_kernel, dim3(a.M), dim3(512), 0, st, a, (bf16*)h, L.router_dl ? L.router_dl : (const bf16*)L.router, L.router_dl != nullptr,
                       L.corr, L.s.experts, L.s.top, L.s.groups, L.s.keep, idx, wt);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

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

int launch_lm_plan(const LmLayer& L, int M, int tile_m, const int32_t* idx, int32_t* perm, int4* tiles, int32_t* n_tiles, int32_t* hist, hipStream_t st) {
    if (L.s.experts > MAX_E) return cr_fail(CR_ERR_ARG, "routing: %d experts (at most %d)", L.s.experts, MAX_E);
    const int n = M * L.s.top, E = L.s.experts, most = lm_max_tiles(n, E, tile_m);
    if (n <= LM_PLAN_ONE) {
        hipLaunchKernelGGL(lm_plan_kernel, dim3(1), dim3(1024), 0, st, idx, n, E, tile_m, perm, tiles, n_tiles, most);
    } else {
        if (!hist) return cr_fail(CR_ERR_ARG, "routing: %d assignments without a place for their counts", n);
        hipLaunchKernelGGL(lm_plan_count_kernel, dim3(PLAN_PARTS), dim3(1024), 0, st, idx, n, E, hist);
        hipLaunchKernelGGL(lm_plan_place_kernel, dim3(PLAN_PARTS), dim3(1024), 0, st, idx, n, E, tile_m, hist, perm, tiles, n_tiles, most);
    }
    CR_HIP(hipGetLastError());
    return CR_OK;
}

size_t lm_plan_ints(int M, int top, int experts) { return M * top <= LM_PLAN_ONE ? 0 : (size_t)PLAN_PARTS * experts; }
