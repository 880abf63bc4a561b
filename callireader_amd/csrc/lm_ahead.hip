// Few-row products that form their own activations: the residual update and norm between two products (lm_post_kernel, lm_rows.hip) done by every workgroup of the second one, on rows it
// keeps in LDS, while its first weights travel.  One launch less and one round trip through memory less: with one or two rows a launch of that kernel is 2.2 us of a pass of 45, nearly all of
// it waiting, and a workgroup reads the few KiB of slices from L2 in about the time its weights take to arrive.  With many rows every workgroup would read megabytes: see lm_ahead_supported.
//
// Sums, norms and products have the order of the kernels they stand for (lm_post_kernel; gemm_skinny.hip; lm_gemm_rows.hip), so a row's bits do not depend on which of them ran.
#include "diag.hpp"
#include "lm_ahead.hpp"

bool gemm_stream_supported(int epi, const GemmParams& p, int splits);      // gemm_stream.hip

namespace {

// bf16: gemm_skinny_kernel's EPI_PARTIAL and EPI_RELU2 with one tile of rows, weights in the decode layout
template <int EPI, int RT>
__global__ __launch_bounds__(512) void ahead_skinny_kernel(const LmAhead a, const bf16* __restrict__ W, void* __restrict__ C, int N) {
    touch_args<(int)(sizeof(LmAhead) + 20)>();
    extern __shared__ __attribute__((aligned(16))) bf16 hs[];  // [M][K + 8]
    __shared__ float red[8][RT][16][17], sums[AHEAD_SEGS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.Wp, n0 = blockIdx.x * 16 * RT, ksteps = K / (256 * (int)gridDim.y), k0 = ((int)blockIdx.y * 8 + wave) * ksteps;
    constexpr int UR = 8 / RT;                                 // k-steps a batch; K = 2048 and one slice are eight
    const bf16* wp[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) wp[r] = W + ((int64_t)min(n0 / 16 + r, (N + 15) / 16 - 1) * (K / 32) + k0) * 512 + lane * 8;
    bf16x8 w[RT][UR];
    auto load = [&](int ks) {
#pragma unroll
        for (int u = 0; u < UR; u++) {
            if (ks + u >= ksteps) break;                      // (uniform)
#pragma unroll
            for (int r = 0; r < RT; r++) w[r][u] = __builtin_nontemporal_load((const bf16x8*)(wp[r] + (ks + u) * 512));
        }
    };
    load(0);
    __builtin_amdgcn_sched_barrier(0);
    update_rows<bf16>(a, 0, a.M, hs, K + 8, sums, blockIdx.x == 0 && blockIdx.y == 0);
    f32x4 acc[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16* xr = hs + min(lane & 15, a.M - 1) * (K + 8) + (lane >> 4) * 8 + k0 * 32;
    for (int ks = 0; ks < ksteps; ks += UR) {
        if (ks) load(ks);
#pragma unroll
        for (int u = 0; u < UR; u++) {
            if (ks + u >= ksteps) break;
            const bf16x8 x = *(const bf16x8*)(xr + (ks + u) * 32);
#pragma unroll
            for (int r = 0; r < RT; r++) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r][u], x, acc[r], 0, 0, 0);
        }
    }
    // C^T tile: row (n) = (lane >> 4) * 4 + e, column (m) = lane & 15; the waves' partials are added in wave order
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[wave][r][(lane >> 4) * 4 + e][lane & 15] = acc[r][e];
    __syncthreads();
    for (int i = tid; i < RT * a.M * 16; i += 512) {
        const int n = i & 15, r = (i >> 4) % RT, m = (i >> 4) / RT, gn = n0 + r * 16 + n;
        if (gn >= N) continue;
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < 8; q++) s += red[q][r][n][m];
        if (EPI == EPI_PARTIAL) ((float*)C)[((int64_t)blockIdx.y * a.M + m) * N + gn] = s;
        else ((bf16*)C)[(int64_t)m * N + gn] = f2bf(relu2(s));
    }
}

// fp32: lm_rows_kernel's LM_RAW32 (slices), LM_RELU2 and LM_SIDE with one tile of rows
template <int EPI>
__global__ __launch_bounds__(512) void ahead_rows_kernel(const LmAhead a, const float* __restrict__ W, float* __restrict__ C, int N, const float* __restrict__ gate, int64_t ldg,
                                                         const int32_t* __restrict__ tok) {
    touch_args<(int)(sizeof(LmAhead) + 48)>();
    constexpr int U = 8;
    extern __shared__ __attribute__((aligned(16))) float hf[];      // [M][K + 4]
    __shared__ __attribute__((aligned(16))) char sm[8 * U * 1024];
    __shared__ float sums[AHEAD_SEGS];
    auto red = (float (*)[16][17])sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.Wp, n0 = blockIdx.x * 16, slice = blockIdx.y, blocks = lm_part_blocks(K, gridDim.y), steps = 2 * blocks;
    const int per = 2 * lm_chain_blocks(blocks), s0 = slice * steps + min(wave * per, steps), s1 = slice * steps + min(wave * per + per, steps);
    const float* w = W + (int64_t)min(n0 + (lane >> 2), N - 1) * K + 4 * ((lane & 3) ^ (((lane >> 2) >> 3) << 1));
    char* ring = sm + wave * U * 1024;
    const char* frag = ring + (lane & 15) * 64 + ((lane >> 4) ^ (((lane & 15) >> 3) << 1)) * 16;
    auto load = [&](int s) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < s1) {
                CR_DIAG_POISON(ring + u * 1024)
                __builtin_amdgcn_global_load_lds(CR_GLB(w + (s + u) * 16), CR_LDS(ring + u * 1024), 16, 0, 0);
            }
    };
    if (s0 < s1) load(s0);
    update_rows<float>(a, 0, a.M, hf, K + 4, sums, blockIdx.x == 0 && blockIdx.y == 0);
    const float* xr = hf + min(lane & 15, a.M - 1) * (K + 4) + 4 * (lane >> 4);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += U) {
        if (s != s0) load(s);
        f32x4 wf[U], af[U];
#pragma unroll
        for (int u = 0; u < U; u++) af[u] = *(const f32x4*)(xr + min(s + u, s1 - 1) * 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++) wf[u] = *(const f32x4*)(frag + u * 1024);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (the next round's loads overwrite what was read here)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < s1)
#pragma unroll
                for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][e], af[u][e], acc, 0, 0, 0);
    }
    __syncthreads();                                          // every wave has read its last steps
#pragma unroll
    for (int e = 0; e < 4; e++) red[wave][lane & 15][4 * (lane >> 4) + e] = acc[e];
    __syncthreads();
    for (int i = tid; i < a.M * 16; i += 512) {
        const int r = i >> 4, c = i & 15, n = n0 + c;
        if (n >= N) continue;
        float v = red[0][r][c];
#pragma unroll
        for (int q = 1; q < 8; q++) v += red[q][r][c];
        float* o = C + ((int64_t)slice * a.M + r) * N + n;
        if (EPI == LM_SIDE) *o = gelu_tanh(v) * gate[(int64_t)tok[r] * ldg + n];
        else if (EPI == LM_RELU2) *o = relu2(v);
        else *o = v;
    }
}

template <int EPI, int RT>
int launch_skinny(const LmAhead& a, const void* W, void* C, int N, int splits, hipStream_t st) {
    hipLaunchKernelGGL((ahead_skinny_kernel<EPI, RT>), dim3((N + 16 * RT - 1) / (16 * RT), splits), dim3(512), a.M * (a.Wp + 8) * 2, st, a, (const bf16*)W, C, N);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
template <int EPI>
int launch_rows(const LmAhead& a, const void* W, void* C, int N, int slices, const void* gate, int64_t ldg, const int32_t* tok, hipStream_t st) {
    static std::atomic<uint64_t> attr_done{0};
    if (!cr_dyn_lds_once(attr_done, (const void*)ahead_rows_kernel<EPI>, 32 * 1024)) return cr_fail(CR_ERR_HIP, "product behind a residual update: LDS");
    hipLaunchKernelGGL((ahead_rows_kernel<EPI>), dim3((N + 15) / 16, slices), dim3(512), a.M * (a.Wp + 4) * 4, st, a, (const float*)W, (float*)C, N, (const float*)gate, ldg, tok);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace

bool lm_ahead_supported(bool f32, int M, int Wp, int N, int epi, bool decode_layout) {
    // Every workgroup reads all rows' slices, about 10 KiB a segment of 256 columns.  Eight segments travel beside the weights (one row of 2048: a step of 8 layers 0.463 -> 0.435 ms); with
    // sixteen (one row of 4096, 4 layers) it went from 0.658 to 0.677, and with 32 (four rows of 2048) the 8192-column product alone took 21.5 us for 8.3 + 3.
    if (M * ((Wp + 255) / 256) > AHEAD_SEGS) return false;
    if (f32) return epi == LM_RAW32 || epi == LM_RELU2 || epi == LM_SIDE;
    if (!decode_layout || Wp % 256) return false;
    GemmParams p{};
    p.M = M; p.N = N; p.K = p.lda = p.ldw = Wp; p.ldc = N; p.wsw = 1; p.raw32 = epi == LM_RAW32;
    // the products that gemm_skinny.hip would take with eight waves
    if (epi == LM_RAW32) return !gemm_stream_supported(EPI_F32, p, 1) && gemm_partial_splits(N, Wp) > 0;
    return epi == LM_RELU2 && N <= 8192 && !gemm_stream_supported(EPI_RELU2, p, 1);
}

int launch_lm_ahead(bool f32, const LmAhead& a, int epi, const void* W, void* C, int N, const void* gate, int64_t ldg, const int32_t* tok, hipStream_t st) {
    if (a.M <= 0 || N <= 0 || !a.Y || !a.x || !a.x_out || a.x == a.x_out || !W || !C || !lm_ahead_supported(f32, a.M, a.Wp, N, epi, true) || (epi == LM_SIDE && (!gate || !tok)))
        return cr_fail(CR_ERR_ARG, "product behind a residual update: %d rows, %d x %d, epilogue %d", a.M, N, a.Wp, epi);
    if (f32) {
        if (epi == LM_RAW32) return launch_rows<LM_RAW32>(a, W, C, N, lm_rows_slices(N, a.Wp), nullptr, 0, nullptr, st);
        if (epi == LM_RELU2) return launch_rows<LM_RELU2>(a, W, C, N, 1, nullptr, 0, nullptr, st);
        return launch_rows<LM_SIDE>(a, W, C, N, 1, gate, ldg, tok, st);
    }
    if (epi == LM_RELU2) return launch_skinny<EPI_RELU2, 1>(a, W, C, N, 1, st);
    const int splits = gemm_partial_splits(N, a.Wp);
    switch (gemm_partial_tiles(N, a.Wp)) {
        case 1: return launch_skinny<EPI_PARTIAL, 1>(a, W, C, N, splits, st);
        case 2: return launch_skinny<EPI_PARTIAL, 2>(a, W, C, N, splits, st);
        case 3: return launch_skinny<EPI_PARTIAL, 3>(a, W, C, N, splits, st);
    }
    return launch_skinny<EPI_PARTIAL, 4>(a, W, C, N, splits, st);
}
