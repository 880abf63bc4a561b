// Few-row products of described decoders in true fp32: C = epi(A[M,K] . W[N,K]^T), M <= 64 (per expert where grouped), every weight read once.
//
// Bound by the weights' bytes.  A workgroup owns 16 rows of W (one v_mfma_f32_16x16x4_f32 operand tile) and the K range of its slice; its eight waves divide that range, so a product
// of 1024 rows keeps 64 x slices x 8 waves of loads in flight where 64 x 64 tiles give 16 workgroups that walk all of K alone (two rows, products of 1024 x 1536 .. 4096: 46 us there,
// 5.5 here; 3584 x 1024: 27 and 7.2; 4096 x 1024 with the squared relu: 27 and 7.1; token side's 64 x 1024: 28 and 4.6).
// W comes by LDS-DMA, a KiB of 16 rows x 16 k an instruction, four neighbouring lanes a row's 64 bytes; loaded straight as operands, four neighbouring lanes hold four rows and a KiB takes
// 64 clocks of the CU's load path instead of 16 (two rows: 1024 x 1536 .. 4096 6.9 us -> 5.5, 3584 x 1024 10.3 -> 7.2, 4096 x 1024 8.8 -> 7.1, 64 x 1024 6.0 -> 4.6).
// A lane multiplies with k = 4 (lane >> 4) .. + 3 of a 16-deep step of its weight row and of its activation row: the four multiplications of a step take one element
// of each, which permutes k inside the step for both operands alike.  Partial tiles of the waves meet in LDS and are added in wave order; slices go to the consumer, which adds them
// in slice order: the order of lm.hpp, a wave a chain.
#include "diag.hpp"
#include "lm.hpp"

namespace {

constexpr int NW = LM_CHAINS;                // waves of a workgroup, one chain of the sum each

template <int MT, int EPI>
__global__ __launch_bounds__(64 * NW) void lm_rows_kernel(const LmGemmParams p) {
    touch_args<(int)(sizeof(LmGemmParams))>();
    constexpr int U = MT == 4 ? 4 : 8;       // 16-deep steps whose loads are issued together
    constexpr int RED = NW * MT * 16 * 17 * 4, RING = NW * U * 1024;
    __shared__ __attribute__((aligned(16))) char sm[RED > RING ? RED : RING];      // the waves' U steps of W; after the products their partial tiles
    auto red = (float (*)[MT * 16][17])sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * 16;
    const float* A = (const float*)p.A + (int64_t)blockIdx.z * p.a_bs;
    const float* W = (const float*)p.W;
    int rows = p.M, pos0 = 0;
    if (p.tiles) {
        if ((int)blockIdx.y >= *p.n_tiles) return;            // (uniform: the grid is sized for the worst split)
        const int4 t = p.tiles[blockIdx.y];
        W += (int64_t)t.x * p.w_bs;
        pos0 = t.y; rows = min(t.z, MT * 16);
    } else W += (int64_t)blockIdx.z * p.w_bs;
    const int slice = p.tiles ? 0 : blockIdx.y, blocks = lm_part_blocks(p.K, p.slices), steps = 2 * blocks;      // 16-deep steps of this slice
    const int per = 2 * lm_chain_blocks(blocks), s0 = slice * steps + min(wave * per, steps), s1 = slice * steps + min(wave * per + per, steps);

    // a load instruction brings 16 rows x 16 k, four neighbouring lanes a row's 64 bytes, into the wave's own KiB of LDS; the 16-byte chunks of rows 8..15 are exchanged in pairs on both
    // sides (reads without bank conflicts)
    const float* w = W + (int64_t)min(n0 + (lane >> 2), p.N - 1) * p.ldw + 4 * ((lane & 3) ^ (((lane >> 2) >> 3) << 1));
    char* ring = sm + wave * U * 1024;
    const char* frag = ring + (lane & 15) * 64 + ((lane >> 4) ^ (((lane & 15) >> 3) << 1)) * 16;
    const float* a[MT];
#pragma unroll
    for (int j = 0; j < MT; j++) {
        const int m = pos0 + min(16 * j + (lane & 15), rows - 1);
        const int64_t ar = (p.perm && p.gather_div) ? p.perm[m] / p.gather_div : m;
        a[j] = A + ar * p.lda + 4 * (lane >> 4);
    }
    f32x4 acc[MT];
#pragma unroll
    for (int j = 0; j < MT; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += U) {
        f32x4 wf[U], af[U][MT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            // (uniform; K = 1024 in four slices are two steps a wave, and eight of its last one took 0.2 us of 5.3: requests of 2 rows 12.82 -> 12.70 ms, of few latent rows 7.87 -> 7.63)
            if (s + u >= s1) break;
            const int k = (s + u) * 16;
            CR_DIAG_POISON(ring + u * 1024)
            __builtin_amdgcn_global_load_lds(CR_GLB(w + k), CR_LDS(ring + u * 1024), 16, 0, 0);
#pragma unroll
            for (int j = 0; j < MT; j++) af[u][j] = *(const f32x4*)(a[j] + k);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++) wf[u] = *(const f32x4*)(frag + u * 1024);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (the next round's loads overwrite what was read here)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < s1) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int j = 0; j < MT; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][e], af[u][j][e], acc[j], 0, 0, 0);
            }
    }
    __syncthreads();                                          // every wave has read its last steps
    // lane: columns 4 (lane >> 4) + e of row lane & 15
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[wave][16 * j + (lane & 15)][4 * (lane >> 4) + e] = acc[j][e];
    __syncthreads();
    for (int i = tid; i < MT * 256; i += 64 * NW) {
        const int r = i >> 4, c = i & 15, n = n0 + c;
        if (r >= rows) continue;
        auto sum = [&](int col) {
            float v = red[0][r][col];
#pragma unroll
            for (int q = 1; q < NW; q++) v += red[q][r][col];
            return v;
        };
        const int m = pos0 + r;
        const int64_t cr = (p.perm && p.scatter) ? p.perm[m] : m;
        if (EPI == LM_GLU) {                                  // columns 0..7 of a tile are gates, 8..15 the matching ups
            if (c >= 8 || n >= p.N) continue;
            const float g = fminf(sum(c), p.limit), up = fminf(fmaxf(sum(c + 8), -p.limit), p.limit);
            ((float*)p.C)[cr * p.ldc + n0 / 2 + c] = g / (1.0f + expf(-1.702f * g)) * (up + 1.0f);
            continue;
        }
        if (n >= p.N) continue;
        const float v = sum(c);
        float* o = (float*)p.C + (int64_t)blockIdx.z * p.c_bs + ((int64_t)slice * p.M + cr) * p.ldc + n;
        if (EPI == LM_RAW32) *o = p.softcap > 0.f ? p.softcap * tanhf(v / p.softcap) : v;
        else if (EPI == LM_GATE) *o = v / (1.0f + expf(-((const float*)p.gate)[(int64_t)blockIdx.z * p.g_bs + cr * p.ldg + n]));
        else if (EPI == LM_SIDE) *o = gelu_tanh(v) * ((const float*)p.gate)[(int64_t)p.tok[cr] * p.ldg + n];
        else if (EPI == LM_RELU2) *o = relu2(v);
        else *o = v;
    }
}

template <int MT>
int launch_t(int epi, const LmGemmParams& p, hipStream_t st) {
    const dim3 grid((p.N + 15) / 16, p.tiles ? p.max_tiles : std::max(p.slices, 1), p.batch > 0 ? p.batch : 1), block(64 * NW);
    switch (epi) {
        case LM_STORE: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_STORE>), grid, block, 0, st, p); break;
        case LM_RAW32: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_RAW32>), grid, block, 0, st, p); break;
        case LM_GLU: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_GLU>), grid, block, 0, st, p); break;
        case LM_GATE: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_GATE>), grid, block, 0, st, p); break;
        case LM_RELU2: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_RELU2>), grid, block, 0, st, p); break;
        case LM_SIDE: hipLaunchKernelGGL((lm_rows_kernel<MT, LM_SIDE>), grid, block, 0, st, p); break;
        default: return cr_fail(CR_ERR_ARG, "lm_gemm_rows: epilogue %d", epi);
    }
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace

// Slices of a product whose consumer adds them: enough 16-row tiles for one workgroup per CU, at least 16 steps (two per wave) a slice, whole blocks of 32.
int lm_rows_slices(int N, int K) {
    int s = 1;
    while (s < LM_ROWS_MAX_SLICES && (N + 15) / 16 * s < 256 && K % (64 * s) == 0 && K / (2 * s) >= 256) s *= 2;
    return s;
}

int launch_lm_gemm_rows(int epi, const LmGemmParams& p, hipStream_t st) {      // (checked by launch_lm_gemm)
    const int most = p.tiles ? std::min(p.M, LM_TILE_M) : p.M;
    if (p.M <= 0 || most > LM_ROWS_MAX || (p.slices > 1 && (p.tiles || p.batch > 1 || epi != LM_RAW32 || p.softcap > 0.f)))
        return cr_fail(CR_ERR_ARG, "lm_gemm_rows(epi=%d M=%d N=%d K=%d slices=%d): bad argument", epi, p.M, p.N, p.K, p.slices);
    return most <= 16 ? launch_t<1>(epi, p, st) : most <= 32 ? launch_t<2>(epi, p, st) : launch_t<4>(epi, p, st);
}
