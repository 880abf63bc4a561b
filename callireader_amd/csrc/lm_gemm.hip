// Matrix products of described decoders that the dense kernels do not take.  C = epi(A[M,K] . W[N,K]^T), K % 64 == 0.  Here: bf16, batched over heads (a query carried into the latent
// space, an attended latent carried back behind its gate).  Everything in fp32 comes through this entry too: decode batches by lm_gemm_rows.hip, the rest by lm_gemm_tiles.hip.
//
// 64 x 64 tile, 4 waves of 32 x 32 (2 x 2 accumulators of 16 x 16), K in steps of 32 through LDS.  The weights are the MFMA's A operand, so a lane's accumulator holds four
// consecutive output columns of one row (the same roles as gemm256 / gemm_skinny).  A row's sum runs over K in ascending steps whatever tile it sits in.
#include "lm.hpp"

namespace {

constexpr int BM = 64, BN = 64, BK = 32, LD = BK + 8;      // LD: elements per LDS row, 80 bytes, 16-byte aligned, rows spread over the banks

template <bool GATE>
__global__ __launch_bounds__(256) void lm_gemm_kernel(const LmGemmParams p) {
    __shared__ __attribute__((aligned(16))) bf16 sA[BM][LD];
    __shared__ __attribute__((aligned(16))) bf16 sW[BN][LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
    const int r = tid >> 2, c = (tid & 3) * 8;                // a vector of eight per thread and operand
    const bf16* ga = (const bf16*)p.A + (int64_t)blockIdx.z * p.a_bs + (int64_t)min(m0 + r, p.M - 1) * p.lda + c;
    const bf16* gw = (const bf16*)p.W + (int64_t)blockIdx.z * p.w_bs + (int64_t)min(n0 + r, p.N - 1) * p.ldw + c;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wn = (wave & 1) * 32, wm = (wave >> 1) * 32, k8 = 8 * (lane >> 4);
    bf16x8 ra = *(const bf16x8*)ga, rw = *(const bf16x8*)gw;
    for (int k0 = 0; k0 < p.K; k0 += BK) {
        __syncthreads();
        *(bf16x8*)&sA[r][c] = ra;
        *(bf16x8*)&sW[r][c] = rw;
        __syncthreads();
        if (k0 + BK < p.K) { ra = *(const bf16x8*)(ga + k0 + BK); rw = *(const bf16x8*)(gw + k0 + BK); }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&sW[wn + 16 * i + (lane & 15)][k8], *(const bf16x8*)&sA[wm + 16 * j + (lane & 15)][k8], acc[i][j], 0, 0, 0);
    }

    // lane: columns n0 + wn + 16 i + 4 (lane >> 4) + e of row wm + 16 j + (lane & 15)
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int m = m0 + wm + 16 * j + (lane & 15);
        if (m >= p.M) continue;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int n = n0 + wn + 16 * i + 4 * (lane >> 4);
            bf16* o = (bf16*)p.C + (int64_t)blockIdx.z * p.c_bs + (int64_t)m * p.ldc + n;
            const bf16* g = GATE ? (const bf16*)p.gate + (int64_t)blockIdx.z * p.g_bs + (int64_t)m * p.ldg + n : nullptr;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < p.N) o[e] = (bf16)(GATE ? acc[i][j][e] / (1.0f + expf(-(float)g[e])) : acc[i][j][e]);
        }
    }
}

}  // namespace

int launch_lm_gemm(bool f32, int epi, const LmGemmParams& p, hipStream_t st) {
    const int vec = f32 ? 4 : 8;
    if (p.N <= 0 || p.K <= 0 || p.K % 64 || p.lda % vec || p.ldw % vec || p.a_bs % vec || p.w_bs % vec || (p.tiles ? p.max_tiles <= 0 || p.batch > 1 || !p.n_tiles : p.M <= 0) ||
        (p.gather_div && !p.perm) || (epi == LM_GLU && (p.N % 16 || p.batch > 1)) || ((epi == LM_GATE || epi == LM_SIDE) && !p.gate) || (epi == LM_SIDE && !p.tok) ||
        (p.slices > 1 && p.K % (32 * p.slices)) || (!f32 && (p.tiles || p.perm || p.stream || p.slices > 1 || (epi != LM_STORE && epi != LM_GATE))) || (((uintptr_t)p.A | (uintptr_t)p.W) & 15))
        return cr_fail(CR_ERR_ARG, "lm_gemm(epi=%d M=%d N=%d K=%d): bad argument", epi, p.M, p.N, p.K);
    if (f32) return p.stream ? launch_lm_gemm_rows(epi, p, st) : launch_lm_gemm_tiles(epi, p, st);
    const dim3 grid((p.N + BN - 1) / BN, (p.M + BM - 1) / BM, p.batch > 0 ? p.batch : 1);
    if (epi == LM_GATE) hipLaunchKernelGGL(lm_gemm_kernel<true>, grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(lm_gemm_kernel<false>, grid, dim3(256), 0, st, p);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
