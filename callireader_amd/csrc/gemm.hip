// C = epi(A[M,K] . W[N,K]^T) in bf16 with fused epilogues: which kernel takes a product.
//
// Every dense contraction of the hot path is this shape (nn.Linear keeps W as [N,K], K contiguous):
//   * decode batches (M <= 64): the weight-streaming kernels (gemm_skinny.hip, gemm_stream.hip), their K-slices summed in an order of their own;
//   * everything else: the persistent 256x256 kernel (gemm256.hip) or the tile shapes of gemm_mid.hip, whichever its cost model says is faster.  Both run a row's sum over K in
//     ascending 32-steps of the same MFMA: a row's bits do not depend on the kernel, the tile, or how many rows it comes with.
#include <stdlib.h>

#include "common.hpp"

bool gemm256_supported(int epi, const GemmParams& p);
int launch_gemm_mid(int epi, const GemmParams& p, hipStream_t stream);
double gemm_mid_cost(int epi, const GemmParams& p, int* tile, int* row_tiles);
int launch_gemm256(int epi, const GemmParams& p, hipStream_t stream);
int launch_gemm256_f8(int epi, const GemmParams& p, hipStream_t stream);
bool gemm_skinny_supported(int epi, const GemmParams& p);
int launch_gemm_skinny(int epi, const GemmParams& p, hipStream_t stream);
double gemm256_cost(const GemmParams& p);
double gemm256_round_us(const GemmParams& p);

// Rows of a product that the 256x256 kernel takes, the others go to gemm_mid: all, none, or those up to a multiple of 256, as a few rows past it can cost the persistent kernel a round of tiles (32 ViT tiles are
// 128 x 256 + 32 rows: three rounds for two rounds' work at N = 1024).  Apart only where the laws see a fifth of a round in it: what is cut off leaves mostly rounds that fill the card, which the law prices too
// low.  541 sizes of 300 .. 99 000 rows, us whole | apart, by the saving that the laws see in rounds: 0.00 .. 0.18 800 x 16384 x 14336 315 | 361, 787 x 28672 x 4096 172 | 185, 3162 x 4096 x 4096 80.3 | 85.6, 4180 x
// 8192 x 1024 63.8 | 69.5; 0.20 .. 0.40 632 x 28672 x 4096 143 | 135, 12373 x 2048 x 4096 157 | 152, 41132 x 28672 x 4096 6539 | 6354, 1170 x 16384 x 4096 138 | 125; above 4100 x 4096 x 4096 126 | 99.7, 98400 x 4096 x
// 1024 640 | 627.  By this line the slower one is taken by more than 2 % at ten of the 423 sizes that gemm_mid does not take whole; by the sign of the saving, or by 3 % of the whole, at eighteen (profiles/tiled_products/last_rows.txt).
int gemm_tiled_rows(int epi, const GemmParams& p) {
    constexpr double APART = 0.19;
    int tile, rt;
    const int r = p.M % 256;
    const double whole = gemm256_cost(p), mid = gemm_mid_cost(epi, p, &tile, &rt);
    if (r > 0 && p.M > r && epi != EPI_PATCH && epi != EPI_ARGMAX) {
        GemmParams a = p, b = p;
        a.M = p.M - r;
        b.M = r;
        const double cut = gemm256_cost(a) + gemm_mid_cost(epi, b, &tile, &rt);
        if (whole - cut > APART * gemm256_round_us(p)) return mid < cut ? 0 : a.M;
    }
    return mid < whole ? 0 : p.M;
}

int launch_gemm(int epi, const GemmParams& p, hipStream_t stream) {
    if (p.M <= 0 || p.N <= 0 || p.K <= 0 || (p.K % 64) != 0) return CR_ERR_ARG;
    if ((p.lda & 7) || (p.ldw & 7)) return CR_ERR_ARG;
    if (p.wsw) {                                                 // decode-layout weights: the weight-streaming kernels only (M <= 64; bf16, or e4m3 in plain tile order)
        if ((p.w8 && p.wsw != 1) || p.a8 || p.wsw > 2 || (p.wsw == 2 && epi != EPI_PARTIAL) || ((uintptr_t)p.W & 15) || !gemm_skinny_supported(epi, p)) return CR_ERR_ARG;
        return launch_gemm_skinny(epi, p, stream);
    }
    if (p.a8) return launch_gemm256_f8(epi, p, stream);                                                  // e4m3 x e4m3 on the matrix cores
    if (p.w8) return gemm_skinny_supported(epi, p) ? launch_gemm_skinny(epi, p, stream) : CR_ERR_ARG;   // fp8 weights: decode kernel only
    if (((uintptr_t)p.A & 15) || ((uintptr_t)p.W & 15) || ((uintptr_t)p.C & 15)) return CR_ERR_ARG;
    static const int env_force = [] { const char* e = getenv("CR_GEMM_FORCE"); return e ? atoi(e) : 0; }();   // tuning aid: 128 | 256
    const int force = p.kernel ? p.kernel : env_force;
    if (force == 1) return gemm_skinny_supported(epi, p) ? launch_gemm_skinny(epi, p, stream) : CR_ERR_ARG;
    if (force == 256) return (p.K % 128) == 0 ? launch_gemm256(epi, p, stream) : CR_ERR_ARG;
    if (p.M <= 64 && !force && gemm_skinny_supported(epi, p)) return launch_gemm_skinny(epi, p, stream);   // decode: stream W once from HBM
    switch (epi) {
        case EPI_STORE: case EPI_GELU: case EPI_RELU2: case EPI_F32: case EPI_ARGMAX: break;
        case EPI_PARTIAL: if (p.bias || p.group <= 0 || p.K % (64 * p.group)) return CR_ERR_ARG; break;
        case EPI_LS_RES: if (!p.scale || !p.res) return CR_ERR_ARG; break;
        case EPI_RES: if (!p.res) return CR_ERR_ARG; break;
        case EPI_SWIGLU: if (p.N % 16) return CR_ERR_ARG; break;
        case EPI_PATCH: if (!p.res || p.group <= 0) return CR_ERR_ARG; break;
        default: return CR_ERR_ARG;
    }
    if (force == 128 || !gemm256_supported(epi, p)) return launch_gemm_mid(epi, p, stream);
    const int rows = gemm_tiled_rows(epi, p);
    if (rows == 0) return launch_gemm_mid(epi, p, stream);
    if (rows == p.M) return launch_gemm256(epi, p, stream);
    GemmParams a = p, b = p;
    a.M = rows;
    b.M = p.M - rows;
    b.A = p.A + (int64_t)rows * p.lda;
    b.C = (char*)p.C + (int64_t)rows * p.ldc * (epi == EPI_F32 ? 4 : 2);
    if (p.res) b.res = p.res + (int64_t)rows * p.ldr;
    const int rc = launch_gemm256(epi, a, stream);
    return rc != CR_OK ? rc : launch_gemm_mid(epi, b, stream);
}
