// Expert products of described decoders in bf16: the weights of an expert are kept in ONE layout, 1-KiB blocks of 16 output rows x 32 k in MFMA fragment order
// ([row / 16][k / 32][lane][8], lane = row % 16 + 16 * (k % 32 / 8)), which both forms below read a contiguous KiB at a time.
//
//   moe_tiled_kernel   prompts: 128 x 128 x 64 tiles over the assignments sorted by expert (moe.hip: lm_plan_kernel), operands by LDS-DMA; the activation rows are gathered by
//                      the DMA's per-lane source addresses straight into fragment order, so neither operand is swizzled and every ds_read_b128 is linear;
//   moe_stream_kernel  decode (<= 64 tokens): one workgroup per expert and 64 output rows; it finds its tokens in the routing table itself (no sort), streams the weights once
//                      from HBM straight to registers and splits K over its eight waves.
// Epilogues: GLU (rows of a 16-row block: 8 gates, 8 matching ups) and plain.  A row's sum does not depend on which other rows share its tile.
#include "lm.hpp"

int launch_gemm256_grouped(int epi, const GemmParams& p, hipStream_t stream);      // gemm256.hip

namespace {

// acc: four consecutive rows n .. n + 3 of the weight block at 4 (lane >> 4), for token column lane & 15
template <bool GLU>
__device__ __forceinline__ void store4(bf16* crow, int n16, int lane, f32x4 acc, float limit, bool live) {
    const int g = lane >> 4;
    if (GLU) {
        f32x4 u;
#pragma unroll
        for (int e = 0; e < 4; e++) u[e] = __shfl_xor(acc[e], 32, 64);
        if (!live || g >= 2) return;
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = f2bf(clamped_glu(acc[e], u[e], limit));
        *(bf16x4*)(crow + n16 / 2 + 4 * g) = o;
    } else {
        if (!live) return;
        *(bf16x4*)(crow + n16 + 4 * g) = bf16x4{f2bf(acc[0]), f2bf(acc[1]), f2bf(acc[2]), f2bf(acc[3])};
    }
}

constexpr int TM = MOE_TILE_M, TN = 128;

template <bool GLU>
__global__ __launch_bounds__(256, 2) void moe_tiled_kernel(const MoeGemmParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];       // 2 x (A 16 KiB | W 16 KiB)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntm = *p.n_tiles, ntn = (p.N + TN - 1) / TN;
    const int nwg = ntm * ntn, orig = blockIdx.x;
    if (orig >= nwg) return;                                          // the grid covers the worst split of the assignments
    // XCD-aware order, then groups of 8 row tiles (of one expert, mostly) x all column tiles: 64 neighbours share 8 row panels and 8 weight panels
    const int xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
    const int pid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
    const int per_group = 8 * ntn, first = pid / per_group * 8, gsz = min(ntm - first, 8), in_g = pid % per_group;
    const int4 t = p.tiles[first + in_g % gsz];
    const int n0 = in_g / gsz * TN, rows = t.z, pos0 = t.y;
    const bf16* W = p.W + (int64_t)t.x * p.w_es;
    const int wm = wave >> 1, wn = wave & 1;

    // this wave stages row blocks 2 wave, 2 wave + 1 of both operands (a block = 16 rows; per K-tile of 64 two 1-KiB fragments each)
    const bf16 *ga[2], *gw[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int rb = 2 * wave + i;
        const int pos = pos0 + min(rb * 16 + (lane & 15), rows - 1);
        const int64_t src = p.gather_div ? p.perm[pos] / p.gather_div : pos;
        ga[i] = p.A + src * p.lda + (lane >> 4) * 8;
        gw[i] = W + (int64_t)min(n0 / 16 + rb, p.N / 16 - 1) * (p.K / 32) * 512 + lane * 8;
    }
    auto stage = [&](int buf, int kt) {
        char* base = smem + buf * 32768 + wave * 4096;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                __builtin_amdgcn_global_load_lds(CR_GLB(ga[i] + kt * 64 + s * 32), CR_LDS(base + (i * 2 + s) * 1024), 16, 0, 0);
                __builtin_amdgcn_global_load_lds(CR_GLB(gw[i] + (int64_t)(kt * 2 + s) * 512), CR_LDS(base + 16384 + (i * 2 + s) * 1024), 16, 0, 0);
            }
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nk = p.K / 64;
    stage(0, 0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < nk) stage(cur ^ 1, kt + 1);
        const char* sb = smem + cur * 32768 + lane * 16;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            bf16x8 a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                a[i] = *(const bf16x8*)(sb + ((wm * 4 + i) * 2 + s) * 1024);
                w[i] = *(const bf16x8*)(sb + 16384 + ((wn * 4 + i) * 2 + s) * 1024);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], a[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int rr = wm * 64 + j * 16 + (lane & 15);
        const bool live = rr < rows;
        const int pos = pos0 + (live ? rr : rows - 1);
        bf16* crow = p.C + (int64_t)(p.scatter ? p.perm[pos] : pos) * p.ldc;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n16 = n0 + wn * 64 + i * 16;
            store4<GLU>(crow, n16, lane, acc[i][j], p.limit, live && n16 < p.N);
        }
    }
}

// SRC = true (gate | up): A rows are tokens; false (down): A rows are assignments.  C rows are assignments (token * top + slot) either way.
template <bool GLU, int RT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void moe_stream_kernel(const MoeGemmParams p) {
    touch_args<(int)(sizeof(MoeGemmParams))>();
    __shared__ float red[WAVES][RT][16][17];
    __shared__ int list[64];
    __shared__ int s_count;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = blockIdx.y;
    // the tokens of this expert, in token order: lane t looks through token t's `top` choices
    if (wave == 0) {
        int mine = -1;
        if (lane < p.M)
            for (int k = 0; k < p.top; k++)
                if (p.idx[lane * p.top + k] == e) mine = lane * p.top + k;
        const unsigned long long b = __ballot(mine >= 0);
        if (mine >= 0) list[__popcll(b & ((1ull << lane) - 1))] = mine;
        if (lane == 0) s_count = __popcll(b);
    }
    __syncthreads();
    const int count = s_count;
    if (count == 0) return;
    const int nt = p.N / 16, t0 = blockIdx.x * RT, ks_all = p.K / 32;
    const int per = (ks_all + WAVES - 1) / WAVES, k_lo = min(wave * per, ks_all), k_hi = min(k_lo + per, ks_all);
    const bf16* wp[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) wp[i] = p.W + (int64_t)e * p.w_es + (int64_t)min(t0 + i, nt - 1) * ks_all * 512 + lane * 8;
    constexpr int U = 4;
    for (int m0 = 0; m0 < count; m0 += 16) {
        const int a = list[min(m0 + (lane & 15), count - 1)];
        const bf16* xp = p.A + (int64_t)(p.gather_div ? a / p.gather_div : a) * p.lda + (lane >> 4) * 8;
        f32x4 acc[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        int ks = k_lo;
        for (; ks + U <= k_hi; ks += U) {
            bf16x8 w[RT][U], x[U];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int i = 0; i < RT; i++) w[i][u] = __builtin_nontemporal_load((const bf16x8*)(wp[i] + (int64_t)(ks + u) * 512));
#pragma unroll
            for (int u = 0; u < U; u++) x[u] = *(const bf16x8*)(xp + (ks + u) * 32);
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int i = 0; i < RT; i++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], x[u], acc[i], 0, 0, 0);
        }
        for (; ks < k_hi; ks++) {
            const bf16x8 x = *(const bf16x8*)(xp + ks * 32);
#pragma unroll
            for (int i = 0; i < RT; i++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_nontemporal_load((const bf16x8*)(wp[i] + (int64_t)ks * 512)), x, acc[i], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) red[wave][i][4 * (lane >> 4) + q][lane & 15] = acc[i][q];
        __syncthreads();
        // the waves' K-slices in wave order; wave w finishes block w, w + WAVES, ...
        for (int i = wave; i < RT; i += WAVES) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WAVES; w++)
#pragma unroll
                for (int q = 0; q < 4; q++) s[q] += red[w][i][4 * (lane >> 4) + q][lane & 15];
            const int m = m0 + (lane & 15);
            const bool live = m < count && t0 + i < nt;
            store4<GLU>(p.C + (int64_t)list[min(m, count - 1)] * p.ldc, (t0 + i) * 16, lane, s, p.limit, live);
        }
        __syncthreads();
    }
}

int check(const MoeGemmParams& p) {
    if (!p.A || !p.W || !p.C || p.N <= 0 || p.N % 16 || p.K <= 0 || p.K % 64 || (p.lda & 7) || (p.ldc & 3) || (p.w_es & 7) || (((uintptr_t)p.A | (uintptr_t)p.W) & 15) || ((uintptr_t)p.C & 7))
        return cr_fail(CR_ERR_ARG, "expert product: N = %d, K = %d", p.N, p.K);
    return CR_OK;
}

}  // namespace

bool moe_grouped256(int M, int top, int experts, int N, int K) {
    // the persistent 256 x 256 kernel (gemm256.hip) where the experts' rows fill its tiles and its 32-bit weight offsets reach every expert
    return K % 128 == 0 && N >= 256 && (int64_t)M * top >= (int64_t)experts * 192 && (double)experts * N * K * 2 < 4294967296.0;
}

int launch_moe_tiled(bool glu_epi, const MoeGemmParams& p, hipStream_t st) {
    CR_TRY(check(p));
    if (p.grouped256) {
        GemmParams g{};
        g.A = p.A; g.lda = p.lda; g.W = p.W; g.C = p.C; g.ldc = p.ldc; g.N = p.N; g.K = p.K; g.M = p.max_tiles * 256;
        g.tiles = p.tiles; g.n_tiles = p.n_tiles; g.max_tiles = p.max_tiles; g.perm = p.perm; g.gather_div = p.gather_div; g.scatter = p.scatter; g.expert_stride = p.w_es; g.limit = p.limit;
        const int r = launch_gemm256_grouped(glu_epi ? EPI_X_GLU : EPI_X_ROWS, g, st);
        return r == CR_OK ? CR_OK : cr_fail(r, "expert product (256 x 256): N = %d, K = %d", p.N, p.K);
    }
    if (!p.tiles || !p.n_tiles || p.max_tiles <= 0 || ((p.gather_div || p.scatter) && !p.perm)) return cr_fail(CR_ERR_ARG, "expert product: no plan");
    constexpr int LDS = 65536;
    static std::atomic<uint64_t> d0{0}, d1{0};
    const dim3 grid((unsigned)p.max_tiles * ((p.N + TN - 1) / TN));
    if (glu_epi) {
        if (!cr_dyn_lds_once(d0, (const void*)moe_tiled_kernel<true>, LDS)) return CR_ERR_HIP;
        hipLaunchKernelGGL(moe_tiled_kernel<true>, grid, dim3(256), LDS, st, p);
    } else {
        if (!cr_dyn_lds_once(d1, (const void*)moe_tiled_kernel<false>, LDS)) return CR_ERR_HIP;
        hipLaunchKernelGGL(moe_tiled_kernel<false>, grid, dim3(256), LDS, st, p);
    }
    CR_HIP(hipGetLastError());
    return CR_OK;
}

int launch_moe_stream(bool glu_epi, const MoeGemmParams& p, hipStream_t st) {
    CR_TRY(check(p));
    if (!p.idx || p.M <= 0 || p.M > 64 || p.top <= 0 || p.experts <= 0) return cr_fail(CR_ERR_ARG, "expert product: %d rows", p.M);
    constexpr int RT = 4, WAVES = 8;
    const dim3 grid((p.N / 16 + RT - 1) / RT, p.experts);
    if (glu_epi) hipLaunchKernelGGL((moe_stream_kernel<true, RT, WAVES>), grid, dim3(WAVES * 64), 0, st, p);
    else hipLaunchKernelGGL((moe_stream_kernel<false, RT, WAVES>), grid, dim3(WAVES * 64), 0, st, p);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
