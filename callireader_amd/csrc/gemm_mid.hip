// bf16 MFMA GEMM for the row counts between decode (gemm_skinny.hip) and the persistent 256x256 kernel (gemm256.hip):  C = epi(A[M,K] . W[N,K]^T),  K % 64 == 0.
//
// What bounds these shapes is neither arithmetic nor bytes but the chain of a K-tile's step: a 128x128 grid over M = 1025, N = 1024 is 72 workgroups, and a K loop that waits for each K-tile's
// loads before it asks for the next-but-one pays a memory round trip per 64 of K.  So (a) the tile shape is a template and picked by the grid it gives (gemm_mid_cost below), down to
// 16 x 32 for two waves, (b) NBUF K-tiles live in LDS and up to NBUF - 1 of them are in flight: one barrier per K-tile, counted vmcnt, never a drain before the last tiles, and (c) with four
// buffers and more a step has no branches and no address arithmetic.
//   * one global_load_lds_dwordx4 brings eight rows x 64 k, whole 128-byte lines (pieces of 16 rows x 32 k reach 56 of the 69 GB/s per CU that these do on cold weights);
//     LDS rows of 128 bytes, the 16-byte chunk XORed with (row >> 1) & 7 on both sides: a fragment's ds_read_b128 is free of bank conflicts;
//   * the weights are the MFMA's A operand: a lane's accumulator holds four consecutive columns of one row; what a column can do by itself happens there, and bf16 rows leave in whole
//     16-byte chunks through a stage in the K-tile buffers (epilogue_staged; ragged edges and fp32 straight from the accumulators);
//   * a row tile's fragments past M are neither read nor multiplied (M = 1025: the last row costs a sixteenth of a tile, not a tile);
//   * a row's sum runs over K in ascending 32-steps of the same MFMA as in gemm256, whatever the tile: the same bits from every kernel and every shape here.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "diag.hpp"
#include "k_ring.hpp"

namespace {

// ---- epilogue of four consecutive columns gn .. gn + 3 (gn % 4 == 0) of row gm: the reference's bf16 rounding sequence ----
template <int EPI>
__device__ __forceinline__ void put1(const GemmParams& p, int gm, int gn, float v) {
    const float sum = v + (p.bias ? bf2f(p.bias[gn]) : 0.0f);
    if (EPI == EPI_F32) { ((float*)p.C)[(int64_t)gm * p.ldc + gn] = f32_out(p, sum); return; }
    float x = EPI == EPI_RELU2 ? relu2(sum) : EPI == EPI_STORE ? sum : rbf(sum);
    int64_t orow = gm;
    if (EPI == EPI_GELU) x = gelu_erf(x);
    else if (EPI == EPI_LS_RES) x = bf2f(p.res[(int64_t)gm * p.ldr + gn]) + rbf(x * bf2f(p.scale[gn]));
    else if (EPI == EPI_RES) x = bf2f(p.res[(int64_t)gm * p.ldr + gn]) + x;
    else if (EPI == EPI_PATCH) {
        const int t = gm / p.group, pi = gm - t * p.group;
        orow = (int64_t)t * (p.group + 1) + 1 + pi;
        x = x + bf2f(p.res[(int64_t)(1 + pi) * p.ldr + gn]);
    }
    ((bf16*)p.C)[orow * p.ldc + gn] = f2bf(x);
}
template <int EPI>
__device__ __forceinline__ void put4(const GemmParams& p, int gm, int gn, f32x4 v) {
    constexpr bool ROUND = EPI != EPI_STORE && EPI != EPI_F32 && EPI != EPI_RELU2;
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = v[e];
    if (p.bias) {
        const bf16x4 b = *(const bf16x4*)(p.bias + gn);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] += bf2f(b[e]);
    }
    if (EPI == EPI_F32) {
        *(f32x4*)((float*)p.C + (int64_t)gm * p.ldc + gn) = f32x4{f32_out(p, x[0]), f32_out(p, x[1]), f32_out(p, x[2]), f32_out(p, x[3])};
        return;
    }
    if (ROUND) {
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = rbf(x[e]);
    }
    int64_t orow = gm;
    if (EPI == EPI_RELU2) {
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = relu2(x[e]);
    } else if (EPI == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = gelu_erf(x[e]);
    } else if (EPI == EPI_LS_RES) {
        const bf16x4 s = *(const bf16x4*)(p.scale + gn), r = *(const bf16x4*)(p.res + (int64_t)gm * p.ldr + gn);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = bf2f(r[e]) + rbf(x[e] * bf2f(s[e]));
    } else if (EPI == EPI_RES) {
        const bf16x4 r = *(const bf16x4*)(p.res + (int64_t)gm * p.ldr + gn);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = bf2f(r[e]) + x[e];
    } else if (EPI == EPI_PATCH) {
        const int t = gm / p.group, pi = gm - t * p.group;
        orow = (int64_t)t * (p.group + 1) + 1 + pi;
        const bf16x4 r = *(const bf16x4*)(p.res + (int64_t)(1 + pi) * p.ldr + gn);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = x[e] + bf2f(r[e]);
    }
    *(bf16x4*)((bf16*)p.C + orow * p.ldc + gn) = bf16x4{f2bf(x[0]), f2bf(x[1]), f2bf(x[2]), f2bf(x[3])};
}

// what a column can do by itself, in the accumulator layout: the linear output with its bias, then GELU / LayerScale / squared relu, each on its rounded input
template <int EPI>
__device__ __forceinline__ bf16x4 by_column(f32x4 v, const float (&bias)[4], const float (&scale)[4]) {
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float x = v[e] + bias[e];                             // -0.0f where there is no bias: x + -0 = x, bit for bit
        if (EPI == EPI_RELU2) x = relu2(x);
        if (EPI == EPI_GELU) x = gelu_erf(rbf(x));
        if (EPI == EPI_LS_RES) x = rbf(x) * scale[e];
        o[e] = f2bf(x);
    }
    return o;
}

// bf16 results of a wave's columns, all inside the matrix: 16 rows at a time through 16 x (FN * 16) of the wave's own LDS, so that memory is read and written in whole 16-byte chunks of
// a row by neighbouring lanes (straight from the accumulators every lane writes eight bytes of a row of its own: 5 us a launch more on 128 x 256 tiles).  Rows of FN * 32 + 16 bytes:
// sixteen rows start at sixteen different bank groups.
template <int EPI, int FM, int FN>
__device__ __forceinline__ void epilogue_staged(const GemmParams& p, const f32x4 (&acc)[FM][FN], char* stg, int row0, int live, int col0, int lane) {
    constexpr int LD = FN * 32 + 16, CPR = EPI == EPI_SWIGLU ? FN : 2 * FN, RPP = 64 / CPR < 16 ? 64 / CPR : 16;      // bytes a row, chunks of a row that leave, rows a pass
    float bias[FN][4], scale[FN][4];
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int gn = col0 + j * 16 + 4 * (lane >> 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            bias[j][e] = p.bias ? bf2f(p.bias[gn + e]) : -0.0f;
            scale[j][e] = EPI == EPI_LS_RES ? bf2f(p.scale[gn + e]) : 1.f;
        }
    }
    const int rin = lane / CPR, c = lane % CPR;
#pragma unroll
    for (int i = 0; i < FM; i++) {
        if (i >= live) break;
        char* buf = stg + (i & 1) * 16 * LD;
#pragma unroll
        for (int j = 0; j < FN; j++) *(bf16x4*)(buf + (lane & 15) * LD + j * 32 + (lane >> 4) * 8) = by_column<EPI>(acc[i][j], bias[j], scale[j]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += RPP) {
            const int row = r0 + rin, gm = row0 + i * 16 + row;
            if (rin >= RPP || gm >= p.M) continue;
            if (EPI == EPI_SWIGLU) {                          // [8 gate | 8 up]
                const bf16x8 g = *(const bf16x8*)(buf + row * LD + c * 32), u = *(const bf16x8*)(buf + row * LD + c * 32 + 16);
                bf16x8 o;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = f2bf(rbf(silu(bf2f(g[e]))) * bf2f(u[e]));
                *(bf16x8*)((bf16*)p.C + (int64_t)gm * p.ldc + col0 / 2 + c * 8) = o;
                continue;
            }
            bf16x8 v = *(const bf16x8*)(buf + row * LD + c * 16);
            int64_t orow = gm, rrow = gm;
            if (EPI == EPI_PATCH) {
                const int t = gm / p.group, pi = gm - t * p.group;
                orow = (int64_t)t * (p.group + 1) + 1 + pi;
                rrow = 1 + pi;
            }
            if (EPI == EPI_LS_RES || EPI == EPI_RES || EPI == EPI_PATCH) {
                const bf16x8 r = *(const bf16x8*)(p.res + rrow * p.ldr + col0 + c * 8);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = f2bf(bf2f(r[e]) + bf2f(v[e]));
            }
            *(bf16x8*)((bf16*)p.C + orow * p.ldc + col0 + c * 8) = v;
        }
    }
}

template <int EPI, int FM, int FN>
__device__ __forceinline__ void epilogue(const GemmParams& p, const f32x4 (&acc)[FM][FN], char* stg, int row0, int live, int col0, int lane) {
    if constexpr (EPI != EPI_F32 && EPI != EPI_ARGMAX) {
        constexpr bool ROWS = EPI == EPI_LS_RES || EPI == EPI_RES || EPI == EPI_PATCH;
        if (col0 + FN * 16 <= p.N && (p.ldc & 7) == 0 && (!ROWS || ((p.ldr & 7) == 0 && ((uintptr_t)p.res & 15) == 0))) {      // (wave-uniform; C is 16-byte aligned)
            epilogue_staged<EPI, FM, FN>(p, acc, stg, row0, live, col0, lane);
            return;
        }
    }
    const bool vec = (p.ldc & 3) == 0;
#pragma unroll
    for (int i = 0; i < FM; i++) {
        if (i >= live) break;
        const int gm = row0 + i * 16 + (lane & 15);
        if (EPI == EPI_ARGMAX) {                              // the wave's 64 columns: one partial per row
            float bv = -INFINITY; int bc = 0x7fffffff;
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int n = col0 + j * 16 + 4 * (lane >> 4) + e;
                    float v = rbf(acc[i][j][e] + (p.bias && n < p.N ? bf2f(p.bias[n]) : 0.f));
                    v = n < p.N ? v : -INFINITY;
                    if (v > bv) { bv = v; bc = n; }              // ascending columns inside a lane: strict > keeps the first
                }
#pragma unroll
            for (int o = 16; o <= 32; o <<= 1) argmax_merge(bv, bc, __shfl_xor(bv, o, 64), __shfl_xor(bc, o, 64));
            if (lane < 16 && gm < p.M && col0 < p.N) ((unsigned long long*)p.C)[(int64_t)gm * p.ldc + (col0 >> 6)] = argmax_pack(bv, bc);
            continue;
        }
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int gn = col0 + j * 16 + 4 * (lane >> 4);
            if (EPI == EPI_SWIGLU) {                          // a fragment's columns are [8 gate | 8 up]: the partner sits 32 lanes away
                f32x4 u;
#pragma unroll
                for (int e = 0; e < 4; e++) u[e] = __shfl_xor(acc[i][j][e], 32, 64);
                if (lane >= 32 || gm >= p.M || gn >= p.N) continue;
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = f2bf(rbf(silu(rbf(acc[i][j][e]))) * rbf(u[e]));
                bf16* c = (bf16*)p.C + (int64_t)gm * p.ldc + (col0 + j * 16) / 2 + 4 * (lane >> 4);
                if (vec) *(bf16x4*)c = o;
                else {
#pragma unroll
                    for (int e = 0; e < 4; e++) c[e] = o[e];
                }
                continue;
            }
            if (gm >= p.M || gn >= p.N) continue;
            if (vec && gn + 4 <= p.N) put4<EPI>(p, gm, gn, acc[i][j]);
            else
                for (int e = 0; e < 4 && gn + e < p.N; e++) put1<EPI>(p, gm, gn + e, acc[i][j][e]);
        }
    }
}

template <int N, int I = 0, typename F>
__device__ __forceinline__ void constexpr_for(F f) {
    if constexpr (I < N) { f(std::integral_constant<int, I>{}); constexpr_for<N, I + 1>(f); }
}
// the last J K-tiles after the one being multiplied: each has landed, for every wave, when f(even) reads it
template <int J, int PER, bool EVEN = true, typename F>
__device__ __forceinline__ void ring_tail(F f) {
    if constexpr (J > 0) {
        wait_vm<(J - 1) * PER>();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        f(std::integral_constant<bool, EVEN>{});
        ring_tail<J - 1, PER, !EVEN>(f);
    }
}

// K-tile u of an unrolled round goes to buffer u (of four) or to the one before it (of more: the kernel's loop), by an instruction offset of 128 u that is taken off the LDS address again: bytes ahead of the
// first buffer that keep that address from being negative (none with four buffers: two workgroups of 96 x 64 fill a CU's LDS to the byte)
constexpr int mid_pad(int nbuf, int round, int stage) {
    int pad = 0;
    for (int u = 0; nbuf > 3 && u < round; u++) pad = std::max(pad, u * 128 - (nbuf > 4 ? (u + nbuf - 1) % nbuf : u % nbuf) * stage);
    return (pad + 511) / 512 * 512;
}
// WM x WN waves of FM x FN fragments of 16 x 16
template <int WM, int WN, int FM, int FN, int NBUF>
struct MidGeom {
    static constexpr int BM = WM * FM * 16, BN = WN * FN * 16, WAVES = WM * WN, PIECES = (BM + BN) / 8, PER = (PIECES + WAVES - 1) / WAVES, STAGE = PIECES * 1024, ROUND = NBUF % 2 ? 2 * NBUF : NBUF, PAD = mid_pad(NBUF, ROUND, STAGE), LDS = PAD + NBUF * STAGE;
    static constexpr bool TWO_A_CU = 2 * LDS <= 160 * 1024;
    static_assert(WAVES * 32 * (FN * 32 + 16) <= LDS, "the epilogue's stage lies in the buffers");
    static_assert((NBUF - 1) * PER <= 63 && NBUF >= 3 && LDS <= 160 * 1024, "vmcnt is six bits wide; a CU has 160 KiB");
};

// What a launch's workgroups would divide for: the tiles' order, the fragments of a row tile, a slice's K-tiles
struct MidGrid {
    int epi, ntm, nk;                                         // epilogue; row tiles; K-tiles of a slice
    int xq, xr;                                               // workgroups / 8 and % 8
    int per_group, last;                                      // workgroups of a super-group of eight row tiles; row tiles of the last one
    unsigned group_mul, last_mul;                             // ceil(2^32 / per_group), ceil(2^32 / last): exact where a workgroup's number times the divisor stays below 2^32 (group_mul 0: it does not)
    int fq, fr;                                               // fragments / row tiles and % row tiles
    unsigned rows_mul;                                        // ceil(2^32 / row tiles): exact for ntm^3 < 2^32 (0: it is not, or one row tile)
};

template <int WM, int WN, int FM, int FN, int NBUF, bool FAR>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mid_kernel(const MidGrid g, const GemmParams p) {
    typedef MidGeom<WM, WN, FM, FN, NBUF> G;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    touch_args<(int)(sizeof(MidGrid) + sizeof(GemmParams))>();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, epi = g.epi;

    // ---- workgroup -> tile: bijective XCD remap (an XCD's L2 gets a contiguous run of tiles), then super-groups of 8 row tiles ----
    // (no division: five of them, one in 64 bits, and the arguments' lines one after the other as they were come upon kept a workgroup from its first load for 2 us)
    const int orig = blockIdx.x, nk = g.nk, xcd = orig & 7;
    const int pid = (xcd < g.xr ? xcd * (g.xq + 1) : g.xr * (g.xq + 1) + (xcd - g.xr) * g.xq) + (orig >> 3);
    constexpr int GM = 8;
    const int grp = g.group_mul ? (int)__umulhi((unsigned)pid, g.group_mul) : pid / g.per_group, first_m = grp * GM, in_g = pid - grp * g.per_group;
    int col, in_col;
    if (g.ntm - first_m >= GM) { col = in_g >> 3; in_col = in_g & 7; }
    else {
        col = g.last_mul ? (int)__umulhi((unsigned)in_g, g.last_mul) : in_g / g.last;
        in_col = in_g - col * g.last;
    }
    const int tile_m = first_m + in_col, n0 = col * G::BN;
    // ---- the matrix's fragments of 16 rows dealt evenly over the row tiles (at most WM * FM each), a tile's over its wave rows ----
    auto dealt = [&](int t) { return t * g.fq + (g.rows_mul ? (int)__umulhi((unsigned)(t * g.fr), g.rows_mul) : (int)((int64_t)t * g.fr / g.ntm)); };
    const int f0 = dealt(tile_m), fn = dealt(tile_m + 1) - f0;
    const int m0 = f0 * 16, wf0 = fn * wm / WM, live = fn * (wm + 1) / WM - wf0;

    // ---- this wave's pieces of a K-tile: eight rows of A or W, all 64 k (128 bytes a row); numbers past the last repeat it ----
    // (pieces of rows past the tile's move one lane's 16 bytes: the count of instructions under way stays a constant)
    // A piece's first row is the same for all lanes, so its address is a scalar one; a lane's own row and chunk are 32 bits beyond it.
    // (FAR: rows so far apart that eight of them span 4 GiB; a lane's address is 64 bits then.)
    const char *src[G::PER], *lane_src[FAR ? G::PER : 1];
    unsigned off[G::PER], dst[G::PER];
    uint64_t lanes[G::PER];
    const unsigned smem_base = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
#pragma unroll
    for (int i = 0; i < G::PER; i++) {
        const int piece = min(wave + i * G::WAVES, G::PIECES - 1), row = piece * 8 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
        const bool a = piece * 8 < G::BM;
        const int first = a ? min(m0 + piece * 8, p.M - 1) : min(n0 + piece * 8 - G::BM, p.N - 1), own = a ? min(m0 + row, p.M - 1) : min(n0 + row - G::BM, p.N - 1);
        if (FAR) {
            src[i] = (const char*)((a ? p.A + (int64_t)first * p.lda : p.W + (int64_t)first * p.ldw) + (int64_t)blockIdx.y * nk * 64);
            lane_src[FAR ? i : 0] = src[i] + (int64_t)(own - first) * (a ? p.lda : p.ldw) * 2 + chunk * 16;
        } else {                                              // (eight rows lie within 4 GiB: less than 306 783 370 elements apart, launch_gemm_mid)
            const unsigned ld = (unsigned)(a ? p.lda : p.ldw);
            src[i] = (const char*)((a ? p.A : p.W) + (uint64_t)(unsigned)first * ld + blockIdx.y * nk * 64);
            off[i] = (unsigned)(own - first) * ld * 2 + chunk * 16;
        }
        dst[i] = smem_base + G::PAD + piece * 1024;
        lanes[i] = a && piece >= 2 * fn ? 1 : ~0ull;
    }
    // (u is a K-tile of an unrolled run: G::PAD keeps the LDS address positive)
    auto ask1 = [&](auto i, auto u, unsigned to) __attribute__((always_inline)) {
        constexpr int I = decltype(i)::value, O = decltype(u)::value * 128;
        if constexpr (FAR) ring_ask_far<O>(lane_src[I], dst[I], to, lanes[I]);
        else if constexpr (I * G::WAVES * 8 < G::BM) ring_ask<O>(src[I], off[I], dst[I], to, lanes[I]);
        else ring_ask<O>(src[I], off[I], dst[I], to);
    };
    // K-tile u of the run that `src` stands at, into buffer buf
    auto ask = [&](auto u, int buf) __attribute__((always_inline)) {
        constexpr_for<G::PER>([&](auto i) {
            CR_DIAG_POISON(smem + G::PAD + buf * G::STAGE + (dst[decltype(i)::value] - smem_base - G::PAD))
            ask1(i, u, buf * G::STAGE);
        });
    };
    auto advance = [&](int tiles) {
#pragma unroll
        for (int i = 0; i < G::PER; i++) {
            if (FAR) lane_src[FAR ? i : 0] += tiles * 128;
            else src[i] += tiles * 128;
        }
    };
    constexpr std::integral_constant<int, 0> here{};

    auto arrive = [&](int t) { ring_arrive<NBUF, G::PER>(nk, t); };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int swz = (lane >> 1) & 7;
    const int c_off[2] = {((lane >> 4) ^ swz) * 16, ((4 + (lane >> 4)) ^ swz) * 16};
    const int a_off = (wf0 * 16 + (lane & 15)) * 128, w_off = (G::BM + wn * FN * 16 + (lane & 15)) * 128;

    struct Frags { bf16x8 a[2][FM], w[2][FN]; };
    auto read = [&](Frags& f, int buf, auto count) {
        const char* s = smem + G::PAD + buf * G::STAGE;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int j = 0; j < FN; j++) f.w[h][j] = *(const bf16x8*)(s + w_off + j * 2048 + c_off[h]);
#pragma unroll
            for (int i = 0; i < FM; i++)
                if (i < decltype(count)::value) f.a[h][i] = *(const bf16x8*)(s + a_off + i * 2048 + c_off[h]);
        }
    };
    auto multiply = [&](const Frags& f, auto count) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < FM; i++)
                if (i < decltype(count)::value) {
#pragma unroll
                    for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[h][j], f.a[h][i], acc[i][j], 0, 0, 0);
                }
    };
    // Tile kt's fragments are read a step ahead.  With four buffers the tile asked for in step kt goes where tile kt lay, whose reads the step's barrier waits for; with more (LATE) where tile kt - 1 lay,
    // which was multiplied before the barrier, so that no LDS read has to have come back by then.  These loops are not bound by bytes (64 x 64 tiles, K = 4096: 256 workgroups take little longer than one;
    // a CU brings in 130 GB/s from its L2 and 480 from LDS) but by a step's chain -- branches, addresses, barrier, LDS reads -- and by how far ahead a K-tile is asked for.  So nothing in a step is
    // conditional or computes an address (LEAN; three buffers keep the loop with its conditions), and one workgroup a CU takes all the buffers there are.  1025 x 1024 x 4096 23.5 -> 18.7 us, 1025 x 1024 x
    // 1024 9.0 -> 7.9, 1025 x 3072 x 1024 12.6 -> 11.5, 1531 x 2048 x 2048 20.5 -> 18.0; tiles of 16 x 32 and 32 x 64 on every CU 62 -> 42, 32.8 -> 27.8.
    constexpr bool LATE = NBUF > 4, LEAN = NBUF > 3;
    constexpr int AHEAD = LATE ? NBUF - 1 : NBUF;             // K-tiles asked for beyond the one being multiplied
    auto loop = [&](auto count) {
        Frags f0, f1;
        int kt = 0, buf = 0;                                  // buffer of tile kt
        auto more = [&](int buf) { ask(here, buf); advance(1); };
        if constexpr (!LEAN) {
            for (int t = 0; t < min(NBUF - 1, nk); t++) more(t);
            arrive(0);
            if (NBUF - 1 < nk) more(NBUF - 1);
            read(f0, 0, count);
            auto step = [&](int kt, Frags& now, Frags& next) {
                arrive(kt + 1);
                if (kt + NBUF < nk) more(buf);                // the buffer that tile kt was read from
                buf = buf + 1 == NBUF ? 0 : buf + 1;
                read(next, buf, count);
                __builtin_amdgcn_sched_barrier(0);
                multiply(now, count);
            };
            for (; kt + 2 < nk; kt += 2) {                    // (no read of the loop is conditional: the compiler waited for it ahead of the multiplications then)
                step(kt, f0, f1);
                step(kt + 1, f1, f0);
            }
            if (kt + 1 < nk) {
                step(kt, f0, f1);
                multiply(f1, count);
            } else multiply(f0, count);
            return;
        }
        for (int t = 0; t < min(AHEAD, nk); t++) more(t);
        if (nk < AHEAD) {                                     // all of K is under way at once
            for (; kt < nk; kt++) {
                wait_tail<AHEAD - 2, G::PER>(nk - 1 - kt);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                read(f0, kt, count);
                multiply(f0, count);
            }
            return;
        }
        wait_vm<(AHEAD - 1) * G::PER>();
        __builtin_amdgcn_s_waitcnt(0xC07F);                   // lgkmcnt(0): with a scalar load under way the loop's LDS reads could not be counted
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read(f0, 0, count);
        // now in buffer b, next in the one behind; u: K-tiles since `src` was moved
        auto step = [&](auto u, int b, Frags& now, Frags& next) __attribute__((always_inline)) {
            wait_vm<(AHEAD - 2) * G::PER>();
            if (!LATE) __builtin_amdgcn_s_waitcnt(0xC07F);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            ask(u, !LATE ? b : b == 0 ? NBUF - 1 : b - 1);
            read(next, b + 1 == NBUF ? 0 : b + 1, count);
            __builtin_amdgcn_sched_barrier(0);
            if (LATE) {                                       // `now` has come, `next` is under way
                __builtin_amdgcn_s_waitcnt(0xC07F | std::min(2 * (FN + decltype(count)::value), 15) << 8);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(now, count);
        };
        // a round of the buffers at a time, so that every address is a constant beside its base
        constexpr int ROUND = G::ROUND;
        for (; kt + ROUND + AHEAD <= nk; kt += ROUND) {
            constexpr_for<ROUND / 2>([&](auto h) {
                constexpr int U = 2 * decltype(h)::value;
                step(std::integral_constant<int, U>{}, U % NBUF, f0, f1);
                step(std::integral_constant<int, U + 1>{}, (U + 1) % NBUF, f1, f0);
            });
            advance(ROUND);
        }
        auto one = [&](Frags& now, Frags& next) {
            step(here, buf, now, next);
            advance(1);
            buf = buf + 1 == NBUF ? 0 : buf + 1;
            kt++;
        };
        while (kt + 1 < nk - AHEAD) {
            one(f0, f1);
            one(f1, f0);
        }
        auto tail = [&](Frags& now, Frags& next) {
            ring_tail<AHEAD - 1, G::PER>([&](auto even) {
                constexpr bool E = decltype(even)::value;
                buf = buf + 1 == NBUF ? 0 : buf + 1;
                read(E ? next : now, buf, count);
                __builtin_amdgcn_sched_barrier(0);
                multiply(E ? now : next, count);
            });
            multiply((AHEAD - 1) & 1 ? next : now, count);
        };
        // (an odd K-tile is copied: with a tail for either order of the two sets the compiler joined the tails and held a third set for it, 256 registers and a spill in 160 x 128 where there are 176 now.  us,
        // two tails / one: 160 x 128 1025 x 4096 x 1024 15.8 / 14.7, 2050 x 2048 x 2048 24.7 / 23.5, 4100 x 2048 x 2240 47.7 / 48.0; 128 x 128 1025 x 3072 x 1024 13.0 / 12.9, of 1088 13.9 / 13.9)
        if (kt < nk - AHEAD) {
            one(f0, f1);
            f0 = f1;
        }
        tail(f0, f1);
    };
    if (live == FM) loop(std::integral_constant<int, FM>{});
    else if (FM > 1 && live == FM - 1) loop(std::integral_constant<int, FM - 1>{});
    else if (FM > 2 && live == FM - 2) loop(std::integral_constant<int, (FM > 2 ? FM - 2 : 0)>{});
    else if (FM > 3 && live == FM - 3) loop(std::integral_constant<int, (FM > 3 ? FM - 3 : 0)>{});
    else if (FM > 4 && live == FM - 4) loop(std::integral_constant<int, (FM > 4 ? FM - 4 : 0)>{});
    else loop(std::integral_constant<int, 0>{});

    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();                             // everybody has read the last K-tile: the buffers become the epilogue's stage
    char* stg = smem + wave * (2 * 16 * (FN * 32 + 16));
    const int row0 = m0 + wf0 * 16, col0 = n0 + wn * FN * 16;
    switch (epi) {                                            // (uniform)
        case EPI_STORE: epilogue<EPI_STORE, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_GELU: epilogue<EPI_GELU, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_RELU2: epilogue<EPI_RELU2, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_LS_RES: epilogue<EPI_LS_RES, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_RES: epilogue<EPI_RES, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_SWIGLU: epilogue<EPI_SWIGLU, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_PATCH: epilogue<EPI_PATCH, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_F32: epilogue<EPI_F32, FM, FN>(p, acc, stg, row0, live, col0, lane); break;
        case EPI_PARTIAL: {
            GemmParams s = p;
            s.C = (float*)p.C + (int64_t)blockIdx.y * p.M * p.ldc; s.raw32 = 1; s.softcap = 0.f;
            epilogue<EPI_F32, FM, FN>(s, acc, stg, row0, live, col0, lane);
            break;
        }
        case EPI_ARGMAX:
            if constexpr (FN == 4) epilogue<EPI_ARGMAX, FM, FN>(p, acc, stg, row0, live, col0, lane);
            break;
    }
}

template <int WM, int WN, int FM, int FN, int NBUF, bool FAR = false>
int launch_t(int epi, const GemmParams& p, int rt, hipStream_t stream) {
    typedef MidGeom<WM, WN, FM, FN, NBUF> G;
    static std::atomic<uint64_t> attr_done{0};
    if (!cr_dyn_lds_once(attr_done, (const void*)gemm_mid_kernel<WM, WN, FM, FN, NBUF, FAR>, G::LDS)) return CR_ERR_HIP;
    const int ntm = std::max((p.M + G::BM - 1) / G::BM, rt), ntn = (p.N + G::BN - 1) / G::BN;
    const int slices = epi == EPI_PARTIAL ? p.group : 1, nwg = ntm * ntn, nf = (p.M + 15) / 16, per_group = 8 * ntn, last = ntm % 8 ? ntm % 8 : 8;
    auto mul = [&](int d) { return d > 1 && (int64_t)nwg * d < (1ll << 32) ? (unsigned)(((1ull << 32) + d - 1) / d) : 0u; };
    const MidGrid g{epi, ntm, p.K / 64 / slices, nwg / 8, nwg % 8, per_group, last, mul(per_group), mul(last), nf / ntm, nf % ntm, ntm > 1 && ntm < 1600 ? (unsigned)(((1ull << 32) + ntm - 1) / ntm) : 0u};
    hipLaunchKernelGGL((gemm_mid_kernel<WM, WN, FM, FN, NBUF, FAR>), dim3(nwg, slices), dim3(64 * G::WAVES), G::LDS, stream, g, p);
    return hipGetLastError() == hipSuccess ? CR_OK : CR_ERR_HIP;
}
// DEEP buffers where every workgroup has a CU to itself, as many as let two share one otherwise (by LDS and by registers).  us, few / deep: 16 x 64 tiles (7 / 8 buffers)
// 1025 x 1024 x 1024 (1040 workgroups) 13.9 / 17.6; 64 x 64 (4 / 8) 1024 x 1024 x 4096 (256) 19.8 / 16.1, 1025 x 1024 x 1024 (272) 9.7 / 12.3, 1025 x 4096 x 1024 (1088) 23.0 / 27.0; 96 x 64 (3 / 6) 25000 x 64 x
// 512 (261) 7.8 / 9.5, 1500 x 2048 x 1024 (512) 13.6 / 15.8, 3000 x 2048 x 4096 (1024) 79.5 / 88.8; 128 x 64 (3 / 6) 1025 x 1024 x 4096 (144) 25.7 / 22.5, 1025 x 4096 x 1024 (576) 20.7 / 23.3; 64 x 128 (3 / 6)
// 23.6 / 20.7 and 20.3 / 23.6.  The law below gives these shapes more workgroups than CUs only at the ends of the range: 64 columns or fewer in more than 24 000 rows (96 and 128 x 64), fewer than 65 rows of a K that
// the weight-streaming kernels do not take (16 and 64 x 64, 64 x 128).
template <int WM, int WN, int FM, int FN, int FEW, int DEEP>
int launch_two(int epi, const GemmParams& p, int rt, hipStream_t stream) {
    typedef MidGeom<WM, WN, FM, FN, FEW> G;
    static_assert(G::TWO_A_CU);
    const int64_t wgs = (int64_t)std::max((p.M + G::BM - 1) / G::BM, rt) * ((p.N + G::BN - 1) / G::BN) * (epi == EPI_PARTIAL ? p.group : 1);
    return wgs <= cr_device_cus() ? launch_t<WM, WN, FM, FN, DEEP>(epi, p, rt, stream) : launch_t<WM, WN, FM, FN, FEW>(epi, p, rt, stream);
}

}  // namespace

namespace {

// Tile shapes (launch_gemm_mid's `tile` = index + 1).  Eight waves where the tile is large enough to feed them: two waves a SIMD cover each other's LDS reads and barriers (64 x 64 at
// M = 1025, N = 1024, K = 4096: four waves 27.5 us, eight 26.6, before the loop that is there now; 128 x 128 at N = 3072, K = 1024: 20 and 13.4).
struct MidShape { int bm, bn; double launch = 2.5, row = 1.9e-3, step = -0.02; };      // (the law's: us a launch, a row of A or W in a K-tile, a K-tile)
constexpr MidShape SHAPES[] = {{16, 32}, {16, 64}, {32, 64}, {64, 32}, {64, 64}, {96, 64}, {128, 64}, {64, 128}, {96, 128}, {128, 128}, {96, 256, 2.5, 2e-3, 0.0}, {128, 256, 3.0, 2e-3, 0.02}, {160, 128, 2.5, 1.9e-3, 0.03}};
constexpr int N_SHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

}  // namespace

// A law to choose by, in us, and the tile shape (and number of row tiles) that takes least by it: launch and drain 2.5 us, a round of workgroups 1 us to its first K-tile, 1.9 ns per row of A or W in
// each K-tile of 64 less 20 ns (the three largest shapes more: SHAPES), 0.1 ns an element in the epilogue; a workgroup more on a CU costs its time again (two shallow ones to a CU take 0.8 of that).  It is no
// prediction.  Measured / law, weights cold: 1025 x 1024 x 4096 18.7 / 20.2, 1025 x 1024 x 1024 7.9 / 8.1, 1025 x 3072 x 1024 11.5 / 11.9, 1025 x 4096 x 1024 14.4 / 14.1, 77 x 4096 x 4096 15.0 / 12.1, 333 x
// 4096 x 14336 81 / 68, 1000 x 4096 x 14336 135 / 110, 13325 x 5120 x 1344 199 / 190; no term stands for the rate of HBM itself, which bounds wide weights at few rows (77 x 28672 x 4096 54 / 29).
// Against every way there is, 500 sizes drawn over M 65 .. 16000, N 512 .. 28672, K 256 .. 14336 (profiles/tiled_products/choice.txt): 1.007 times the fastest in geometric mean, above 1.05 at 21 of them.
// The largest shapes' terms decide where a product takes several rounds of one and fewer of the other, above all where K leaves 64 modulo 128, which the 256x256 kernel does not take.  us, 160 x 128 | 128 x
// 256: 3075 x 9216 x 448 48.3 | 39.9, 6124 x 9216 x 2240 260 | 228, 13325 x 5120 x 1344 212 | 199, and one round either way 2050 x 2048 x 2048 24.2 | 29.4; 96 x 128 | 96 x 256: 356 x 12800 x 14336 215 | 177,
// 1923 x 2560 x 14336 186 | 162.
double gemm_mid_cost(int epi, const GemmParams& p, int* tile, int* row_tiles) {
    const int nf = (p.M + 15) / 16, slices = epi == EPI_PARTIAL && p.group > 0 ? p.group : 1, nk = p.K / 64 / slices, cus = cr_device_cus();
    double best = 1e30;
    for (int t = 0; t < N_SHAPES; t++) {
        if (epi == EPI_ARGMAX && SHAPES[t].bn != 256) continue;          // (a wave's columns are a partial's 64)
        const long ntn = (long)((p.N + SHAPES[t].bn - 1) / SHAPES[t].bn) * slices;
        const int cap = SHAPES[t].bm / 16, least = (nf + cap - 1) / cap;
        for (int per_cu = 0; per_cu <= 2; per_cu++) {                    // the fewest row tiles, or as many as make one or two workgroups per CU
            const long want = per_cu == 0 ? least : (long)per_cu * cus / ntn;
            if (want < least || want > nf || (per_cu && want > 2L * least)) continue;
            const int rows = 16 * ((nf + (int)want - 1) / (int)want);
            const double rounds = (double)((want * ntn + cus - 1) / cus);
            const double c = SHAPES[t].launch + rounds * (1.0 + nk * (SHAPES[t].row * (rows + SHAPES[t].bn) + SHAPES[t].step) + 1e-4 * rows * SHAPES[t].bn);
            if (c < best - 1e-9) { best = c; *tile = t + 1; *row_tiles = (int)want; }
        }
    }
    return best;
}

int launch_gemm_mid(int epi, const GemmParams& p, hipStream_t stream) {
    int tile = p.tile, rt = 0;
    if (!tile) gemm_mid_cost(epi, p, &tile, &rt);
    if (tile < 1 || tile > N_SHAPES || (epi == EPI_ARGMAX && SHAPES[tile - 1].bn != 256)) return CR_ERR_ARG;      // (a pin; a wave's columns have to be a partial's 64)
    if (7 * 2 * std::max(p.lda, p.ldw) + 128 > (int64_t)UINT32_MAX) return launch_t<2, 4, 2, 4, 3, true>(epi, p, 0, stream);      // (whatever the epilogue; the same bits)
    switch (tile) {
        case 1: return launch_t<1, 2, 1, 1, 12>(epi, p, rt, stream);
        case 2: return launch_two<1, 4, 1, 1, 7, 8>(epi, p, rt, stream);
        case 3: return launch_t<1, 4, 2, 1, 6>(epi, p, rt, stream);
        case 4: return launch_t<2, 2, 2, 1, 6>(epi, p, rt, stream);
        case 5: return launch_two<2, 4, 2, 1, 4, 8>(epi, p, rt, stream);
        case 6: return launch_two<2, 4, 3, 1, 3, 6>(epi, p, rt, stream);
        case 7: return launch_two<2, 4, 4, 1, 3, 6>(epi, p, rt, stream);
        case 8: return launch_two<2, 4, 2, 2, 3, 6>(epi, p, rt, stream);
        case 9: return launch_t<2, 4, 3, 2, 5>(epi, p, rt, stream);
        case 10: return launch_t<2, 4, 4, 2, 4>(epi, p, rt, stream);
        case 11: return launch_t<2, 4, 3, 4, 3>(epi, p, rt, stream);
        case 12: return launch_t<2, 4, 4, 4, 3>(epi, p, rt, stream);
        case 13: return launch_t<2, 4, 5, 2, 4>(epi, p, rt, stream);
    }
    return CR_ERR_ARG;
}
