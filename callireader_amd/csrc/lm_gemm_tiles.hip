// Prompt products of described decoders in true fp32: C = epi(A[M,K] . W[N,K]^T), K % 64 == 0, optionally batched over heads or grouped over experts with gathered rows and scattered
// results.  (Decode batches: lm_gemm_rows.hip.)
//
// Bound by the matrix cores (v_mfma_f32_16x16x4_f32: 256 operations a clock and CU) where the grid fills the card, by what a K-tile asks for, reads and folds where it does not.  The form of
// gemm_mid.hip: NBUF K-tiles in LDS, NBUF - 1 of them under way, one barrier a K-tile, eight rows of 128 bytes a load instruction; the tile shape is picked by the rounds it gives.
// 402 x 4096 x 1024, 40.5 us on 256 workgroups: multiplications and launch 30.6, folded chains 2.7, LDS reads 2 to 3, asking for K-tiles 4.5, the barriers nothing.  So asking takes a scalar address and three
// other scalar instructions a piece, and both it and the reads go between the multiplications; every SIMD has all of a tile's rows in its two waves (with four wave rows a tile of six fragments left two SIMDs
// with four of them and two with two).  402 rows, us: products of 1024 columns over K = 1536 22.2 -> 19.5, 3584 and 4096 x 1024 42.5 -> 37.3; 1600 x 4096 x 1024 142 -> 127, 800 x 4096 x 1024 77.6 -> 72.5,
// 260 x 4096 x 1024 40.3 -> 31.5, experts of 1600 rows 154 and 85 -> 145 and 79.  (Tiles of half the size, two workgroups a CU: 45; K-tiles twice as deep, six buffers for three: no difference.)
// A lane reads 16 bytes of its row, k = 16 h + 4 (lane >> 4) .. + 3; the four multiplications take one element of each, which permutes k inside 16 for both operands alike.  A row's
// sum has the order of lm.hpp whatever the tile: an accumulator is a chain, and goes to the part's sum and that to the total when it ends.  That costs 1.6 us of the 22 where a chain is one block of 32 (two chains over all of K: 20), nothing on
// the larger tiles, whose waves multiply under each other's additions.
#include <algorithm>
#include <type_traits>

#include "diag.hpp"
#include "k_ring.hpp"
#include "lm.hpp"

namespace {

// four consecutive columns gn .. gn + 3 of row cr (`whole`: all inside N, 16-byte places)
template <int EPI>
__device__ __forceinline__ void put4(const LmGemmParams& p, int64_t cr, int gn, f32x4 v, bool whole) {
    float* c = (float*)p.C + (int64_t)blockIdx.z * p.c_bs + cr * p.ldc + gn;
    const float* g = EPI == LM_GATE ? (const float*)p.gate + (int64_t)blockIdx.z * p.g_bs + cr * p.ldg + gn : EPI == LM_SIDE ? (const float*)p.gate + (int64_t)p.tok[cr] * p.ldg + gn : nullptr;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (EPI == LM_RAW32 && p.softcap > 0.f) v[e] = p.softcap * tanhf(v[e] / p.softcap);
        if (EPI == LM_RELU2) v[e] = relu2(v[e]);
        if ((EPI == LM_GATE || EPI == LM_SIDE) && gn + e < p.N) v[e] = EPI == LM_GATE ? v[e] / (1.0f + expf(-g[e])) : gelu_tanh(v[e]) * g[e];
    }
    if (whole) { *(f32x4*)c = v; return; }
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (gn + e < p.N) c[e] = v[e];
}

template <int EPI, int FM, int FN>
__device__ __forceinline__ void epilogue(const LmGemmParams& p, const f32x4 (&acc)[FM][FN], int row0, int live, int rows, int pos0, int col0, int lane) {
    const bool vec = (p.ldc & 3) == 0 && (p.c_bs & 3) == 0 && ((uintptr_t)p.C & 15) == 0;
#pragma unroll
    for (int i = 0; i < FM; i++) {
        const int r = row0 + i * 16 + (lane & 15);
        if (i >= live) break;
        const int m = pos0 + min(r, rows - 1);
        const int64_t cr = (p.perm && p.scatter) ? p.perm[m] : m;
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int gn = col0 + j * 16 + 4 * (lane >> 4);
            f32x4 v = acc[i][j];
            if (EPI == LM_GLU) {                              // rows 0..7 of a 16-row weight tile are gates, 8..15 the matching ups: the partner's accumulator is 32 lanes away
                f32x4 u;
#pragma unroll
                for (int e = 0; e < 4; e++) u[e] = __shfl_xor(v[e], 32, 64);
                if (r >= rows || lane >= 32 || gn >= p.N) continue;
                float* c = (float*)p.C + cr * p.ldc + (col0 + j * 16) / 2 + 4 * (lane >> 4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float g = fminf(v[e], p.limit), up = fminf(fmaxf(u[e], -p.limit), p.limit);
                    c[e] = g / (1.0f + expf(-1.702f * g)) * (up + 1.0f);
                }
                continue;
            }
            if (r < rows && gn < p.N) put4<EPI>(p, cr, gn, v, vec && gn + 4 <= p.N);
        }
    }
}

// WM x WN waves of FM x FN fragments of 16 x 16; KB blocks of 32 of K a K-tile
template <int WM, int WN, int FM, int FN, int KB, int NBUF>
struct Geom {
    static constexpr int BM = WM * FM * 16, BN = WN * FN * 16, WAVES = WM * WN, ROWS8 = (BM + BN) / 8, PIECES = KB * ROWS8, PER = (PIECES + WAVES - 1) / WAVES, STAGE = PIECES * 1024,
                         LDS = NBUF * STAGE;
    static_assert((NBUF - 2) * PER <= 63 && NBUF >= 2 && LDS <= 160 * 1024, "vmcnt is six bits wide; a CU has 160 KiB");
};

template <int WM, int WN, int FM, int FN, int KB, int NBUF, bool FAR>
__global__ __launch_bounds__(64 * WM * WN) void lm_tiles_kernel(const LmGemmParams p, const int epi, const int ntm) {
    typedef Geom<WM, WN, FM, FN, KB, NBUF> G;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, n0 = blockIdx.x * G::BN;
    const float* A = (const float*)p.A + (int64_t)blockIdx.z * p.a_bs;
    const float* W = (const float*)p.W;
    int pos0 = 0, rows = p.M, m0 = 0, fn;                     // rows pos0 + m0 .. of A (of the sorted assignments), in fn fragments
    if (p.tiles) {
        if ((int)blockIdx.y >= *p.n_tiles) return;            // (uniform: the grid is sized for the worst split)
        const int4 t = p.tiles[blockIdx.y];
        W += (int64_t)t.x * p.w_bs;
        pos0 = t.y; rows = t.z;
        fn = (min(rows, G::BM) + 15) >> 4;
    } else {                                                  // the matrix's fragments dealt evenly over the row tiles (at most WM * FM each)
        const int nf = (p.M + 15) >> 4, f0 = (int)((int64_t)blockIdx.y * nf / ntm);
        fn = (int)((int64_t)(blockIdx.y + 1) * nf / ntm) - f0;
        W += (int64_t)blockIdx.z * p.w_bs;
        m0 = f0 * 16;
    }
    const int wf0 = fn * wm / WM, live = fn * (wm + 1) / WM - wf0;      // a tile's over its wave rows

    // This wave's pieces of a K-tile: eight rows, 128 bytes each; numbers past the last repeat it, pieces past the tile's rows move one lane's 16 bytes (the count of instructions under way stays a
    // constant).  A piece's first row is the same for all lanes, so its address is a scalar one and a lane's own row and chunk are 32 bits beyond it; FAR: gathered rows, and rows so far apart that eight of
    // them span 4 GiB, have 64 bits a lane.
    const char *src[G::PER], *lane_src[FAR ? G::PER : 1];
    unsigned off[G::PER], dst[G::PER];
    uint64_t lanes[G::PER];
    const unsigned smem_base = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
#pragma unroll
    for (int i = 0; i < G::PER; i++) {
        const int at = min(wave + i * G::WAVES, G::PIECES - 1), kb = at / G::ROWS8, piece = at - kb * G::ROWS8, row = piece * 8 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
        const bool a = piece * 8 < G::BM;
        const int first = a ? pos0 + min(m0 + piece * 8, rows - 1) : min(n0 + piece * 8 - G::BM, p.N - 1), own = a ? pos0 + min(m0 + row, rows - 1) : min(n0 + row - G::BM, p.N - 1);
        src[i] = (const char*)((a ? A + (int64_t)first * p.lda : W + (int64_t)first * p.ldw) + kb * 32);
        off[i] = (unsigned)((own - first) * (a ? p.lda : p.ldw) * 4) + chunk * 16;
        if (FAR) {
            const int64_t r = a && p.perm && p.gather_div ? p.perm[own] / p.gather_div : own;
            lane_src[FAR ? i : 0] = (const char*)((a ? A + r * p.lda : W + r * p.ldw) + kb * 32 + chunk * 4);
        }
        dst[i] = smem_base + at * 1024;
        lanes[i] = a && piece >= 2 * fn ? 1 : ~0ull;
    }
    const int nk = p.K / (32 * KB);
    auto ask_piece = [&](int i, int buf) __attribute__((always_inline)) {
        CR_DIAG_POISON(smem + buf * G::STAGE + (dst[i] - smem_base))
        if constexpr (FAR) {
            ring_ask_far<0>(lane_src[FAR ? i : 0], dst[i], buf * G::STAGE, lanes[i]);
            lane_src[FAR ? i : 0] += KB * 128;
        } else {
            ring_ask<0>(src[i], off[i], dst[i], buf * G::STAGE, lanes[i]);
            src[i] += KB * 128;
        }
    };
    // the K-tile that `src` stands at, into buffer buf
    auto ask = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < G::PER; i++) ask_piece(i, buf);
    };
    f32x4 acc[FM][FN], part[FM][FN], total[FM][FN];           // of the chain, of the part, of the whole sum
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = part[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int part_blocks = lm_part_blocks(p.K, p.slices), chain_blocks = lm_chain_blocks(part_blocks);
    int in_part = part_blocks, in_chain = chain_blocks;       // blocks of 32 until they end
    const int swz = (lane >> 1) & 7;
    const int c_off[2] = {((lane >> 4) ^ swz) * 16, ((4 + (lane >> 4)) ^ swz) * 16};
    const int a_off = (wf0 * 16 + (lane & 15)) * 128, w_off = (G::BM + wn * FN * 16 + (lane & 15)) * 128;
    struct Frags { f32x4 a[2 * KB][FM], w[2 * KB][FN]; };
    // fragment x of a K-tile's 2 * KB * (FN + FM): those of 16 k after each other, W's first
    auto read_one = [&](Frags& f, int x, int buf, auto count) {
        const char* s = smem + buf * G::STAGE;
        const int h = x / (FN + FM), c = x % (FN + FM), at = (h >> 1) * G::ROWS8 * 1024 + c_off[h & 1];
        if (c < FN) f.w[h][c] = *(const f32x4*)(s + w_off + c * 2048 + at);
        else if (c - FN < decltype(count)::value) f.a[h][c - FN] = *(const f32x4*)(s + a_off + (c - FN) * 2048 + at);
    };
    auto read = [&](Frags& f, int buf, auto count) {
#pragma unroll
        for (int x = 0; x < 2 * KB * (FN + FM); x++) read_one(f, x, buf, count);
    };
    auto fold = [&](f32x4 (&to)[FM][FN], f32x4 (&from)[FM][FN], auto count) {
#pragma unroll
        for (int i = 0; i < FM; i++)
            if (i < decltype(count)::value) {
#pragma unroll
                for (int j = 0; j < FN; j++) { to[i][j] += from[i][j]; from[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
            }
    };
    // beside(g): what is issued behind the multiplications g of 8 * KB
    auto multiply = [&](const Frags& f, auto count, auto beside) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
#pragma unroll
            for (int h = 2 * kb; h < 2 * kb + 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
#pragma unroll
                    for (int i = 0; i < FM; i++)
                        if (i < decltype(count)::value) {
#pragma unroll
                            for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[h][j][e], f.a[h][i][e], acc[i][j], 0, 0, 0);
                        }
                    beside(4 * h + e);
                }
            in_chain--; in_part--;
            if (in_chain == 0 || in_part == 0) {              // (uniform)
                fold(part, acc, count);
                in_chain = chain_blocks;
                if (in_part == 0) { fold(total, part, count); in_part = part_blocks; }
            }
        }
    };
    auto nothing = [](int) {};
    auto arrive = [&](int t) { ring_arrive<NBUF, G::PER>(nk, t); };
    auto loop = [&](auto count) {
        for (int t = 0; t < min(NBUF - 1, nk); t++) ask(t);
        Frags f0, f1;
        arrive(0);
        if (NBUF - 1 < nk) ask(NBUF - 1);
        read(f0, 0, count);
        int buf = 0;                                          // buffer of K-tile kt
        // What a step reads and asks for goes between its multiplications, which keep the matrix pipe busy for 32 clocks each
        auto step = [&](int kt, Frags& now, Frags& next, auto all) {
            if constexpr (decltype(all)::value) {
                wait_vm<(NBUF - 2) * G::PER>();
                __builtin_amdgcn_s_waitcnt(0xC07F);           // lgkmcnt(0)
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            } else arrive(kt + 1);
            const int into = buf;
            buf = buf + 1 == NBUF ? 0 : buf + 1;
            constexpr int READS = 2 * KB * (FN + FM), GROUPS = 8 * KB, EACH = (READS + G::PER + GROUPS - 2) / (GROUPS - 1);
            multiply(now, count, [&](int g) {
#pragma unroll
                for (int x = g * EACH; x < (g + 1) * EACH; x++) {
                    if (x < READS) read_one(next, x, buf, count);
                    else if (x < READS + G::PER) {
                        if (decltype(all)::value || kt + NBUF < nk) ask_piece(x - READS, into);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        constexpr std::true_type whole{};
        constexpr std::false_type tail{};
        int kt = 0;
        for (; kt + 1 + NBUF < nk; kt += 2) {                 // (no step of the loop is conditional: the compiler waited for the reads ahead of the multiplications then)
            step(kt, f0, f1, whole);
            step(kt + 1, f1, f0, whole);
        }
        for (; kt + 2 < nk; kt += 2) {
            step(kt, f0, f1, tail);
            step(kt + 1, f1, f0, tail);
        }
        if (kt + 1 < nk) {
            step(kt, f0, f1, tail);
            multiply(f1, count, nothing);
        } else multiply(f0, count, nothing);
    };
    // (fewer than FM - 1 live fragments: those past them multiply what an older K-tile left in LDS, and are not stored)
    if (live == FM) loop(std::integral_constant<int, FM>{});
    else if (FM > 1 && live == FM - 1) loop(std::integral_constant<int, FM - 1>{});
    else if (FM > 2 && live > 0) loop(std::integral_constant<int, FM - 2>{});
    else loop(std::integral_constant<int, 0>{});
    const int row0 = m0 + wf0 * 16, col0 = n0 + wn * FN * 16;
    switch (epi) {                                            // (uniform)
        case LM_STORE: epilogue<LM_STORE, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
        case LM_RAW32: epilogue<LM_RAW32, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
        case LM_GLU: epilogue<LM_GLU, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
        case LM_GATE: epilogue<LM_GATE, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
        case LM_RELU2: epilogue<LM_RELU2, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
        case LM_SIDE: epilogue<LM_SIDE, FM, FN>(p, total, row0, live, rows, pos0, col0, lane); break;
    }
}

template <int WM, int WN, int FM, int FN, int KB, int NBUF, bool FAR = false>
int launch_t(int epi, const LmGemmParams& p, int ntm, hipStream_t st) {
    typedef Geom<WM, WN, FM, FN, KB, NBUF> G;
    static std::atomic<uint64_t> attr_done{0};
    if (!cr_dyn_lds_once(attr_done, (const void*)lm_tiles_kernel<WM, WN, FM, FN, KB, NBUF, FAR>, G::LDS)) return CR_ERR_HIP;
    hipLaunchKernelGGL((lm_tiles_kernel<WM, WN, FM, FN, KB, NBUF, FAR>), dim3((p.N + G::BN - 1) / G::BN, ntm, p.batch > 0 ? p.batch : 1), dim3(64 * G::WAVES), G::LDS, st, p, epi, ntm);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

struct Shape { int bm, bn; };
constexpr Shape SHAPES[] = {{16, 32}, {32, 32}, {32, 64}, {64, 64}, {128, 64}, {64, 128}, {128, 128}};

}  // namespace

// The shape that a cost model says is fastest (us): a K-tile of a workgroup 0.05 + the longer of its loads (2.1 ns a row of A or W, as in gemm_mid.hip) and its multiplications (0.12 ns
// an element of the tile); a workgroup more on a CU costs its time again.
int launch_lm_gemm_tiles(int epi, const LmGemmParams& p, hipStream_t st) {      // (checked by launch_lm_gemm)
    static_assert(LM_TILE_M == 64, "an expert's list of rows is one row tile");
    if (epi < LM_STORE || epi > LM_SIDE) return cr_fail(CR_ERR_ARG, "lm_gemm: epilogue %d", epi);
    const int nf = (p.M + 15) / 16, batch = std::max(p.batch, 1), nk = p.K / 32, cus = cr_device_cus();
    // 64 bits a lane, whatever the epilogue and with the same bits: rows that a list names, and operands eight of whose rows (and an XOR that keeps to a row's 128 bytes) are not within 32 bits of each other
    if (p.tiles || (p.perm && p.gather_div) || 8 * std::max(p.lda, p.ldw) * 4 >= (1ll << 32)) return launch_t<2, 4, 2, 1, 1, 4, true>(epi, p, p.tiles ? p.max_tiles : (nf + 3) / 4, st);
    int tile = 0, ntm = 0;
    double best = 1e30;
    for (int t = 0; t < (int)(sizeof(SHAPES) / sizeof(SHAPES[0])); t++) {
        const int cap = SHAPES[t].bm / 16, rt = (nf + cap - 1) / cap, rows = 16 * ((nf + rt - 1) / rt);
        const long wgs = (long)((p.N + SHAPES[t].bn - 1) / SHAPES[t].bn) * batch * rt;
        const double c = (double)((wgs + cus - 1) / cus) * (nk * (0.05 + std::max(0.0021 * (rows + SHAPES[t].bn), 0.00012 * rows * SHAPES[t].bn)) + 1.0);
        if (c < best) { best = c; tile = t; ntm = rt; }
    }
    switch (tile) {
        case 0: return launch_t<1, 2, 1, 1, 2, 5>(epi, p, ntm, st);
        case 1: return launch_t<2, 2, 1, 1, 2, 4>(epi, p, ntm, st);
        case 2: return launch_t<2, 4, 1, 1, 2, 4>(epi, p, ntm, st);
        case 3: return launch_t<2, 4, 2, 1, 1, 4>(epi, p, ntm, st);
        case 4: return launch_t<2, 4, 4, 1, 1, 3>(epi, p, ntm, st);
        case 5: return launch_t<2, 4, 2, 2, 1, 3>(epi, p, ntm, st);
    }
    return launch_t<4, 2, 2, 4, 1, 4>(epi, p, ntm, st);
}
