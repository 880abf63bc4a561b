// Attention over a cache of latents: key and value of a token are both linear in one cached row c, so with the query carried into the latent space (W_uk^T q per head) the
// scores are q' . c and the attended latents sum p c are carried back by W_uv -- every head reads the same rows.  Scores, softmax weights and their sums are fp32.
#include <algorithm>
#include <type_traits>

#include "attention_plain.hpp"
#include "lm.hpp"

namespace {

// Any size, either element type: one workgroup per (row, head), the cached row as key and value (attention_plain.hpp).
template <typename T, int TPB>
__global__ __launch_bounds__(TPB) void latent_attn_plain_kernel(const LatentAttnParams p) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ float red[PLAIN_RED];
    const int row = blockIdx.x, head = blockIdx.y;
    const int seq = p.ix.row_seq ? p.ix.row_seq[row] : p.ix.seqs[row];
    const int n = (p.ix.row_pos ? p.ix.row_pos[row] : p.ix.lens[seq]) + 1;
    const T* C = (const T*)p.C + (int64_t)seq * p.max_tokens * p.Rp;
    const int64_t at = ((int64_t)row * p.H + head) * p.Rp;
    T* O = (T*)p.O + at;
    plain_attend<T, TPB>((const T*)p.Q + at, C, p.Rp, C, p.Rp, n, p.Rp, p.Rp, p.scale, 0.f, sm, red, [&](int i, float v) { O[i] = (T)v; });
}
template <typename T>
void launch_plain_t(const LatentAttnParams& p, hipStream_t st) {
    if (!p.ix.row_pos) hipLaunchKernelGGL((latent_attn_plain_kernel<T, 1024>), dim3(p.M, p.H), dim3(1024), plain_lds_floats(p.Rp, 1024) * 4, st, p);
    else hipLaunchKernelGGL((latent_attn_plain_kernel<T, 256>), dim3(p.M, p.H), dim3(256), plain_lds_floats(p.Rp, 256) * 4, st, p);
}

// ---- bf16 decode --------------------------------------------------------------------------------------------------------
constexpr float LOG2E = 1.4426950408889634f;
__device__ __forceinline__ unsigned pack2(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
// LDS rows of a key tile: 16-byte chunk c of row r sits at c ^ swz(r).  Two readers: K . q takes 16 consecutive rows at one chunk (swz is a bijection of r mod 16), the transposed
// reads of P . V take rows {0..3, 8..11} + 4 j at a chunk pair (the upper bits of swz differ over those eight rows).
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 1) | ((r >> 2) & 1) | (r & 8); }
// reductions over the lanes that share a head: a DPP row of 16 (HT = 1) or half of one (HT = 2)
template <int HT, typename F> __device__ __forceinline__ float head_reduce(float x, F f) {
    x = f(x, dpp<0xB1>(x));                            // quad_perm 1 0 3 2
    x = f(x, dpp<0x4E>(x));                            // quad_perm 2 3 0 1
    x = f(x, dpp<0x141>(x));                           // row_half_mirror
    return HT == 2 ? x : f(x, dpp<0x128>(x));          // row_ror 8
}
template <int HT> __device__ __forceinline__ float head_max(float x) { return head_reduce<HT>(x, [](float a, float b) { return fmaxf(a, b); }); }
template <int HT> __device__ __forceinline__ float head_sum(float x) { return head_reduce<HT>(x, [](float a, float b) { return a + b; }); }
// LDS-only barrier: the next tile's fill stays in flight across it;
// ... and the tile's closing barrier, behind which the next tile has landed for every wave
#define TILE_BARRIER() asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory")
#define LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// One workgroup of 4 waves = one token, one split of the keys, 16 HT heads; two workgroups fit a CU (the loads of one run under the products of the other).  Key tiles of 32 in two
// LDS buffers, the next one filled under the current one.  S^T = C . q'^T: wave = 16 keys x half of the latent columns, all heads; the halves meet in LDS.
// Softmax: a wave owns 4 HT heads (running maximum and sum stay in its registers) and leaves their weights in LDS as two bf16 halves (hi + lo) with the rescale factors.
// O^T += C^T . P^T: each wave owns a quarter of the latent columns, C^T by transposed LDS reads.  Three LDS-only barriers per tile.
template <int R, int HT>
__global__ __launch_bounds__(256, 2) void latent_decode_kernel(const LatentDecodeParams p) {
    touch_args<(int)(sizeof(LatentDecodeParams))>();
    constexpr int KT = LATENT_TILE, CH = R / 8, KS = R / 64, DT = R / 64, SLD = KT + 4, PLD = KT + 8;
    extern __shared__ __attribute__((aligned(16))) char smem[];            // 2 key tiles | scores | weights | rescale factors
    float* sS = (float*)(smem + 2 * KT * R * 2);                           // [2][16 HT][SLD]
    bf16* sP = (bf16*)(sS + 2 * 16 * HT * SLD);                            // [hi, lo][16 HT][PLD]
    float* sAl = (float*)(sP + 2 * 16 * HT * PLD);                         // [16 HT]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = p.a.H, groups = (H + 16 * HT - 1) / (16 * HT);
    const int row = blockIdx.y / groups, h0 = blockIdx.y % groups * 16 * HT, split = blockIdx.x;
    if (row >= p.a.M) {                                        // (uniform)
        const int linear = blockIdx.x + gridDim.x * blockIdx.y, nth = l2_ahead_nth(linear, (int)gridDim.x * p.a.M * groups);
        if (nth >= 0 && nth < L2_AHEAD_GROUPS) l2_ahead(p.ahead, linear, nth);
        return;
    }
    const int seq = p.a.ix.row_seq ? p.a.ix.row_seq[row] : p.a.ix.seqs[row];
    const int n = (p.a.ix.row_pos ? p.a.ix.row_pos[row] : p.a.ix.lens[seq]) + 1;
    const int lo = split * p.split, hi = min(lo + p.split, n);
    if (lo >= n) return;
    const bf16* C = (const bf16*)p.a.C + (int64_t)seq * p.a.max_tokens * R;
    const int g = lane >> 4, li = lane & 15;
    const int kt16 = (wave & 1) * 16, half = wave >> 1;

    // staging by LDS-DMA, NP 1-KiB pieces per wave and tile (RPP rows each); the swizzle sits on the source side.  Issued from inline asm (M0 = LDS base, saved and restored inside the
    // statement) so that the compiler does not order this tile's LDS reads behind the next tile's fill; its landing is waited for in front of the tile's closing barrier.
    constexpr int NP = R / 64, RPP = 512 / R;
    const unsigned smem_base = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
    int prow[NP], pchunk[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        prow[i] = (wave * NP + i) * RPP + lane / CH;
        pchunk[i] = ((lane % CH) ^ (swz(prow[i]) & (CH - 1))) * 16;
    }
    auto stage = [&](int buf, int k0) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const unsigned off = (unsigned)min(k0 + prow[i], hi - 1) * (unsigned)(R * 2) + pchunk[i];
            const unsigned dst = smem_base + buf * (KT * R * 2) + (wave * NP + i) * 1024;
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(C), "s"(dst) : "memory");
        }
    };
    stage(0, lo);
    bf16x8 qf[HT][KS];
#pragma unroll
    for (int h = 0; h < HT; h++) {
        const bf16* q = (const bf16*)p.a.Q + ((int64_t)row * H + min(h0 + h * 16 + li, H - 1)) * R + half * (R / 2) + g * 8;
#pragma unroll
        for (int s = 0; s < KS; s++) qf[h][s] = *(const bf16x8*)(q + s * 32);
    }
    f32x4 acc[DT][HT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int h = 0; h < HT; h++) acc[d][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;                                  // of head shead; l_run: this lane's keys
    const int shead = HT == 2 ? 8 * wave + (lane >> 3) : (4 * wave + g), skey = HT == 2 ? 4 * (lane & 7) : 2 * li;
    const float sc2 = p.a.scale * LOG2E;
    const int krow = kt16 + li, ksw = swz(krow) & (CH - 1);
    const int tq = li >> 2, tp = li & 3, vr0 = 8 * g + tq, vr1 = vr0 + 4, vs0 = swz(vr0) & (CH - 1), vs1 = swz(vr1) & (CH - 1);
    const int col0 = wave * (DT * 16);

    __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0) the compiler sees: without it the queries' first use, inside the loop, waits for the loop's own fills
    TILE_BARRIER();
    int buf = 0;
    for (int k0 = lo; k0 < hi; k0 += KT, buf ^= 1) {
        const bool more = k0 + KT < hi;
        if (more) stage(buf ^ 1, k0 + KT);
        const char* kb = smem + buf * (KT * R * 2);
        // ---- S^T ----
        {
            f32x4 s4[HT];
#pragma unroll
            for (int h = 0; h < HT; h++) s4[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const bf16x8 kf = *(const bf16x8*)(kb + krow * (R * 2) + (((half * (CH / 2) + s * 4 + g) ^ ksw) * 16));
#pragma unroll
                for (int h = 0; h < HT; h++) s4[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[h][s], s4[h], 0, 0, 0);
            }
#pragma unroll
            for (int h = 0; h < HT; h++) *(f32x4*)(sS + (half * 16 * HT + h * 16 + li) * SLD + kt16 + 4 * g) = s4[h];
        }
        LDS_BARRIER();
        // ---- softmax weights: HT = 2: 8 heads a wave, 8 lanes a head, 4 keys a lane; HT = 1: 4 heads, 16 lanes, 2 keys ----
        {
            constexpr int KL = 2 * HT;
            float t[KL];
            const float *s0 = sS + shead * SLD + skey, *s1 = s0 + 16 * HT * SLD;
#pragma unroll
            for (int e = 0; e < KL; e++) t[e] = more || k0 + skey + e < hi ? (s0[e] + s1[e]) * sc2 : -INFINITY;
            float mx = fmaxf(t[0], t[1]);
            if (HT == 2) mx = fmaxf(mx, fmaxf(t[KL - 2], t[KL - 1]));
            const float m_new = fmaxf(m_run, head_max<HT>(mx));
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < KL; e++) { t[e] = __builtin_amdgcn_exp2f(t[e] - m_new); sum += t[e]; }
            l_run = l_run * alpha + sum;
#pragma unroll
            for (int e = 0; e < KL; e += 2) {
                const unsigned hw = pack2(t[e], t[e + 1]);
                *(unsigned*)(sP + shead * PLD + skey + e) = hw;
                *(unsigned*)(sP + (16 * HT + shead) * PLD + skey + e) = pack2(t[e] - __uint_as_float(hw << 16), t[e + 1] - __uint_as_float(hw & 0xffff0000u));
            }
            if (skey == 0) sAl[shead] = alpha;
        }
        LDS_BARRIER();
        // ---- O^T += C^T . P^T on this wave's columns ----
        {
            bf16x8 ph[HT], pl[HT];
#pragma unroll
            for (int h = 0; h < HT; h++) {
                ph[h] = *(const bf16x8*)(sP + (h * 16 + li) * PLD + 8 * g);
                pl[h] = *(const bf16x8*)(sP + (16 * HT + h * 16 + li) * PLD + 8 * g);
                const float alpha = sAl[h * 16 + li];
#pragma unroll
                for (int d = 0; d < DT; d++) acc[d][h] *= alpha;
            }
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const int c0 = (col0 + d * 16) / 8 + (tp >> 1);
                const char* base = kb + (tp & 1) * 8;
                const bf16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)CR_LDS(base + vr0 * (R * 2) + ((c0 ^ vs0) * 16)));
                const bf16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)CR_LDS(base + vr1 * (R * 2) + ((c0 ^ vs1) * 16)));
                const bf16x8 vf = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
#pragma unroll
                for (int h = 0; h < HT; h++) acc[d][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph[h], acc[d][h], 0, 0, 0);
#pragma unroll
                for (int h = 0; h < HT; h++) acc[d][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl[h], acc[d][h], 0, 0, 0);
            }
        }
        TILE_BARRIER();
    }
    const float l_sum = head_sum<HT>(l_run);
    if (skey == 0 && h0 + shead < H) {
        const int64_t pr = ((int64_t)row * H + h0 + shead) * p.nsplit + split;
        p.part_ml[pr * 2] = m_run; p.part_ml[pr * 2 + 1] = l_sum;
    }
#pragma unroll
    for (int h = 0; h < HT; h++) {
        const int head = h0 + h * 16 + li;
        if (head >= H) continue;
        const int64_t pr = ((int64_t)row * H + head) * p.nsplit + split;
#pragma unroll
        for (int d = 0; d < DT; d++) *(f32x4*)(p.part_o + pr * R + col0 + d * 16 + 4 * g) = acc[d][h];
    }
}

// RW tokens of one head: 8 / RW waves per token merge its splits (each in index order) and the attended latent is rounded once; then the row block is carried back by W_uv, gated and stored
// Bound by its chain of loads: the splits' rows are asked for first, then W_uv (fragment-ordered, a contiguous KiB an instruction; as rows a fragment's four neighbouring lanes hold four of them and a KiB
// takes 64 clocks) and the gates, which all travel under the merge.  gridDim.z workgroups share a row block's columns at few splits (each merges for itself, see the launch).  24 rows of 16 heads, latent
// of 512: 6.3 us with rows, weights first and gates last, 5.2 now; a step of 8 layers 953 / 948 / 944 us with 1 / 2 / 4 workgroups a row block.
template <int R, int RW>
__global__ __launch_bounds__(512) void latent_combine_kernel(const LatentDecodeParams p) {
    touch_args<(int)(sizeof(LatentDecodeParams))>();
    __shared__ __attribute__((aligned(16))) bf16 sA[RW][R + 8];
    __shared__ float sO[RW == 1 ? 8 : 1][RW == 1 ? R : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), H = p.a.H, head = blockIdx.x, m0 = blockIdx.y * RW;      // (head fastest: the row blocks of a head share an XCD's L2)
    constexpr int CPL = R / 64, SW = 8 / RW, JB = RW == 1 ? 8 : 4096 / R < 32 ? 4096 / R : 32;                   // columns per lane: CPL lane + 0 ..; waves per row (wave w takes every SW-th split); splits in flight
    typedef __attribute__((ext_vector_type(CPL < 2 ? 2 : CPL))) float vecf_;
    struct one { float x; __device__ float& operator[](int) { return x; } __device__ const float& operator[](int) const { return x; } };
    typedef typename std::conditional<CPL == 1, one, vecf_>::type vecf;
    const int g = lane >> 4, li = lane & 15, out_row = m0 + (li & (RW - 1));       // (the product's other token columns repeat the first RW)
    const int cw = 8 / (int)gridDim.z, col0 = wave < cw ? ((int)blockIdx.z * cw + wave) * 16 : p.vdim;      // waves that take columns: col0, col0 + 128, ..
    bf16x8 wf[R / 32];
    auto weights = [&](int n16) {
        const bf16* w = p.wuv_dl ? p.wuv_dl + (int64_t)head * p.uv_hs + (int64_t)n16 * R + lane * 8 : p.wuv + (int64_t)head * p.uv_hs + (int64_t)min(n16 + li, p.vdim - 1) * R + g * 8;
        const int step = p.wuv_dl ? 512 : 32;
#pragma unroll
        for (int k = 0; k < R / 32; k++) wf[k] = *(const bf16x8*)(w + k * step);
    };
    float gates[4];
    auto gate = [&](int n16) {
#pragma unroll
        for (int e = 0; e < 4; e++) gates[e] = bf2f(p.gate[(int64_t)min(out_row, p.a.M - 1) * p.ldg + head * p.vdim + min(n16 + 4 * g + e, p.vdim - 1)]);
    };
    {
        const int row = min(m0 + wave / SW, p.a.M - 1), sw = wave % SW;
        const int64_t base = ((int64_t)row * H + head) * p.nsplit;
        vecf o, v[JB];
#pragma unroll
        for (int c = 0; c < CPL; c++) o[c] = 0.f;
        // the first splits' rows are requested before anything about the row is known (splits it does not have are dropped below)
#pragma unroll
        for (int j = 0; j < JB; j++) v[j] = *(const vecf*)(p.part_o + (base + min(sw + SW * j, p.nsplit - 1)) * R + lane * CPL);
        const float m0s = p.part_ml[(base + min(lane, p.nsplit - 1)) * 2], l0s = p.part_ml[(base + min(lane, p.nsplit - 1)) * 2 + 1];
        // the projection's weights of this wave's first column block, and its gates, travel under the merge
        __builtin_amdgcn_sched_barrier(0);
        if (col0 < p.vdim) { weights(col0); gate(col0); }
        __builtin_amdgcn_sched_barrier(0);
        const int seq = p.a.ix.row_seq ? p.a.ix.row_seq[row] : p.a.ix.seqs[row];
        const int n = (p.a.ix.row_pos ? p.a.ix.row_pos[row] : p.a.ix.lens[seq]) + 1, ns = (n + p.split - 1) / p.split;
        float M = lane < ns ? m0s : -INFINITY;
        for (int s = lane + 64; s < ns; s += 64) M = fmaxf(M, p.part_ml[(base + s) * 2]);
        M = wave_max_s(M);
        float L = 0.f;
        for (int s0 = 0; s0 < ns; s0 += 64) {
            const int s = s0 + lane;
            float m = m0s, l = l0s;
            if (s0 > 0 && s < ns) { m = p.part_ml[(base + s) * 2]; l = p.part_ml[(base + s) * 2 + 1]; }
            const float w = s < ns ? __builtin_amdgcn_exp2f(m - M) : 0.f;
            L += wave_sum_s(s < ns ? w * l : 0.f);
            const int cnt = min(64, ns - s0);
            for (int j0 = sw; j0 < cnt; j0 += SW * JB) {
                if (s0 + j0 > sw)
#pragma unroll
                    for (int j = 0; j < JB; j++) v[j] = *(const vecf*)(p.part_o + (base + min(s0 + j0 + SW * j, ns - 1)) * R + lane * CPL);
#pragma unroll
                for (int j = 0; j < JB; j++) {
                    const float wj = lane_value(w, min(j0 + SW * j, 63));
#pragma unroll
                    for (int c = 0; c < CPL; c++) o[c] += j0 + SW * j < cnt ? wj * v[j][c] : 0.f;
                }
            }
        }
        const float inv = 1.0f / L;
#pragma unroll
        for (int c = 0; c < CPL; c++) {
            if constexpr (RW == 1) sO[wave][lane * CPL + c] = o[c] * inv;
            else sA[wave][lane * CPL + c] = f2bf(o[c] * inv);
        }
    }
    __syncthreads();
    if constexpr (RW == 1) {
        for (int c = tid; c < R; c += 512) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < 8; w++) t += sO[w][c];
            sA[0][c] = f2bf(t);
        }
        __syncthreads();
    }
    for (int n16 = col0; n16 < p.vdim; n16 += 128) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (n16 >= 128) { weights(n16); gate(n16); }           // heads wider than a block per wave
#pragma unroll
        for (int k = 0; k < R / 32; k++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[k], *(const bf16x8*)&sA[li & (RW - 1)][k * 32 + g * 8], acc, 0, 0, 0);
        if (li >= RW || out_row >= p.a.M) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = n16 + 4 * g + e;
            if (c < p.vdim) p.out[(int64_t)out_row * p.ldo + head * p.vdim + c] = f2bf(acc[e] / (1.0f + __builtin_amdgcn_exp2f(-LOG2E * gates[e])));
        }
    }
}

// q'[m][h][:] = W_uk^T q[m][h] for 16 MT tokens of one head and 128 latent columns: the query's K-slices are added in slice order and rounded once on their way into LDS
template <int MT>
__global__ __launch_bounds__(256) void latent_absorb_kernel(const float* __restrict__ part, int slices, int M, int H, int Ap, int Rp, const bf16* __restrict__ ukT, int dl, bf16* __restrict__ out) {
    touch_args<56>();
    extern __shared__ __attribute__((aligned(16))) char smem[];
    bf16* sq = (bf16*)smem;                            // [16 MT][Ap + 8]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15, head = blockIdx.y, ld = Ap + 8;
    const int per = Ap / 4;                            // vectors of four per row
    // 16 columns' weights from column k on: fragment-ordered (dl), or rows
    auto frag = [&](int n16, int k) { return *(const bf16x8*)(ukT + ((int64_t)head * Rp + n16) * Ap + (dl ? k * 16 + lane * 8 : li * Ap + k + g * 8)); };
    bf16x8 w0[2][2], w1[2][2];                         // the weights' first 128 columns travel under the sums below (24 rows of 16 heads: 5.7 us -> 5.0; fragment-ordered 4.5)
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int n16 = min((int)blockIdx.x * 128 + (wave * 2 + t) * 16, Rp - 16), c = min(k * 64, Ap - 64);
            w0[t][k] = frag(n16, c);
            w1[t][k] = frag(n16, c + 32);
        }
    for (int v = tid; v < 16 * MT * per; v += 256) {
        const int m = v / per, c = (v % per) * 4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        if (m < M) {
            const float* q = part + ((int64_t)m * H + head) * Ap + c;
#pragma unroll 4
            for (int k = 0; k < slices; k++) s += *(const f32x4*)(q + (int64_t)k * M * H * Ap);
        }
        *(bf16x4*)(sq + m * ld + c) = bf16x4{f2bf(s[0]), f2bf(s[1]), f2bf(s[2]), f2bf(s[3])};
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int n16 = blockIdx.x * 128 + (wave * 2 + t) * 16;
        if (n16 >= Rp) continue;                       // (uniform per wave; no barrier follows)
        f32x4 acc[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto step = [&](int k, const bf16x8& a, const bf16x8& b) {
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const bf16* q = sq + (m * 16 + li) * ld + k + g * 8;
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, *(const bf16x8*)q, acc[m], 0, 0, 0);
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, *(const bf16x8*)(q + 32), acc[m], 0, 0, 0);
            }
        };
        step(0, w0[t][0], w1[t][0]);
        if (Ap > 64) step(64, w0[t][1], w1[t][1]);
        for (int k = 128; k < Ap; k += 64) step(k, frag(n16, k), frag(n16, k + 32));
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int row = m * 16 + li;
            if (row < M) *(bf16x4*)(out + ((int64_t)row * H + head) * Rp + n16 + 4 * g) = bf16x4{f2bf(acc[m][0]), f2bf(acc[m][1]), f2bf(acc[m][2]), f2bf(acc[m][3])};
        }
    }
}

template <int R, int HT>
int launch_decode_t(const LatentDecodeParams& p, hipStream_t st) {
    constexpr int LDS = 2 * LATENT_TILE * R * 2 + 2 * 16 * HT * (LATENT_TILE + 4) * 4 + 2 * 16 * HT * (LATENT_TILE + 8) * 2 + 16 * HT * 4;
    static_assert(LDS <= 81920, "two workgroups per CU");
    static std::atomic<uint64_t> done{0};
    if (!cr_dyn_lds_once(done, (const void*)latent_decode_kernel<R, HT>, LDS)) return CR_ERR_HIP;
    const int rows = p.a.M * ((p.a.H + 16 * HT - 1) / (16 * HT));
    const bool ahead = p.ahead.at && l2_ahead_bytes(p.ahead) <= l2_ahead_beside_latent((int64_t)p.nsplit * rows, cr_device_cus());
    hipLaunchKernelGGL((latent_decode_kernel<R, HT>), dim3(p.nsplit, rows + (ahead ? (l2_ahead_extra(p.nsplit * rows) + p.nsplit - 1) / p.nsplit : 0)), dim3(256), LDS, st, p);
    const bool few = p.a.M * p.a.H <= cr_device_cus();        // few rows: eight waves share one row's splits
    const int wgs = p.a.H * (few ? p.a.M : (p.a.M + 7) / 8);
    const int z = p.nsplit > 4 ? 1 : 4 * wgs <= cr_device_cus() ? 4 : 2 * wgs <= cr_device_cus() ? 2 : 1;      // (past four splits merging them again costs more than the columns save: 8 rows of 16 heads, 1000 keys, a step 790 / 788 / 810 us with 1 / 2 / 4)
    if (few) hipLaunchKernelGGL((latent_combine_kernel<R, 1>), dim3(p.a.H, p.a.M, z), dim3(512), 0, st, p);
    else hipLaunchKernelGGL((latent_combine_kernel<R, 8>), dim3(p.a.H, (p.a.M + 7) / 8, z), dim3(512), 0, st, p);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

}  // namespace

// Two workgroups fill a CU, so the splits of the whole batch should come to about that many workgroups -- but a split of fewer than four tiles costs more in partials than it saves.
int latent_split_keys(int heads, int64_t keys) {
    const int64_t groups = heads > 16 ? (heads + 31) / 32 : 1, wgs = std::max<int64_t>(2 * cr_device_cus() / groups, 1);
    const int64_t per = (keys + wgs - 1) / wgs;
    const int64_t tiles = std::min<int64_t>(std::max<int64_t>((per + LATENT_TILE - 1) / LATENT_TILE, 4), 128);
    return (int)tiles * LATENT_TILE;
}

int launch_latent_absorb(const LmLayer& L, int M, const float* part, int slices, void* out, hipStream_t st) {
    if (M <= 0 || M > 64 || !part || slices <= 0 || L.Ap > 512) return cr_fail(CR_ERR_ARG, "latent absorb: rows %d, head size %d", M, L.Ap);
    const int mt = (M + 15) / 16;
    const size_t lds = (size_t)16 * mt * (L.Ap + 8) * 2;
    const dim3 grid((L.Rp + 127) / 128, L.s.heads), block(256);
    static std::atomic<uint64_t> d3{0}, d4{0};
    if (lds > 65536) {
        if (mt == 3 && !cr_dyn_lds_once(d3, (const void*)latent_absorb_kernel<3>, 131072)) return CR_ERR_HIP;
        if (mt == 4 && !cr_dyn_lds_once(d4, (const void*)latent_absorb_kernel<4>, 131072)) return CR_ERR_HIP;
    }
#define ABSORB(MT) hipLaunchKernelGGL(latent_absorb_kernel<MT>, grid, block, lds, st, part, slices, M, L.s.heads, L.Ap, L.Rp, L.wukT_dl ? L.wukT_dl : (const bf16*)L.wukT, L.wukT_dl != nullptr, (bf16*)out)
    switch (mt) {
        case 1: ABSORB(1); break;
        case 2: ABSORB(2); break;
        case 3: ABSORB(3); break;
        default: ABSORB(4); break;
    }
#undef ABSORB
    CR_HIP(hipGetLastError());
    return CR_OK;
}

bool latent_decode_supported(int Rp) { return Rp == 64 || Rp == 128 || Rp == 256 || Rp == 512; }

int launch_latent_decode(const LatentDecodeParams& p, hipStream_t st) {
    if (p.a.M <= 0 || p.a.H <= 0 || p.nsplit <= 0 || p.split <= 0 || p.split % LATENT_TILE || !p.part_o || !p.part_ml || !p.wuv || !p.gate || !p.out || p.vdim <= 0 || !latent_decode_supported(p.a.Rp))
        return cr_fail(CR_ERR_ARG, "latent decode attention: rows %d, heads %d, latent %d", p.a.M, p.a.H, p.a.Rp);
    const bool two = p.a.H > 16;
    switch (p.a.Rp) {
        case 64: return two ? launch_decode_t<64, 2>(p, st) : launch_decode_t<64, 1>(p, st);
        case 128: return two ? launch_decode_t<128, 2>(p, st) : launch_decode_t<128, 1>(p, st);
        case 256: return two ? launch_decode_t<256, 2>(p, st) : launch_decode_t<256, 1>(p, st);
        default: return two ? launch_decode_t<512, 2>(p, st) : launch_decode_t<512, 1>(p, st);
    }
}

int launch_latent_attn_plain(bool f32, const LatentAttnParams& p, hipStream_t st) {
    if (p.M <= 0 || p.H <= 0 || p.Rp <= 0 || p.Rp % 64 || p.Rp > PLAIN_MAX_COLS) return cr_fail(CR_ERR_ARG, "latent attention: rows %d, heads %d, latent %d", p.M, p.H, p.Rp);
    if (f32) launch_plain_t<float>(p, st);
    else launch_plain_t<bf16>(p, st);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
