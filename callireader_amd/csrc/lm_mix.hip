// One decode step's mixers in one launch: from the fused projection's K-slices to the output projection's input.  A workgroup takes a (row, key head, split of keys) of the attention or a
// (row, head) of retention, forms its own queries, keys, values and gate from the slices (lm_heads.hpp), and goes on with them on the chip; the caches and states it needs travel meanwhile.
// What all layers of a step share -- a row's sequence and position, the cos and sin of its angles -- is there already (lm_embed_step_kernel).
//
// Bound by latency: with few rows none of it fills the chip, so the chain from the slices to the result is what counts.
//
// Attention in bf16 (heads of 64 or 128, any number of keys): a wave forms the scores of 32 of the split's 256 keys, which go from the cache straight into its registers as the A operand;
// the values come by LDS-DMA.  Scores of a query lie in LDS before its softmax starts, so a wave takes a whole query (four keys a lane) instead of an accumulator's 32 query places of which a
// group fills a few.  Weights go through LDS as the P.V product's fragments (two bf16 terms, as in attention.hip), a wave of the first D / 32 takes 32 value columns.
// The arithmetic is flash_attn_kernel's over the split's tiles of 64 keys (attention.hip, SPLIT with WIDE), bit for bit: its running reference point, which a vote over the unit's queries moves, its
// rescaling, its order of sums (one row of 8 heads of 128 on 2, 49 .. 80 keys: 7.2 us; with one reference point a split and sums across the wave 7.0, and other bits).  The token's own key and value never come from memory: they replace the stale row in the registers and in LDS.  Attention in fp32: attention_plain.hpp on the token's
// freshly written cache row, which every workgroup of a group of query heads writes for itself -- the same bits.
#include "attention_merge.hpp"
#include "attention_plain.hpp"
#include "diag.hpp"
#include "lm_heads.hpp"
#include "retention.hpp"

namespace {

typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
__device__ __forceinline__ unsigned pack_bf16x2(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

constexpr int MIX_THREADS16 = 512, MIX_THREADS32 = 1024, MIX_SC = 260;      // floats between the queries of a split's scores: 256 keys, the rows four banks apart
constexpr int MIX_TILES = 4;                     // tiles of 64 keys a split: eight waves of 32 keys
static_assert(MIX_TILES == ATTN_SPLIT_TILES, "the caller counts splits of ATTN_SPLIT_TILES tiles (lm.hip: HEADS_SPLIT)");

struct MixArgs {
    const float* part; const int2* where; const float* ang; void* ao;      // K-slices; {sequence, position} and angles of every row
    int slices, M, Na, ang_ld, ldo, pad0, pad1, pad2, pad3;
    int col[LM_REGIONS];                         // first column of a region by kind
    int att, ret;                                // workgroups of a row: attention, retention; those behind them merge splits
    // attention: R query heads of a key head a workgroup, `units` of them a row, kv_group a key head (fp32: R = 1)
    void *K, *V; const float *nq, *nk;
    float *part_o, *part_ml;
    int D, G, R, units, kv_group, nsplit, ring, chunk, dim, vdim, half_a, off_a, merge;
    float eps, s_mul, softcap, out_mul;
    // retention
    void* ao_r; RetHead ret_head;
    int half_r, off_r;
    float k_scale;
    L2AheadList ahead;                           // weights of the products behind, brought into L2 by the workgroups past the rows
};
__device__ __forceinline__ const float* mix_cos(const MixArgs& p, int row, int off) { return p.ang + (int64_t)row * p.ang_ld + off; }

__device__ __forceinline__ void lds_barrier() {               // LDS writes are seen by all waves; loads from memory stay under way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// eight columns of a row of the projection: the first four slices are asked for at once, the others behind them; added in slice order
struct Columns {
    const float* at; int64_t step; int slices;
    f32x4 w[4][2];
    __device__ __forceinline__ void load(int k0) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (k0 + k < slices) { w[k][0] = *(const f32x4*)(at + (k0 + k) * step); w[k][1] = *(const f32x4*)(at + (k0 + k) * step + 4); }
    }
    __device__ __forceinline__ void ask(const MixArgs& p, int64_t row, int col) {
        step = (int64_t)p.M * p.Na; slices = p.slices;
        at = p.part + row * p.Na + col;
        load(0);
    }
    __device__ __forceinline__ void sum(float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = 0.f;
        for (int k0 = 0; k0 < slices; k0 += 4) {
            if (k0) load(k0);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k0 + k < slices)
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] += w[k][e >> 2][e & 3];
        }
    }
};

// bytes: value tiles, weights, scores (before them, in the same place, the waves' columns), queries, own key and value, maxima of the tiles
template <int D> constexpr int mix_lds16(int rows) { return MIX_TILES * 64 * D * 2 + 1024 * rows + MIX_SC * 4 * rows + (rows + 2) * D * 2 + MIX_TILES * 32 * 4; }

template <int D>
__device__ __forceinline__ void mix_attend16(const MixArgs& p, int u, int row, char* smem) {
    constexpr int KS = D / 16, DB = D / 32, ROWB = D * 2, TILE = 64 * ROWB, CPR = D / 8, RPI = 1024 / ROWB;
    constexpr float LOG2E = 1.4426950408889634f;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l31 = lane & 31, hh = lane >> 5;
    const int unit = u / p.nsplit, split = u - unit * p.nsplit, g = unit / p.kv_group, R = p.R, heads = R + 2;
    char *vt = smem, *pt = vt + MIX_TILES * TILE;              // [tile][64][D] bf16, chunks swizzled; [32-key block][16-key step][term][half wave][query] x 16 bytes
    float* sc = (float*)(pt + 1024 * R);                       // [R][MIX_SC]
    bf16 *q = (bf16*)(sc + MIX_SC * R), *nk = q + R * D, *nv = nk + D;
    float *mx = (float*)(nv + D), *sx = (float*)pt;      // [tile][32 queries]; [wave][512]: (R + 2) * D floats in whole waves, at most 4096

    // the unit's query heads, its key and its value: D / 8 lanes each
    const int e0 = (lane % CPR) * 8;
    auto ask = [&](int hd, Columns& cols, HeadLane& hl) {
        hd = min(hd, heads - 1);
        cols.ask(p, row, (hd < R ? p.col[LM_Q] + (unit * R + hd) * D : (hd == R ? p.col[LM_K] : p.col[LM_V]) + g * D) + e0);
        hl.ask(e0, hd < R ? p.nq : hd == R ? p.nk : nullptr, hd <= R ? p.half_a : 0, mix_cos(p, row, p.off_a), mix_cos(p, row, p.off_a) + (p.half_a + 7) / 8 * 8);
    };
    const int2 at = p.where[row];
    const int64_t cache = ((int64_t)at.x * p.G + g) * p.ring * D;
    bf16 *Kb = (bf16*)p.K + cache, *Vb = (bf16*)p.V + cache;
    const int n = at.y % p.chunk + 1, key0 = split * 256;      // keys of the row, the token's own among them; first of this split
    const int here = max(0, min(256, n - key0)), tiles = (here + 63) / 64, old = max(n - 2, 0);      // (rows past `old` hold nothing yet of this sequence)
    const int r0 = (7 - wave) * 32;                            // the wave's keys: the first waves project, so theirs are the last
    bf16x8 kf[KS];
    auto caches = [&]() {
        if (r0 < here) {
            const bf16* r = Kb + (int64_t)min(key0 + r0 + l31, old) * D + hh * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kf[ks] = *(const bf16x8*)(r + ks * 16);
        }
        if (r0 < 64 * tiles) {
#pragma unroll
            for (int i = 0; i < 32 / RPI; i++) {
                const int r = r0 + i * RPI + lane / CPR;
                CR_DIAG_POISON(vt + (r0 + i * RPI) * ROWB)
                __builtin_amdgcn_global_load_lds(CR_GLB(Vb + (int64_t)min(key0 + r, old) * D + (((lane % CPR) ^ attn_vswz<D>(r)) * 8)), CR_LDS(vt + (r0 + i * RPI) * ROWB), 16, 0, 0);
            }
        }
    };
    const int h0 = wave * (64 / CPR);
    if (h0 < heads) {
        const bool keep = unit % p.kv_group == 0 && n - 1 >= key0 && n - 1 < key0 + 256;
        for (int h = h0; h < heads; h += 512 / CPR) {          // (whole waves)
            const int hd = h + lane / CPR;
            Columns cols;
            HeadLane hl;
            ask(hd, cols, hl);
            float v[8];
            cols.sum(v);
            hl.apply(D, p.dim, p.eps, sx + tid * 8, v);
            if (hd < R) st8(q + hd * D + e0, v);
            else if (hd < heads) {
                st8((hd == R ? nk : nv) + e0, v);
                if (keep) st8((hd == R ? Kb : Vb) + (int64_t)(n - 1) * D + e0, v);
            }
        }
    }
    caches();
    lds_barrier();

    if (r0 < here) {
        if (key0 + r0 + 32 >= n && key0 + r0 + l31 == n - 1)   // the token's own key
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kf[ks] = *(const bf16x8*)(nk + hh * 8 + ks * 16);
        const bf16* qr = q + min(l31, R - 1) * D + hh * 8;
        f32x16 s;
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], *(const bf16x8*)(qr + ks * 16), s, 0, 0, 0);
        if (l31 < R)                                           // lane (query, half): keys 8 i + 4 half + 0..3
#pragma unroll
            for (int i = 0; i < 4; i++) *(f32x4*)(sc + l31 * MIX_SC + r0 + 8 * i + 4 * hh) = f32x4{s[4 * i], s[4 * i + 1], s[4 * i + 2], s[4 * i + 3]};
    }
    lds_barrier();
    // a wave's queries, every eighth: four scores a lane, sixteen lanes a tile
    const bool capped = p.softcap > 0.f;
    f32x4 z[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = wave + 8 * j;
        if (i >= R) break;
        z[j] = *(const f32x4*)(sc + i * MIX_SC + 4 * lane);
        if (capped) {                                          // softcap * tanh(z / softcap) = softcap - 2 softcap / (1 + exp(2 z / softcap))
            const float cap2 = -2.0f * p.softcap, capx = 2.0f * LOG2E * p.s_mul / p.softcap;
#pragma unroll
            for (int e = 0; e < 4; e++) z[j][e] = fmaf(cap2, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z[j][e] * capx)), p.softcap);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) z[j][e] = 4 * lane + e < here ? z[j][e] : -INFINITY;
        float m = fmaxf(fmaxf(z[j][0], z[j][1]), fmaxf(z[j][2], z[j][3]));
        m = fmaxf(m, dpp<0xB1>(m)); m = fmaxf(m, dpp<0x4E>(m)); m = fmaxf(m, dpp<0x141>(m)); m = fmaxf(m, dpp<0x128>(m));      // over the tile's lanes
        if ((lane & 15) == 0) mx[(lane >> 4) * 32 + i] = capped ? m : m * p.s_mul;
    }
    lds_barrier();

    // the reference point of each tile's exponentials (it stays while no query's maximum grows by more than 8) and what the sums ahead of the tile are scaled by; lane: query
    float m = -INFINITY, ref[MIX_TILES] = {}, alpha[MIX_TILES] = {};
    const int qi = min(l31, R - 1);
#pragma unroll
    for (int t = 0; t < MIX_TILES; t++) {
        if (t >= tiles) break;                                 // (uniform)
        const float top = mx[32 * t + qi], was = m;
        const bool move = !__all(top - m <= 8.0f);
        if (move) m = fmaxf(m, top);
        ref[t] = m;
        alpha[t] = move ? __builtin_amdgcn_exp2f((was - m) * LOG2E) : 1.0f;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = wave + 8 * j;
        if (i >= R) break;
        float at_tile = 0.f;                                   // query i's reference point in the lane's tile
#pragma unroll
        for (int t = 0; t < MIX_TILES; t++) {
            const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ref[t]), i));
            at_tile = lane >> 4 == t ? r : at_tile;
        }
        const float scale = capped ? LOG2E : p.s_mul * LOG2E, m2 = at_tile * LOG2E;
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = __builtin_amdgcn_exp2f(fmaf(z[j][e], scale, -m2));
        *(f32x4*)(sc + i * MIX_SC + 4 * lane) = w;             // (for their sums)
        u32x2 hi, lo;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            hi[e] = pack_bf16x2(w[2 * e], w[2 * e + 1]);
            lo[e] = pack_bf16x2(w[2 * e] - __uint_as_float(hi[e] << 16), w[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u));
        }
        // the lane's four keys in the product's fragment: of a 16-key step the half waves hold keys {0..3, 8..11} and {4..7, 12..15}
        char* d = pt + ((lane >> 2) * 4 + (lane & 1)) * R * 16 + i * 16 + (lane >> 1 & 1) * 8;
        *(u32x2*)d = hi;
        *(u32x2*)(d + 2 * R * 16) = lo;
    }
    if (r0 < 64 * tiles) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the wave's values are in LDS, for all waves behind the barrier
        // the token's own value, also over what lies behind it (its weights are zero, but the rows hold anything)
        for (int r = max(r0, n - 1 - key0) + lane / CPR; r < r0 + 32; r += RPI)
            *(bf16x8*)(vt + r * ROWB + (((lane % CPR) ^ attn_vswz<D>(r)) * 16)) = *(const bf16x8*)(nv + e0);
    }
    __syncthreads();
    if (wave >= DB) return;
    const int db = wave, tq = (lane & 15) >> 2, tp = lane & 3, v_row = 4 * hh + tq;
    const int v_at = v_row * ROWB + (tp & 1) * 8 + ((((db * 4) ^ attn_vswz<D>(v_row)) | (((lane >> 4) & 1) * 2 + (tp >> 1))) * 16);
    f32x16 o;
#pragma unroll
    for (int e = 0; e < 16; e++) o[e] = 0.f;
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < MIX_TILES; t++) {
        if (t >= tiles) break;
        if (t)
#pragma unroll
            for (int e = 0; e < 16; e++) o[e] *= alpha[t];
        float even = 0.f, odd = 0.f;                           // the tile's weights, as the lanes of its keys add them
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const char* w = pt + (((t * 4 + st) * 4 + hh) * R + qi) * 16;
            const bf16x8 hi = *(const bf16x8*)w, lo = *(const bf16x8*)(w + 2 * R * 16);
            const char* vp = vt + t * TILE + 16 * st * ROWB + v_at;
            const bf16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)CR_LDS(vp));
            const bf16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)CR_LDS(vp + 8 * ROWB));
            const bf16x8 vf = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, hi, o, 0, 0, 0);
            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, lo, o, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const f32x4 z = *(const f32x4*)(sc + qi * MIX_SC + 64 * t + 16 * st + 8 * i + 4 * hh);
                even += z[0]; odd += z[1];
                even += z[2]; odd += z[3];
            }
        }
        l = fmaf(l, alpha[t], even + odd);
    }
    l += __shfl_xor(l, 32, 64);
    if (l31 >= R) return;
    // lane (query, half) owns columns 32 db + 8 g4 + 4 hh + 0..3
    if (p.nsplit > 1) {
        const int64_t pr = (((int64_t)row * p.units + unit) * p.nsplit + split) * R + l31;
        if (db == 0 && hh == 0) { p.part_ml[pr * 2] = m; p.part_ml[pr * 2 + 1] = l; }
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) *(f32x4*)(p.part_o + pr * D + 32 * db + 8 * g4 + 4 * hh) = f32x4{o[4 * g4], o[4 * g4 + 1], o[4 * g4 + 2], o[4 * g4 + 3]};
        return;
    }
    bf16* out = (bf16*)p.ao + (int64_t)row * p.ldo + (int64_t)(unit * R + l31) * p.vdim;
#pragma unroll
    for (int g4 = 0; g4 < 4; g4++) {
        const int d = 32 * db + 8 * g4 + 4 * hh;
        bf16 r[4];
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = f2bf(p.out_mul != 0.f ? p.out_mul * o[4 * g4 + e] / l : o[4 * g4 + e] / l);
        if ((p.vdim & 3) == 0) { if (d < p.vdim) *(bf16x4*)(out + d) = bf16x4{r[0], r[1], r[2], r[3]}; }
        else
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (d + e < p.vdim) out[d + e] = r[e];
    }
}

constexpr int mix_lds32(int cols) { return (plain_lds_floats(cols, MIX_THREADS32) + cols + 3 * 512) * 4; }      // bytes: attention_plain's, query, the columns' exchange

// head: query head
__device__ __forceinline__ void mix_attend32(const MixArgs& p, int head, int row, char* smem) {
    __shared__ float red[PLAIN_RED];
    const int tid = threadIdx.x, g = head / p.kv_group, D = p.D;
    float *sm = (float*)smem, *q = sm + plain_lds_floats(D, MIX_THREADS32), *sx = q + D;
    const int hd = tid * 8 / D, e0 = tid * 8 % D;              // the query, its key and its value
    const bool projects = (tid & ~63) * 8 < 3 * D;             // (whole waves)
    Columns cols;
    HeadLane hl;
    if (projects) {
        const int h = min(hd, 2);
        cols.ask(p, row, p.col[h == 0 ? LM_Q : h == 1 ? LM_K : LM_V] + (h == 0 ? head : g) * D + e0);
        hl.ask(e0, h == 0 ? p.nq : h == 1 ? p.nk : nullptr, h < 2 ? p.half_a : 0, mix_cos(p, row, p.off_a), mix_cos(p, row, p.off_a) + (p.half_a + 7) / 8 * 8);
    }
    const int2 at = p.where[row];
    const int n = at.y % p.chunk + 1;
    const int64_t base = ((int64_t)at.x * p.G + g) * p.ring * D;
    float *K = (float*)p.K + base, *V = (float*)p.V + base;
    if (projects) {
        float v[8];
        cols.sum(v);
        hl.apply(D, p.dim, p.eps, sx + tid * 8, v);
        if (hd < 3) st8(hd == 0 ? q + e0 : (hd == 1 ? K : V) + (int64_t)(n - 1) * D + e0, v);
    }
    __syncthreads();                                            // (the workgroup reads its own cache row)
    float* O = (float*)p.ao + (int64_t)row * p.ldo + (int64_t)head * p.vdim;
    plain_attend<float, MIX_THREADS32>(q, K, D, V, D, n, D, p.vdim, p.s_mul, p.softcap, sm, red, [&](int i, float x) { O[i] = x * p.out_mul; });
}

// floats of LDS: rotated queries and keys, values, gate, ret_step's outputs and sums, the columns' exchange
__host__ __device__ constexpr int mix_ret_floats(int Kp, int Vp) { return 2 * Kp + 3 * Vp + LM_MAX_HEAD / 16 + (2 * Kp + 2 * Vp + 511) / 512 * 512; }

template <typename T, int NR>
__device__ __forceinline__ void mix_retain(const MixArgs& p, int h, int row, float* sm) {
    const int tid = threadIdx.x, Kp = NR * 16, Vp = p.ret_head.Vp, wide = max(Kp, Vp), thin = min(Kp, Vp);
    float *q = sm, *k = q + Kp, *v = k + Kp, *g = v + Vp, *so = g + Vp, *red = so + Vp, *sx = red + LM_MAX_HEAD / 16;
    // the widest heads first: every head's lanes start at a multiple of their number
    const int at = tid * 8, P = at < 2 * wide ? wide : thin, which = at < 2 * wide ? at / wide : 2 + (at - 2 * wide) / thin, e0 = at & (P - 1);
    const int kind = which > 3 ? LM_RG : (which < 2) == (Vp >= Kp) ? LM_RV + (which & 1) : LM_RQ + (which & 1);
    const bool projects = (tid & ~63) * 8 < 2 * (Kp + Vp);     // (whole waves)
    Columns cols;
    HeadLane hl;
    if (projects) {
        cols.ask(p, row, p.col[kind] + h * P + e0);
        hl.ask(e0, nullptr, kind == LM_RQ || kind == LM_RK ? p.half_r : 0, mix_cos(p, row, p.off_r), mix_cos(p, row, p.off_r) + (p.half_r + 7) / 8 * 8);
    }
    const int2 sp = p.where[row];
    RetStep<NR> step(p.ret_head, sp.x, h);
    step.ask();
    if (projects) {
        float x[8];
        cols.sum(x);
        hl.apply(P, p.dim, p.eps, sx + at, x);
        if (kind == LM_RK)
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] *= p.k_scale;
        if (kind == LM_RV || kind == LM_RG)
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = (float)(T)x[e];
        if (which < 4) st8((kind == LM_RQ ? q : kind == LM_RK ? k : kind == LM_RV ? v : g) + e0, x);
    }
    lds_barrier();
    step.run(sp.y == 0, q, k, [&](int c) { return *(const f32x4*)(v + c); }, so, red);
    __syncthreads();
    T* out = (T*)p.ao_r + (int64_t)row * p.ldo + (int64_t)h * p.ret_head.vdim;
    step.finish(so, red, [&](int c, float o) { out[c] = (T)(o * silu32(g[c])); });
}

template <typename T, int D, int NR>
__global__ __launch_bounds__(sizeof(T) == 4 ? MIX_THREADS32 : MIX_THREADS16, 4) void lm_mix_kernel(const MixArgs p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    touch_args<(int)sizeof(MixArgs)>();
    const int x = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
    if (row >= p.M) {                                          // (uniform)
        const int linear = x + (int)gridDim.x * row, nth = l2_ahead_nth(linear, (int)gridDim.x * p.M);
        // (bf16: about 1.1 us for the rows' own reads first: 1 row of 1024 443 us a step for 453, 4 rows 553 for 558; float32, whose weights take longer than that leaves, 8 rows 803 for 795)
        if (sizeof(T) == 2) __builtin_amdgcn_s_sleep(40);
        if (nth >= 0 && nth < L2_AHEAD_GROUPS) l2_ahead(p.ahead, linear, nth);
        return;
    }
    if (x < p.att) {
        if constexpr (sizeof(T) == 4) mix_attend32(p, x, row, smem);
        else mix_attend16<D>(p, x, row, smem);
    } else if (x < p.att + p.ret) mix_retain<T, NR>(p, x - p.att, row, (float*)smem);
    else if constexpr (sizeof(T) == 2) {
        AttnParams a{};
        a.H = p.units; a.Sq = p.R; a.nsplit = p.nsplit; a.part_o = p.part_o; a.part_ml = p.part_ml; a.wide = 1; a.vdim = p.vdim; a.out_mul = p.out_mul;
        a.O = (bf16*)p.ao; a.o_bs = p.ldo; a.o_rs = p.vdim; a.o_hs = (int64_t)p.R * p.vdim;
        const int u = (x - p.att - p.ret) * (MIX_THREADS16 / 64) + (tid >> 6), hq = u / (D / 64);
        if (hq < p.units * p.R) attn_merge_splits(a, D, row, hq / p.R, hq % p.R, (u % (D / 64)) * 64 + (tid & 63));
    }
    if (x == 0 && !p.merge) {                                  // the output projection's input: padding columns
        T* ao = (T*)p.ao + (int64_t)row * p.ldo;
        for (int i = p.pad0 + tid; i < p.pad1; i += blockDim.x) ao[i] = (T)0.f;
        for (int i = p.pad2 + tid; i < p.pad3; i += blockDim.x) ao[i] = (T)0.f;
    }
}

template <typename T, int D, int NR>
int launch_mix_n(const MixArgs& a, int merge, int lds, hipStream_t st) {
    static std::atomic<uint64_t> attr_done{0};
    if (!cr_dyn_lds_once(attr_done, (const void*)lm_mix_kernel<T, D, NR>, 160 * 1024 - 256)) return cr_fail(CR_ERR_HIP, "decode mixer: LDS");
    const int X = a.att + a.ret + merge;
    hipLaunchKernelGGL((lm_mix_kernel<T, D, NR>), dim3(X, a.M + (a.ahead.n ? (l2_ahead_extra(X * a.M) + X - 1) / X : 0)), dim3(sizeof(T) == 4 ? MIX_THREADS32 : MIX_THREADS16), lds, st, a);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
int launch_mix_part(bool f32, int Kp, const MixArgs& a, int merge, int lds, hipStream_t st) {
    if (f32) return Kp <= 64 ? launch_mix_n<float, 0, 4>(a, merge, lds, st) : launch_mix_n<float, 0, 8>(a, merge, lds, st);
    if (a.D == 64) return Kp <= 64 ? launch_mix_n<bf16, 64, 4>(a, merge, lds, st) : launch_mix_n<bf16, 64, 8>(a, merge, lds, st);
    return Kp <= 64 ? launch_mix_n<bf16, 128, 4>(a, merge, lds, st) : launch_mix_n<bf16, 128, 8>(a, merge, lds, st);
}

}  // namespace

bool lm_mix_supported(bool f32, const LmLayer& L) {
    // heads of retention of up to 128 keys: a wave's piece of the state stays in registers beside the rest; attention in bf16: sizes with an instance
    if (L.retention() && L.Kp > 128) return false;
    return !L.heads() || f32 || (L.s.attn.scale > 0.f && L.Ap <= 128);
}

// One launch saves two others and their round trips, 6 to 15 us a layer while the chip is not full.  Beyond that the separate kernels' smaller workgroups count.  Us of a layer's step saved:
//   fp32: a workgroup of 16 waves has its CU to itself, so a second round of them loses: heads of 8 on 2 x 128 + 8 of retention, 16 rows +6.5 / +2.8 / -1.1 at 60 / 900 / 2500 keys, 20 rows
//   +1.4 / -11, 64 rows -5 / -37.  Wide heads over many keys are bound by reading them, which a group's heads share better in the separate kernel's order: 16 on 4 x 128, 12 rows (216 workgroups)
//   +6.7 / -2 / -10 at 60 / 900 / 2500; 4 x 256, 32 rows (256) +6.7 at 60, -3.4 at 400; 24 rows (192) +7 / +2.3 / +0.6 / -9 at 60 / 400 / 900 / 2500, 16 rows (128) +6 at 2500.
//   bf16, one workgroup a CU (their LDS: groups of 8 of 128 and more, of 32 of 64): 16 on 2 x 128, 24 x 900 (192) +6.5, 24 x 2500 (480) -0.6, 64 x 2500 -6.6; 32 on 1 x 64, 64 x 900 (256) +2,
//   40 x 2500 (400) -5.  Two a CU: heads of 128 gain throughout (16 on 16, 64 x 2500 +20); of 64, whose cache rows of 128 bytes come in pieces of 32, up to four rounds: 32 on 32,
//   9 x 900 (1152) +1.7, 64 x 200 (2048) +4.5, 9 x 2500 (2880) -1.4, 64 x 900 (8192) -15; 32 on 2 (groups of 16), 64 x 900 (512) +0.6, 64 x 2500 (1280) -2.
bool lm_mix_pays(bool f32, const LmLayer& L, int M, int rows, int splits) {
    const int64_t cus = cr_device_cus();
    const int64_t att = L.heads() ? (int64_t)M * (L.s.attn.heads / rows) * (f32 ? 1 : splits) : 0, ret = L.retention() ? (int64_t)M * L.s.ret.heads : 0;
    if (f32) return att + ret <= (!L.heads() || L.Ap <= 64 || splits <= 1 ? cus : cus * ((L.Ap <= 128 ? 4 : 3) - (splits > 4)) / 4);
    if (!L.heads()) return true;
    const int lds = L.Ap == 64 ? mix_lds16<64>(rows) : mix_lds16<128>(rows);
    if (2 * lds > 160 * 1024) return att <= cus;
    return L.Ap == 128 || att <= (rows > 8 ? 4 : 8) * cus;
}

int launch_lm_mix(bool f32, const Lm& lm, const LmLayer& L, const LmMixIn& in, hipStream_t st) {
    const cr_lm_heads& s = L.s.attn;
    const cr_lm_retention& r = L.s.ret;
    if (in.M <= 0 || in.M > 65535 || !in.part || in.slices <= 0 || !in.where || !in.ang || !in.ao || !lm_mix_supported(f32, L) || (L.retention() && !in.state)) return cr_fail(CR_ERR_ARG, "decode mixer: operands");
    MixArgs a{};
    a.part = in.part; a.where = in.where; a.ang = in.ang; a.ao = in.ao; a.slices = in.slices; a.M = in.M; a.Na = L.Na; a.ang_ld = (int)lm.rot.size(); a.ldo = L.Gp;
    a.pad0 = L.heads() ? s.heads * s.vdim : 0; a.pad1 = L.off_r; a.pad2 = L.off_r + (L.retention() ? r.heads * r.vdim : 0); a.pad3 = L.Gp;
    for (int i = 0; i < L.n_regions; i++) a.col[L.regions[i].kind] = L.regions[i].off;
    a.eps = lm.d.eps;
    if (in.ahead) a.ahead = *in.ahead;
    int lds = 0, merge = 0;
    if (L.heads()) {
        if (!in.cache_k || !in.cache_v || in.ring <= 0 || in.chunk <= 0 || in.rows <= 0 || in.rows > 32 || s.heads / s.kv_heads % in.rows || in.nsplit <= 0 || (in.nsplit > 1 && (f32 || !in.part_o || !in.part_ml)) ||
            (f32 && in.rows != 1)) return cr_fail(CR_ERR_ARG, "decode mixer: attention");
        a.K = in.cache_k; a.V = in.cache_v; a.nq = L.nq; a.nk = L.nc; a.part_o = in.part_o; a.part_ml = in.part_ml;
        a.D = L.Ap; a.G = s.kv_heads; a.R = in.rows; a.units = s.heads / in.rows; a.kv_group = s.heads / s.kv_heads / in.rows; a.nsplit = in.nsplit; a.ring = in.ring; a.chunk = in.chunk;
        a.dim = s.dim; a.vdim = s.vdim; a.half_a = s.rot_dims / 2; a.off_a = L.rot_a; a.s_mul = s.scale; a.softcap = s.softcap; a.out_mul = s.out_scale;
        a.att = a.units * in.nsplit;
        lds = f32 ? mix_lds32(L.Ap) : L.Ap == 64 ? mix_lds16<64>(in.rows) : mix_lds16<128>(in.rows);
        if (in.nsplit > 1) merge = (s.heads * (L.Ap / 64) + MIX_THREADS16 / 64 - 1) / (MIX_THREADS16 / 64);
    }
    const int ret_lds = L.retention() ? mix_ret_floats(L.Kp, L.Vp) * 4 : 0, heads_r = L.retention() ? r.heads : 0;
    if (L.retention()) {
        a.ao_r = (char*)in.ao + (size_t)L.off_r * lm.esz(); a.half_r = r.rot_dims / 2; a.off_r = L.rot_r; a.k_scale = r.k_scale;
        a.ret_head = RetHead{in.state, L.pw, r.heads, L.Kp, L.Vp, r.vdim, lm.d.eps, r.out_scale};
    }
    if (!merge) {
        a.ret = heads_r;
        return launch_mix_part(f32, L.Kp, a, 0, std::max(lds, ret_lds), st);
    }
    // rows of several splits: retention goes with the merge, so that two launches do
    CR_TRY(launch_mix_part(f32, L.Kp, a, 0, lds, st));
    a.att = 0; a.ret = heads_r; a.merge = 1; a.ahead.n = 0;
    return launch_mix_part(f32, L.Kp, a, merge, ret_lds, st);
}
