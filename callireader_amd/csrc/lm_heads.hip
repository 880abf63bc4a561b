// Attention over grouped heads and retention, the parts around their cores: one kernel turns a row of the fused input projection into normed, rotated queries and keys, cache rows
// and retention operands; a copy kernel fetches the cached start of a chunk; an attention kernel for any size and type (the matrix-core forms are in attention.hip).
//
// Row kernel: a wave takes 512 columns of one region, eight per lane.  A head's padded size is a power of two (64 .. 512), so a head is a run of lanes of one wave: its norm is a lane
// reduction, its rotation partner (half a rotation away, at any distance) comes through 2 KiB of the wave's own LDS.  Angles are fp32 and are computed once per row.
// Bound, in prompts, by vector issue before it is by memory: so what a region is -- its kind, whether it is normed or rotated -- is known to a wave in scalars and costs it a branch, regions
// that pass through unchanged (retention's values and gate of a prompt) have no waves, and a row's places are found by 32-bit divisions or none.  The next columns travel under the
// current ones.  8192 rows of 16 + 2 x 4 heads of 128 and retention's 8 of 128 + 256: 77.7 -> 55.4 us a layer.
#include <algorithm>
#include <climits>

#include "attention_plain.hpp"
#include "lm_heads.hpp"

namespace {

struct HeadsArgs {
    LmHeadsIn in;
    int M, Na, tasks;
    LmRegion reg[LM_REGIONS];                    // those with work, and the first of the 512-column tasks of each (INT_MAX: there are no more)
    int first[LM_REGIONS];
    float eps, k_scale;
    int dim, G, Ap, half_a, half_r;              // half a rotation's entries, 0 = no rotation
    const float *nq, *nk, *fq_a, *fq_r;          // nq null: no query / key norm
    int pad0, pad1, pad2, pad3, ldo;             // columns [pad0, pad1) and [pad2, pad3) of `ao` are padding
    int64_t rplane;                              // elements of one term of rq2 / rk2
};

template <typename T> struct Row8;                       // eight entries on their way
template <> struct Row8<bf16> {
    bf16x8 x;
    __device__ __forceinline__ void load(const bf16* p) { x = *(const bf16x8*)p; }
    __device__ __forceinline__ void get(float (&v)[8]) const {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (float)x[e];
    }
};
template <> struct Row8<float> {
    f32x4 a, b;
    __device__ __forceinline__ void load(const float* p) { a = *(const f32x4*)p; b = *(const f32x4*)(p + 4); }
    __device__ __forceinline__ void get(float (&v)[8]) const {
#pragma unroll
        for (int e = 0; e < 4; e++) { v[e] = a[e]; v[4 + e] = b[e]; }
    }
};

template <typename T>
__global__ __launch_bounds__(512) void lm_heads_kernel(const HeadsArgs p) {
    __shared__ __attribute__((aligned(16))) float cs[2][2][LM_MAX_HEAD / 2];      // [attention, retention][cos, sin][pair], read as 16-byte vectors
    extern __shared__ __attribute__((aligned(16))) float sx[];                    // 512 floats a wave
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x, waves = threads >> 6;
    const int64_t row = blockIdx.x;
    // task t's region; at: the lane's first column of it (past its end: none)
    auto region = [&](int t, int& at) -> LmRegion {
        int i = 0;
#pragma unroll
        for (int j = 1; j < LM_REGIONS; j++) i += t >= p.first[j];
        at = (t - p.first[i]) * 512 + lane * 8;
        return p.reg[i];
    };
    Row8<T> raw;
    auto fetch = [&](int t) {
        int at;
        if (t >= p.tasks) return;
        const LmRegion rg = region(t, at);
        if (at < rg.heads * rg.P) raw.load((const T*)p.in.a + row * p.in.lda + rg.off + at);
    };
    int t = blockIdx.y * waves + wave, next, at;
    if (!p.in.part) fetch(t);
    const int seq = p.in.ix.row_seq ? p.in.ix.row_seq[row] : p.in.ix.seqs[row];
    const int pos = p.in.ix.row_pos ? p.in.ix.row_pos[row] : p.in.ix.lens[seq];
    for (int i = tid; i < p.half_a + p.half_r; i += threads) {
        const bool r = i >= p.half_a;
        const int j = r ? i - p.half_a : i;
        float s, c;
        sincosf((float)pos * (r ? p.fq_r[j] : p.fq_a[j]), &s, &c);
        cs[r][0][j] = c; cs[r][1][j] = s;
    }
    if (blockIdx.y == 0) {
        T* ao = (T*)p.in.ao + row * p.ldo;
        for (int i = p.pad0 + tid; i < p.pad1; i += threads) ao[i] = (T)0.f;
        for (int i = p.pad2 + tid; i < p.pad3; i += threads) ao[i] = (T)0.f;
    }
    __syncthreads();
    // cache row of the token, < 0: not kept
    int64_t crow = -1;
    if (p.in.row_slot) {
        const int slot = p.in.row_slot[row];
        if (slot >= 0) crow = (int64_t)(slot / p.in.ring) * p.G * p.in.ring + slot % p.in.ring;
    } else crow = (int64_t)seq * p.G * p.in.ring + pos % p.in.chunk;
    for (; t < p.tasks; t = next) {
        next = t + gridDim.y * waves;
        const LmRegion rg = region(t, at);
        const bool in = at < rg.heads * rg.P, rq = rg.kind == LM_RQ || rg.kind == LM_RK;
        const int e0 = at & (rg.P - 1), here = at;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (!p.in.part) {
            if (in) raw.get(v);
            fetch(next);
        } else if (in)
            for (int k = 0; k < p.in.slices; k++) {
                float w[8];
                ld8<float>(p.in.part + ((int64_t)k * p.M + row) * p.Na + rg.off + here, w);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] += w[e];
            }
        HeadLane hl;
        hl.ask(e0, rg.kind == LM_Q ? p.nq : rg.kind == LM_K ? p.nk : nullptr, rg.kind == LM_Q || rg.kind == LM_K ? p.half_a : rq ? p.half_r : 0, cs[rq][0], cs[rq][1]);
        hl.apply(rg.P, p.dim, p.eps, &sx[wave * 512 + lane * 8], v);
        if (!in) continue;
        if (rg.kind == LM_Q) st8((T*)p.in.q + row * ((int64_t)rg.heads * rg.P) + here, v);
        else if (rg.kind == LM_K || rg.kind == LM_V) {
            if (p.in.kv) st8((T*)p.in.kv + ((int64_t)p.in.row_key[row] * 2 + (rg.kind == LM_V)) * p.G * p.Ap + here, v);
            if (crow >= 0) st8((T*)(rg.kind == LM_K ? p.in.cache_k : p.in.cache_v) + (crow + (int64_t)(here >> __builtin_ctz(rg.P)) * p.in.ring) * p.Ap + e0, v);
        } else if (rq) {
            if (rg.kind == LM_RK) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= p.k_scale;
            }
            const int64_t o = row * ((int64_t)rg.heads * rg.P) + here;
            if (p.in.rq2) {
                bf16* d = (rg.kind == LM_RQ ? p.in.rq2 : p.in.rk2) + o;
                float lo[8];
#pragma unroll
                for (int e = 0; e < 8; e++) lo[e] = v[e] - rbf(v[e]);
                st8(d, v);
                st8(d + p.rplane, lo);
            } else st8((rg.kind == LM_RQ ? p.in.rq : p.in.rk) + o, v);
        } else if (p.in.part) st8((T*)const_cast<void*>(p.in.a) + row * p.in.lda + rg.off + here, v);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void lm_prefix_kernel(const int32_t* __restrict__ key_rows, const int32_t* __restrict__ cache_rows, T* __restrict__ kv, const T* __restrict__ ck,
                                                        const T* __restrict__ cv, int G, int Ap, int ring) {
    const int64_t k = key_rows[blockIdx.x], slot = cache_rows[blockIdx.x];
    const int64_t crow = slot / ring * G * ring + slot % ring;
    for (int i = threadIdx.x * 8; i < G * Ap; i += 2048) {
        const int64_t src = (crow + (int64_t)(i / Ap) * ring) * Ap + i % Ap;
        float a[8], b[8];
        ld8<T>(ck + src, a);
        ld8<T>(cv + src, b);
        st8(kv + k * 2 * G * Ap + i, a);
        st8(kv + (k * 2 + 1) * G * Ap + i, b);
    }
}

template <typename T, int TPB>
__global__ __launch_bounds__(TPB) void heads_attn_plain_kernel(const HeadsAttnParams p) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ float red[PLAIN_RED];
    const int row = blockIdx.x, head = blockIdx.y;
    const int g = head / (p.H / p.G);
    const int seq = p.ix.row_seq ? p.ix.row_seq[row] : p.ix.seqs[row];
    const int n = (p.ix.row_pos ? p.ix.row_pos[row] : p.ix.lens[seq]) % p.chunk + 1;
    const int64_t base = p.row_key ? (int64_t)(p.row_key[row] - n + 1) * p.k_rs + g * p.k_hs : ((int64_t)seq * p.G + g) * p.ring * p.Ap;
    T* O = (T*)p.O + (int64_t)row * p.ldo + (int64_t)head * p.vdim;
    plain_attend<T, TPB>((const T*)p.Q + ((int64_t)row * p.H + head) * p.Ap, (const T*)p.K + base, p.k_rs, (const T*)p.V + base, p.k_rs, n, p.Ap, p.vdim, p.scale, p.softcap, sm, red,
                         [&](int i, float v) { O[i] = (T)(v * p.out_scale); });
}

template <typename T>
void launch_plain_t(const HeadsAttnParams& p, hipStream_t st) {
    // decode: few workgroups, sixteen waves each (a row's chain of loads is what counts); prompts: four, the chip is full.  The same bits either way.
    if (!p.ix.row_pos) hipLaunchKernelGGL((heads_attn_plain_kernel<T, 1024>), dim3(p.M, p.H), dim3(1024), plain_lds_floats(p.Ap, 1024) * 4, st, p);
    else hipLaunchKernelGGL((heads_attn_plain_kernel<T, 256>), dim3(p.M, p.H), dim3(256), plain_lds_floats(p.Ap, 256) * 4, st, p);
}

}  // namespace

int launch_lm_heads(bool f32, const Lm& lm, const LmLayer& L, int M, const LmHeadsIn& in, hipStream_t st) {
    const cr_lm_heads& a = L.s.attn;
    const cr_lm_retention& r = L.s.ret;
    HeadsArgs p{};
    p.in = in; p.M = M; p.Na = L.Na;
    int n = 0;
    std::fill(p.first, p.first + LM_REGIONS, INT_MAX);
    for (int i = 0; i < L.n_regions; i++) {
        const LmRegion& g = L.regions[i];
        if (!in.part && (g.kind == LM_RV || g.kind == LM_RG)) continue;      // (read where the projection left them)
        p.reg[n] = g;
        p.first[n++] = p.tasks;
        p.tasks += (g.heads * g.P + 511) / 512;
    }
    p.eps = lm.d.eps; p.k_scale = r.k_scale; p.G = a.kv_heads; p.Ap = L.Ap; p.dim = a.dim;
    p.half_a = L.heads() ? a.rot_dims / 2 : 0; p.half_r = L.retention() ? r.rot_dims / 2 : 0;
    p.nq = L.nq; p.nk = L.nc; p.fq_a = L.fq_a; p.fq_r = L.fq_r;
    p.pad0 = L.heads() ? a.heads * a.vdim : 0; p.pad1 = L.off_r; p.pad2 = L.off_r + (L.retention() ? r.heads * r.vdim : 0); p.pad3 = L.Gp; p.ldo = L.Gp;
    p.rplane = (int64_t)M * r.heads * L.Kp;
    if (!L.heads()) { p.in.ring = p.in.chunk = 1; }
    // Waves of a workgroup.  Up to 512 rows: four, the tasks beside each other in workgroups.  Then a row is one workgroup, angles computed once: a wave for every task (or every second ...,
    // eight at most) while such workgroups are resident at once, 22 waves a CU; then four while these are, and past that even shares of four waves' rounds, so that none stands by while
    // the last task runs (five or six tasks: three waves).  Two layers, four waves -> these: 700 rows, five tasks 7.2 -> 6.3 us, six 7.1 -> 6.4; 2000 rows, five 11.3 -> 9.9, six 12.1 -> 10.4
    // (a wave each: 13.0, 15.0); 1000 rows, six: 7.7 with four, 8.0 with three, 9.2 with six.
    constexpr int RESIDENT = 22 * 256;
    auto shared = [&](int most) { const int rounds = (p.tasks + most - 1) / most; return (p.tasks + rounds - 1) / rounds; };
    int waves = 4;
    if (M > 512) {
        if ((int64_t)M * shared(8) <= RESIDENT) waves = shared(8);
        else if ((int64_t)M * 4 > RESIDENT) waves = shared(4);
    }
    const int y = M <= 512 ? (p.tasks + 3) / 4 : 1;
    if (f32) hipLaunchKernelGGL(lm_heads_kernel<float>, dim3((unsigned)M, y), dim3(64 * waves), 2048 * waves, st, p);
    else hipLaunchKernelGGL(lm_heads_kernel<bf16>, dim3((unsigned)M, y), dim3(64 * waves), 2048 * waves, st, p);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

int launch_lm_prefix(bool f32, const LmLayer& L, int n, const int32_t* key_rows, const int32_t* cache_rows, void* kv, const void* cache_k, const void* cache_v, int ring, hipStream_t st) {
    if (n <= 0) return CR_OK;
    const int G = L.s.attn.kv_heads;
    if (f32) hipLaunchKernelGGL(lm_prefix_kernel<float>, dim3((unsigned)n), dim3(256), 0, st, key_rows, cache_rows, (float*)kv, (const float*)cache_k, (const float*)cache_v, G, L.Ap, ring);
    else hipLaunchKernelGGL(lm_prefix_kernel<bf16>, dim3((unsigned)n), dim3(256), 0, st, key_rows, cache_rows, (bf16*)kv, (const bf16*)cache_k, (const bf16*)cache_v, G, L.Ap, ring);
    CR_HIP(hipGetLastError());
    return CR_OK;
}

int launch_heads_attn_plain(bool f32, const HeadsAttnParams& p, hipStream_t st) {
    if (p.M <= 0 || p.H <= 0 || p.G <= 0 || p.H % p.G || p.Ap <= 0 || p.Ap > LM_MAX_HEAD || p.vdim > p.Ap || p.chunk <= 0)
        return cr_fail(CR_ERR_ARG, "attention over heads: rows %d, heads %d / %d, size %d / %d", p.M, p.H, p.G, p.Ap, p.vdim);
    if (f32) launch_plain_t<float>(p, st);
    else launch_plain_t<bf16>(p, st);
    CR_HIP(hipGetLastError());
    return CR_OK;
}
