// Weights that the launch behind this one reads, brought into the L2 cache that will be asked for them by workgroups of a launch that leaves compute units and memory idle.
//
// Only the L2 of the reading XCD counts: 32 MiB read again take 2.6 us less there than cold, after another XCD's read (in the memory-side cache) 0.8 less.  A workgroup's number modulo 8 is its XCD, so
// a workgroup of the consumer finds what one of the launch before with the same remainder has read.  What is fetched should be all that the consumer reads, even if it is a little more than
// the eight L2 caches hold (34 MB of wo, us of the launch with 0 / 64 / 96 / 128 KiB of every workgroup's 128: 8.0 / 6.4 / 5.5 / 4.8): its slowest workgroup counts.
#pragma once
#include "common.hpp"

// units of unit_bytes side by side, unit u read by workgroups whose numbers leave u % 8; fetched in pieces (of a multiple of 16 bytes), a workgroup each.  at null: nothing
struct L2Ahead { const void* at; int units, unit_bytes, pieces; };
constexpr int L2_AHEAD_GROUPS = 256, L2_AHEAD_PIECES = 8, L2_AHEAD_MOST = 5;      // fetching workgroups, pieces of a unit, products of a list

// `bytes` of weights in `units` equal parts, or nothing where they cannot be cut so.  A power of two of pieces, as long as every fetching workgroup gets at most one.  (The count that just goes round, six for
// 40 units, cuts at odd addresses and leaves the rest of the division out.  Us a step without fetching / so / in powers of two: float32, 768 wide, 4 and 12 rows 289 / 301 / 282 and 326 / 347 / 328; 640 wide,
// 4 rows 257 / 270 / 250; bf16, 768 wide, 48 rows 369 / 383 / 371.)
inline L2Ahead l2_ahead_of(const void* at, int64_t bytes, int units) {
    if (!at || bytes <= 0 || units <= 0 || bytes % units || bytes / units % 16 || bytes / units > INT32_MAX) return {};
    L2Ahead a{at, units, (int)(bytes / units), 1};
    while (a.pieces < L2_AHEAD_PIECES && 2 * a.pieces * units <= L2_AHEAD_GROUPS && a.unit_bytes % (32 * a.pieces) == 0) a.pieces *= 2;
    return a;
}
inline int64_t l2_ahead_bytes(const L2Ahead& a) { return (int64_t)a.units * a.unit_bytes; }
// Whether wo's 34 MB go beside `own` workgroups of 256 keys each of the chat model's attention.  A step of four layers and the head with fetching over one without: 72 .. 2560 own 1.02 .. 1.04, 4096 (64 rows of
// 2000 keys) and 4608 1.01, 4992 and 5760 1.00, 6656 and 8192 (64 rows of 3164 and 3900) 0.99.
// Measured again, with rows of unequal length: profiles/read_ahead/chat.txt (up to 4608 1.01 .. 1.04, 5632 and 6656 1.01; 64 rows of 100 to 3164 keys, 6656 launched, 1.01).
inline bool l2_ahead_beside_attention(int64_t own, int cus) { return own <= 20 * cus; }
// Most bytes that go beside `own` workgroups of latent attention.  What the caches do not hold is read twice, and where every second CU has a workgroup of its own the two share its load path.  A step with
// fetching over one without, few experts, wo of 8 / 32 / 40 / 80 MiB: 1 .. 64 own 1.01 / 1.02 .. 1.05 / 1.04 / 0.98, 96 .. 128 1.01 / 1.00 / 1.02 / 0.96, 192 .. 256 1.00 / 0.98 / 0.99 / 0.94, 448 1.00 /
// 0.99 / 0.97 / 0.88 (235 MB of 128 heads 0.85 throughout).  Again, with rows of unequal length: profiles/read_ahead/latent.txt.
inline int64_t l2_ahead_beside_latent(int64_t own, int cus) { return (int64_t)(2 * own <= cus ? 40 : 8) << 20; }
// The same beside `own` workgroups of a decode mixer (lm_mix.hip), with how little it must be to go at all and how many products it may be.  A step with all that fits over one without (bf16 again, with rows of
// unequal length: profiles/read_ahead/mixer.txt):
//   bf16, one key split: up to 256 own 0.98 .. 1.07; 288 .. 960 0.95 .. 1.05 with 34 MiB, 0.97 .. 1.05 with 26; where all that there is are 7 MiB, 320 .. 512 0.97 .. 0.99.
//   Several splits (retention then streams its states through the caches before the weights' reader starts): up to 256 0.97 .. 1.05, 320 0.98 .. 1.04, 384 .. 1024 0.93 .. 1.03, mostly below one.
//   float32, whose workgroups have a CU each: up to 128 0.99 .. 1.04; 144 .. 192 0.95 .. 1.03, the first product alone 1.00 .. 1.03 (of 32 MiB 0.99 .. 1.02); 200 .. 256 0.95 .. 1.03 and 0.98 .. 1.03.
//   float32 with heads of 128 and more, by the bytes of keys and values that its workgroups read (profiles/read_ahead/float32_keys.txt): 2048 wide up to 26 MB 0.99 .. 1.03, 33 .. 164 (5 rows of 400 keys, 4 of 520
//   and more) 0.98 .. 1.00; 1024 wide, 14 passes, up to 26 MB 1.00 .. 1.05, 34 .. 131 0.99 .. 1.00.  Heads of 64 lose nothing by 98 MB (0.99 .. 1.06).
struct L2AheadRoom { int64_t most, least; int products; };
inline L2AheadRoom l2_ahead_beside_mixer(bool f32, int64_t own, int splits, int cus, int dim = 0, int64_t key_bytes = 0) {
    constexpr int64_t MiB = 1 << 20;
    if (f32 && dim >= 128 && key_bytes > 30 * MiB) return {};
    if (f32) return 2 * own <= cus ? L2AheadRoom{34 * MiB, 0, L2_AHEAD_MOST} : 4 * own <= 3 * cus ? L2AheadRoom{16 * MiB, 0, 1} : L2AheadRoom{};
    if (own <= cus) return {34 * MiB, 0, L2_AHEAD_MOST};
    return splits > 1 && 4 * own > 5 * cus ? L2AheadRoom{} : L2AheadRoom{26 * MiB, 8 * MiB, L2_AHEAD_MOST};
}
// A fetching workgroup takes pieces j = nth >> 3, then every L2_AHEAD_GROUPS / 8 further, of the units of its remainder: the offset of piece j's first byte, negative past the last unit
__host__ __device__ inline int64_t l2_ahead_piece(const L2Ahead& a, int linear, int j) {
    const int u = (linear & 7) + 8 * (j / a.pieces);
    return u < a.units ? (int64_t)u * a.unit_bytes + j % a.pieces * (a.unit_bytes / a.pieces) : -1;
}

// linear: the workgroup's number in its launch; nth: its number among those that do this (linear and nth alike modulo 8), < L2_AHEAD_GROUPS
__device__ __forceinline__ void l2_ahead(const L2Ahead& a, int linear, int nth) {
    typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;
    u32x4_t s = {0u, 0u, 0u, 0u};
    const int bytes = a.unit_bytes / a.pieces, step = (int)blockDim.x * 16;
    for (int j = nth >> 3; j < (a.units + 7) / 8 * a.pieces; j += L2_AHEAD_GROUPS / 8) {
        const int64_t off = l2_ahead_piece(a, linear, j);
        if (off < 0) break;
        const char* p = (const char*)a.at + off;
        for (int i = threadIdx.x * 16; i < bytes; i += 8 * step) {
            u32x4_t v[8];                                     // (past a short piece's end its last vector again; fewer loads there: 1024 wide, a row 440 us a step -> 451)
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = *(const u32x4_t*)(p + min(i + q * step, bytes - 16));
#pragma unroll
            for (int q = 0; q < 8; q++) s |= v[q];
        }
    }
    asm volatile("" ::"v"(s));                                // (the loads have a reader)
}

// several, one behind the other
struct L2AheadList {
    L2Ahead w[L2_AHEAD_MOST];
    int n;
};
__device__ __forceinline__ void l2_ahead(const L2AheadList& l, int linear, int nth) {
    for (int i = 0; i < l.n; i++) l2_ahead(l.w[i], linear, nth);
}
// workgroups behind the `groups` of a launch's own that make L2_AHEAD_GROUPS fetching ones, which start at a multiple of eight
inline int l2_ahead_extra(int groups) { return (groups + 7) / 8 * 8 - groups + L2_AHEAD_GROUPS; }
// number of workgroup `linear` among them (negative, or L2_AHEAD_GROUPS and more: none of them)
__host__ __device__ inline int l2_ahead_nth(int linear, int groups) { return linear - (groups + 7) / 8 * 8; }
