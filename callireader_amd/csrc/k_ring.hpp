// What the kernels share that keep NBUF K-tiles in LDS with up to NBUF - 1 of them under way by LDS-DMA (gemm_mid.hip, lm_gemm_tiles.hip): how a wave asks for a piece of a K-tile, and the waits.  One barrier a
// K-tile, counted vmcnt, never a drain before the last tiles.  A wave issues PER load instructions a K-tile, always (the counts are constants).  (The loop around them is each kernel's own: shared as a
// function over its lambdas it took 9 registers more, and a workgroup a CU with them.)
//   step t: wait until K-tile t + 1 has landed (this wave's pieces), barrier (everybody's have, and everybody holds tile t in registers), ask for tile t + NBUF into the buffer that tile t
//   leaves, read the fragments of t + 1, multiply t: the LDS reads' latency runs under the MFMAs.  (gemm_mid.hip with five buffers and more: tile t + NBUF - 1 into the buffer of t - 1, which everybody has
//   multiplied by then, so that no read has to have come back ahead of the barrier.)
#pragma once
#include "common.hpp"

template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// ... with `behind` <= R K-tiles of PER instructions left under way
template <int R, int PER> __device__ __forceinline__ void wait_tail(int behind) {
    if (behind >= R) wait_vm<R * PER>();
    else if constexpr (R > 0) wait_tail<R - 1, PER>(behind);
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"               // (m0 is a reserved register: nothing else in these kernels uses it)
// A piece, eight rows of 128 bytes, to LDS address dst + to, its addresses O bytes further on: the instruction's offset is added to both, so O is taken off the LDS one first, and dst + to >= O.  Inline asm,
// because the compiler lets every LDS read wait for all others while a load into LDS that it knows of is under way, and from the builtin a piece came with 64-bit sums, a copy of m0 and a branch on the lanes;
// the loops wait for its landing by hand.  All lanes are on before and after.  A piece's first row is the same for all lanes, so its address is a scalar one (base), a lane's own row and chunk 32 bits beyond (off).
template <int O> __device__ __forceinline__ void ring_ask(const char* base, unsigned off, unsigned dst, unsigned to) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%4" ::"v"(off), "s"(base), "s"(dst), "s"(to - O), "n"(O) : "m0", "scc", "memory");
}
// ... of which only some lanes are wanted
template <int O> __device__ __forceinline__ void ring_ask(const char* base, unsigned off, unsigned dst, unsigned to, uint64_t lanes) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_mov_b64 exec, %4\n\tglobal_load_lds_dwordx4 %0, %1 offset:%5\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(dst), "s"(to - O), "s"(lanes), "n"(O) : "m0", "scc", "memory");
}
// ... from rows that 32 bits do not reach from each other: a lane's whole address
template <int O> __device__ __forceinline__ void ring_ask_far(const char* at, unsigned dst, unsigned to, uint64_t lanes) {
    asm volatile("s_add_u32 m0, %1, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, off offset:%4\n\ts_mov_b64 exec, -1" ::"v"(at), "s"(dst), "s"(to - O), "s"(lanes), "n"(O) : "m0", "scc", "memory");
}
#pragma clang diagnostic pop

// K-tile t of nk has landed in every wave's pieces, and every wave holds tile t - 1 in registers
template <int NBUF, int PER> __device__ __forceinline__ void ring_arrive(int nk, int t) {
    const int behind = nk - 1 - t;                            // tiles after t: at most NBUF - 2 of them are under way
    if (behind >= NBUF - 2) wait_vm<(NBUF - 2) * PER>();
    else if constexpr (NBUF > 2) wait_tail<NBUF - 3, PER>(behind);
    __builtin_amdgcn_s_waitcnt(0xC07F);                       // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}
