// The waits of the kernels that keep NBUF K-tiles in LDS with NBUF - 1 of them under way by LDS-DMA (gemm_mid.hip, lm_gemm_tiles.hip): one barrier a K-tile, counted vmcnt, never a drain
// before the last tiles.  A wave issues PER load instructions a K-tile, always (the counts are constants).  (The loop around them is each kernel's own: shared as a function over its
// lambdas it took 9 registers more, and a workgroup a CU with them.)
//   step t: wait until K-tile t + 1 has landed (this wave's pieces), barrier (everybody's have, and everybody holds tile t in registers), ask for tile t + NBUF into the buffer that tile t
//   leaves, read the fragments of t + 1, multiply t: the LDS reads' latency runs under the MFMAs.
#pragma once
#include "common.hpp"

template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// ... with `behind` <= R K-tiles of PER instructions left under way
template <int R, int PER> __device__ __forceinline__ void wait_tail(int behind) {
    if (behind >= R) wait_vm<R * PER>();
    else if constexpr (R > 0) wait_tail<R - 1, PER>(behind);
}

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
