/*
 * gf_sync.hpp -- the workgroup barrier of every kernel here.
 */
#ifndef GF_SYNC_HPP_
#define GF_SYNC_HPP_

namespace gf {

/* __syncthreads with this wave's LDS accesses done first.  Said in so many
 * words: the compiler (ROCm 7.2, AMD clang 22.0.0git 7b800a19) leaves the wait
 * out before some barriers that a loop's back edge or a long branch-free
 * stretch leads to, and another wave then reads the old words now and then
 * (k_advance_packed, whose six instances all have such barriers with a plain
 * __syncthreads, lost 17 of 4.2e6 slots).  Which kernels it strikes depends on
 * how their loops are laid out, so all of them use this; where the compiler's
 * own wait is there, it costs nothing. */
__device__ __forceinline__ void sync_lds() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
    __syncthreads();
}

} /* namespace gf */

#endif /* GF_SYNC_HPP_ */
