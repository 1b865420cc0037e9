// amx_device.hpp -- device helpers shared by the kernels (HIP sources only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "amx_solver.hpp"

namespace amx {

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
// b % 8).  Return a logical block index such that XCD x gets the contiguous
// logical range [x*q + min(x, r), ... + q + (x < r)), q = nb / 8, r = nb % 8.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb)
{
    const uint32_t x = b & 7u, i = b >> 3;
    const uint32_t q = nb >> 3, r = nb & 7u;
    return x * q + (x < r ? x : r) + i;
}

// index of the entry that owns work item x: the largest j < n with prefix[j] <= x
// (x wave-uniform, every lane active).  The lanes compare 64 entries at once:
// one memory latency for up to 64 jobs, where a binary search took log2(n).
__device__ __forceinline__ uint32_t job_of(const uint32_t* __restrict__ prefix, uint32_t n, uint32_t x)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = 0, cnt = n;
    while (cnt > 64u) {
        const uint32_t step = (cnt + 63u) / 64u, i = lane * step;
        const bool le = i < cnt && prefix[lo + min(i, cnt - 1u)] <= x;
        const uint32_t k = (uint32_t)__popcll(__ballot(le)) - 1u;
        lo += k * step;
        cnt = min(step, cnt - k * step);
    }
    const bool le = lane < cnt && prefix[lo + min(lane, cnt - 1u)] <= x;
    return __builtin_amdgcn_readfirstlane(lo + (uint32_t)__popcll(__ballot(le)) - 1u);
}

// ---- deterministic reductions over the blocks of a launch ------------------
// The order is fixed: a tree over a block's 256 sums (stride 128, 64, ... 1), a
// tree over the sums of each 32 blocks (zero-padded), a tree over those sums.

// tree over sh[0..255]; called by the 64 threads of one wave (lane 0 has it)
__device__ __forceinline__ double block_tree(const double* sh)
{
    const uint32_t l = threadIdx.x & 63u;
    double x = (sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192]);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) x += __shfl_down(x, s, 64);
    return x;
}

__device__ __forceinline__ double tree32(double x)
{
    x += 0.0;  // the zero-padded strides above 32
#pragma unroll
    for (int s = 16; s > 0; s >>= 1) x += __shfl_down(x, s, 32);
    return x;
}

// totals of NV block sums that an earlier launch of nblk blocks left at
// part[k * kMaxRedBlocks + block]; every one of the caller's 256 threads gets
// them.  A launch that needs them sums them again in every block: the few
// loads and shuffles cost less than a last block that collects the sums behind
// atomics while the others have gone (cg_pq on 117 k DoFs 7.6 us, most of it
// that chain).  sh: NV * 32 doubles.
template <int NV>
__device__ __forceinline__ void block_totals(const double* part, uint32_t nblk, double* sh, double (&tot)[NV])
{
    constexpr uint32_t R = kMaxRedBlocks / 256u;
    const uint32_t tid = threadIdx.x & 255u;
    double v[NV][R];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t i = r * 256u + tid;
            const double x = part[k * kMaxRedBlocks + min(i, nblk - 1u)];
            v[k][r] = i < nblk ? x : 0.0;
        }
    const uint32_t ng = (nblk + 31u) / 32u;
#pragma unroll
    for (uint32_t r = 0; r < R; r++) {
        if (r * 256u >= nblk) break;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const double x = tree32(v[k][r]);
            const uint32_t g = r * 8u + tid / 32u;
            if ((tid & 31u) == 0u && g < ng) sh[k * 32 + g] = x;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t l = threadIdx.x & 31u;
        tot[k] = __shfl(tree32(l < ng ? sh[k * 32 + l] : 0.0), 0, 64);
    }
}

__device__ __forceinline__ void lds_sync_wave()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace amx
