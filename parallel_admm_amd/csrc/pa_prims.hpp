// Device primitives shared by the detector and the solver: fill, exclusive
// scan and a stable least-significant-digit radix sort of 32-bit keys with a
// 32-bit payload (8-bit digits, wave64 ballot ranking in LDS).
#pragma once

#include "pa_common.hpp"

namespace pa {

template <class T> __global__ void k_fill(T* __restrict__ p, T v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Kernel fill instead of hipMemsetAsync so the same code can sit in a captured graph.
template <class T> inline void fill(T* p, T v, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill<T>, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
    PA_LAUNCH_CHECK();
}

// Two fills in one launch: p[0..n) and q[0..m) = v.
template <class T> __global__ void k_fill2(T* __restrict__ p, int64_t n, T* __restrict__ q, int64_t m, T v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
    else if (i - n < m) q[i - n] = v;
}
template <class T> inline void fill2(T* p, int64_t n, T* q, int64_t m, T v, hipStream_t s) {
    if (n + m <= 0) return;
    hipLaunchKernelGGL(k_fill2<T>, dim3(grid_for(n + m, 256)), dim3(256), 0, s, p, n, q, m, v);
    PA_LAUNCH_CHECK();
}

// Rank of this lane's 8-bit digit d among the wave's equal digits of this and
// earlier calls (cnt: the wave's digit counts in LDS, updated); lanes with
// valid = false take no part.
__device__ inline uint32_t rs_rank(uint32_t d, bool valid, uint32_t* cnt) {
    unsigned long long match = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const bool bit = (d >> b) & 1u;
        const unsigned long long m = __ballot(bit);
        match &= bit ? m : ~m;
    }
    const uint32_t before = __builtin_amdgcn_mbcnt_hi((unsigned)(match >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)match, 0u));
    const uint32_t start = valid ? cnt[d] : 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // every lane reads before the first of its digit adds
    if (valid && before == 0) cnt[d] = start + (uint32_t)__popcll(match);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return start + before;
}

// Scratch for scan/sort; grown on demand.
struct PrimScratch {
    DBuf<uint32_t> sums, hist, keys_alt, vals_alt;
};

// out[i] = sum_{j<i} in[j]; if total != nullptr, *total (device) = sum of all.
// in and out are 16-byte aligned and may alias; total is outside both.  host3
// (pinned host memory, with total): the same launch also writes total[0..2]
// there, so the caller reads them after a stream synchronisation without a
// copy.
void scan_exclusive(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* total, PrimScratch& s, hipStream_t st,
                    uint32_t* host3 = nullptr);

// Sorts (keys, vals) by the low `bits` bits of keys, stably.  Result in keys/vals.
void radix_sort_pairs(uint32_t* keys, uint32_t* vals, int64_t n, int bits, PrimScratch& s, hipStream_t st);

} // namespace pa
