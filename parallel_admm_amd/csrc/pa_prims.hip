// Scan and radix sort for gfx950 (wave64).
#include "pa_prims.hpp"

namespace pa {
namespace {

// Exclusive scan.  Up to SCAN_ONE values: one workgroup, one launch.  Above:
// two launches, k_scan_sums (each tile's sum) and k_scan_apply, where every
// tile adds up the sums before it (a few thousand values at most here, read by
// 1024 lanes) and scans itself.  Launches bound these scans, not bytes: the
// scans here are over 1e3 to 1e6 counts, and a launch costs 2-3 us and its
// dependent dispatch as much again; a recursive tile scan takes up to five.
constexpr int SCAN_BLOCK = 1024;
constexpr int SCAN_TILE = 4 * SCAN_BLOCK;
constexpr int SCAN_ONE = 16 * SCAN_BLOCK;

// Four consecutive values from i on, 0 past n (in is 16-byte aligned).
__device__ inline uint4 scan_load(const uint32_t* in, int64_t i, int64_t n) {
    if (i + 4 <= n) return *reinterpret_cast<const uint4*>(in + i);
    return make_uint4(i < n ? in[i] : 0u, i + 1 < n ? in[i + 1] : 0u, i + 2 < n ? in[i + 2] : 0u, 0u);
}
__device__ inline void scan_store(uint32_t* out, int64_t i, int64_t n, uint4 v) {
    if (i + 4 <= n) {
        *reinterpret_cast<uint4*>(out + i) = v;
        return;
    }
    if (i < n) out[i] = v.x;
    if (i + 1 < n) out[i + 1] = v.y;
    if (i + 2 < n) out[i + 2] = v.z;
}

// Block-wide exclusive scan of one value per thread (16 waves).
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh_wave, uint32_t* block_total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v; // inclusive scan inside the wave
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh_wave[wave] = x;
    __syncthreads();
    uint32_t base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / 64; w++) {
        if (w < wave) base += sh_wave[w];
        all += sh_wave[w];
    }
    *block_total = all;
    return base + x - v;
}

__device__ inline void scan_publish(uint32_t t, uint32_t* total, uint32_t* host3) {
    if (total) *total = t;
    if (host3) {
        host3[0] = t;
        host3[1] = total[1];
        host3[2] = total[2];
    }
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_one(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* total, uint32_t* host3) {
    __shared__ uint32_t sh_wave[SCAN_BLOCK / 64];
    const int64_t i0 = 16 * (int64_t)threadIdx.x;
    uint4 v[4];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = scan_load(in, i0 + 4 * k, n);
        sum += v[k].x + v[k].y + v[k].z + v[k].w;
    }
    uint32_t all;
    uint32_t ex = block_exclusive_scan(sum, sh_wave, &all); // its barrier: every load is done before a store
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint4 o = make_uint4(ex, ex + v[k].x, ex + v[k].x + v[k].y, ex + v[k].x + v[k].y + v[k].z);
        scan_store(out, i0 + 4 * k, n, o);
        ex = o.w + v[k].w;
    }
    if (threadIdx.x == 0) scan_publish(all, total, host3);
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_sums(const uint32_t* __restrict__ in, int64_t n, uint32_t* __restrict__ sums) {
    __shared__ uint32_t sh_wave[SCAN_BLOCK / 64];
    const uint4 v = scan_load(in, (int64_t)blockIdx.x * SCAN_TILE + 4 * (int64_t)threadIdx.x, n);
    uint32_t all;
    block_exclusive_scan(v.x + v.y + v.z + v.w, sh_wave, &all);
    if (threadIdx.x == 0) sums[blockIdx.x] = all;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_apply(const uint32_t* in, uint32_t* out, int64_t n, const uint32_t* __restrict__ sums,
                                                          uint32_t* total, uint32_t* host3) {
    __shared__ uint32_t sh_base[SCAN_BLOCK / 64], sh_wave[SCAN_BLOCK / 64];
    const int64_t i = (int64_t)blockIdx.x * SCAN_TILE + 4 * (int64_t)threadIdx.x;
    const uint4 v = scan_load(in, i, n);
    uint32_t before = 0;
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += SCAN_BLOCK) before += sums[b];
    uint32_t base, all;
    block_exclusive_scan(before, sh_base, &base);
    uint32_t ex = base + block_exclusive_scan(v.x + v.y + v.z + v.w, sh_wave, &all);
    scan_store(out, i, n, make_uint4(ex, ex + v.x, ex + v.x + v.y, ex + v.x + v.y + v.z));
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) scan_publish(base + all, total, host3);
}

// Histogram of one 8-bit digit per tile; hist is digit-major [256][ntiles].
constexpr int RS_BLOCK = 256;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_BLOCK * RS_ITEMS;

__global__ void __launch_bounds__(RS_BLOCK) k_rs_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                     uint32_t* __restrict__ hist, int ntiles) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RS_TILE;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        int64_t e = base + (int64_t)k * RS_BLOCK + threadIdx.x;
        if (e < n) atomicAdd(&h[(keys[e] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter of one tile.  Wave w takes the tile's w-th quarter in rounds of
// 64, so a wave ranks its elements by itself: 8 ballots find the lanes with the
// same digit, and a digit count per wave in LDS carries over the rounds.  Only
// then do the waves add up their counts: two barriers and 5-6 us a tile (with
// all waves on each round and a barrier between, 24 barriers and 8-15 us).
__global__ void __launch_bounds__(RS_BLOCK) k_rs_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                        uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int64_t n,
                                                        int shift, const uint32_t* __restrict__ offs, int ntiles) {
    constexpr int WV = RS_BLOCK / 64;
    __shared__ uint32_t cnt[WV][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t base0 = offs[(int64_t)tid * ntiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < WV; w++) cnt[w][tid] = 0;
    const int64_t first = (int64_t)blockIdx.x * RS_TILE + (int64_t)wave * (RS_TILE / WV) + lane;
    uint32_t key[RS_ITEMS], val[RS_ITEMS], pos[RS_ITEMS];
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        const int64_t e = first + 64 * k;
        key[k] = e < n ? kin[e] : 0u;
        val[k] = e < n ? vin[e] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) pos[k] = rs_rank((key[k] >> shift) & 255u, first + 64 * k < n, cnt[wave]);
    __syncthreads();
    uint32_t run = base0; // digit tid: where each wave's elements start
#pragma unroll
    for (int w = 0; w < WV; w++) {
        const uint32_t c = cnt[w][tid];
        cnt[w][tid] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++)
        if (first + 64 * k < n) {
            const uint32_t p = cnt[wave][(key[k] >> shift) & 255u] + pos[k];
            kout[p] = key[k];
            vout[p] = val[k];
        }
}

} // namespace

void scan_exclusive(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* total, PrimScratch& s, hipStream_t st, uint32_t* host3) {
    PA_CHECK(!host3 || total, PA_ERR_INVALID, "scan: host3 needs total");
    PA_CHECK(((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0, PA_ERR_INVALID, "scan: unaligned array");
    if (n <= SCAN_ONE) { // also n <= 0: the total is 0
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(SCAN_BLOCK), 0, st, in, out, n, total, host3);
        PA_LAUNCH_CHECK();
        return;
    }
    const int64_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    s.sums.reserve((size_t)tiles);
    hipLaunchKernelGGL(k_scan_sums, dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, st, in, n, s.sums.p);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, st, in, out, n, (const uint32_t*)s.sums.p, total, host3);
    PA_LAUNCH_CHECK();
}

void radix_sort_pairs(uint32_t* keys, uint32_t* vals, int64_t n, int bits, PrimScratch& s, hipStream_t st) {
    if (n <= 1) return;
    const int ntiles = (int)((n + RS_TILE - 1) / RS_TILE);
    s.keys_alt.reserve((size_t)n);
    s.vals_alt.reserve((size_t)n);
    s.hist.reserve((size_t)ntiles * 256);
    DBuf<uint32_t>& hist = s.hist;
    uint32_t *ka = keys, *va = vals, *kb = s.keys_alt.p, *vb = s.vals_alt.p;
    int passes = (bits + 7) / 8;
    for (int pss = 0; pss < passes; pss++) {
        const int shift = 8 * pss;
        hipLaunchKernelGGL(k_rs_hist, dim3(ntiles), dim3(RS_BLOCK), 0, st, ka, n, shift, hist.p, ntiles);
        PA_LAUNCH_CHECK();
        scan_exclusive(hist.p, hist.p, (int64_t)ntiles * 256, nullptr, s, st);
        hipLaunchKernelGGL(k_rs_scatter, dim3(ntiles), dim3(RS_BLOCK), 0, st, ka, va, kb, vb, n, shift, hist.p, ntiles);
        PA_LAUNCH_CHECK();
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    if (ka != keys) {
        PA_HIP(hipMemcpyAsync(keys, ka, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
        PA_HIP(hipMemcpyAsync(vals, va, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
    }
}

} // namespace pa
