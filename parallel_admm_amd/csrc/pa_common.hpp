// Shared host/device helpers for the gfx950 backend: error propagation,
// RAII device buffers, small vector math.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

#include "pa_admm.h"

namespace pa {

// Internal errors carry a pa_status; the C ABI converts them to return codes.
struct Error : std::runtime_error {
    pa_status code;
    Error(pa_status c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define PA_HIP(call)                                                                                          \
    do {                                                                                                      \
        hipError_t e_ = (call);                                                                               \
        if (e_ != hipSuccess)                                                                                 \
            throw ::pa::Error(PA_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_) + " (" __FILE__ ":" + \
                                              std::to_string(__LINE__) + ")");                                \
    } while (0)

#define PA_CHECK(cond, code, msg)                                                                             \
    do {                                                                                                      \
        if (!(cond)) throw ::pa::Error((code), (msg));                                                        \
    } while (0)

#define PA_LAUNCH_CHECK() PA_HIP(hipGetLastError())

// Device buffer owning `n` elements of T.
template <class T> struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    DBuf() = default;
    explicit DBuf(size_t count) { alloc(count); }
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept : p(o.p), n(o.n) {
        o.p = nullptr;
        o.n = 0;
    }
    DBuf& operator=(DBuf&& o) noexcept {
        if (this != &o) {
            release();
            p = o.p;
            n = o.n;
            o.p = nullptr;
            o.n = 0;
        }
        return *this;
    }
    ~DBuf() { release(); }
    // A failed allocation leaves an empty buffer (n is set by a successful one
    // only), so a later reserve() tries again.
    void alloc(size_t count) {
        release();
        if (!count) return;
        T* q = nullptr;
        PA_HIP(hipMalloc(&q, sizeof(T) * count));
        p = q;
        n = count;
    }
    // Grow-only reallocation (contents not preserved).
    void reserve(size_t count) {
        if (count > n) alloc(count);
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    // Copies from pageable host memory and waits, so the caller may free or
    // reuse `h` on return (uploads happen at set-up and on state transfers).
    void upload(const T* h, size_t count, hipStream_t s) {
        PA_CHECK(count <= n, PA_ERR_INVALID, "upload larger than buffer");
        if (count) {
            PA_HIP(hipMemcpyAsync(p, h, sizeof(T) * count, hipMemcpyHostToDevice, s));
            PA_HIP(hipStreamSynchronize(s));
        }
    }
    void upload(const std::vector<T>& h, hipStream_t s) {
        reserve(h.size());
        upload(h.data(), h.size(), s);
    }
    void download(T* h, size_t count, hipStream_t s) const {
        PA_CHECK(count <= n, PA_ERR_INVALID, "download larger than buffer");
        if (count) PA_HIP(hipMemcpyAsync(h, p, sizeof(T) * count, hipMemcpyDeviceToHost, s));
    }
    void zero(hipStream_t s) {
        if (n) PA_HIP(hipMemsetAsync(p, 0, sizeof(T) * n, s));
    }
};

inline int grid_for(int64_t n, int block) { return (int)((n + block - 1) / block); }

} // namespace pa

// ---------------------------------------------------------------------------
// float3 math (device and host)
// ---------------------------------------------------------------------------
__host__ __device__ inline float3 f3(float x, float y, float z) { return make_float3(x, y, z); }
__host__ __device__ inline float3 operator+(float3 a, float3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
__host__ __device__ inline float3 operator-(float3 a, float3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
__host__ __device__ inline float3 operator*(float s, float3 a) { return f3(s * a.x, s * a.y, s * a.z); }
__host__ __device__ inline float dot3(float3 a, float3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ inline float3 ld3(const float* p, int64_t i) { return f3(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
__device__ inline void st3(float* p, int64_t i, float3 v) {
    p[3 * i] = v.x;
    p[3 * i + 1] = v.y;
    p[3 * i + 2] = v.z;
}

// double3 math: positions and velocities are kept in FP64, so differences of
// nearby positions (edge vectors, per-step displacements) carry full FP32
// precision relative to their own size when rounded.
__host__ __device__ inline double3 d3(double x, double y, double z) { return make_double3(x, y, z); }
__host__ __device__ inline double3 operator+(double3 a, double3 b) { return d3(a.x + b.x, a.y + b.y, a.z + b.z); }
__host__ __device__ inline double3 operator-(double3 a, double3 b) { return d3(a.x - b.x, a.y - b.y, a.z - b.z); }
__host__ __device__ inline double3 operator*(double s, double3 a) { return d3(s * a.x, s * a.y, s * a.z); }
__device__ inline double3 ld3(const double* p, int64_t i) { return d3(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
__device__ inline void st3(double* p, int64_t i, double3 v) {
    p[3 * i] = v.x;
    p[3 * i + 1] = v.y;
    p[3 * i + 2] = v.z;
}
__host__ __device__ inline float3 to_f3(double3 a) { return f3((float)a.x, (float)a.y, (float)a.z); }
__host__ __device__ inline double3 to_d3(float3 a) { return d3(a.x, a.y, a.z); }

// XCD-contiguous block numbering.  The dispatcher deals workgroups to the
// eight XCDs round-robin (workgroup b runs on XCD b % 8) and each XCD has its
// own L2, so with blockIdx.x as the work index every XCD would touch every
// part of the mesh.  This bijection of [0, gridDim.x) hands XCD x one
// contiguous range of logical blocks instead (XCD x holds q + (x < r) of the
// grid's workgroups, q = grid / 8, r = grid % 8): neighbouring rows and
// queries, whose gathers share vertices and tree nodes, then share an L2.
__device__ inline int xcd_block() {
    const int g = (int)gridDim.x, b = (int)blockIdx.x;
    const int q = g >> 3, r = g & 7, x = b & 7, k = b >> 3;
    return x * q + min(x, r) + k;
}

// Chunked variant for grids whose work per block differs along the grid (the
// element kernels: triangles, then cheaper bending rows): rounds of 8 C
// logical blocks, each round dealt as 8 chunks of C consecutive blocks, chunk
// x to XCD x, so each XCD keeps C neighbouring blocks in its L2 and every XCD
// gets work from the whole grid.  Blocks past the last full round keep their
// index.  A bijection of [0, gridDim.x).
template <int C> __device__ inline int xcd_block_chunked() {
    const int g = (int)gridDim.x, b = (int)blockIdx.x;
    constexpr int R = 8 * C;
    if (b >= g / R * R) return b;
    const int j = b % R;
    return b - j + (j & 7) * C + (j >> 3);
}
