// ADMM time step on gfx950.
//
// One time step (reference ADMMImplGPU::step, src/solver/backend_gpu/admm_impl_gpu.cu:256-344,
// with damping kept in the matrix and the right-hand side as the CPU backend
// does, src/solver/backend_cpu/admm_impl_cpu.cpp:264-359):
//   prologue        k_begin_step (+ k_spmv_add for Damp x0)
//   per iteration   [detection every dcd_interval]
//                   [k_elem        z = prox(D x + Ue) per constraint (tri/tet/bend/pin in one launch), first iteration]
//                   k_vertex_p     p += Gamma r_c                       (contact on; p = (x - x0 + Uc)/h before)
//                   G x (k_contact_du, k_vertex_gather)                  (friction-cone sweeps;
//                                  up to 2048 contacts all of this in k_contact_sweeps_wg)
//                   k_rhs          b = M x~ + Damp x0 + h^2 D^T We^2 (z - Ue) + h^2 Wc (h p + x0 - Uc)
//                                  (and b - A x with the direct solve)
//                   global solve   A x = b: FP64 residual + FP32 correction (the direct factor, or PCG
//                                  with a smoothed-aggregation AMG V-cycle or Jacobi preconditioner)
//                   k_dual_vert    x += correction, Uc += x - x0 - h p, p = (x - x0 + Uc)/h (+ residual sums)
//                   k_elem         Ue += D x - z (+ residual sums), then z of the next iteration
//                   k_resid_final  residual check (the stop test on the device with the direct solve)
//   epilogue        k_end_step     v = (x - x0)/h
// D is applied matrix-free from the constraint rest data; D^T We^2 is a
// per-vertex gather (CSR over vertices) so every sum has a fixed order and the
// step is deterministic (the reference scatters p with float atomics,
// src/solver/contact_solver.cu:316-335).
#include "pa_backend.hpp"
#include "pa_chol.hpp"

#include <roctracer/roctx.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <limits>
#include <new>
#include <thread>
#include <type_traits>

namespace pa {
namespace {

constexpr int BLK = 256;
// Upper bound on the grid of kernels that emit per-block partial sums: every
// consumer block re-reduces all partials, so their number stays modest.
constexpr int CG_MAX_BLOCKS = 256;
// Block size of every kernel that writes or re-reduces the PCG partial sums.
constexpr int PBLK = 1024;

// Lanes per CSR row: about three entries per lane, so each lane's dependent
// gather chain is short and the wave has many rows in flight.
int lanes_per_row(int64_t nnz, int rows) {
    const double avg = rows > 0 ? (double)nnz / rows : 0.0;
    int l = 2;
    while (l < 32 && l * 3 < avg) l *= 2;
    return l;
}

template <class F> void with_lpr(int lpr, F&& f) {
    switch (lpr) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    default: f(std::integral_constant<int, 32>{}); break;
    }
}

// ---------------------------------------------------------------------------
// Block reduction of K doubles (fixed order -> identical result in every block).
// ---------------------------------------------------------------------------
// The partials go to slot `blk` (default blockIdx.x); kernels numbered by
// xcd_block() pass that, so the slots keep the logical block order.
template <int K, int NT = BLK>
__device__ inline void block_sum_write(double (&v)[K], double* __restrict__ part, int stride, int offset, int blk = -1) {
    __shared__ double sh[K][NT / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) {
        double s = v[k];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) sh[k][wave] = s;
    }
    __syncthreads();
    // thread k sums component k over the waves (same order in every block)
    if (threadIdx.x < K) {
        double s = 0;
#pragma unroll 1
        for (int w = 0; w < NT / 64; w++) s += sh[threadIdx.x][w];
        part[(size_t)(blk < 0 ? (int)blockIdx.x : blk) * stride + offset + threadIdx.x] = s;
    }
}

// Every block sums the same partials in the same order.
template <int K, int NT = BLK>
__device__ inline void block_reduce_parts(const double* __restrict__ part, int nparts, int stride, int offset, double (&out)[K],
                                          int3 npair = make_int3(1 << 30, 1 << 30, 1 << 30)) {
    __shared__ double sh[K][NT / 64];
    __shared__ double fin[K];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double v[K];
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = 0;
    // not unrolled: K accumulators per thread, and nparts <= NT in practice
    // component k counts the first npair[k / 2] parts (every part by default)
    const int lim[3] = {npair.x, npair.y, npair.z};
#pragma unroll 1
    for (int b = threadIdx.x; b < nparts; b += NT)
#pragma unroll
        for (int k = 0; k < K; k++)
            if (b < lim[min(k / 2, 2)]) v[k] += part[(size_t)b * stride + offset + k];
#pragma unroll
    for (int k = 0; k < K; k++) {
        double s = v[k];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) sh[k][wave] = s;
    }
    __syncthreads();
    if (threadIdx.x < K) {
        double s = 0;
#pragma unroll 1
        for (int w = 0; w < NT / 64; w++) s += sh[threadIdx.x][w];
        fin[threadIdx.x] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) out[k] = fin[k];
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Prologue / epilogue (reference do_integration_kernel / do_post_process_kernel,
// src/solver/jacobi_solver.cu:183-252).
// ---------------------------------------------------------------------------
// Positions and velocities are FP64: x~ = x0 + h v and v = (x - x0)/h are
// formed without the cancellation an FP32 position would carry.  bconst =
// M x~ + bpin, bpin holding the pins' targets (the pin rows of z are kept
// relative to the pin position).  p starts as the velocity on static vertices
// and as (x~ - x0 + Uc) / h, the first iteration's value, on dynamic ones.
__global__ void k_begin_step(int n_all, int n, double h, float hinv, double g, const uint8_t* __restrict__ pinned, double* __restrict__ x,
                             const double* __restrict__ v, double* __restrict__ x0, float* __restrict__ p, double* __restrict__ bconst,
                             const double* __restrict__ mass, const double* __restrict__ bpin, const float* __restrict__ Uc) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_all) return;
    const double3 xi = ld3(x, i);
    st3(x0, i, xi);
    double3 vi = ld3(v, i);
    if (i < n) {
        if (pinned[i]) vi = d3(0.0, 0.0, 0.0);
        else vi.y -= g * h;
        const double3 xt = xi + h * vi;
        st3(x, i, xt);
        const double mi = mass[i];
        bconst[3 * i] = mi * xt.x + bpin[3 * i];
        bconst[3 * i + 1] = mi * xt.y + bpin[3 * i + 1];
        bconst[3 * i + 2] = mi * xt.z + bpin[3 * i + 2];
        st3(p, i, hinv * (to_f3(xt - xi) + ld3(Uc, i)));
    } else {
        st3(p, i, to_f3(vi));
    }
}

// flag[0] |= 1 if any of x (3 n_all) or v (3 n_all) is not finite.
__global__ void k_nonfinite(int64_t m, const double* __restrict__ x, const double* __restrict__ v, uint32_t* __restrict__ flag) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    if (!isfinite(x[i]) || !isfinite(v[i])) atomicOr(flag, 1u);
}

__global__ void k_end_step(int n, double h, const double* __restrict__ x, const double* __restrict__ x0, double* __restrict__ v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double3 d = ld3(x, i) - ld3(x0, i);
    st3(v, i, d3(d.x / h, d.y / h, d.z / h));
}

// y += A x (full CSR, 3 interleaved columns), FP64
__global__ void k_spmv_add(int n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col, const double* __restrict__ val,
                           const double* __restrict__ xin, double* __restrict__ y) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s0 = 0, s1 = 0, s2 = 0;
    for (int e = ptr[i]; e < ptr[i + 1]; e++) {
        const double a = val[e];
        const int c = col[e];
        s0 += a * xin[3 * c];
        s1 += a * xin[3 * c + 1];
        s2 += a * xin[3 * c + 2];
    }
    y[3 * i] += s0;
    y[3 * i + 1] += s1;
    y[3 * i + 2] += s2;
}

// ---------------------------------------------------------------------------
// Elastic constraints: D x per constraint and the prox operators.
// Reference prox: TriProxFunctor (src/constraint/triangle_constraint_device.cu:111-201),
// TetProxFunctor (tetrahedral_constraint_device.cu:56-104), BendProxFunctor
// (bending_constraint_device.cu:31-78), PinProxFunctor (pin_constraint_device.cu:69-93).
// ---------------------------------------------------------------------------
struct ElemArgs {
    int n_tri, n_tet, n_bend, n_pin;
    int tri_row0, tet_row0, bend_row0, pin_row0;
    int blk_tri, blk_tet, blk_bend; // block offsets
    const int4* tri_v;
    const float4* tri_binv;
    const float* tri_w;
    const int4* tet_v;
    const float* tet_binv;
    const float* tet_w;
    const int32_t* bend_ptr;
    const int32_t* bend_idx;
    const float* bend_coef;
    const double* bend_sum; // FP64 row sum of each bending row's coefficients
    const float* bend_w;
    const int32_t* pin_v;
    const double* pin_pos; // 3 per pin
    const float* pin_w;
};

// Maps (block, thread) to (type, constraint index).  type: 0 tri, 1 tet, 2 bend, 3 pin, -1 none.
__device__ inline int elem_of(const ElemArgs& a, int* c) {
    const int b = xcd_block_chunked<32>(); // neighbouring elements share vertices: one L2 per chunk
    if (b < a.blk_tri) {
        *c = b * BLK + threadIdx.x;
        return *c < a.n_tri ? 0 : -1;
    }
    if (b < a.blk_tet) {
        *c = (b - a.blk_tri) * BLK + threadIdx.x;
        return *c < a.n_tet ? 1 : -1;
    }
    if (b < a.blk_bend) {
        *c = (b - a.blk_tet) * BLK + threadIdx.x;
        return *c < a.n_bend ? 2 : -1;
    }
    *c = (b - a.blk_bend) * BLK + threadIdx.x;
    return *c < a.n_pin ? 3 : -1;
}

// D x for constraint c of type TYPE: ELEM_ROWS<TYPE> rows into dx[]; returns the
// first row.  Edge vectors and the bending sum are formed from the FP64
// positions and rounded once.  A pin row is kept relative to its target:
// dx = x_v - pin position (its z is 0, and the target enters the right-hand
// side through bpin), so no FP32 value holds an absolute position.
template <int TYPE> constexpr int ELEM_ROWS = TYPE == 0 ? 2 : TYPE == 1 ? 3 : 1;
template <int TYPE>
__device__ inline int elem_dx(const ElemArgs& a, int c, const double* __restrict__ x, float3 (&dx)[ELEM_ROWS<TYPE>], float* w) {
    if constexpr (TYPE == 0) {
        int4 t = a.tri_v[c];
        float4 B = a.tri_binv[c]; // row-major 2x2
        *w = a.tri_w[c];
        const double3 xa = ld3(x, t.x);
        const float3 e1 = to_f3(ld3(x, t.y) - xa), e2 = to_f3(ld3(x, t.z) - xa);
        dx[0] = B.x * e1 + B.z * e2;
        dx[1] = B.y * e1 + B.w * e2;
        return a.tri_row0 + 2 * c;
    } else if constexpr (TYPE == 1) {
        int4 t = a.tet_v[c];
        const float* B = a.tet_binv + 9 * c; // row-major 3x3
        *w = a.tet_w[c];
        const double3 xa = ld3(x, t.x);
        const float3 e1 = to_f3(ld3(x, t.y) - xa), e2 = to_f3(ld3(x, t.z) - xa), e3 = to_f3(ld3(x, t.w) - xa);
#pragma unroll
        for (int r = 0; r < 3; r++) dx[r] = (B[r] * e1 + B[3 + r] * e2) + B[6 + r] * e3;
        return a.tet_row0 + 3 * c;
    } else if constexpr (TYPE == 2) {
        // sum_e coef_e x_e = sum_e coef_e (x_e - x_ref) + (sum_e coef_e) x_ref with
        // the row sum in FP64: the FP32 coefficients then multiply only
        // differences of nearby positions.  The ring is read four entries at a
        // time (a padded entry has coefficient 0 and the reference vertex).
        const int e0 = a.bend_ptr[c], e1 = a.bend_ptr[c + 1];
        *w = a.bend_w[c];
        const int ref = e1 > e0 ? a.bend_idx[e0] : 0;
        const double3 xr = e1 > e0 ? ld3(x, ref) : d3(0.0, 0.0, 0.0);
        double3 s = a.bend_sum[c] * xr;
        for (int e = e0 + 1; e < e1; e += 4) {
            int id[4];
            float cf[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                id[u] = e + u < e1 ? a.bend_idx[e + u] : ref;
                cf[u] = e + u < e1 ? a.bend_coef[e + u] : 0.f;
            }
            double3 q[4];
#pragma unroll
            for (int u = 0; u < 4; u++) q[u] = ld3(x, id[u]);
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (e + u < e1) s = s + (double)cf[u] * (q[u] - xr);
        }
        dx[0] = to_f3(s);
        return a.bend_row0 + c;
    } else {
        *w = a.pin_w[c];
        dx[0] = to_f3(ld3(x, a.pin_v[c]) - ld3(a.pin_pos, c));
        return a.pin_row0 + c;
    }
}

// Stiefel polar factor of F = [y0 y1] (3x2): P = F (F^T F)^{-1/2}, using the
// closed-form square root of a 2x2 SPD matrix C: sqrt(C) = (C + sI)/t with
// s = sqrt(det C), t = sqrt(tr C + 2s).
__device__ inline void prox_tri(float3& y0, float3& y1) {
    float a = dot3(y0, y0), b = dot3(y0, y1), c = dot3(y1, y1);
    float s = sqrtf(fmaxf(a * c - b * b, 0.f));
    float t = sqrtf(a + c + 2.f * s);
    float m00 = (a + s) / t, m01 = b / t, m11 = (c + s) / t;
    float det = m00 * m11 - m01 * m01;
    float i00 = m11 / det, i01 = -m01 / det, i11 = m00 / det;
    float3 p0 = i00 * y0 + i01 * y1;
    float3 p1 = i01 * y0 + i11 * y1;
    y0 = 0.5f * (p0 + y0);
    y1 = 0.5f * (p1 + y1);
}

// Closest rotation R to F = [y0 y1 y2]: cyclic Jacobi eigen-decomposition of
// F^T F (V sorted by descending eigenvalue, det V = +1), U by Gram-Schmidt of
// F V with u2 = u0 x u1, R = U V^T (det R = +1, so inverted elements map to
// the nearest rotation).
__device__ inline void prox_tet(float3& y0, float3& y1, float3& y2) {
    float F[3][3] = {{y0.x, y1.x, y2.x}, {y0.y, y1.y, y2.y}, {y0.z, y1.z, y2.z}};
    float A[3][3], V[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) A[i][j] = (F[0][i] * F[0][j] + F[1][i] * F[1][j]) + F[2][i] * F[2][j];
    for (int sweep = 0; sweep < 6; sweep++) {
#pragma unroll
        for (int pq = 0; pq < 3; pq++) {
            const int p = pq == 2 ? 1 : 0, q = pq == 0 ? 1 : 2;
            float apq = A[p][q];
            if (fabsf(apq) < 1e-30f) continue;
            float theta = (A[q][q] - A[p][p]) / (2.f * apq);
            float t = (theta >= 0.f ? 1.f : -1.f) / (fabsf(theta) + sqrtf(theta * theta + 1.f));
            float c = 1.f / sqrtf(t * t + 1.f), s = t * c;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                float akp = A[k][p], akq = A[k][q];
                A[k][p] = c * akp - s * akq;
                A[k][q] = s * akp + c * akq;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                float apk = A[p][k], aqk = A[q][k];
                A[p][k] = c * apk - s * aqk;
                A[q][k] = s * apk + c * aqk;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                float vkp = V[k][p], vkq = V[k][q];
                V[k][p] = c * vkp - s * vkq;
                V[k][q] = s * vkp + c * vkq;
            }
        }
    }
    // sort eigenpairs descending
    float w[3] = {A[0][0], A[1][1], A[2][2]};
    int o0 = 0, o1 = 1, o2 = 2;
    if (w[o0] < w[o1]) { int tq = o0; o0 = o1; o1 = tq; }
    if (w[o1] < w[o2]) { int tq = o1; o1 = o2; o2 = tq; }
    if (w[o0] < w[o1]) { int tq = o0; o0 = o1; o1 = tq; }
    float3 v0 = f3(V[0][o0], V[1][o0], V[2][o0]);
    float3 v1 = f3(V[0][o1], V[1][o1], V[2][o1]);
    float3 v2 = f3(V[0][o2], V[1][o2], V[2][o2]);
    float3 vc = f3(v0.y * v1.z - v0.z * v1.y, v0.z * v1.x - v0.x * v1.z, v0.x * v1.y - v0.y * v1.x);
    if (dot3(vc, v2) < 0.f) v2 = -1.f * v2;
    auto Fv = [&](float3 vv) {
        return f3((F[0][0] * vv.x + F[0][1] * vv.y) + F[0][2] * vv.z, (F[1][0] * vv.x + F[1][1] * vv.y) + F[1][2] * vv.z,
                  (F[2][0] * vv.x + F[2][1] * vv.y) + F[2][2] * vv.z);
    };
    auto unit = [](float3 u) {
        float q = dot3(u, u);
        if (q > 0.f) {
            float l = sqrtf(q);
            return f3(u.x / l, u.y / l, u.z / l);
        }
        return u;
    };
    float3 b0 = Fv(v0), b1 = Fv(v1);
    float3 u0 = unit(b0);
    float3 u1 = unit(b1 - dot3(u0, b1) * u0);
    float3 u2 = f3(u0.y * u1.z - u0.z * u1.y, u0.z * u1.x - u0.x * u1.z, u0.x * u1.y - u0.y * u1.x);
    // R[:, r] = sum_k u_k * v_k[r]
    float3 r0 = (v0.x * u0 + v1.x * u1) + v2.x * u2;
    float3 r1 = (v0.y * u0 + v1.y * u1) + v2.y * u2;
    float3 r2 = (v0.z * u0 + v1.z * u1) + v2.z * u2;
    y0 = 0.5f * (r0 + y0);
    y1 = 0.5f * (r1 + y1);
    y2 = 0.5f * (r2 + y2);
}

// The elastic part of the iterations, one pass over the constraints at a
// given x.  DUAL (the end of iteration k): Ue += D x - z, and with want_res the
// residual sums w^2 |Dx - z|^2 and w^2 |Dx|^2 into part[blk*6 + 0..1] (for a
// pin row |Dx|^2 is the absolute |x_v|^2, as D x = x_v in the residual's
// definition).  LOCAL (the start of iteration k + 1, at the same x):
// z = prox(D x + Ue), zprev <- the old z where it is wanted; a pin row's prox is
// its target, which is 0 in the relative form of elem_dx.  Both together read
// the constraint, its vertices, z and Ue once: 10.4 us per iteration at 256x256
// vertices against 22.7 + 21.2 us as two passes with a runtime row count.
enum { ELEM_DUAL = 1, ELEM_LOCAL = 2 };
template <int MODE, int TYPE>
__device__ inline void elem_pass(const ElemArgs& a, int c, bool keep, const double* __restrict__ x, float* __restrict__ Ue,
                                 float* __restrict__ z, float* __restrict__ zprev, double (&acc)[2]) {
    constexpr int NR = ELEM_ROWS<TYPE>;
    float3 dx[NR], u[NR], zz[NR];
    float w;
    const int row0 = elem_dx<TYPE>(a, c, x, dx, &w);
#pragma unroll
    for (int r = 0; r < NR; r++) {
        u[r] = ld3(Ue, row0 + r);
        if constexpr ((MODE & ELEM_DUAL) != 0) zz[r] = ld3(z, row0 + r);
    }
    if constexpr ((MODE & ELEM_DUAL) != 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const float3 d = dx[r] - zz[r];
            u[r] = u[r] + d;
            if (!keep) st3(Ue, row0 + r, u[r]);
            if ((MODE & ELEM_LOCAL) && zprev) st3(zprev, row0 + r, zz[r]);
            const double w2 = (double)w * (double)w;
            acc[0] += w2 * (((double)d.x * d.x + (double)d.y * d.y) + (double)d.z * d.z);
            const double3 da = TYPE == 3 ? ld3(x, a.pin_v[c]) : to_d3(dx[r]);
            acc[1] += w2 * ((da.x * da.x + da.y * da.y) + da.z * da.z);
        }
    }
    if constexpr ((MODE & ELEM_LOCAL) != 0) {
        float3 y[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) y[r] = dx[r] + u[r];
        if constexpr (TYPE == 0) prox_tri(y[0], y[1]);
        else if constexpr (TYPE == 1) prox_tet(y[0], y[1], y[2]);
        else if constexpr (TYPE == 2) y[0] = 0.5f * y[0];
        else y[0] = f3(0.f, 0.f, 0.f);
#pragma unroll
        for (int r = 0; r < NR; r++) st3(z, row0 + r, y[r]);
    }
}

template <int MODE>
__global__ void __launch_bounds__(BLK) k_elem(ElemArgs a, int want_res, const double* __restrict__ x, float* __restrict__ Ue,
                                              float* __restrict__ z, float* __restrict__ zprev, double* __restrict__ part,
                                              const int32_t* __restrict__ stop) {
    const bool keep = stop && stop[0]; // the iteration runs past the stop: Ue stays
    int c;
    const int type = elem_of(a, &c);
    double acc[2] = {0, 0};
    if (type == 0) elem_pass<MODE, 0>(a, c, keep, x, Ue, z, zprev, acc);
    else if (type == 1) elem_pass<MODE, 1>(a, c, keep, x, Ue, z, zprev, acc);
    else if (type == 2) elem_pass<MODE, 2>(a, c, keep, x, Ue, z, zprev, acc);
    else if (type == 3) elem_pass<MODE, 3>(a, c, keep, x, Ue, z, zprev, acc);
    if constexpr ((MODE & ELEM_DUAL) != 0)
        if (want_res) block_sum_write<2>(acc, part, 6, 0, xcd_block_chunked<32>());
}

// ---------------------------------------------------------------------------
// Contacts (reference src/solver/contact_solver.cu:90-431).
// ---------------------------------------------------------------------------
// Contact counts per vertex (all vertices), and each contact's place among its
// vertices' contacts (any order): what the detection's last kernel does itself
// within a step.
__global__ void k_contact_count(int nc, const int4* __restrict__ cv, uint32_t* __restrict__ cnt, int4* __restrict__ loc) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    int4 v = cv[c], l;
    l.x = (int)atomicAdd(&cnt[v.x], 1u);
    l.y = (int)atomicAdd(&cnt[v.y], 1u);
    l.z = (int)atomicAdd(&cnt[v.z], 1u);
    l.w = (int)atomicAdd(&cnt[v.w], 1u);
    loc[c] = l;
}

// The entries of dynamic vertices into their runs, unsorted (vraw), and per
// contact S_c = eps + sum_i b_i^2 w_i^-1 cnt_i; Gamma_ci = b_i / (S_c w_i); K_c = h^-1 h_cN gamma n
// with the contact's friction coefficient (that of its first vertex) in K.w; r_c = 0.
__global__ void k_contact_fill(int nc, int n, float eps, float gam, float hinv, const int4* __restrict__ cv, const int4* __restrict__ loc,
                               const uint32_t* __restrict__ vptr, uint32_t* __restrict__ vraw, const float4* __restrict__ bary,
                               const float4* __restrict__ nrm, const uint32_t* __restrict__ cnt, const float* __restrict__ wc,
                               const float* __restrict__ wc_inv, const float* __restrict__ mu_v, float4* __restrict__ G,
                               float4* __restrict__ K, float4* __restrict__ rc) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const int4 v = cv[c], l = loc[c];
    const int vs[4] = {v.x, v.y, v.z, v.w}, ls[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (vs[k] < n) vraw[vptr[vs[k]] + ls[k]] = (uint32_t)(4 * c + k);
    float4 b = bary[c];
    float Sc = eps;
    Sc += b.x * b.x * wc_inv[v.x] * (float)cnt[v.x];
    Sc += b.y * b.y * wc_inv[v.y] * (float)cnt[v.y];
    Sc += b.z * b.z * wc_inv[v.z] * (float)cnt[v.z];
    Sc += b.w * b.w * wc_inv[v.w] * (float)cnt[v.w];
    float4 g;
    g.x = v.x < n ? b.x / (Sc * wc[v.x]) : 0.f;
    g.y = v.y < n ? b.y / (Sc * wc[v.y]) : 0.f;
    g.z = v.z < n ? b.z / (Sc * wc[v.z]) : 0.f;
    g.w = v.w < n ? b.w / (Sc * wc[v.w]) : 0.f;
    G[c] = g;
    float4 nn = nrm[c];
    float s = hinv * nn.w * gam;
    K[c] = make_float4(s * nn.x, s * nn.y, s * nn.z, mu_v[v.x]);
    rc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Sorts every vertex's entries ascending (contact order, so that gathers sum in
// a fixed order), one lane per (contact, vertex): the entry's place is the
// number of smaller entries in its run.  vent gets the sorted entries, slot[c].k
// the place of (contact c, vertex k), -1 for static vertices, and erun[e]
// (vertex, end of its entries) on a vertex's first entry, (-1, 0) on the
// others.  Counting reads a run eight entries at a time (3.9 us at 256x256
// vertices); an insertion sort by one lane per vertex is a chain of dependent
// loads and stores over runs of 10 to 40 entries, 32-85 us per detection on
// single scenes.
__global__ void k_contact_rank(int nc, int n, const int4* __restrict__ cv, const uint32_t* __restrict__ vptr,
                               const uint32_t* __restrict__ vraw, uint32_t* __restrict__ vent, int32_t* __restrict__ slot,
                               int2* __restrict__ erun) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * nc) return;
    const int v = reinterpret_cast<const int32_t*>(cv)[i];
    if (v >= n) {
        slot[i] = -1;
        return;
    }
    const int begin = (int)vptr[v], end = (int)vptr[v + 1];
    int rank = 0;
    for (int q = begin; q < end; q += 8) {
        uint32_t k[8];
#pragma unroll
        for (int u = 0; u < 8; u++) k[u] = vraw[min(q + u, end - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++) rank += q + u < end && k[u] < (uint32_t)i ? 1 : 0;
    }
    const int e = begin + rank;
    vent[e] = (uint32_t)i;
    slot[i] = e;
    erun[e] = rank == 0 ? make_int2(v, end) : make_int2(-1, 0);
}

// p += Gamma r_c on the vertices with contacts (p holds (x - x0 + Uc) / h from
// k_begin_step or k_dual_vert), one lane per entry of the sorted list: the lane
// of a vertex's first entry sums its run in contact order, eight entries read
// at a time (160 merged cloths: 11.5 us, with four at a time 38).
__global__ void k_vertex_p(int ne_max, int n, float* __restrict__ p, const uint32_t* __restrict__ vptr, const int2* __restrict__ erun,
                           const uint32_t* __restrict__ vent, const float4* __restrict__ G, const float4* __restrict__ rc) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne_max) return;
    const int ne = (int)vptr[n];
    const int2 run = erun[e];
    if (e >= ne || run.x < 0) return;
    const float3 pv = ld3(p, run.x);
    float3 s = f3(0.f, 0.f, 0.f);
    for (int q = e; q < run.y; q += 8) {
        float gk[8];
        float4 d[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint32_t ent = vent[min(q + u, run.y - 1)];
            gk[u] = reinterpret_cast<const float*>(G)[ent]; // Gamma of (contact ent / 4, vertex ent % 4)
            d[u] = rc[ent >> 2];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (q + u < run.y) s = s + gk[u] * f3(d[u].x, d[u].y, d[u].z);
    }
    st3(p, run.x, pv + s);
}

// The friction-cone projection of one contact with barycentric weights b, its
// vertices' p values p0..p3, normal n4, K (the friction coefficient in K.w)
// and dual r4 (formula of ADMMImplCPU::_project_one_contact,
// admm_impl_cpu.cpp:411-448): returns du, the change of r_c.
__device__ __forceinline__ float3 contact_du_core(float4 b, float3 p0, float3 p1, float3 p2, float3 p3, float4 n4, float4 kk, float4 r4) {
    float3 u = f3(0.f, 0.f, 0.f);
    u = u + b.x * p0;
    u = u + b.y * p1;
    u = u + b.z * p2;
    u = u + b.w * p3;
    u = u + f3(kk.x, kk.y, kk.z);
    const float mu = kk.w;
    float3 r = f3(r4.x, r4.y, r4.z);
    float3 nn = f3(n4.x, n4.y, n4.z);
    float3 us = u - r;
    float uN = dot3(nn, us);
    float3 uT = us - uN * nn;
    if (uN < 0.f) {
        float tau = sqrtf(dot3(uT, uT));
        float alpha = -mu * uN;
        uN = 0.f;
        if (tau <= alpha) uT = f3(0.f, 0.f, 0.f);
        else uT = (1.f - alpha / tau) * uT;
    }
    float3 unew = uN * nn + uT;
    return unew - u;
}

// One Jacobi sweep of the friction-cone projection, one lane per contact.
__global__ void k_contact_du(int nc, const int4* __restrict__ cv, const float4* __restrict__ bary,
                             const float4* __restrict__ nrm, const float4* __restrict__ K, const float* __restrict__ p,
                             float4* __restrict__ rc, const float4* __restrict__ G, const int4* __restrict__ slot,
                             float4* __restrict__ gdu, const int32_t* __restrict__ stop) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const bool keep = stop && stop[0]; // the iteration runs past the stop: r_c stays
    const int4 v = cv[c];
    const float4 r = rc[c];
    const float3 d = contact_du_core(bary[c], ld3(p, v.x), ld3(p, v.y), ld3(p, v.z), ld3(p, v.w), nrm[c], K[c], r);
    if (!keep) rc[c] = make_float4(r.x + d.x, r.y + d.y, r.z + d.z, 0.f);
    // Gamma_k du goes straight into the entry slot of vertex k (dynamic
    // vertices only), so the per-vertex gather reads contiguous entries
    const float4 g = G[c];
    const int4 sl = slot[c];
    const float gk[4] = {g.x, g.y, g.z, g.w};
    const int sk[4] = {sl.x, sl.y, sl.z, sl.w};
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (sk[k] >= 0) gdu[sk[k]] = make_float4(gk[k] * d.x, gk[k] * d.y, gk[k] * d.z, 0.f);
}

// p_v += sum of the Gamma du entries of v (contact order), one lane per
// entry of the sorted list: the lane of a vertex's first entry sums its run,
// the others exit.  A run's entries are read eight at a time before they are
// added; one at a time the longest run, 30 and more entries, sets the kernel's
// time (9.9 us against 7.4 on a 256x256 cloth with a folded flap, 9.6 against
// 6.0 on 160 merged cloths).  Lanes past the entry count read stale (allocated) run
// markers beside the count and drop them.
__global__ void k_vertex_gather(int ne_max, int n, float* __restrict__ p, const uint32_t* __restrict__ vptr,
                                const int2* __restrict__ erun, const float4* __restrict__ gdu) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne_max) return;
    const int ne = (int)vptr[n];
    const int2 r = erun[e];
    if (e >= ne || r.x < 0) return;
    const float3 pv = ld3(p, r.x);
    float3 s = f3(0.f, 0.f, 0.f);
    for (int q = e; q < r.y; q += 8) {
        float4 g[8];
#pragma unroll
        for (int u = 0; u < 8; u++) g[u] = gdu[min(q + u, r.y - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (q + u < r.y) s = s + f3(g[u].x, g[u].y, g[u].z);
    }
    st3(p, r.x, pv + s);
}

// Every Jacobi sweep of one contact projection in a single 1024-lane
// workgroup, for contact sets of at most 1024 NPT contacts: the Gamma r_c term
// of k_vertex_p, then per sweep the update of k_contact_du and the gather of
// k_vertex_gather, with the same arithmetic in the same order (bit-identical
// results), separated by workgroup barriers instead of kernel boundaries.
// A projection is a chain of 2 sweeps dependent rounds on one CU, so what
// bounds it is a round's latency and instruction count.  What a round
// exchanges lives in LDS (through L2 a sweep took 4-7 us), what only its lane
// reads in registers:
// - lane t owns contacts t + 1024 k (k < NPT): weights, normal, K, Gamma, r_c
//   and the p of its static vertices;
// - a vertex's entries are one run of the sorted entry list; lane t owns runs
//   t + 1024 j and adds each one's entries, in order, to its vertex's p.  A
//   run is read eight entries at a time before they are added (the cap of a
//   draped cloth has runs of 30 and more, and a read per add was 2 us a
//   sweep);
// - buf holds one float4 per entry (Gamma_k du), then the p of each run.  Runs
//   that no longer fit behind the entries (only possible with over 1024
//   contacts, most of whose vertices are distinct) keep p in global memory.
// Ten sweeps (gs_max_iter 10), against everything through L2: a side-16 cloth
// draped over its sphere 17.1 us (36.6), cloth256 landing (about 600
// contacts) 27.8 (38-48), a side-95 cloth 24 (47) with up to 1024 contacts
// and 36 (68) above, where two contacts per lane spill 18 registers.
constexpr int CONTACT_WG_SLOTS = 10000;
template <int NPT>
__global__ void __launch_bounds__(1024) k_contact_sweeps_wg(int nc, int n, int sweeps, const int4* __restrict__ cv,
                                                            const float4* __restrict__ bary, const float4* __restrict__ nrm,
                                                            const float4* __restrict__ K, float* p, float4* __restrict__ rc,
                                                            const float4* __restrict__ G, const int4* __restrict__ slot,
                                                            const uint32_t* __restrict__ vptr, const int2* __restrict__ erun,
                                                            const int32_t* __restrict__ stop) {
    constexpr int EPT = 4 * NPT, NE = 1024 * EPT, SLOTS = NPT == 1 ? 2 * NE : CONTACT_WG_SLOTS;
    constexpr unsigned NONE = 0xffffu;
    __shared__ float4 buf[SLOTS];
    __shared__ int wsum[16];
    uint16_t* const map = reinterpret_cast<uint16_t*>(buf); // set-up: run number of a run-start entry,
    uint16_t* const first = map + NE;                       // and a run's first entry
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool keep = stop && stop[0]; // the iteration runs past the stop: r_c stays
    const int ne = (int)vptr[n];
    const int e0 = EPT * t;

    // contacts of this lane: what every sweep reads, once
    int4 v[NPT], sl[NPT];
    float4 b[NPT], n4[NPT], kk[NPT], g4[NPT], r4[NPT];
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int c = t + 1024 * k;
        const bool on = c < nc;
        v[k] = on ? cv[c] : make_int4(0, 0, 0, 0);
        sl[k] = on ? slot[c] : make_int4(-1, -1, -1, -1);
        b[k] = on ? bary[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        n4[k] = on ? nrm[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        kk[k] = on ? K[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        g4[k] = on ? G[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        r4[k] = on ? rc[c] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // number the runs: an exclusive scan of the run starts among each lane's EPT entries
    unsigned starts = 0;
#pragma unroll
    for (int j = 0; j < EPT; j++)
        if (e0 + j < ne && erun[e0 + j].x >= 0) starts |= 1u << j;
    int inc = __popc(starts);
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int rbase = inc - __popc(starts), nrun = 0;
    for (int w = 0; w < 16; w++) {
        if (w < wave) rbase += wsum[w];
        nrun += wsum[w];
    }
#pragma unroll
    for (int j = 0; j < EPT; j++)
        if (starts >> j & 1) {
            const int r = rbase + __popc(starts & ((1u << j) - 1));
            map[e0 + j] = (uint16_t)r;
            first[r] = (uint16_t)(e0 + j);
        }
    __syncthreads();
    const int pcap = SLOTS - ne; // runs whose p fits behind the entries
    // per contact vertex: its run and its entry (dynamic, two packed per
    // register) or its p (static)
    unsigned run[NPT][2], ent[NPT][2];
    float3 ps[NPT][4];
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int vk[4] = {v[k].x, v[k].y, v[k].z, v[k].w}, sk[4] = {sl[k].x, sl[k].y, sl[k].z, sl[k].w};
        unsigned rk[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            rk[q] = sk[q] >= 0 ? (unsigned)map[vptr[vk[q]]] : NONE;
            ps[k][q] = t + 1024 * k < nc && sk[q] < 0 ? ld3(p, vk[q]) : f3(0.f, 0.f, 0.f);
        }
        run[k][0] = rk[0] | rk[1] << 16;
        run[k][1] = rk[2] | rk[3] << 16;
        ent[k][0] = ((unsigned)sk[0] & NONE) | (unsigned)sk[1] << 16;
        ent[k][1] = ((unsigned)sk[2] & NONE) | (unsigned)sk[3] << 16;
    }
    auto half = [](const unsigned(&w)[2], int q) { return q & 1 ? w[q >> 1] >> 16 : w[q >> 1] & 0xffffu; };
    // this lane's runs: entries [se & 0xffff, se >> 16), empty where it has none
    unsigned se[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) {
        const int r = t + 1024 * j;
        se[j] = r < nrun ? (unsigned)first[r] | (unsigned)(r + 1 < nrun ? first[r + 1] : ne) << 16 : 0u;
    }
    __syncthreads();
    // entries hold (r_c, Gamma_k): p += Gamma r_c (k_vertex_p has written the rest of p)
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const float gk[4] = {g4[k].x, g4[k].y, g4[k].z, g4[k].w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const unsigned e = half(ent[k], q);
            if (e != NONE) buf[e] = make_float4(r4[k].x, r4[k].y, r4[k].z, gk[q]);
        }
    }
    __syncthreads();
    // s = the run's entries folded in order by add, eight read at a time
    auto sum_run = [&](unsigned w, auto add) {
        float3 s = f3(0.f, 0.f, 0.f);
        const int end = (int)(w >> 16);
        for (int e = (int)(w & 0xffffu); e < end; e += 8) {
            float4 g[8];
#pragma unroll
            for (int u = 0; u < 8; u++) g[u] = buf[e + u]; // past the run's end: other entries or p, dropped below
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float3 a = add(s, g[u]);
                if (e + u < end) s = a;
            }
        }
        return s;
    };
#pragma unroll
    for (int j = 0; j < EPT; j++) {
        const int r = t + 1024 * j;
        if (r >= nrun) break;
        const int vtx = erun[se[j] & 0xffffu].x;
        const float3 s = sum_run(se[j], [](float3 s, float4 g) { return s + g.w * f3(g.x, g.y, g.z); });
        const float3 pv = ld3(p, vtx) + s;
        if (r < pcap) buf[ne + r] = make_float4(pv.x, pv.y, pv.z, 0.f);
        else st3(p, vtx, pv);
    }
    __syncthreads();
    for (int sw = 0; sw < sweeps; sw++) {
#pragma unroll
        for (int k = 0; k < NPT; k++)
            if (t + 1024 * k < nc) {
                float3 pv[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int r = (int)half(run[k], q);
                    const float4 w = buf[ne + (r < pcap ? r : 0)];
                    pv[q] = f3(w.x, w.y, w.z);
                    if (r == (int)NONE) {
                        pv[q] = ps[k][q];
                    } else if (NPT > 1 && r >= pcap) {
                        const int4 vv = cv[t + 1024 * k];
                        pv[q] = ld3(p, q == 0 ? vv.x : q == 1 ? vv.y : q == 2 ? vv.z : vv.w);
                    }
                }
                const float3 d = contact_du_core(b[k], pv[0], pv[1], pv[2], pv[3], n4[k], kk[k], r4[k]);
                r4[k] = make_float4(r4[k].x + d.x, r4[k].y + d.y, r4[k].z + d.z, 0.f);
                const float gk[4] = {g4[k].x, g4[k].y, g4[k].z, g4[k].w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const unsigned e = half(ent[k], q);
                    if (e != NONE) buf[e] = make_float4(gk[q] * d.x, gk[q] * d.y, gk[q] * d.z, 0.f);
                }
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < EPT; j++) {
            const int r = t + 1024 * j;
            if (r >= nrun) break;
            const float3 s = sum_run(se[j], [](float3 s, float4 g) { return s + f3(g.x, g.y, g.z); });
            if (NPT == 1 || r < pcap) {
                const float4 w = buf[ne + r];
                buf[ne + r] = make_float4(w.x + s.x, w.y + s.y, w.z + s.z, 0.f);
            } else {
                const int vtx = erun[se[j] & 0xffffu].x;
                st3(p, vtx, ld3(p, vtx) + s);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < EPT; j++) {
        const int r = t + 1024 * j;
        if (r < nrun && r < pcap) {
            const float4 w = buf[ne + r];
            st3(p, erun[se[j] & 0xffffu].x, f3(w.x, w.y, w.z));
        }
    }
    if (!keep)
#pragma unroll
        for (int k = 0; k < NPT; k++)
            if (t + 1024 * k < nc) rc[t + 1024 * k] = r4[k];
}

// ---------------------------------------------------------------------------
// Warm start of the contact duals (no counterpart in the reference, whose
// duals restart from zero at every detection, contact_solver.cu:243).
// ---------------------------------------------------------------------------
__device__ inline bool key_less(int t0, int a0, int b0, int t1, int a1, int b1) {
    return t0 != t1 ? t0 < t1 : (a0 != a1 ? a0 < a1 : b0 < b1);
}

// The 10 features of contact c at the start of its window (definitions in
// pa_admm.h, pa_warm_start), the tangent t of the feature frame, and the index
// of the same contact (type, prim0, prim1) in the previous window's list,
// which is in the same canonical order, by binary search.
__global__ void k_ws_features(int nc, int n, int nprev, float h, float dhat, const int32_t* __restrict__ type,
                              const int32_t* __restrict__ prim0, const int32_t* __restrict__ prim1, const int4* __restrict__ cv,
                              const float4* __restrict__ bary, const float4* __restrict__ nrm, const float4* __restrict__ K,
                              const double* __restrict__ x, const double* __restrict__ x0, const float* __restrict__ Uc,
                              const float* __restrict__ p, const double* __restrict__ vel, const int32_t* __restrict__ ptype,
                              const int32_t* __restrict__ pp0, const int32_t* __restrict__ pp1, const float4* __restrict__ prc,
                              int normalise, const float* __restrict__ consts, float* __restrict__ feat, float* __restrict__ norm,
                              float4* __restrict__ tan, int32_t* __restrict__ match) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const float s = h / dhat, hinv = 1.f / h;
    const int4 v = cv[c];
    const float4 b = bary[c];
    const int vs[4] = {v.x, v.y, v.z, v.w};
    const float bs[4] = {b.x, b.y, b.z, b.w};
    const float4 k4 = K[c];
    float3 u = f3(k4.x, k4.y, k4.z), vr = f3(0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = vs[k];
        const float3 pk = i < n ? hinv * (to_f3(ld3(x, i) - ld3(x0, i)) + ld3(Uc, i)) : ld3(p, i);
        u = u + bs[k] * pk;
        vr = vr + bs[k] * to_f3(ld3(vel, i));
    }
    const float4 n4 = nrm[c];
    const float3 nn = f3(n4.x, n4.y, n4.z);
    const float un = dot3(nn, u);
    const float3 ut = u - un * nn;
    const float utn = sqrtf(dot3(ut, ut));
    float3 t;
    if (utn > 1e-30f) {
        t = (1.f / utn) * ut;
    } else { // n x (the axis of n's smallest component), normalised
        const float ax = fabsf(nn.x), ay = fabsf(nn.y), az = fabsf(nn.z);
        const float3 a = (ax <= ay && ax <= az) ? f3(1.f, 0.f, 0.f) : (ay <= az ? f3(0.f, 1.f, 0.f) : f3(0.f, 0.f, 1.f));
        const float3 cr = f3(nn.y * a.z - nn.z * a.y, nn.z * a.x - nn.x * a.z, nn.x * a.y - nn.y * a.x);
        t = (1.f / sqrtf(dot3(cr, cr))) * cr;
    }
    const float vn = dot3(nn, vr);
    const float3 vt = vr - vn * nn;
    const int kt = type[c], ka = prim0[c], kb = prim1[c];
    int lo = 0, hi = nprev;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (key_less(ptype[mid], pp0[mid], pp1[mid], kt, ka, kb)) lo = mid + 1;
        else hi = mid;
    }
    const int j = (lo < nprev && ptype[lo] == kt && pp0[lo] == ka && pp1[lo] == kb) ? lo : -1;
    float ln = 0.f, lt = 0.f;
    if (j >= 0) {
        const float4 r4 = prc[j];
        const float3 r = f3(r4.x, r4.y, r4.z);
        ln = s * dot3(nn, r);
        lt = s * dot3(t, r);
    }
    const float f[10] = {n4.w / dhat, s * un, s * utn, s * vn, s * sqrtf(dot3(vt, vt)), k4.w, (float)kt, j >= 0 ? 1.f : 0.f, ln, lt};
#pragma unroll
    for (int k = 0; k < 10; k++) {
        feat[(size_t)c * 10 + k] = f[k];
        if (normalise) norm[(size_t)c * 10 + k] = (f[k] - consts[k]) * consts[10 + k];
    }
    tan[c] = make_float4(t.x, t.y, t.z, 0.f);
    match[c] = j;
}

// Seeds r_c: mode 1 from the network outputs y (s lambda.n, s lambda.t after
// out_scale; non-finite -> 0, clamped), mode 2 the previous window's dual of
// the same contact.
__global__ void k_ws_seed(int nc, int mode, float inv_s, float clampv, const float* __restrict__ Y, const float* __restrict__ consts,
                          const float4* __restrict__ nrm, const float4* __restrict__ tan, const int32_t* __restrict__ match,
                          const float4* __restrict__ prc, float4* __restrict__ rc, float4* __restrict__ seed) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    float3 l = f3(0.f, 0.f, 0.f);
    if (mode == 1) {
        float a = Y[2 * (size_t)c] * consts[20], b = Y[2 * (size_t)c + 1] * consts[21];
        a = isfinite(a) ? fminf(fmaxf(a, -clampv), clampv) : 0.f;
        b = isfinite(b) ? fminf(fmaxf(b, -clampv), clampv) : 0.f;
        const float4 n4 = nrm[c], t4 = tan[c];
        l = inv_s * (a * f3(n4.x, n4.y, n4.z) + b * f3(t4.x, t4.y, t4.z));
    } else {
        const int j = match[c];
        if (j >= 0) {
            const float4 r = prc[j];
            l = f3(r.x, r.y, r.z);
        }
    }
    const float4 o = make_float4(l.x, l.y, l.z, 0.f);
    rc[c] = o;
    seed[c] = o;
}

// Judge of a seeded window: partial sums of |r_c - seed|^2 and |r_c|^2.
__global__ void __launch_bounds__(BLK) k_ws_judge(int nc, const float4* __restrict__ rc, const float4* __restrict__ seed,
                                                   double* __restrict__ part) {
    double acc[2] = {0.0, 0.0};
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += gridDim.x * blockDim.x) {
        const float4 r = rc[c], q = seed[c];
        const double dx = (double)r.x - q.x, dy = (double)r.y - q.y, dz = (double)r.z - q.z;
        acc[0] += dx * dx + dy * dy + dz * dz;
        acc[1] += (double)r.x * r.x + (double)r.y * r.y + (double)r.z * r.z;
    }
    block_sum_write<2>(acc, part, 2, 0);
}

// Log rows: the window's features, then s (r_c.n), s (r_c.t).
__global__ void k_ws_log(int nc, float s, const float* __restrict__ feat, const float4* __restrict__ rc, const float4* __restrict__ nrm,
                         const float4* __restrict__ tan, float* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    float* o = out + (size_t)c * 12;
#pragma unroll
    for (int k = 0; k < 10; k++) o[k] = feat[(size_t)c * 10 + k];
    const float4 r = rc[c], n4 = nrm[c], t4 = tan[c];
    o[10] = s * ((r.x * n4.x + r.y * n4.y) + r.z * n4.z);
    o[11] = s * ((r.x * t4.x + r.y * t4.y) + r.z * t4.z);
}

// System matrix rows for the residual of the global solve (off-diagonal CSR
// and diagonal, A = hi + lo), and where r goes: row i to place ipos[i].
struct ResidArgs {
    const int32_t* ptr;
    const int32_t* col;
    const float *val, *val_lo, *diag, *diag_lo;
    const double* x;
    float* r;
    const int32_t* ipos;
};

// b = bconst + sum_e coef_e (z - Ue)[row_e] + h^2 wc (h p + x0 - Uc), accumulated in FP64.
// With want_res, also |sum coef (z - zprev)|^2 and |sum coef z|^2 into part[blk*6 + 4..5],
// with the pins' targets (bpin) added back to z (and to z - zprev on the
// first iteration, where zprev is 0), as the pin rows of z are relative.
// LPR lanes share a vertex (each takes every LPR-th entry of its D^T row
// list, RU at a time) and combine with shuffles, so a vertex's dependent
// gathers of z and Ue are spread over LPR lanes.
// RESID (the direct solve): the row's residual r = b - A x in FP64 as well, so
// that b need not go through memory (store_b: later refinement passes read it).
// Both sums of a row are chains of dependent loads of like length; the matrix
// row's are issued first and its vertices arrive during the gather of z and Ue.
// At 256x256 vertices 31 us (checked, RES) against 21.7 + 12.7 us in two
// launches, at 16x16 5.8 against 4.9 + 9.4 (k_cg_resid64 also forms the norms
// that only PCG uses), on a 160-scene batch 134 against 110 + 77.  The matrix
// row is read ahead only without the residual sums: with them it would take
// 106 registers and half the waves.
constexpr int RU = 3;
template <int LPR, bool RESID, bool RES>
__global__ void __launch_bounds__(BLK) k_rhs(int n, float h, int contact, int first_iter, int store_b,
                                             const int32_t* __restrict__ dt_ptr,
                                             const int32_t* __restrict__ dt_row, const float* __restrict__ dt_coef,
                                             const float* __restrict__ z, const float* __restrict__ zprev, const float* __restrict__ Ue,
                                             const double* __restrict__ bconst, const double* __restrict__ wch2, const float* __restrict__ p,
                                             const double* __restrict__ x0, const float* __restrict__ Uc, const double* __restrict__ bpin,
                                             double* __restrict__ b, double* __restrict__ part, ResidArgs A) {
    // XCD-contiguous numbering: neighbouring vertices gather shared rows from one L2
    const int t = xcd_block() * blockDim.x + threadIdx.x;
    const int i = t / LPR, sub = t % LPR;
    constexpr bool AHEAD = RESID && !RES;
    double acc[2] = {0, 0};
    double s[3] = {0, 0, 0}, s1[3] = {0, 0, 0}, s2[3] = {0, 0, 0}, ax[3] = {0, 0, 0};
    if (i < n) {
        // entries ae .. of the matrix row, RU at a time: (value, x of its column)
        int ae = 0, ae1 = 0;
        double av[RU], xv[RU][3];
        auto a_load = [&]() {
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int e = ae + u * LPR;
                const int c = e < ae1 ? A.col[e] : i;
                av[u] = e < ae1 ? (double)A.val[e] + (double)A.val_lo[e] : 0.0;
#pragma unroll
                for (int a = 0; a < 3; a++) xv[u][a] = A.x[3 * c + a];
            }
        };
        if (RESID) {
            ae = A.ptr[i] + sub;
            ae1 = A.ptr[i + 1];
            if (AHEAD) a_load();
        }
        const int e1 = dt_ptr[i + 1];
        for (int e0 = dt_ptr[i] + sub; e0 < e1; e0 += RU * LPR) {
            int r[RU];
            double cf[RU];
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int e = e0 + u * LPR;
                r[u] = dt_row[min(e, e1 - 1)];
                cf[u] = e < e1 ? (double)dt_coef[e] : 0.0;
            }
            float zr[RU][3], ur[RU][3], pr[RU][3];
#pragma unroll
            for (int u = 0; u < RU; u++)
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    zr[u][a] = z[3 * r[u] + a];
                    ur[u][a] = Ue[3 * r[u] + a];
                    pr[u][a] = RES && !first_iter ? zprev[3 * r[u] + a] : 0.f;
                }
#pragma unroll
            for (int u = 0; u < RU; u++)
                if (e0 + u * LPR < e1)
#pragma unroll
                    for (int a = 0; a < 3; a++) {
                        s[a] += cf[u] * ((double)zr[u][a] - (double)ur[u][a]);
                        if (RES) {
                            s1[a] += cf[u] * ((double)zr[u][a] - (double)pr[u][a]);
                            s2[a] += cf[u] * (double)zr[u][a];
                        }
                    }
        }
        if (RESID)
            for (bool loaded = AHEAD; ae < ae1; ae += RU * LPR, loaded = false) {
                if (!loaded) a_load();
#pragma unroll
                for (int u = 0; u < RU; u++)
#pragma unroll
                    for (int a = 0; a < 3; a++) ax[a] += av[u] * xv[u][a];
            }
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1)
#pragma unroll
        for (int a = 0; a < 3; a++) {
            s[a] += __shfl_xor(s[a], o, LPR);
            if (RESID) ax[a] += __shfl_xor(ax[a], o, LPR);
            if (RES) {
                s1[a] += __shfl_xor(s1[a], o, LPR);
                s2[a] += __shfl_xor(s2[a], o, LPR);
            }
        }
    if (i < n && sub == 0) {
        const double wv = contact ? wch2[i] : 0.0;
        const double di = RESID ? (double)A.diag[i] + (double)A.diag_lo[i] : 0.0;
        const int64_t o = RESID ? A.ipos[i] : 0;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            double bi = bconst[3 * i + a] + s[a];
            if (wv != 0.0) bi += wv * (((double)h * p[3 * i + a] + x0[3 * i + a]) - (double)Uc[3 * i + a]);
            if (!RESID || store_b) b[3 * i + a] = bi;
            if (RESID) A.r[3 * o + a] = (float)(bi - (ax[a] + di * A.x[3 * i + a]));
        }
        if (RES) {
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const double bp = bpin[3 * i + a];
                s2[a] += bp;
                if (first_iter) s1[a] += bp;
            }
            acc[0] = (s1[0] * s1[0] + s1[1] * s1[1]) + s1[2] * s1[2];
            acc[1] = (s2[0] * s2[0] + s2[1] * s2[1]) + s2[2] * s2[2];
        }
    }
    if (RES) block_sum_write<2>(acc, part, 6, 4, xcd_block());
}

// Uc += x - x0 - h p; residual sums wc |x - x0 - h p|^2, wc |x - x0|^2 into part[blk*6 + 2..3].
// With dxg non-null the direct solve's last correction (in elimination order,
// vertex i at ipos[i]) is applied here first: x += dxg (what k_axpy_d would have
// done), then the dual update on the new x.  p becomes the next iteration's (x - x0 + Uc) / h.
__global__ void __launch_bounds__(BLK) k_dual_vert(int n, float h, float hinv, int contact, int want_res, double* __restrict__ x,
                                                   const double* __restrict__ x0, float* __restrict__ p, const double* __restrict__ wch2,
                                                   float* __restrict__ Uc, double* __restrict__ part, double h2inv,
                                                   const int32_t* __restrict__ stop, const float* __restrict__ dxg,
                                                   const int32_t* __restrict__ ipos) {
    const bool keep = stop && stop[0]; // the iteration runs past the stop: x and Uc stay
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[2] = {0, 0};
    if (i < n && dxg && !keep) {
        const int64_t o = ipos[i];
#pragma unroll
        for (int a = 0; a < 3; a++) x[3 * i + a] += (double)dxg[3 * o + a];
    }
    if (i < n && contact) {
        const float3 dx = to_f3(ld3(x, i) - ld3(x0, i));
        float3 d = dx - h * ld3(p, i);
        const float3 uc = ld3(Uc, i) + d;
        if (!keep) st3(Uc, i, uc);
        st3(p, i, hinv * (dx + uc));
        const double w = wch2[i] * h2inv;
        if (want_res && w != 0.0) {
            acc[0] = w * (((double)d.x * d.x + (double)d.y * d.y) + (double)d.z * d.z);
            acc[1] = w * (((double)dx.x * dx.x + (double)dx.y * dx.y) + (double)dx.z * dx.z);
        }
    }
    if (want_res) block_sum_write<2>(acc, part, 6, 2);
}

// Residual check of one ADMM iteration: out[0..5] the six sums, out[6] the
// primal residual sqrt(s0 + s2) / max(1, sqrt(s1 + s3)), out[7] the dual
// residual sqrt(s4) / max(1, sqrt(s5)).  With stop non-null, a residual
// max(r_p, r_d) <= tol sets stop[0] (the iterations enqueued after this one
// then leave the state alone), and a check after that leaves out untouched.
// Component pair q of the partials (0-1 k_elem, 2-3 k_dual_vert, 4-5
// k_rhs) is read from its kernel's first nq[q] blocks only, so the slots need
// no clearing between checks (the skipped slots would add zeros).
__global__ void __launch_bounds__(BLK) k_resid_final(const double* __restrict__ part, int3 nq, double* __restrict__ out, double tol,
                                                     int32_t* __restrict__ stop) {
    if (stop && stop[0]) return;
    double s[6];
    block_reduce_parts<6>(part, max(nq.x, max(nq.y, nq.z)), 6, 0, s, nq);
    if (threadIdx.x == 0) {
        for (int k = 0; k < 6; k++) out[k] = s[k];
        const double rp = sqrt(s[0] + s[2]) / fmax(1.0, sqrt(s[1] + s[3]));
        const double rd = sqrt(s[4]) / fmax(1.0, sqrt(s[5]));
        out[6] = rp;
        out[7] = rd;
        const double r = rp < rd ? rd : rp; // the host's std::max(rp, rd)
        if (stop && r <= tol) stop[0] = 1;
    }
}

// ---------------------------------------------------------------------------
// Preconditioned conjugate gradients on A = M + h^2 D^T We^2 D + h^2 Wc + Damp
// (replaces the fixed-count Jacobi sweeps of cu_jacobi_global,
// src/solver/jacobi_solver.cu:141-180).  Three right-hand sides (xyz) share
// each SpMV; FP32 vectors, FP64 dot products.  cg_state layout (two slots s,
// ping-pong by iteration parity): [s*8 + 0..2] rz, [s*8 + 3..5] done flags;
// [16..18] stop thresholds tol^2 |r_0|^2; [19] iterations; [20..22] |b|^2.
// ---------------------------------------------------------------------------
// Row groups: LPR consecutive lanes share one CSR row, each taking every
// LPR-th entry, and combine with shuffles (width LPR).  Many short dependent
// gather chains in flight instead of one long chain per lane.  Kernels that
// emit dot-product partials run on a fixed grid (grid-stride over rows) so the
// number of partials stays small for the redundant per-block reductions.
template <int LPR> __device__ inline float3 group_sum(float3 s) {
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) {
        s.x += __shfl_xor(s.x, o, LPR);
        s.y += __shfl_xor(s.y, o, LPR);
        s.z += __shfl_xor(s.z, o, LPR);
    }
    return s;
}

// Calls f(val, col) for the entries of row i that lane `sub` of the row group
// owns (every LPR-th), loading up to RU entries' column ids and values before
// any gather, so the row costs one chain of dependent loads
// (ptr -> col/val -> gathered vector) instead of one per entry.  Unused slots
// pass value 0 and column 0, an index every matrix here has (the row index
// would not do: the prolongators have more rows than columns).
template <int LPR, class F>
__device__ inline void row_foreach(int i, int rows, int sub, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                   const float* __restrict__ val, F&& f) {
    if (i >= rows) return;
    const int e1 = ptr[i + 1];
    for (int b = ptr[i] + sub; b < e1; b += RU * LPR) {
        int c[RU];
        float v[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            const int e = b + u * LPR;
            const bool ok = e < e1;
            c[u] = ok ? col[e] : 0;
            v[u] = ok ? val[e] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < RU; u++) f(v[u], c[u]);
    }
}

// sum_e val[e] * in[col[e]] over row r (lanes of the group split the entries)
template <int LPR> __device__ inline float3 row_dot(int r, int rows, int sub, const int32_t* __restrict__ ptr,
                                                    const int32_t* __restrict__ col, const float* __restrict__ val,
                                                    const float* __restrict__ in) {
    float3 s = f3(0.f, 0.f, 0.f);
    row_foreach<LPR>(r, rows, sub, ptr, col, val, [&](float v, int c) { s = s + v * ld3(in, c); });
    return group_sum<LPR>(s);
}

// Start of one refinement pass: r = b - A x with A = hi + lo and FP64
// accumulation (the exact residual of the FP64 iterate); the FP32 PCG for the
// correction d starts from d = 0 with r32 = r.  Partials: |b|^2 at 0..2,
// |r|^2 at 3..5.  With ipos (the direct solve) row i of r goes to place
// ipos[i], and d is left alone.
template <int LPR>
__global__ void __launch_bounds__(PBLK) k_cg_resid64(int n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                    const float* __restrict__ val, const float* __restrict__ val_lo,
                                                    const float* __restrict__ diag, const float* __restrict__ diag_lo,
                                                    const double* __restrict__ bvec, const double* __restrict__ x, float* __restrict__ r,
                                                    float* __restrict__ d, double* __restrict__ part, const int32_t* __restrict__ ipos) {
    const int sub = threadIdx.x % LPR;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int r0 = xcd_block() * (PBLK / LPR); r0 < n; r0 += gridDim.x * (PBLK / LPR)) {
        const int i = r0 + threadIdx.x / LPR;
        double ax[3] = {0, 0, 0};
        if (i < n) {
            const int e1 = ptr[i + 1];
            for (int b = ptr[i] + sub; b < e1; b += RU * LPR) {
                int c[RU];
                double a[RU];
#pragma unroll
                for (int u = 0; u < RU; u++) {
                    const int e = b + u * LPR;
                    const bool ok = e < e1;
                    c[u] = ok ? col[e] : 0;
                    a[u] = ok ? (double)val[e] + (double)val_lo[e] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < RU; u++) {
                    ax[0] += a[u] * x[3 * c[u]];
                    ax[1] += a[u] * x[3 * c[u] + 1];
                    ax[2] += a[u] * x[3 * c[u] + 2];
                }
            }
        }
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < 3; k++) ax[k] += __shfl_xor(ax[k], o, LPR);
        if (i < n && sub == 0) {
            const double di = (double)diag[i] + (double)diag_lo[i];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double bk = bvec[3 * i + k];
                const double rk = bk - (ax[k] + di * x[3 * i + k]);
                r[3 * (int64_t)(ipos ? ipos[i] : i) + k] = (float)rk;
                if (!ipos) d[3 * i + k] = 0.f;
                acc[k] += bk * bk;
                acc[3 + k] += rk * rk;
            }
        }
    }
    block_sum_write<6, PBLK>(acc, part, 9, 0);
}

// Jacobi preconditioner z = D^-1 r; partial r.z at 6..8.
__global__ void __launch_bounds__(PBLK) k_jacobi_prec(int n, const float* __restrict__ dinv, const float* __restrict__ r,
                                                     float* __restrict__ z, double* __restrict__ part) {
    double acc[3] = {0, 0, 0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float di = dinv[i];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float rk = r[3 * i + k], zk = di * rk;
            z[3 * i + k] = zk;
            acc[k] += (double)rk * zk;
        }
    }
    block_sum_write<3, PBLK>(acc, part, 9, 6);
}

// Pass state from the partials: rz, |b|^2 and the stop threshold
// tol^2 |r_0|^2 per column (|b|^2 when r_0 = 0); a column whose r_0 is zero
// is done at once.
__global__ void __launch_bounds__(PBLK) k_cg_init_state(const double* __restrict__ part, int nparts, double tol2,
                                                       double* __restrict__ st) {
    double s[9];
    block_reduce_parts<9, PBLK>(part, nparts, 9, 0, s);
    if (threadIdx.x == 0) {
        for (int k = 0; k < 3; k++) {
            st[k] = s[6 + k];
            st[16 + k] = tol2 * s[3 + k];
            st[20 + k] = s[k];
            st[3 + k] = (s[3 + k] <= 1e-24 * s[k] || s[3 + k] == 0.0) ? 1.0 : 0.0;
        }
        st[19] = 0;
    }
}

__global__ void k_copy(int64_t m, const float* __restrict__ a, float* __restrict__ b) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) b[i] = a[i];
}

// x += d, skipped once stop[0] is set (stop may be null).
__global__ void k_axpy_d(int n, const float* __restrict__ d, const int32_t* __restrict__ ipos, double* __restrict__ x,
                         const int32_t* __restrict__ stop) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n || (stop && stop[0])) return;
    x[i] += (double)(ipos ? d[3 * (int64_t)ipos[i / 3] + i % 3] : d[i]);
}

// q = A pd (off-diagonal CSR + diagonal); partial p.q at 0..2
template <int LPR>
__global__ void __launch_bounds__(PBLK) k_cg_spmv(int n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                 const float* __restrict__ val, const float* __restrict__ diag,
                                                 const float* __restrict__ pd, float* __restrict__ q, double* __restrict__ part) {
    const int sub = threadIdx.x % LPR;
    double acc[3] = {0, 0, 0};
    for (int r0 = xcd_block() * (PBLK / LPR); r0 < n; r0 += gridDim.x * (PBLK / LPR)) {
        const int i = r0 + threadIdx.x / LPR;
        float3 s = row_dot<LPR>(i, n, sub, ptr, col, val, pd);
        if (i < n && sub == 0) {
            const float3 pi = ld3(pd, i);
            s = s + diag[i] * pi;
            st3(q, i, s);
            acc[0] += (double)pi.x * s.x;
            acc[1] += (double)pi.y * s.y;
            acc[2] += (double)pi.z * s.z;
        }
    }
    block_sum_write<3, PBLK>(acc, part, 9, 0);
}

// alpha = rz / pq; d += alpha pd; r -= alpha q; partial |r|^2 at 3..5
__global__ void __launch_bounds__(PBLK) k_cg_update(int n, int slot, int nparts, const double* __restrict__ st_in,
                                                   const float* __restrict__ pd, const float* __restrict__ q, float* __restrict__ x,
                                                   float* __restrict__ r, double* __restrict__ part) {
    double pq[3];
    block_reduce_parts<3, PBLK>(part, nparts, 9, 0, pq);
    const double* s = st_in + slot * 8;
    float al[3];
    for (int k = 0; k < 3; k++) al[k] = (s[3 + k] != 0.0 || pq[k] == 0.0) ? 0.f : (float)(s[k] / pq[k]);
    double acc[3] = {0, 0, 0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float3 pi = ld3(pd, i), qi = ld3(q, i);
        float3 xi = ld3(x, i), ri = ld3(r, i);
        xi = f3(xi.x + al[0] * pi.x, xi.y + al[1] * pi.y, xi.z + al[2] * pi.z);
        ri = f3(ri.x - al[0] * qi.x, ri.y - al[1] * qi.y, ri.z - al[2] * qi.z);
        st3(x, i, xi);
        st3(r, i, ri);
        acc[0] += (double)ri.x * ri.x;
        acc[1] += (double)ri.y * ri.y;
        acc[2] += (double)ri.z * ri.z;
    }
    block_sum_write<3, PBLK>(acc, part, 9, 3);
}

// beta = rz_new / rz_old (rz at 6..8), done when |r|^2 (3..5) <= threshold;
// pd = zc + beta pd; block 0 advances the state slot.
__global__ void __launch_bounds__(PBLK) k_cg_dir(int n, int slot, int nparts, double* __restrict__ st,
                                                const float* __restrict__ zc, float* __restrict__ pd, const double* __restrict__ part) {
    double s6[6];
    block_reduce_parts<6, PBLK>(part, nparts, 9, 3, s6); // s6[0..2] = |r|^2, s6[3..5] = r.z
    const double* so = st + slot * 8;
    float be[3];
    double done[3];
    bool all_done_before = true;
    for (int k = 0; k < 3; k++) {
        be[k] = (so[k] == 0.0) ? 0.f : (float)(s6[3 + k] / so[k]);
        all_done_before = all_done_before && so[3 + k] != 0.0;
        done[k] = (so[3 + k] != 0.0 || s6[k] <= st[16 + k]) ? 1.0 : 0.0;
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float3 zi = ld3(zc, i), pi = ld3(pd, i);
        st3(pd, i, f3(zi.x + be[0] * pi.x, zi.y + be[1] * pi.y, zi.z + be[2] * pi.z));
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        double* sn = st + (slot ^ 1) * 8;
        for (int k = 0; k < 3; k++) {
            sn[k] = s6[3 + k];
            sn[3 + k] = done[k];
        }
        if (!all_done_before) st[19] += 1.0;
    }
}

// ---------------------------------------------------------------------------
// Fused PCG iteration for the AMG preconditioner (two kernels plus the rest of
// the V-cycle instead of four plus a full V-cycle):
//   k_cg_dir_spmv:   beta from the previous iteration's partials, then
//                    p' = z + beta p and q = A p' with p' formed on the fly for
//                    every gathered neighbour (p' goes to the other p buffer);
//   k_cg_update_pre: alpha = rz / p'.q, d += alpha p', r' = r - alpha q, and the
//                    level-0 pre-smoothing of r' (again on the fly from r and q;
//                    r' goes to the other r buffer).
// ---------------------------------------------------------------------------
// Next state slot (slot_old ^ 1) from |r|^2 at 3..5 and r.z at 6..8; every
// thread gets beta, block 0 thread 0 writes the slot.
template <int NT>
__device__ inline void cg_advance(const double* __restrict__ part, int nparts, double* __restrict__ st, int slot_old, float (&be)[3]) {
    double s6[6];
    block_reduce_parts<6, NT>(part, nparts, 9, 3, s6);
    const double* so = st + slot_old * 8;
    double done[3];
    for (int k = 0; k < 3; k++) {
        be[k] = (so[k] == 0.0) ? 0.f : (float)(s6[3 + k] / so[k]);
        done[k] = (so[3 + k] != 0.0 || s6[k] <= st[16 + k]) ? 1.0 : 0.0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        double* sn = st + (slot_old ^ 1) * 8;
        for (int k = 0; k < 3; k++) {
            sn[k] = s6[3 + k];
            sn[3 + k] = done[k];
        }
    }
}

// State update alone (before a convergence read-back); idempotent with the
// one k_cg_dir_spmv does at the start of the next iteration.
__global__ void __launch_bounds__(PBLK) k_cg_state(int slot_old, int nparts, double* __restrict__ st, const double* __restrict__ part) {
    float be[3];
    cg_advance<PBLK>(part, nparts, st, slot_old, be);
}

// Up to RU entries of row i that lane `sub` of its row group owns (every
// LPR-th), loaded before any gather; e_tail..e_end is the rest of the lane's
// entries (rows longer than RU * LPR).  Unused slots: value 0, column 0.
// Entry range (ptr[i], ptr[i+1]) of row i, (0, 0) past the last row.
__device__ inline int2 row_ptr(int i, int rows, const int32_t* __restrict__ ptr) {
    return i < rows ? make_int2(ptr[i], ptr[i + 1]) : make_int2(0, 0);
}

template <int LPR> struct RowSlot {
    int c[RU];
    float v[RU];
    int e_tail, e_end;
    __device__ inline void load(int i, int rows, int sub, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                const float* __restrict__ val) {
        load_range(row_ptr(i, rows, ptr), sub, col, val);
    }
    // from a row range loaded beforehand (one dependent load less per row)
    __device__ inline void load_range(int2 pr, int sub, const int32_t* __restrict__ col, const float* __restrict__ val) {
        const int e0 = pr.x + sub, e1 = pr.y;
#pragma unroll
        for (int u = 0; u < RU; u++) {
            const int e = e0 + u * LPR;
            const bool ok = e < e1;
            c[u] = ok ? col[e] : 0;
            v[u] = ok ? val[e] : 0.f;
        }
        e_tail = e0 + RU * LPR;
        e_end = e1;
    }
};

__device__ inline float3 ld3_or0(const float* __restrict__ a, int i, bool ok) { return ok ? ld3(a, i) : f3(0.f, 0.f, 0.f); }

// The fused kernels below take PF = true when their grid makes more than one
// pass over the rows: each pass then loads the next pass's row ranges while
// its own gathers are in flight, one dependent load less per pass.  A single
// pass keeps the variant without the extra registers.
inline bool multi_pass(int rows, int grid, int lpr) { return (int64_t)rows > 2 * (int64_t)grid * (PBLK / lpr); }

// They run on workgroups of NT = 256 threads up to SMALL_LANES lanes (rows
// times lanes per row) and of PBLK above.  4096 rows fill 16 workgroups of
// PBLK, on 16 of the 256 CUs; a quarter of the size spreads the same waves over
// 64 CUs.  At SMALL_LANES the grid leaves 256 partial sums, still one load per
// thread and the cap of the grid; larger systems would need more passes.
// AMG steps of a falling cloth (100 iterations), PBLK against SBLK: 4096 rows
// 6.78 -> 5.56 ms (direction 12.1 -> 8.1 us, update 12.6 -> 7.8, post-smoothing
// 8.9 -> 5.5), 16129 rows 8.47 -> 7.13 ms, 576 rows 3.08 -> 2.83 ms.
constexpr int SBLK = 256;
constexpr int64_t SMALL_LANES = 256 * 2 * SBLK;
inline bool small_rows(int rows, int lpr) { return (int64_t)rows * lpr <= SMALL_LANES; }

// The three SpMV-type kernels of the fused PCG iteration process two rows per
// lane group (i and i + one grid's worth of rows) and issue every load that
// does not depend on the reduced scalars (row pointers, entries, gathers, the
// row's own values) before reducing the previous kernel's partial sums.

template <int LPR, bool PF, int NT>
__global__ void __launch_bounds__(NT) k_cg_dir_spmv(int n, int first, int slot_old, int nparts, double* __restrict__ st,
                                                     const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                     const float* __restrict__ val, const float* __restrict__ diag,
                                                     const float* __restrict__ z, const float* __restrict__ p_old,
                                                     float* __restrict__ p_new, float* __restrict__ q, double* __restrict__ part) {
    const int sub = threadIdx.x % LPR;
    const int rpb = NT / LPR, stride = gridDim.x * rpb;
    float be[3] = {0.f, 0.f, 0.f};
    bool need_be = !first;
    double acc[3] = {0, 0, 0};
    auto comb = [&](float3 zc, float3 pc) { return f3(zc.x + be[0] * pc.x, zc.y + be[1] * pc.y, zc.z + be[2] * pc.z); };
    const int r_first = xcd_block() * rpb;
    int2 pra = make_int2(0, 0), prb = make_int2(0, 0);
    if constexpr (PF) {
        pra = row_ptr(r_first + threadIdx.x / LPR, n, ptr);
        prb = row_ptr(r_first + threadIdx.x / LPR + stride, n, ptr);
    }
    for (int r0 = r_first; r0 < n; r0 += 2 * stride) {
        const int ia = r0 + threadIdx.x / LPR, ib = ia + stride;
        const bool ha = ia < n, hb = ib < n;
        RowSlot<LPR> A, B;
        if constexpr (PF) {
            A.load_range(pra, sub, col, val);
            B.load_range(prb, sub, col, val);
            pra = row_ptr(ia + 2 * stride, n, ptr); // the next pass's row ranges, in flight meanwhile
            prb = row_ptr(ib + 2 * stride, n, ptr);
        } else {
            A.load(ia, n, sub, ptr, col, val);
            B.load(ib, n, sub, ptr, col, val);
        }
        const float3 zia = ld3_or0(z, ia, ha), zib = ld3_or0(z, ib, hb);
        const float3 pia = first ? zia : ld3_or0(p_old, ia, ha), pib = first ? zib : ld3_or0(p_old, ib, hb);
        const float dia = ha ? diag[ia] : 0.f, dib = hb ? diag[ib] : 0.f;
        float3 za[RU], zb[RU], pa[RU], pb[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            za[u] = ld3(z, A.c[u]);
            zb[u] = ld3(z, B.c[u]);
            pa[u] = first ? za[u] : ld3(p_old, A.c[u]);
            pb[u] = first ? zb[u] : ld3(p_old, B.c[u]);
        }
        if (need_be) { // uniform per block (first row pass)
            cg_advance<NT>(part, nparts, st, slot_old, be);
            need_be = false;
        }
        float3 sa = f3(0.f, 0.f, 0.f), sb = f3(0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < RU; u++) {
            sa = sa + A.v[u] * (first ? za[u] : comb(za[u], pa[u]));
            sb = sb + B.v[u] * (first ? zb[u] : comb(zb[u], pb[u]));
        }
        for (int e = A.e_tail; e < A.e_end; e += LPR) {
            const int c = col[e];
            sa = sa + val[e] * (first ? ld3(z, c) : comb(ld3(z, c), ld3(p_old, c)));
        }
        for (int e = B.e_tail; e < B.e_end; e += LPR) {
            const int c = col[e];
            sb = sb + val[e] * (first ? ld3(z, c) : comb(ld3(z, c), ld3(p_old, c)));
        }
        sa = group_sum<LPR>(sa);
        sb = group_sum<LPR>(sb);
        if (sub == 0) {
            if (ha) {
                const float3 pn = first ? zia : comb(zia, pia);
                const float3 qv = sa + dia * pn;
                st3(p_new, ia, pn);
                st3(q, ia, qv);
                acc[0] += (double)pn.x * qv.x;
                acc[1] += (double)pn.y * qv.y;
                acc[2] += (double)pn.z * qv.z;
            }
            if (hb) {
                const float3 pn = first ? zib : comb(zib, pib);
                const float3 qv = sb + dib * pn;
                st3(p_new, ib, pn);
                st3(q, ib, qv);
                acc[0] += (double)pn.x * qv.x;
                acc[1] += (double)pn.y * qv.y;
                acc[2] += (double)pn.z * qv.z;
            }
        }
    }
    if (need_be) cg_advance<NT>(part, nparts, st, slot_old, be); // a block without rows still takes part
    block_sum_write<3, NT>(acc, part, 9, 0);
}

template <int LPR, bool PF, int NT>
__global__ void __launch_bounds__(NT) k_cg_update_pre(int n, int slot, int nparts, double* __restrict__ st,
                                                       const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                       const float* __restrict__ val, const float* __restrict__ dinv, float w,
                                                       const float* __restrict__ pd, const float* __restrict__ q,
                                                       float* __restrict__ d, const float* __restrict__ r_old,
                                                       float* __restrict__ r_new, float* __restrict__ x0, float* __restrict__ res,
                                                       double* __restrict__ part) {
    const int sub = threadIdx.x % LPR;
    const int rpb = NT / LPR, stride = gridDim.x * rpb;
    float al[3] = {0.f, 0.f, 0.f};
    bool need_al = true;
    auto take_alpha = [&] {
        double pq[3];
        block_reduce_parts<3, NT>(part, nparts, 9, 0, pq);
        const double* s = st + slot * 8;
        bool all_done = true;
        for (int k = 0; k < 3; k++) {
            al[k] = (s[3 + k] != 0.0 || pq[k] == 0.0) ? 0.f : (float)(s[k] / pq[k]);
            all_done = all_done && s[3 + k] != 0.0;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0 && !all_done) st[19] += 1.0;
        need_al = false;
    };
    auto rnew = [&](float3 rc, float3 qc) { return f3(rc.x - al[0] * qc.x, rc.y - al[1] * qc.y, rc.z - al[2] * qc.z); };
    double acc[3] = {0, 0, 0};
    const int r_first = xcd_block() * rpb;
    int2 pra = make_int2(0, 0), prb = make_int2(0, 0);
    if constexpr (PF) {
        pra = row_ptr(r_first + threadIdx.x / LPR, n, ptr);
        prb = row_ptr(r_first + threadIdx.x / LPR + stride, n, ptr);
    }
    for (int r0 = r_first; r0 < n; r0 += 2 * stride) {
        const int ia = r0 + threadIdx.x / LPR, ib = ia + stride;
        const bool ha = ia < n, hb = ib < n;
        RowSlot<LPR> A, B;
        if constexpr (PF) {
            A.load_range(pra, sub, col, val);
            B.load_range(prb, sub, col, val);
            pra = row_ptr(ia + 2 * stride, n, ptr); // the next pass's row ranges, in flight meanwhile
            prb = row_ptr(ib + 2 * stride, n, ptr);
        } else {
            A.load(ia, n, sub, ptr, col, val);
            B.load(ib, n, sub, ptr, col, val);
        }
        const float3 ria = ld3_or0(r_old, ia, ha), qia = ld3_or0(q, ia, ha), pia = ld3_or0(pd, ia, ha), dia = ld3_or0(d, ia, ha);
        const float3 rib = ld3_or0(r_old, ib, hb), qib = ld3_or0(q, ib, hb), pib = ld3_or0(pd, ib, hb), dib = ld3_or0(d, ib, hb);
        const float wia = ha ? w * dinv[ia] : 0.f, wib = hb ? w * dinv[ib] : 0.f;
        float3 ra[RU], qa[RU], rb[RU], qb[RU];
        float wa[RU], wb[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            ra[u] = ld3(r_old, A.c[u]);
            qa[u] = ld3(q, A.c[u]);
            wa[u] = dinv[A.c[u]];
            rb[u] = ld3(r_old, B.c[u]);
            qb[u] = ld3(q, B.c[u]);
            wb[u] = dinv[B.c[u]];
        }
        if (need_al) take_alpha(); // uniform per block (first row pass)
        float3 sa = f3(0.f, 0.f, 0.f), sb = f3(0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < RU; u++) {
            sa = sa + (A.v[u] * (w * wa[u])) * rnew(ra[u], qa[u]);
            sb = sb + (B.v[u] * (w * wb[u])) * rnew(rb[u], qb[u]);
        }
        for (int e = A.e_tail; e < A.e_end; e += LPR) {
            const int c = col[e];
            sa = sa + (val[e] * (w * dinv[c])) * rnew(ld3(r_old, c), ld3(q, c));
        }
        for (int e = B.e_tail; e < B.e_end; e += LPR) {
            const int c = col[e];
            sb = sb + (val[e] * (w * dinv[c])) * rnew(ld3(r_old, c), ld3(q, c));
        }
        sa = group_sum<LPR>(sa);
        sb = group_sum<LPR>(sb);
        if (sub == 0) {
            if (ha) {
                const float3 rn = rnew(ria, qia);
                st3(d, ia, f3(dia.x + al[0] * pia.x, dia.y + al[1] * pia.y, dia.z + al[2] * pia.z));
                st3(r_new, ia, rn);
                st3(x0, ia, wia * rn);
                st3(res, ia, rn - sa);
                acc[0] += (double)rn.x * rn.x;
                acc[1] += (double)rn.y * rn.y;
                acc[2] += (double)rn.z * rn.z;
            }
            if (hb) {
                const float3 rn = rnew(rib, qib);
                st3(d, ib, f3(dib.x + al[0] * pib.x, dib.y + al[1] * pib.y, dib.z + al[2] * pib.z));
                st3(r_new, ib, rn);
                st3(x0, ib, wib * rn);
                st3(res, ib, rn - sb);
                acc[0] += (double)rn.x * rn.x;
                acc[1] += (double)rn.y * rn.y;
                acc[2] += (double)rn.z * rn.z;
            }
        }
    }
    if (need_al) take_alpha(); // a block without rows still takes part (block 0 counts the iteration)
    block_sum_write<3, NT>(acc, part, 9, 3);
}

// ---------------------------------------------------------------------------
// Smoothed-aggregation AMG V-cycle (one weighted-Jacobi pre- and post-sweep per
// level, dense inverse on the coarsest level); symmetric, so usable as the PCG
// preconditioner.  Level matrices hold the diagonal.
// ---------------------------------------------------------------------------
// Pre-smoothing from a zero guess: x = w D^-1 b; r = b - A x.  The scaled
// input w D^-1 b is formed on the fly for each gathered neighbour.
template <int LPR>
__global__ void __launch_bounds__(BLK) k_amg_pre(int n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                 const float* __restrict__ val, const float* __restrict__ dinv, float w,
                                                 const float* __restrict__ b, float* __restrict__ x, float* __restrict__ r) {
    const int sub = threadIdx.x % LPR;
    const int i = xcd_block() * (BLK / LPR) + threadIdx.x / LPR;
    float3 s = f3(0.f, 0.f, 0.f);
    row_foreach<LPR>(i, n, sub, ptr, col, val, [&](float v, int c) { s = s + (v * (w * dinv[c])) * ld3(b, c); });
    s = group_sum<LPR>(s);
    if (i < n && sub == 0) {
        const float3 bi = ld3(b, i);
        st3(x, i, (w * dinv[i]) * bi);
        st3(r, i, bi - s);
    }
}

// out = base + M in (M a CSR with `rows` rows); base may be null.
template <int LPR>
__global__ void __launch_bounds__(BLK) k_amg_spmv(int rows, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                  const float* __restrict__ val, const float* __restrict__ in,
                                                  const float* __restrict__ base, float* __restrict__ out) {
    const int sub = threadIdx.x % LPR;
    const int i = xcd_block() * (BLK / LPR) + threadIdx.x / LPR;
    float3 s = row_dot<LPR>(i, rows, sub, ptr, col, val, in);
    if (i < rows && sub == 0) st3(out, i, base ? ld3(base, i) + s : s);
}

// Post-smoothing: xo = xi + w D^-1 (b - A xi); with part != null also b.xo at
// 6..8 (on the finest level b is the PCG residual, so this is r.z).  Two rows
// per lane group, as the fused PCG kernels.
template <int LPR, bool PF, int NT>
__global__ void __launch_bounds__(NT) k_amg_post(int n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                                  const float* __restrict__ val, const float* __restrict__ dinv, float w,
                                                  const float* __restrict__ b, const float* __restrict__ xi, float* __restrict__ xo,
                                                  double* __restrict__ part) {
    const int sub = threadIdx.x % LPR;
    const int rpb = NT / LPR, stride = gridDim.x * rpb;
    double acc[3] = {0, 0, 0};
    const int r_first = xcd_block() * rpb;
    int2 pra = make_int2(0, 0), prb = make_int2(0, 0);
    if constexpr (PF) {
        pra = row_ptr(r_first + threadIdx.x / LPR, n, ptr);
        prb = row_ptr(r_first + threadIdx.x / LPR + stride, n, ptr);
    }
    for (int r0 = r_first; r0 < n; r0 += 2 * stride) {
        const int ia = r0 + threadIdx.x / LPR, ib = ia + stride;
        const bool ha = ia < n, hb = ib < n;
        RowSlot<LPR> A, B;
        if constexpr (PF) {
            A.load_range(pra, sub, col, val);
            B.load_range(prb, sub, col, val);
            pra = row_ptr(ia + 2 * stride, n, ptr); // the next pass's row ranges, in flight meanwhile
            prb = row_ptr(ib + 2 * stride, n, ptr);
        } else {
            A.load(ia, n, sub, ptr, col, val);
            B.load(ib, n, sub, ptr, col, val);
        }
        const float3 bia = ld3_or0(b, ia, ha), xia = ld3_or0(xi, ia, ha), bib = ld3_or0(b, ib, hb), xib = ld3_or0(xi, ib, hb);
        const float wia = ha ? w * dinv[ia] : 0.f, wib = hb ? w * dinv[ib] : 0.f;
        float3 xa[RU], xb[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            xa[u] = ld3(xi, A.c[u]);
            xb[u] = ld3(xi, B.c[u]);
        }
        float3 sa = f3(0.f, 0.f, 0.f), sb = f3(0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < RU; u++) {
            sa = sa + A.v[u] * xa[u];
            sb = sb + B.v[u] * xb[u];
        }
        for (int e = A.e_tail; e < A.e_end; e += LPR) sa = sa + val[e] * ld3(xi, col[e]);
        for (int e = B.e_tail; e < B.e_end; e += LPR) sb = sb + val[e] * ld3(xi, col[e]);
        sa = group_sum<LPR>(sa);
        sb = group_sum<LPR>(sb);
        if (sub == 0) {
            if (ha) {
                const float3 v = xia + wia * (bia - sa);
                st3(xo, ia, v);
                acc[0] += (double)bia.x * v.x;
                acc[1] += (double)bia.y * v.y;
                acc[2] += (double)bia.z * v.z;
            }
            if (hb) {
                const float3 v = xib + wib * (bib - sb);
                st3(xo, ib, v);
                acc[0] += (double)bib.x * v.x;
                acc[1] += (double)bib.y * v.y;
                acc[2] += (double)bib.z * v.z;
            }
        }
    }
    if (part) block_sum_write<3, NT>(acc, part, 9, 6);
}

// Partial r.z at 6..8.
__global__ void __launch_bounds__(PBLK) k_rz_part(int n, const float* __restrict__ r, const float* __restrict__ z,
                                                 double* __restrict__ part) {
    double acc[3] = {0, 0, 0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        for (int k = 0; k < 3; k++) acc[k] += (double)r[3 * i + k] * z[3 * i + k];
    block_sum_write<3, PBLK>(acc, part, 9, 6);
}

// Coarsest level: x = A_c^-1 b with the dense inverse (nc <= 2048, rows
// padded with zeros to ncp, a multiple of 4, so every lane reads float4).
// b is staged in LDS as three column vectors (zero beyond nc), so a lane's float4 of
// the inverse meets one float4 of each; every wave computes CROWS rows at once
// (independent accumulators), which also cuts the number of workgroups that
// stage b.
constexpr int CROWS = 2;
constexpr int CSLOTS = 2048 / 4 / 64; // float4 slots per lane for ncp <= 2048
__global__ void __launch_bounds__(BLK) k_amg_coarse(int nc, int ncp, const float4* __restrict__ inv, const float* __restrict__ b,
                                                    float* __restrict__ x) {
    __shared__ float4 sb[3][512]; // 3 x 2048 columns
    float* sbf = &sb[0][0].x;
    for (int j = threadIdx.x; j < ncp; j += BLK) {
        const bool in = j < nc;
        sbf[j] = in ? b[3 * j] : 0.f;
        sbf[2048 + j] = in ? b[3 * j + 1] : 0.f;
        sbf[4096 + j] = in ? b[3 * j + 2] : 0.f;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int row0 = (blockIdx.x * (BLK / 64) + (threadIdx.x >> 6)) * CROWS;
    if (row0 >= nc) return;
    float s[CROWS][3];
#pragma unroll
    for (int r = 0; r < CROWS; r++) s[r][0] = s[r][1] = s[r][2] = 0.f;
    const int q4 = ncp / 4;
    // all of a lane's loads first (up to CSLOTS per row in flight), then the sums
    float4 a[CROWS][CSLOTS];
#pragma unroll
    for (int r = 0; r < CROWS; r++) {
        const int row = min(row0 + r, nc - 1); // rows past nc repeat the last one and are not stored
#pragma unroll
        for (int k = 0; k < CSLOTS; k++) {
            const int j4 = lane + 64 * k;
            a[r][k] = j4 < q4 ? inv[(size_t)row * q4 + j4] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
#pragma unroll
    for (int k = 0; k < CSLOTS; k++) {
        const int j4 = lane + 64 * k;
        if (j4 >= q4) break;
        const float4 bx = sb[0][j4], by = sb[1][j4], bz = sb[2][j4];
#pragma unroll
        for (int r = 0; r < CROWS; r++) {
            const float4 v = a[r][k];
            s[r][0] += v.x * bx.x + v.y * bx.y + v.z * bx.z + v.w * bx.w;
            s[r][1] += v.x * by.x + v.y * by.y + v.z * by.z + v.w * by.w;
            s[r][2] += v.x * bz.x + v.y * bz.y + v.z * bz.z + v.w * bz.w;
        }
    }
#pragma unroll
    for (int r = 0; r < CROWS; r++)
#pragma unroll
        for (int k = 0; k < 3; k++)
            for (int o = 32; o > 0; o >>= 1) s[r][k] += __shfl_xor(s[r][k], o, 64);
    if (lane == 0)
#pragma unroll
        for (int r = 0; r < CROWS; r++)
            if (row0 + r < nc) {
                x[3 * (row0 + r)] = s[r][0];
                x[3 * (row0 + r) + 1] = s[r][1];
                x[3 * (row0 + r) + 2] = s[r][2];
            }
}

// ---------------------------------------------------------------------------
// Direct global solve with the prefactored supernodal Cholesky (pa_chol.hpp).
// Every vector is in elimination order and a supernode's columns are
// consecutive there.  With F the right-hand side of a supernode's front (r on
// its columns plus the children's update vectors), D = (L11 L11^T)^-1 and
// W = L21 L11^-1 of its factor blocks, one launch per tree level below the
// dense tops:
//   up (leaves first):        u = F(below) - W F(cols), to the parent
//   down (from the tops on):  x(cols) = D F(cols) - W^T x(below)
// and between them every tree's dense top: f = r(top) + the update vectors its
// boundary children send up, x(top) = S^-1 f.
//
// What bounds a level is its chain of dependent loads, not its bytes (below
// 3 MB but for the leaves), so a level is one product in each direction: with
// the triangular blocks L11^-1 and L21 themselves a level needed y = L11^-1 F
// before u and L21^T x before x, in two phases with a barrier (or, spread over
// tiles, two launches).  D and W take no more storage than L11^-1 and L21,
// and up reads only W.  A supernode's panel [D; -W] is column-major with its
// rows padded to whole float4s.  Everything a tile needs to find its data is
// in one descriptor, and where a row of F comes from is a table, so the chain
// is descriptor -> (panel, table, r) -> children's u -> product.
//
// At 256x256 vertices (6 levels and the top): up 6 x 5.5-6.1 us, down 5 x
// 4.5-4.8 and the leaves 10.1 us.  With L11^-1 and L21, over the 7 levels of
// smaller leaves: up 4 x 13.3 + 3 x 11.0, down 4 x (7.4 + 4.3) + 3 x 9.5 us.
// ---------------------------------------------------------------------------
struct CholTile {
    int64_t panel;     // the supernode's [D; -W] in the panel array
    int32_t c0, w, nb; // its columns' first position, their number, rows below
    int32_t first;     // up: first row of u of this tile; down: first column
    int32_t below;     // its rows below in chol_below and chol_u
    int32_t gat, kids; // its table in chol_gat_rows: kids entries per row of the front (-1: none)
    int32_t pad;
};
constexpr int CHOL_BLK = 256;
// Dissection leaves hold up to 160 unknowns in systems of up to this many, 64
// above.  Larger leaves save a level, two launches of about 6 us, and cost
// host set-up (about 25,000 more flops per unknown).  Step with 160 against 64:
// side-95 cloth 3.67 against 4.03 ms, tet box 3.84 / 4.31, 256x256 cloth 12.1 /
// 12.5, 362x362 (131,044 unknowns) 7.1 / 7.2; above the line 420x420 9.4 / 9.4,
// batches of 157,000 unknowns 6.6 / 7.1, of 304,000 11.2 / 11.7, of 500,000
// 36.3 / 36.9.  Set-up is 2 to 5% longer throughout.  So the line gives up 0 to
// 6% of a large system's step for 0.1 to 0.2 s of its set-up.
constexpr int CHOL_BIG_LEAF_N = 1 << 17;
constexpr int CHOL_INFLIGHT = 8; // float4 panel loads in flight per lane

__device__ inline int chol_pad4(int v) { return (v + 3) & ~3; }

// Adds the children's update-vector entries of front row `row` to v, in child order.
__device__ inline float3 chol_gather(const CholTile& T, int row, const int32_t* __restrict__ gat, const float* u, float3 v) {
    const int32_t* g = gat + T.gat + (int64_t)row * T.kids;
    int k = 0;
    for (; k + 2 <= T.kids; k += 2) {
        const int a = g[k], b = g[k + 1];
        const float3 ua = a >= 0 ? ld3(u, a) : f3(0.f, 0.f, 0.f), ub = b >= 0 ? ld3(u, b) : f3(0.f, 0.f, 0.f);
        v = v + ua;
        v = v + ub;
    }
    if (k < T.kids && g[k] >= 0) v = v + ld3(u, g[k]);
    return v;
}

// Rows first .. first + 4 RG of u.  RG lanes take four rows each (one float4 of
// a panel column), 256 / RG groups of lanes share the columns.  A small RG
// gives a level more tiles, a large one gathers F fewer times.
template <int RG>
__global__ void __launch_bounds__(CHOL_BLK) k_chol_up(const CholTile* __restrict__ tiles, const float* __restrict__ panels,
                                                      const int32_t* __restrict__ gat, const float* __restrict__ r, float* __restrict__ F,
                                                      float* u) {
    constexpr int PARTS = CHOL_BLK / RG, RT = 4 * RG, U = CHOL_INFLIGHT;
    extern __shared__ float4 chol_sh4[];
    __shared__ float red[CHOL_BLK / 64][3 * RT];
    float4* const Fs = chol_sh4; // w: F of the columns
    const CholTile T = tiles[blockIdx.x];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wp = chol_pad4(T.w), ld = wp + chol_pad4(T.nb);
    const int j = T.first + 4 * (t % RG), part = t / RG;
    const float* P = panels + T.panel + wp + j;
    float4 pv[U];
    auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int k = k0 + part + q * PARTS;
            pv[q] = j < T.nb && k < T.w ? *reinterpret_cast<const float4*>(P + (int64_t)k * ld) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    load(0);
    for (int i = t; i < T.w; i += CHOL_BLK) {
        const float3 f = chol_gather(T, i, gat, u, ld3(r, T.c0 + i));
        Fs[i] = make_float4(f.x, f.y, f.z, 0.f);
        if (T.first == 0) st3(F, T.c0 + i, f);
    }
    float3 fb = f3(0.f, 0.f, 0.f);
    if (t < RT && T.first + t < T.nb) fb = chol_gather(T, T.w + T.first + t, gat, u, fb);
    __syncthreads();
    if (T.nb == 0) return;
    float3 acc[4];
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q] = f3(0.f, 0.f, 0.f);
    for (int k0 = 0; k0 < T.w; k0 += U * PARTS) {
        if (k0 > 0) load(k0);
#pragma unroll
        for (int q = 0; q < U; q++) {
            const float4 g = Fs[min(k0 + part + q * PARTS, T.w - 1)];
            const float3 fk = f3(g.x, g.y, g.z);
            acc[0] = acc[0] + pv[q].x * fk;
            acc[1] = acc[1] + pv[q].y * fk;
            acc[2] = acc[2] + pv[q].z * fk;
            acc[3] = acc[3] + pv[q].w * fk;
        }
    }
#pragma unroll
    for (int o = RG; o < 64; o <<= 1)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            acc[q].x += __shfl_xor(acc[q].x, o, 64);
            acc[q].y += __shfl_xor(acc[q].y, o, 64);
            acc[q].z += __shfl_xor(acc[q].z, o, 64);
        }
    if (lane < RG)
#pragma unroll
        for (int q = 0; q < 4; q++) st3(red[wave], 4 * lane + q, acc[q]);
    __syncthreads();
    if (t < RT && T.first + t < T.nb) {
#pragma unroll
        for (int q = 0; q < CHOL_BLK / 64; q++) fb = fb + ld3(red[q], t);
        st3(u, T.below + T.first + t, fb);
    }
}

// Columns first .. first + 256 / LP of x: LP lanes share a column of the panel,
// four rows each, and combine with shuffles.
template <int LP>
__global__ void __launch_bounds__(CHOL_BLK) k_chol_down(const CholTile* __restrict__ tiles, const float* __restrict__ panels,
                                                        const int32_t* __restrict__ below, const float* __restrict__ F, float* x) {
    constexpr int U = CHOL_INFLIGHT;
    extern __shared__ float4 chol_sh4[];
    const CholTile T = tiles[blockIdx.x];
    const int t = threadIdx.x, s = t % LP, col = T.first + t / LP;
    const int wp = chol_pad4(T.w), ld = wp + chol_pad4(T.nb);
    float* const v = reinterpret_cast<float*>(chol_sh4); // 3 x ld: [F(cols); x(below)], zeros in the padding
    const float* P = panels + T.panel + (int64_t)col * ld + 4 * s;
    float4 pv[U];
    auto load = [&](int l0) {
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int l = l0 + q * 4 * LP;
            pv[q] = col < T.w && l + 4 * s < ld ? *reinterpret_cast<const float4*>(P + l) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    load(0);
    for (int l = t; l < ld; l += CHOL_BLK) {
        float3 e = f3(0.f, 0.f, 0.f);
        if (l < T.w) e = ld3(F, T.c0 + l);
        else if (l >= wp && l - wp < T.nb) e = ld3(x, below[T.below + l - wp]);
        v[l] = e.x;
        v[ld + l] = e.y;
        v[2 * ld + l] = e.z;
    }
    __syncthreads();
    float3 acc = f3(0.f, 0.f, 0.f);
    for (int l0 = 0; l0 < ld; l0 += U * 4 * LP) {
        if (l0 > 0) load(l0);
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int l = min(l0 + q * 4 * LP + 4 * s, ld - 4);
            const float4 p = pv[q], vx = *reinterpret_cast<const float4*>(v + l), vy = *reinterpret_cast<const float4*>(v + ld + l),
                         vz = *reinterpret_cast<const float4*>(v + 2 * ld + l);
            acc.x += (p.x * vx.x + p.y * vx.y) + (p.z * vx.z + p.w * vx.w);
            acc.y += (p.x * vy.x + p.y * vy.y) + (p.z * vy.z + p.w * vy.w);
            acc.z += (p.x * vz.x + p.y * vz.y) + (p.z * vz.z + p.w * vz.w);
        }
    }
#pragma unroll
    for (int o = LP / 2; o > 0; o >>= 1) {
        acc.x += __shfl_xor(acc.x, o, LP);
        acc.y += __shfl_xor(acc.y, o, LP);
        acc.z += __shfl_xor(acc.z, o, LP);
    }
    if (s == 0 && col < T.w) st3(x, T.c0 + col, acc);
}

// Dense tops.  k_chol_top_f assembles every top entry's right-hand side once:
// f = r at its position plus the update-vector entries the boundary children
// send up (at most gmax each, in a fixed order).  Where there is no level
// below the tops f is r itself (pos non-null) and the launch falls away.
// k_chol_top: workgroup (block, row0) forms CHOL_TOP_ROWS rows of S^-1 f for
// its tree's top, one wave per row.  A row is up to NV float4s per lane (rows
// padded to whole float4s), all in flight before f arrives in LDS; the lanes'
// sums combine with shuffles.  NV follows the largest top, so a small one does
// not step over the loads of a large one.  256x256 vertices (3036 columns,
// 37 MB): 11.9 us against 15.5 with scalar loads and lane 0 adding 64 sums from
// LDS; a 256-column top 3.5 against 8.0.
constexpr int CHOL_TOP_ROWS = 4;   // rows of S^-1 per workgroup (one per wave)
constexpr int CHOL_TOP_BLK = 256;
constexpr int CHOL_TOP_MAX = 4096; // largest dense top (16 float4s per lane)
constexpr int CHOL_TOP_GMAX = 8;   // most update-vector entries gathered into one top entry

__global__ void k_chol_top_f(int ntop, const int32_t* __restrict__ pos, const int64_t* __restrict__ gat_fix, int gmax,
                             const float* __restrict__ r, const float* __restrict__ u, float* __restrict__ ftop) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ntop) return;
    int64_t ge[CHOL_TOP_GMAX];
#pragma unroll
    for (int k = 0; k < CHOL_TOP_GMAX; k++) ge[k] = k < gmax ? gat_fix[(int64_t)q * gmax + k] : -1;
    float3 fv = ld3(r, pos[q]);
#pragma unroll
    for (int k = 0; k < CHOL_TOP_GMAX; k++)
        if (ge[k] >= 0) fv = fv + ld3(u, ge[k]);
    st3(ftop, q, fv);
}

template <int NV>
__global__ void __launch_bounds__(CHOL_TOP_BLK) k_chol_top(const int2* __restrict__ tiles, const int64_t* __restrict__ top_ptr,
                                                           const int32_t* __restrict__ top_pos, const int64_t* __restrict__ sinv_off,
                                                           const float* __restrict__ sinv, const float* __restrict__ f,
                                                           const int32_t* __restrict__ pos, float* __restrict__ x) {
    extern __shared__ float4 chol_sh4[];
    const int2 tl = tiles[blockIdx.x];
    const int64_t p0 = top_ptr[tl.x];
    const int m = (int)(top_ptr[tl.x + 1] - p0), mp = chol_pad4(m);
    const int lane = threadIdx.x & 63, i0 = tl.y + (threadIdx.x >> 6);
    const float* S = sinv + sinv_off[tl.x] + (int64_t)i0 * mp + 4 * lane;
    float4 s0[NV];
#pragma unroll
    for (int t = 0; t < NV; t++)
        s0[t] = i0 < m && 4 * lane + 256 * t < mp ? *reinterpret_cast<const float4*>(S + 256 * t) : make_float4(0.f, 0.f, 0.f, 0.f);
    float* const v = reinterpret_cast<float*>(chol_sh4); // 3 x mp
#pragma unroll
    for (int t = 0; t < NV; t++) {
        const int q = threadIdx.x + CHOL_TOP_BLK * t;
        if (q < mp) {
            const float3 e = q < m ? ld3(f, pos ? (int64_t)pos[p0 + q] : p0 + q) : f3(0.f, 0.f, 0.f);
            v[q] = e.x;
            v[mp + q] = e.y;
            v[2 * mp + q] = e.z;
        }
    }
    __syncthreads();
    float3 a = f3(0.f, 0.f, 0.f);
#pragma unroll
    for (int t = 0; t < NV; t++) {
        const int j = min(4 * lane + 256 * t, mp - 4);
        const float4 p = s0[t], vx = *reinterpret_cast<const float4*>(v + j), vy = *reinterpret_cast<const float4*>(v + mp + j),
                     vz = *reinterpret_cast<const float4*>(v + 2 * mp + j);
        a.x += (p.x * vx.x + p.y * vx.y) + (p.z * vx.z + p.w * vx.w);
        a.y += (p.x * vy.x + p.y * vy.y) + (p.z * vy.z + p.w * vy.w);
        a.z += (p.x * vz.x + p.y * vz.y) + (p.z * vz.z + p.w * vz.w);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a.x += __shfl_xor(a.x, o, 64);
        a.y += __shfl_xor(a.y, o, 64);
        a.z += __shfl_xor(a.z, o, 64);
    }
    if (lane == 0 && i0 < m) st3(x, top_pos[p0 + i0], a);
}

// Rigid animation of static vertices (reference ScriptAnimator::animate_rigid,
// src/solver/animator.cpp:83-130): x = t + q (x) rest with the unit quaternion
// rotation v' = v + w T + u x T, T = 2 (u x v); v_static = (x - x_prev) / h,
// or 0 once the track has ended.  FP64 throughout.
__global__ void k_animate_rigid(int first, int count, const double* __restrict__ rest, double* __restrict__ prev, double tx,
                                double ty, double tz, double qw, double qx, double qy, double qz, double hinv, int zero_v,
                                double* __restrict__ x, double* __restrict__ v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const double rx = rest[3 * i], ry = rest[3 * i + 1], rz = rest[3 * i + 2];
    const double Tx = 2.0 * (qy * rz - qz * ry), Ty = 2.0 * (qz * rx - qx * rz), Tz = 2.0 * (qx * ry - qy * rx);
    const double nx = tx + (rx + qw * Tx + (qy * Tz - qz * Ty));
    const double ny = ty + (ry + qw * Ty + (qz * Tx - qx * Tz));
    const double nz = tz + (rz + qw * Tz + (qx * Ty - qy * Tx));
    const int g = first + i;
    if (x) { // without x and v only the placed positions are kept (resuming at a frame)
        x[3 * g] = nx;
        x[3 * g + 1] = ny;
        x[3 * g + 2] = nz;
        v[3 * g] = zero_v ? 0.0 : (nx - prev[3 * i]) * hinv;
        v[3 * g + 1] = zero_v ? 0.0 : (ny - prev[3 * i + 1]) * hinv;
        v[3 * g + 2] = zero_v ? 0.0 : (nz - prev[3 * i + 2]) * hinv;
    }
    prev[3 * i] = nx;
    prev[3 * i + 1] = ny;
    prev[3 * i + 2] = nz;
}

// Point-sequence animation of static vertices (reference
// ScriptAnimator::animate_points, src/solver/animator.cpp:132-178): x = the
// frame's positions, v = (x - x_prev) / h, or 0 once the sequence has ended.
__global__ void k_animate_points(int first, int count, const double* __restrict__ frame, double* __restrict__ prev, double hinv,
                                 int zero_v, double* __restrict__ x, double* __restrict__ v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int g = first + i;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double p = frame[3 * i + k];
        if (x) {
            x[3 * g + k] = p;
            v[3 * g + k] = zero_v ? 0.0 : (p - prev[3 * i + k]) * hinv;
        }
        prev[3 * i + k] = p;
    }
}

} // namespace

// ===========================================================================
// Host side
// ===========================================================================
Backend::Backend(const pa_device_opts* o) : Backend() {
    device = o ? o->device : 0;
    verbose = o ? o->verbose : 0;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    PA_CHECK(e == hipSuccess && count > 0, PA_ERR_NO_DEVICE, "no HIP device visible");
    PA_CHECK(device >= 0 && device < count, PA_ERR_INVALID, "device ordinal out of range");
    PA_HIP(hipSetDevice(device));
    PA_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    for (auto& e : ev_chk) PA_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    PA_HIP(hipHostMalloc((void**)&chk_host, 16 * sizeof(double), hipHostMallocDefault));
    pa_admm_config_default(&cfg);
}

Backend::~Backend() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto& g : pcg_graph)
        if (g) (void)hipGraphExecDestroy(g);
    for (auto e : ev_pool) (void)hipEventDestroy(e);
    // an attached external detector goes back to its own stream
    if (det && det != own_det.get()) det->stream = det->own_stream;
    own_det.reset();
    ws_mlp.reset(); // uses the stream
    for (auto e : ev_chk)
        if (e) (void)hipEventDestroy(e);
    if (chk_host) (void)hipHostFree(chk_host);
    if (stream) (void)hipStreamDestroy(stream);
}

void Backend::apply_config(const pa_admm_config& c) {
    PA_CHECK(c.dt > 0, PA_ERR_INVALID, "dt must be positive");
    PA_CHECK(c.admm_max_iter >= 1, PA_ERR_INVALID, "admm_max_iter must be >= 1");
    PA_CHECK(c.dcd_interval >= 1, PA_ERR_INVALID, "dcd_interval must be >= 1");
    PA_CHECK(c.gs_max_iter >= 0, PA_ERR_INVALID, "gs_max_iter must be >= 0");
    PA_CHECK(c.global_max_iter >= 1, PA_ERR_INVALID, "global_max_iter must be >= 1");
    PA_CHECK(c.max_contacts >= 1, PA_ERR_INVALID, "max_contacts must be >= 1");
    PA_CHECK(c.precond >= 0 && c.precond <= 2, PA_ERR_INVALID, "precond must be 0 (Jacobi), 1 (AMG) or 2 (direct)");
    PA_CHECK(!initialized, PA_ERR_INVALID, "apply_config must precede init");
    cfg = c;
    if (cfg.residual_interval < 1) cfg.residual_interval = 1;
    use_graphs = cfg.graphs != 0;
    have_cfg = true;
}

void Backend::set_constraints(const pa_constraint_soa& c) {
    PA_CHECK(!finalized, PA_ERR_INVALID, "constraints already finalized");
    HostConstraints h;
    h.n_tri = c.n_tri;
    h.n_tet = c.n_tet;
    h.n_bend = c.n_bend;
    h.n_pin = c.n_pin;
    PA_CHECK(h.n_tri >= 0 && h.n_tet >= 0 && h.n_bend >= 0 && h.n_pin >= 0, PA_ERR_INVALID, "negative constraint count");
    h.tri_row0 = c.tri_row0;
    h.tet_row0 = c.tet_row0;
    h.bend_row0 = c.bend_row0;
    h.pin_row0 = c.pin_row0;
    auto cp_i = [](const int32_t* p, size_t n, std::vector<int32_t>& out) {
        PA_CHECK(n == 0 || p, PA_ERR_INVALID, "null constraint array");
        out.assign(p, p + n);
    };
    auto cp_d = [](const double* p, size_t n, std::vector<double>& out) {
        PA_CHECK(n == 0 || p, PA_ERR_INVALID, "null constraint array");
        out.assign(p, p + n);
    };
    cp_i(c.tri_inds, 3 * (size_t)h.n_tri, h.tri_inds);
    cp_d(c.tri_binv, 4 * (size_t)h.n_tri, h.tri_binv);
    cp_d(c.tri_w, h.n_tri, h.tri_w);
    cp_i(c.tet_inds, 4 * (size_t)h.n_tet, h.tet_inds);
    cp_d(c.tet_binv, 9 * (size_t)h.n_tet, h.tet_binv);
    cp_d(c.tet_w, h.n_tet, h.tet_w);
    cp_i(c.bend_ptr, h.n_bend ? (size_t)h.n_bend + 1 : 0, h.bend_ptr);
    if (h.n_bend == 0) h.bend_ptr = {0};
    size_t nbe = h.bend_ptr.back();
    cp_i(c.bend_inds, nbe, h.bend_inds);
    cp_d(c.bend_coef, nbe, h.bend_coef);
    cp_d(c.bend_w, h.n_bend, h.bend_w);
    cp_i(c.pin_inds, h.n_pin, h.pin_inds);
    cp_d(c.pin_pos, 3 * (size_t)h.n_pin, h.pin_pos);
    cp_d(c.pin_w, h.n_pin, h.pin_w);
    hc = std::move(h);
    have_constraints = true;
}

void Backend::finalize_constraints() {
    PA_CHECK(have_constraints, PA_ERR_INVALID, "finalize_constraints before set_constraints");
    PA_CHECK(m_declared >= 0, PA_ERR_INVALID, "finalize_constraints before set_constraint_dim");
    // Rows must tile [0, m): tri, tet, bend, pin blocks, each contiguous.
    struct Blk {
        int row0, rows;
    } blks[4] = {{hc.tri_row0, 2 * hc.n_tri}, {hc.tet_row0, 3 * hc.n_tet}, {hc.bend_row0, hc.n_bend}, {hc.pin_row0, hc.n_pin}};
    std::vector<std::pair<int, int>> iv;
    for (auto& b : blks)
        if (b.rows > 0) iv.push_back({b.row0, b.rows});
    std::sort(iv.begin(), iv.end());
    int cur = 0;
    for (auto& q : iv) {
        PA_CHECK(q.first == cur, PA_ERR_INVALID, "constraint rows must tile [0, m) without gaps or overlap");
        cur += q.second;
    }
    PA_CHECK(cur == m_declared, PA_ERR_INVALID, "constraint dimension does not match the constraints");
    for (size_t i = 1; i < hc.bend_ptr.size(); i++)
        PA_CHECK(hc.bend_ptr[i] >= hc.bend_ptr[i - 1], PA_ERR_INVALID, "bend_ptr must be non-decreasing");
    m = m_declared;
    finalized = true;
}

void Backend::init(const double* x0h, const double* massh, int n_all_, int n_dyn, const uint8_t* surface, int n_pins, const int32_t* pins) {
    PA_CHECK(have_cfg, PA_ERR_INVALID, "init before apply_config");
    PA_CHECK(finalized, PA_ERR_INVALID, "init before finalize_constraints");
    PA_CHECK(!initialized, PA_ERR_INVALID, "init called twice");
    PA_CHECK(n_all_ > 0 && n_dyn > 0 && n_dyn <= n_all_, PA_ERR_INVALID, "bad vertex counts");
    if (det) { // attached before these sizes were known: what attach_detector could not check
        PA_CHECK(det->n_all <= n_all_, PA_ERR_INVALID, "attached detector has more vertices than the backend");
        PA_CHECK(det->c.cap <= cfg.max_contacts, PA_ERR_INVALID, "detector capacity exceeds max_contacts");
    }
    n_all = n_all_;
    n = n_dyn;
    auto chk_v = [&](int v) { PA_CHECK(v >= 0 && v < n, PA_ERR_INVALID, "constraint references a non-dynamic vertex"); };
    for (int v : hc.tri_inds) chk_v(v);
    for (int v : hc.tet_inds) chk_v(v);
    for (int v : hc.bend_inds) chk_v(v);
    for (int v : hc.pin_inds) chk_v(v);
    mass_h.assign(massh, massh + n_all);
    for (int i = 0; i < n; i++) PA_CHECK(mass_h[i] > 0, PA_ERR_INVALID, "dynamic vertex with non-positive mass");
    surface_h.assign(n_all, 0);
    if (surface)
        for (int i = 0; i < n_all; i++) surface_h[i] = surface[i] ? 1 : 0;
    pinned_h.assign(n_all, 0);
    for (int i = 0; i < n_pins; i++) {
        PA_CHECK(pins[i] >= 0 && pins[i] < n_all, PA_ERR_INVALID, "pin out of range");
        pinned_h[pins[i]] = 1;
    }
    assemble_and_upload(x0h);
    x_init_h.assign(x0h, x0h + 3 * (size_t)n_all);
    bad_flag.alloc(1);
    initialized = true;
    save_good_state();
    PA_HIP(hipStreamSynchronize(stream));
}

// Registers a rigid track and places its vertices at frame 0 with zero
// velocity, as the reference's initial animate_all does (admm_impl_gpu.cu:143-144).
void Backend::add_rigid_track(int first, int count, int frames, const double* pos, const double* quat_xyzw, int fps) {
    PA_CHECK(initialized, PA_ERR_INVALID, "add_rigid_track before init");
    PA_CHECK(pos && quat_xyzw, PA_ERR_INVALID, "null track data");
    PA_CHECK(first >= n && count > 0 && (int64_t)first + count <= n_all, PA_ERR_INVALID, "track range must lie within the static vertices");
    PA_CHECK(frames >= 3, PA_ERR_INVALID, "track needs at least 3 frames");
    PA_CHECK(fps >= 1, PA_ERR_INVALID, "frames per step must be >= 1");
    for (const auto& t : tracks)
        PA_CHECK(first + count <= t->first || t->first + t->count <= first, PA_ERR_INVALID, "tracks overlap");
    auto T = std::make_unique<RigidTrack>();
    T->first = first;
    T->count = count;
    T->frames = frames;
    T->fps = fps;
    T->trans.assign(pos, pos + 3 * (size_t)frames);
    T->quat.resize(4 * (size_t)frames);
    for (int f = 0; f < frames; f++) { // npz order (x, y, z, w) -> (w, x, y, z), animator.cpp:32
        const double* q = quat_xyzw + 4 * (size_t)f;
        const double nq = std::sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        PA_CHECK(nq > 0.5 && nq < 2.0, PA_ERR_INVALID, "track quaternion far from unit length");
        T->quat[4 * f] = q[3] / nq;
        T->quat[4 * f + 1] = q[0] / nq;
        T->quat[4 * f + 2] = q[1] / nq;
        T->quat[4 * f + 3] = q[2] / nq;
    }
    T->rest.alloc(3 * (size_t)count);
    T->rest.upload(x_init_h.data() + 3 * (size_t)first, 3 * (size_t)count, stream);
    T->prev.alloc(3 * (size_t)count);
    tracks.push_back(std::move(T));
    animate_tracks(true);
    save_good_state(); // with the tracked vertices at frame 0
    PA_HIP(hipStreamSynchronize(stream));
}

// A point-sequence track for static vertices [first, first + count): frame
// k places them at points[k] (frames x count x 3, world positions; the mesh's
// transform T + R (s p) already applied, animator.cpp:149-172); registered at
// frame 0 with zero velocity, like a rigid track.
void Backend::add_point_track(int first, int count, int frames, const double* points, int fps) {
    PA_CHECK(initialized, PA_ERR_INVALID, "add_point_track before init");
    PA_CHECK(points, PA_ERR_INVALID, "null track data");
    PA_CHECK(first >= n && count > 0 && (int64_t)first + count <= n_all, PA_ERR_INVALID, "track range must lie within the static vertices");
    PA_CHECK(frames >= 1, PA_ERR_INVALID, "point track needs at least one frame");
    PA_CHECK(fps >= 1, PA_ERR_INVALID, "frames per step must be >= 1");
    for (const auto& t : tracks)
        PA_CHECK(first + count <= t->first || t->first + t->count <= first, PA_ERR_INVALID, "tracks overlap");
    const size_t total = (size_t)frames * count * 3;
    for (size_t i = 0; i < total; i++) PA_CHECK(std::isfinite(points[i]), PA_ERR_INVALID, "non-finite point-track position");
    auto T = std::make_unique<RigidTrack>();
    T->first = first;
    T->count = count;
    T->frames = frames;
    T->fps = fps;
    T->points = true;
    T->pts.alloc(total);
    T->pts.upload(points, total, stream);
    T->prev.alloc(3 * (size_t)count);
    tracks.push_back(std::move(T));
    animate_tracks(true);
    save_good_state(); // with the tracked vertices at frame 0
    PA_HIP(hipStreamSynchronize(stream));
}

// Per step (before the prologue): frame counter += frames per step; past the
// end the vertices stay at the last frame with zero velocity.  A rigid track
// counts as ended once its counter reaches the frame count (it places frame
// counter - 1, animator.cpp:89-103); a point sequence places frame counter - 1
// too but ends only past its last frame (animate_points reads frame counter
// before the rigid tracks' increment, animator.cpp:135-160).  With
// place_first_frame every track is put at frame 0.
void Backend::animate_tracks(bool place_first_frame) {
    const double hinv = 1.0 / cfg.dt;
    for (auto& tp : tracks) {
        RigidTrack& T = *tp;
        int f;
        bool zero_v;
        if (place_first_frame) {
            T.cur = 1;
            f = 0;
            zero_v = true;
        } else if (T.points) {
            T.cur = std::min(T.cur + T.fps, T.frames + 1);
            zero_v = T.cur - 1 >= T.frames;
            f = std::min(T.cur - 1, T.frames - 1);
        } else {
            T.cur += T.fps;
            zero_v = T.cur >= T.frames;
            if (zero_v) T.cur = T.frames;
            f = T.cur - 1;
        }
        if (T.points) {
            hipLaunchKernelGGL(k_animate_points, dim3(grid_for(T.count, BLK)), dim3(BLK), 0, stream, T.first, T.count,
                               (const double*)T.pts.p + (size_t)f * T.count * 3, T.prev.p, hinv, zero_v ? 1 : 0, x.p, v.p);
            PA_LAUNCH_CHECK();
            continue;
        }
        const double* t = T.trans.data() + 3 * (size_t)f;
        const double* q = T.quat.data() + 4 * (size_t)f;
        hipLaunchKernelGGL(k_animate_rigid, dim3(grid_for(T.count, BLK)), dim3(BLK), 0, stream, T.first, T.count, T.rest.p, T.prev.p,
                           t[0], t[1], t[2], q[0], q[1], q[2], q[3], hinv, zero_v ? 1 : 0, x.p, v.p);
        PA_LAUNCH_CHECK();
    }
}

// Frame counters of the tracks (registration order), for checkpoints.
// Setting them also re-places each track's last-placed positions at that
// frame (FP64, as the step that reached it did), so the next step's static
// velocities are the ones an uninterrupted run computes.
void Backend::get_track_frames(int32_t* frames) const {
    for (size_t k = 0; k < tracks.size(); k++) frames[k] = tracks[k]->cur;
}

void Backend::set_track_frames(const int32_t* frames, int count) {
    PA_CHECK(count == (int)tracks.size(), PA_ERR_INVALID, "one frame counter per track");
    for (int k = 0; k < count; k++)
        PA_CHECK(frames[k] >= 1 && frames[k] <= tracks[k]->frames + (tracks[k]->points ? 1 : 0), PA_ERR_INVALID,
                 "frame counter out of range");
    for (int k = 0; k < count; k++) {
        RigidTrack& T = *tracks[k];
        T.cur = frames[k];
        if (T.points) {
            const int fp = std::min(T.cur - 1, T.frames - 1);
            hipLaunchKernelGGL(k_animate_points, dim3(grid_for(T.count, BLK)), dim3(BLK), 0, stream, T.first, T.count,
                               (const double*)T.pts.p + (size_t)fp * T.count * 3, T.prev.p, 0.0, 0, (double*)nullptr, (double*)nullptr);
            PA_LAUNCH_CHECK();
            continue;
        }
        const int f = T.cur - 1;
        const double* t = T.trans.data() + 3 * (size_t)f;
        const double* q = T.quat.data() + 4 * (size_t)f;
        hipLaunchKernelGGL(k_animate_rigid, dim3(grid_for(T.count, BLK)), dim3(BLK), 0, stream, T.first, T.count, T.rest.p, T.prev.p,
                           t[0], t[1], t[2], q[0], q[1], q[2], q[3], 0.0, 0, (double*)nullptr, (double*)nullptr);
        PA_LAUNCH_CHECK();
    }
    PA_HIP(hipStreamSynchronize(stream));
}

void Backend::assemble_and_upload(const double* x0h) {
    const double h = cfg.dt, h2 = h * h;
    const bool contact = cfg.enable_contact != 0;
    // ---- per-row D coefficients (row, vertex, G) ----
    struct Ent {
        int row, v;
        double g, w;
        bool pin;
    };
    std::vector<Ent> ents;
    ents.reserve(6 * (size_t)hc.n_tri + 12 * (size_t)hc.n_tet + hc.bend_inds.size() + hc.n_pin);
    for (int c = 0; c < hc.n_tri; c++) {
        const double* B = &hc.tri_binv[4 * c];
        const int* t = &hc.tri_inds[3 * c];
        for (int r = 0; r < 2; r++) {
            int row = hc.tri_row0 + 2 * c + r;
            ents.push_back({row, t[0], -(B[r] + B[2 + r]), hc.tri_w[c], false});
            ents.push_back({row, t[1], B[r], hc.tri_w[c], false});
            ents.push_back({row, t[2], B[2 + r], hc.tri_w[c], false});
        }
    }
    for (int c = 0; c < hc.n_tet; c++) {
        const double* B = &hc.tet_binv[9 * c];
        const int* t = &hc.tet_inds[4 * c];
        for (int r = 0; r < 3; r++) {
            int row = hc.tet_row0 + 3 * c + r;
            ents.push_back({row, t[0], -((B[r] + B[3 + r]) + B[6 + r]), hc.tet_w[c], false});
            for (int q = 0; q < 3; q++) ents.push_back({row, t[q + 1], B[3 * q + r], hc.tet_w[c], false});
        }
    }
    for (int c = 0; c < hc.n_bend; c++)
        for (int e = hc.bend_ptr[c]; e < hc.bend_ptr[c + 1]; e++)
            ents.push_back({hc.bend_row0 + c, hc.bend_inds[e], hc.bend_coef[e], hc.bend_w[c], false});
    for (int c = 0; c < hc.n_pin; c++) ents.push_back({hc.pin_row0 + c, hc.pin_inds[c], 1.0, hc.pin_w[c], true});
    // group by row (entries of one row are consecutive already)
    // ---- A = M + h^2 D^T We^2 D + h^2 Wc + h (kL D^T Wd D + kM M);  Damp separately ----
    struct T3 {
        int r, c;
        double v;
    };
    std::vector<T3> ta, td;
    ta.reserve(ents.size() * 8);
    std::vector<double> adiag(mass_h.begin(), mass_h.begin() + n); // diagonal of M + h^2 D^T We^2 D + Damp
    for (size_t s = 0; s < ents.size();) {
        size_t e = s;
        while (e < ents.size() && ents[e].row == ents[s].row) e++;
        const double w = ents[s].w;
        for (size_t a = s; a < e; a++)
            for (size_t bb = s; bb < e; bb++) {
                double gg = ents[a].g * ents[bb].g;
                ta.push_back({ents[a].v, ents[bb].v, h2 * w * w * gg});
                const bool on_diag = ents[a].v == ents[bb].v;
                if (on_diag) adiag[ents[a].v] += h2 * w * w * gg;
                if (!ents[s].pin && cfg.damp_kl != 0) {
                    double dv = h * cfg.damp_kl * w * gg;
                    ta.push_back({ents[a].v, ents[bb].v, dv});
                    td.push_back({ents[a].v, ents[bb].v, dv});
                    if (on_diag) adiag[ents[a].v] += dv;
                }
            }
        s = e;
    }
    // Contact weights w_c (solver_config_applier.cpp:34-47): m / h^2 * w_scale
    // on every dynamic vertex, or with use_heu_wc the GPU precompute's
    // heuristic on the dynamic surface vertices (admm_impl_gpu.cu:205-218),
    // max(sigma a_ii, min(beta m_i, a_ii)) * 10 / h^2, the others keeping 1e12.
    std::vector<double> wch2_h(n_all, 0.0);
    std::vector<float> wc_h(n_all, 1e12f), wcinv_h(n_all, 0.f);
    for (int i = 0; i < n; i++) {
        if (cfg.damp_km != 0) adiag[i] += h * cfg.damp_km * mass_h[i];
        double wci = mass_h[i] / h2 * cfg.w_scale;
        if (cfg.use_heu_wc) {
            wci = surface_h[i] ? std::max(cfg.wc_sigma * adiag[i], std::min(cfg.wc_beta * mass_h[i], adiag[i])) * 10.0 / h2 : 1e12;
            PA_CHECK(wci > 0, PA_ERR_INVALID, "heuristic contact weight is not positive (wc_sigma, wc_beta)");
        }
        wc_h[i] = (float)wci;
        wcinv_h[i] = wci >= 1e12 ? 0.f : (float)(1.0 / wci);
        ta.push_back({i, i, mass_h[i]});
        if (contact && surface_h[i]) {
            ta.push_back({i, i, h2 * wci});
            wch2_h[i] = h2 * wci; // the same FP64 value the matrix holds
        }
        if (cfg.damp_km != 0) {
            ta.push_back({i, i, h * cfg.damp_km * mass_h[i]});
            td.push_back({i, i, h * cfg.damp_km * mass_h[i]});
        }
    }
    auto to_csr = [&](std::vector<T3>& t, std::vector<int32_t>& ptr, std::vector<int32_t>& col, std::vector<double>& val) {
        std::sort(t.begin(), t.end(), [](const T3& a, const T3& b) { return a.r != b.r ? a.r < b.r : a.c < b.c; });
        ptr.assign(n + 1, 0);
        col.clear();
        val.clear();
        for (size_t s = 0; s < t.size();) {
            size_t e = s;
            double acc = 0;
            while (e < t.size() && t[e].r == t[s].r && t[e].c == t[s].c) acc += t[e++].v;
            col.push_back(t[s].c);
            val.push_back(acc);
            ptr[t[s].r + 1]++;
            s = e;
        }
        for (int i = 0; i < n; i++) ptr[i + 1] += ptr[i];
    };
    std::vector<int32_t> aptr, acol, dptr, dcol;
    std::vector<double> aval, dval;
    to_csr(ta, aptr, acol, aval);
    to_csr(td, dptr, dcol, dval);
    // split A into diagonal + off-diagonal
    std::vector<int32_t> optr(n + 1, 0), ocol;
    std::vector<float> oval, oval_lo, diag(n, 0.f), diag_lo(n, 0.f), dinv(n, 0.f);
    for (int i = 0; i < n; i++) {
        for (int e = aptr[i]; e < aptr[i + 1]; e++) {
            const float hi = (float)aval[e];
            const float lo = (float)(aval[e] - (double)hi);
            if (acol[e] == i) {
                diag[i] = hi;
                diag_lo[i] = lo;
            } else {
                ocol.push_back(acol[e]);
                oval.push_back(hi);
                oval_lo.push_back(lo);
            }
        }
        optr[i + 1] = (int32_t)ocol.size();
        PA_CHECK(diag[i] > 0, PA_ERR_NOT_SPD, "system matrix has a non-positive diagonal");
        dinv[i] = 1.f / diag[i];
    }
    nnz_a_off = (int64_t)ocol.size();
    nnz_dm = (int64_t)dcol.size();
    // AMG hierarchy on the full double-precision matrix
    use_amg = false;
    amg.clear();
    amg_sizes.clear();
    if (cfg.precond == 1) {
        HostCsr Ah;
        Ah.rows = Ah.cols = n;
        Ah.ptr.assign(aptr.begin(), aptr.end());
        Ah.col.assign(acol.begin(), acol.end());
        Ah.val.assign(aval.begin(), aval.end());
        AmgHierarchy H;
        bool ok = true;
        try {
            H = amg_build(Ah);
        } catch (const std::exception&) {
            ok = false;
        }
        if (ok && H.coarse_n <= 2048) {
            // the device kernels index vectors by these columns: check them once
            auto cols_ok = [](const HostCsr& M) {
                if ((int)M.ptr.size() != M.rows + 1 || M.ptr[M.rows] != (int32_t)M.col.size()) return false;
                for (int32_t c : M.col)
                    if (c < 0 || c >= M.cols) return false;
                return M.cols > 0;
            };
            for (size_t l = 0; l < H.levels.size(); l++) {
                const AmgLevel& L = H.levels[l];
                PA_CHECK(cols_ok(L.A) && (l + 1 == H.levels.size() || (cols_ok(L.P) && cols_ok(L.R))), PA_ERR_INVALID,
                         "AMG level with column indices out of range");
                auto D = std::make_unique<DevLevel>();
                D->n = L.A.rows;
                D->omega = (float)L.omega_smooth;
                D->lpr_a = lanes_per_row(L.A.nnz(), L.A.rows);
                amg_sizes.push_back(D->n);
                std::vector<float> av(L.A.val.begin(), L.A.val.end()), dv(L.dinv.begin(), L.dinv.end());
                D->aptr.upload(L.A.ptr, stream);
                D->acol.upload(L.A.col, stream);
                D->aval.upload(av, stream);
                D->dinv.upload(dv, stream);
                if (l + 1 < H.levels.size()) {
                    D->nnext = L.P.cols;
                    D->lpr_p = lanes_per_row(L.P.nnz(), L.P.rows);
                    D->lpr_r = lanes_per_row(L.R.nnz(), L.R.rows);
                    std::vector<float> pv(L.P.val.begin(), L.P.val.end()), rv(L.R.val.begin(), L.R.val.end());
                    D->pptr.upload(L.P.ptr, stream);
                    D->pcol.upload(L.P.col, stream);
                    D->pval.upload(pv, stream);
                    D->rptr.upload(L.R.ptr, stream);
                    D->rcol.upload(L.R.col, stream);
                    D->rval.upload(rv, stream);
                }
                D->b.alloc(3 * (size_t)D->n);
                D->x.alloc(3 * (size_t)D->n);
                D->x2.alloc(3 * (size_t)D->n);
                D->r.alloc(3 * (size_t)D->n);
                amg.push_back(std::move(D));
            }
            amg_nc = H.coarse_n;
            amg_ncp = (amg_nc + 3) & ~3;
            std::vector<float> ci((size_t)amg_nc * amg_ncp, 0.f);
            for (int i = 0; i < amg_nc; i++)
                for (int j = 0; j < amg_nc; j++) ci[(size_t)i * amg_ncp + j] = (float)H.coarse_inv[(size_t)i * amg_nc + j];
            amg_cinv.upload(ci, stream);
            use_amg = true;
        }
    }
    use_chol = false;
    if (cfg.precond == 2) chol_setup(aptr, acol, aval, x0h);
    // D^T We^2 h^2 gather, per vertex sorted by row
    std::vector<std::array<double, 3>> dt; // (v, row, coef)
    dt.reserve(ents.size());
    for (auto& e : ents) dt.push_back({(double)e.v, (double)e.row, h2 * e.w * e.w * e.g});
    std::sort(dt.begin(), dt.end(), [](const std::array<double, 3>& a, const std::array<double, 3>& b) {
        return a[0] != b[0] ? a[0] < b[0] : a[1] < b[1];
    });
    std::vector<int32_t> dtptr(n + 1, 0), dtrow(dt.size());
    std::vector<float> dtcoef(dt.size());
    for (size_t k = 0; k < dt.size(); k++) {
        dtptr[(int)dt[k][0] + 1]++;
        dtrow[k] = (int32_t)dt[k][1];
        dtcoef[k] = (float)dt[k][2];
    }
    for (int i = 0; i < n; i++) dtptr[i + 1] += dtptr[i];

    // ---- upload ----
    hipStream_t s = stream;
    
    x.alloc(3 * (size_t)n_all);
    x.upload(x0h, 3 * (size_t)n_all, s);
    x0.alloc(3 * (size_t)n_all);
    x0.upload(x0h, 3 * (size_t)n_all, s); // a step that fails before its prologue restores x from x0
    v.alloc(3 * (size_t)n_all);
    fill<double>(v.p, 0.0, 3 * (int64_t)n_all, s);
    {
        // pin targets in FP64: bpin_v = sum over the pins of v of h^2 w^2 x_pin (the pin rows of z are relative)
        std::vector<double> bp(3 * (size_t)n, 0.0);
        for (int c = 0; c < hc.n_pin; c++) {
            const int vtx = hc.pin_inds[c];
            const double cf = h2 * hc.pin_w[c] * hc.pin_w[c];
            for (int k = 0; k < 3; k++) bp[3 * (size_t)vtx + k] += cf * hc.pin_pos[3 * c + k];
        }
        bpin.upload(bp, s);
    }
    p.alloc(3 * (size_t)n_all);
    Ue.alloc(3 * (size_t)std::max(m, 1));
    fill<float>(Ue.p, 0.f, 3 * (int64_t)m, s);
    Uc.alloc(3 * (size_t)n);
    fill<float>(Uc.p, 0.f, 3 * (int64_t)n, s);
    z.alloc(3 * (size_t)std::max(m, 1));
    fill<float>(z.p, 0.f, 3 * (int64_t)m, s);
    zprev.alloc(3 * (size_t)std::max(m, 1));
    fill<float>(zprev.p, 0.f, 3 * (int64_t)m, s);
    b.alloc(3 * (size_t)n);
    bconst.alloc(3 * (size_t)n);
    mass.upload(mass_h, s);
    wc.upload(wc_h, s);
    wc_inv.upload(wcinv_h, s);
    mu_v.alloc(n_all);
    fill<float>(mu_v.p, (float)cfg.mu, n_all, s);
    wch2.upload(wch2_h, s);
    pinned.upload(pinned_h, s);
    // constraints
    {
        std::vector<int4> tv(hc.n_tri);
        std::vector<float4> tb(hc.n_tri);
        std::vector<float> tw(hc.n_tri);
        for (int c = 0; c < hc.n_tri; c++) {
            tv[c] = make_int4(hc.tri_inds[3 * c], hc.tri_inds[3 * c + 1], hc.tri_inds[3 * c + 2], 0);
            tb[c] = make_float4((float)hc.tri_binv[4 * c], (float)hc.tri_binv[4 * c + 1], (float)hc.tri_binv[4 * c + 2],
                                (float)hc.tri_binv[4 * c + 3]);
            tw[c] = (float)hc.tri_w[c];
        }
        tri_v.upload(tv, s);
        tri_binv.upload(tb, s);
        tri_w.upload(tw, s);
        std::vector<int4> qv(hc.n_tet);
        std::vector<float> qb(9 * (size_t)hc.n_tet), qw(hc.n_tet);
        for (int c = 0; c < hc.n_tet; c++) {
            qv[c] = make_int4(hc.tet_inds[4 * c], hc.tet_inds[4 * c + 1], hc.tet_inds[4 * c + 2], hc.tet_inds[4 * c + 3]);
            for (int k = 0; k < 9; k++) qb[9 * c + k] = (float)hc.tet_binv[9 * c + k];
            qw[c] = (float)hc.tet_w[c];
        }
        tet_v.upload(qv, s);
        tet_binv.upload(qb, s);
        tet_w.upload(qw, s);
        std::vector<float> bc(hc.bend_coef.begin(), hc.bend_coef.end()), bw(hc.bend_w.begin(), hc.bend_w.end());
        std::vector<double> bs(std::max(hc.n_bend, 1), 0.0);
        for (int c = 0; c < hc.n_bend; c++)
            for (int e = hc.bend_ptr[c]; e < hc.bend_ptr[c + 1]; e++) bs[c] += hc.bend_coef[e];
        bend_ptr.upload(hc.bend_ptr, s);
        bend_idx.upload(hc.bend_inds, s);
        bend_coef.upload(bc, s);
        bend_sum.upload(bs, s);
        bend_w.upload(bw, s);
        std::vector<float> pw(hc.n_pin);
        for (int c = 0; c < hc.n_pin; c++) pw[c] = (float)hc.pin_w[c];
        pin_v.upload(hc.pin_inds, s);
        pin_pos.upload(hc.pin_pos, s);
        pin_w.upload(pw, s);
    }
    dt_ptr.upload(dtptr, s);
    dt_row.upload(dtrow, s);
    dt_coef.upload(dtcoef, s);
    a_ptr.upload(optr, s);
    a_col.upload(ocol, s);
    a_val.upload(oval, s);
    a_val_lo.upload(oval_lo, s);
    a_diag.upload(diag, s);
    a_diag_lo.upload(diag_lo, s);
    a_dinv.upload(dinv, s);
    {
        dm_ptr.upload(dptr, s);
        dm_col.upload(dcol, s);
        dm_val.upload(dval, s);
    }
    cg_r.alloc(3 * (size_t)n);
    cg_z.alloc(3 * (size_t)n);
    cg_p.alloc(3 * (size_t)n);
    cg_q.alloc(3 * (size_t)n);
    cg_d.alloc(3 * (size_t)n);
    cg_r2.alloc(3 * (size_t)n);
    cg_p2.alloc(3 * (size_t)n);
    a_lpr = lanes_per_row(nnz_a_off + n, n);
    // two rows per lane group in the fused PCG kernels
    cg_blocks = std::max(1, std::min(grid_for((int64_t)n * a_lpr, 2 * (small_rows(n, a_lpr) ? SBLK : PBLK)), CG_MAX_BLOCKS));
    cg_part.alloc(9 * (size_t)cg_blocks);
    cg_state.alloc(24);
    int elem_blocks = grid_for(hc.n_tri, BLK) + grid_for(hc.n_tet, BLK) + grid_for(hc.n_bend, BLK) + grid_for(hc.n_pin, BLK);
    rhs_lpr = lanes_per_row((int64_t)dtrow.size(), n);
    res_blocks = std::max(std::max(elem_blocks, grid_for((int64_t)n * rhs_lpr, BLK)), 1); // >= every grid writing res_part
    res_part.alloc(6 * (size_t)res_blocks);
    res_sum.alloc(8);
    stop_ctl.alloc(1);
    // contact buffers sized by capacity
    const int cap = cfg.max_contacts;
    gam.alloc(cap);
    kc.alloc(cap);
    rc.alloc(cap);
    cslot.alloc(4 * (size_t)cap);
    gdu.alloc(4 * (size_t)cap);
    vcnt.alloc(n_all);
    vptr.alloc((size_t)n + 1);
    vloc.alloc(cap);
    vraw.alloc(4 * (size_t)cap);
    vent.alloc(4 * (size_t)cap);
    erun.alloc(4 * (size_t)cap);
    x_host.assign(x0h, x0h + 3 * (size_t)n_all);
    v_host.assign(3 * (size_t)n_all, 0.0);
    PA_HIP(hipStreamSynchronize(s));
}

// Attaching a detector to an initialised backend runs the reference's set-up
// check of the surface mesh against the contact distance
// (thickness_validation_check, src/contact/dcd_validation.h:8-33, enforced at
// app_initializer.cpp:186-188): a surface edge whose first vertex is dynamic
// must be at least d-hat long in the positions given to init, else the pair
// tests between neighbours would see the mesh's own edges as contacts.
void Backend::attach_detector(Detector* d) {
    PA_CHECK(d, PA_ERR_INVALID, "null detector");
    if (initialized) PA_CHECK(d->n_all == n_all, PA_ERR_INVALID, "detector vertex count differs from the backend");
    PA_CHECK(d->c.cap <= cfg.max_contacts, PA_ERR_INVALID, "detector capacity exceeds max_contacts");
    if (initialized) {
        double shortest = std::numeric_limits<double>::infinity();
        for (size_t k = 0; k + 1 < d->edges_h.size(); k += 2) {
            const int a = d->edges_h[k], b = d->edges_h[k + 1];
            if (a >= n) continue; // a static edge (static vertices follow the dynamic ones)
            double l2 = 0;
            for (int q = 0; q < 3; q++) {
                const double t = x_init_h[3 * (size_t)a + q] - x_init_h[3 * (size_t)b + q];
                l2 += t * t;
            }
            shortest = std::min(shortest, std::sqrt(l2));
        }
        PA_CHECK(!(shortest < d->dhat), PA_ERR_GEOMETRY,
                 "surface edge shorter than the contact distance (thickness): length " + std::to_string(shortest) + " < " +
                     std::to_string(d->dhat));
    }
    // work still queued on the detector's previous stream (the tail of a
    // detection) must finish before the backend's stream reads its lists
    if (d->stream && d->stream != stream) PA_HIP(hipStreamSynchronize(d->stream));
    det = d;
    det->set_stream(stream);
}

void Backend::detach_detector(const Detector* d) {
    if (!d || det != d) return;
    if (stream) (void)hipStreamSynchronize(stream); // no queued work may still read its lists
    det->stream = det->own_stream;
    det = nullptr;
    nc = 0;
    ws_forget();
}

static ElemArgs make_elem_args(const Backend& B) {
    ElemArgs a;
    const HostConstraints& h = B.hc;
    a.n_tri = h.n_tri;
    a.n_tet = h.n_tet;
    a.n_bend = h.n_bend;
    a.n_pin = h.n_pin;
    a.tri_row0 = h.tri_row0;
    a.tet_row0 = h.tet_row0;
    a.bend_row0 = h.bend_row0;
    a.pin_row0 = h.pin_row0;
    a.blk_tri = grid_for(h.n_tri, BLK);
    a.blk_tet = a.blk_tri + grid_for(h.n_tet, BLK);
    a.blk_bend = a.blk_tet + grid_for(h.n_bend, BLK);
    a.tri_v = B.tri_v.p;
    a.tri_binv = B.tri_binv.p;
    a.tri_w = B.tri_w.p;
    a.tet_v = B.tet_v.p;
    a.tet_binv = B.tet_binv.p;
    a.tet_w = B.tet_w.p;
    a.bend_ptr = B.bend_ptr.p;
    a.bend_idx = B.bend_idx.p;
    a.bend_coef = B.bend_coef.p;
    a.bend_w = B.bend_w.p;
    a.pin_v = B.pin_v.p;
    a.pin_pos = B.pin_pos.p;
    a.bend_sum = B.bend_sum.p;
    a.pin_w = B.pin_w.p;
    return a;
}

static int elem_grid(const ElemArgs& a, int n_pin) { return a.blk_bend + grid_for(n_pin, BLK); }

// z = prox(D x + Ue) at the step's first x.
void Backend::local_step() {
    ElemArgs a = make_elem_args(*this);
    int g = elem_grid(a, hc.n_pin);
    if (g == 0) return;
    hipLaunchKernelGGL(k_elem<ELEM_LOCAL>, dim3(g), dim3(BLK), 0, stream, a, 0, x.p, Ue.p, z.p, (float*)nullptr, (double*)nullptr,
                       (const int32_t*)nullptr);
    PA_LAUNCH_CHECK();
}

// Applies a deferred global-solve correction to x as well, which elem_update
// then reads.
void Backend::dual_vertices(bool want_res) {
    hipLaunchKernelGGL(k_dual_vert, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, n, (float)cfg.dt, (float)(1.0 / cfg.dt),
                       cfg.enable_contact, want_res ? 1 : 0, x.p, x0.p, p.p, wch2.p, Uc.p, res_part.p, 1.0 / (cfg.dt * cfg.dt),
                       (const int32_t*)stop_guard, dx_pending ? (const float*)chol_x.p : nullptr, (const int32_t*)chol_ipos.p);
    PA_LAUNCH_CHECK();
    dx_pending = false;
}

// The elastic dual update of this iteration and, unless it is the last, the
// local step of the next one (next_check: that one's residual needs zprev).
void Backend::elem_update(bool want_res, bool last, bool next_check) {
    ElemArgs a = make_elem_args(*this);
    const int g = elem_grid(a, hc.n_pin);
    if (g == 0) return;
    hipLaunchKernelGGL((last ? k_elem<ELEM_DUAL> : k_elem<ELEM_DUAL | ELEM_LOCAL>), dim3(g), dim3(BLK), 0, stream, a, want_res ? 1 : 0, x.p, Ue.p,
                       z.p, next_check ? zprev.p : (float*)nullptr, res_part.p, (const int32_t*)stop_guard);
    PA_LAUNCH_CHECK();
}

// counted: the detection has filled vcnt and vloc.
void Backend::contact_setup(float eps, float gamma_, float hinv, bool counted) {
    nc = det ? det->n_contacts : 0;
    if (nc == 0) return;
    if (!counted) {
        fill<uint32_t>(vcnt.p, 0u, n_all, stream);
        hipLaunchKernelGGL(k_contact_count, dim3(grid_for(nc, BLK)), dim3(BLK), 0, stream, nc, (const int4*)det->c.v.p, vcnt.p, vloc.p);
        PA_LAUNCH_CHECK();
    }
    // per-vertex contact entries over dynamic vertices; static vertices keep
    // their counts (they enter S_c) but get no entries
    scan_exclusive(vcnt.p, vptr.p, n, vptr.p + n, scratch, stream);
    hipLaunchKernelGGL(k_contact_fill, dim3(grid_for(nc, BLK)), dim3(BLK), 0, stream, nc, n, eps, gamma_, hinv, (const int4*)det->c.v.p,
                       (const int4*)vloc.p, (const uint32_t*)vptr.p, vraw.p, (const float4*)det->c.bary.p, (const float4*)det->c.nrm.p,
                       (const uint32_t*)vcnt.p, (const float*)wc.p, (const float*)wc_inv.p, (const float*)mu_v.p, gam.p, kc.p, rc.p);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_contact_rank, dim3(grid_for(4 * (int64_t)nc, BLK)), dim3(BLK), 0, stream, nc, n, (const int4*)det->c.v.p,
                       (const uint32_t*)vptr.p, (const uint32_t*)vraw.p, vent.p, cslot.p, erun.p);
    PA_LAUNCH_CHECK();
}

void Backend::contact_project(bool) {
    if (nc == 0) return;
    if (nc <= contact_wg_max) { // the whole projection in one workgroup: no launch per sweep
        hipLaunchKernelGGL((nc <= 1024 ? k_contact_sweeps_wg<1> : k_contact_sweeps_wg<2>), dim3(1), dim3(1024), 0, stream, nc, n,
                           cfg.gs_max_iter, det->c.v.p, det->c.bary.p, det->c.nrm.p, kc.p, p.p, rc.p, (const float4*)gam.p,
                           (const int4*)cslot.p, (const uint32_t*)vptr.p, (const int2*)erun.p, (const int32_t*)stop_guard);
        PA_LAUNCH_CHECK();
        return;
    }
    hipLaunchKernelGGL(k_vertex_p, dim3(grid_for(4 * (int64_t)nc, BLK)), dim3(BLK), 0, stream, 4 * nc, n, p.p, (const uint32_t*)vptr.p,
                       (const int2*)erun.p, (const uint32_t*)vent.p, (const float4*)gam.p, (const float4*)rc.p);
    PA_LAUNCH_CHECK();
    for (int g = 0; g < cfg.gs_max_iter; g++) contact_sweep_once();
}

void Backend::contact_sweep_once() {
    hipLaunchKernelGGL(k_contact_du, dim3(grid_for(nc, BLK)), dim3(BLK), 0, stream, nc, det->c.v.p, det->c.bary.p,
                       det->c.nrm.p, kc.p, p.p, rc.p, (const float4*)gam.p, (const int4*)cslot.p, gdu.p, (const int32_t*)stop_guard);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_vertex_gather, dim3(grid_for(4 * (int64_t)nc, BLK)), dim3(BLK), 0, stream, 4 * nc, n, p.p,
                       (const uint32_t*)vptr.p, (const int2*)erun.p, (const float4*)gdu.p);
    PA_LAUNCH_CHECK();
}

// The right-hand side, and with the direct solve also the residual of its
// first pass (cg_r): global_solve then starts from it.
void Backend::rhs(bool want_res, bool first_iter) {
    const ResidArgs A{a_ptr.p, a_col.p, a_val.p, a_val_lo.p, a_diag.p, a_diag_lo.p, x.p, cg_r.p, chol_ipos.p};
    const int store_b = cfg.global_refine > 1 ? 1 : 0;
    with_lpr(rhs_lpr, [&](auto c) {
        constexpr int P = decltype(c)::value;
        hipLaunchKernelGGL((use_chol ? (want_res ? k_rhs<P, true, true> : k_rhs<P, true, false>)
                                     : (want_res ? k_rhs<P, false, true> : k_rhs<P, false, false>)),
                           dim3(grid_for((int64_t)n * P, BLK)), dim3(BLK), 0, stream, n, (float)cfg.dt, cfg.enable_contact,
                           first_iter ? 1 : 0, store_b, dt_ptr.p, dt_row.p, dt_coef.p,
                           z.p, zprev.p, Ue.p, bconst.p, wch2.p, p.p, x0.p, Uc.p, bpin.p, b.p, res_part.p, A);
    });
    PA_LAUNCH_CHECK();
}

// Per-launch time (ms) of the measured solver kernel (PCG SpMV, or the direct
// solve's dense-top product): `reps` launches back-to-back
// on the backend's stream between two events, on the current device vectors
// (run between steps: it only writes PCG scratch).  This is the kernel's own
// duration plus the gap between consecutive launches; an event pair around a
// single launch inside the solve also holds the dispatch latency.
double Backend::spmv_time_ms(int reps) {
    PA_CHECK(initialized, PA_ERR_INVALID, "init first");
    PA_CHECK(reps > 0 && reps <= 100000, PA_ERR_INVALID, "reps out of range");
    const int nb = cg_blocks;
    const bool fused = use_amg && amg.size() >= 2;
    PA_CHECK(!use_chol || chol_top_tiles > 0, PA_ERR_INVALID, "the direct solve has no dense top to time");
    hipEvent_t e0, e1;
    PA_HIP(hipEventCreate(&e0));
    PA_HIP(hipEventCreate(&e1));
    float ms = 0.f;
    try {
        PA_HIP(hipEventRecord(e0, stream));
        for (int r = 0; r < reps; r++) {
            if (use_chol) { // the dense-top product on the last solve's vectors
                chol_top_launch(cg_r.p);
                continue;
            }
            with_lpr(a_lpr, [&](auto c) {
                constexpr int P = decltype(c)::value;
                if (fused)
                    hipLaunchKernelGGL((small_rows(n, a_lpr)     ? k_cg_dir_spmv<P, false, SBLK>
                                        : multi_pass(n, nb, P) ? k_cg_dir_spmv<P, true, PBLK>
                                                               : k_cg_dir_spmv<P, false, PBLK>),
                                       dim3(nb), dim3(small_rows(n, a_lpr) ? SBLK : PBLK), 0, stream, n, 0, 0, nb, cg_state.p, a_ptr.p, a_col.p,
                                       a_val.p, a_diag.p, (const float*)cg_z.p, (const float*)cg_p.p, cg_p2.p, cg_q.p, cg_part.p);
                else
                    hipLaunchKernelGGL(k_cg_spmv<P>, dim3(nb), dim3(PBLK), 0, stream, n, a_ptr.p, a_col.p, a_val.p, a_diag.p,
                                       (const float*)cg_p.p, cg_q.p, cg_part.p);
            });
            PA_LAUNCH_CHECK();
        }
        PA_HIP(hipEventRecord(e1, stream));
        PA_HIP(hipEventSynchronize(e1));
        PA_HIP(hipEventElapsedTime(&ms, e0, e1));
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return (double)ms / reps;
}

hipEvent_t Backend::next_event() {
    if (ev_next >= ev_pool.size()) {
        hipEvent_t e;
        PA_HIP(hipEventCreate(&e));
        ev_pool.push_back(e);
    }
    return ev_pool[ev_next++];
}

// z = P^-1 r for the PCG: Jacobi, or one AMG V-cycle (downward pre-smoothing
// and restriction, dense coarse solve, upward prolongation and
// post-smoothing).  Both variants leave the r.z partials at 6..8 of cg_part.
void Backend::precondition(const float* r, bool skip_pre0) {
    const int nb = cg_blocks;
    if (!use_amg) {
        hipLaunchKernelGGL(k_jacobi_prec, dim3(nb), dim3(PBLK), 0, stream, n, a_dinv.p, r, cg_z.p, cg_part.p);
        PA_LAUNCH_CHECK();
        return;
    }
    const int nl = (int)amg.size();
    // downward: level 0 takes b = cg_r
    for (int l = 0; l + 1 < nl; l++) {
        DevLevel& L = *amg[l];
        DevLevel& C = *amg[l + 1];
        const float* bl = l == 0 ? r : L.b.p;
        if (!(l == 0 && skip_pre0)) {
            with_lpr(L.lpr_a, [&](auto c) {
                constexpr int P = decltype(c)::value;
                hipLaunchKernelGGL(k_amg_pre<P>, dim3(grid_for((int64_t)L.n * P, BLK)), dim3(BLK), 0, stream, L.n, L.aptr.p, L.acol.p,
                                   L.aval.p, L.dinv.p, L.omega, bl, L.x.p, L.r.p);
            });
            PA_LAUNCH_CHECK();
        }
        with_lpr(L.lpr_r, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL(k_amg_spmv<P>, dim3(grid_for((int64_t)L.nnext * P, BLK)), dim3(BLK), 0, stream, L.nnext, L.rptr.p,
                               L.rcol.p, L.rval.p, (const float*)L.r.p, (const float*)nullptr, C.b.p);
        });
        PA_LAUNCH_CHECK();
    }
    DevLevel& Cl = *amg[nl - 1];
    const float* bc = nl == 1 ? r : Cl.b.p;
    float* xc = nl == 1 ? cg_z.p : Cl.x2.p;
    hipLaunchKernelGGL(k_amg_coarse, dim3(grid_for(amg_nc, (BLK / 64) * CROWS)), dim3(BLK), 0, stream, amg_nc, amg_ncp,
                       (const float4*)amg_cinv.p, bc, xc);
    PA_LAUNCH_CHECK();
    if (nl == 1) { // the whole system is the coarse level: exact solve, then r.z partials
        hipLaunchKernelGGL(k_rz_part, dim3(nb), dim3(PBLK), 0, stream, n, r, cg_z.p, cg_part.p);
        PA_LAUNCH_CHECK();
        return;
    }
    // upward: x_l += P x_{l+1}, then post-smooth into x2_l (cg_z on level 0)
    for (int l = nl - 2; l >= 0; l--) {
        DevLevel& L = *amg[l];
        const float* bl = l == 0 ? r : L.b.p;
        with_lpr(L.lpr_p, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL(k_amg_spmv<P>, dim3(grid_for((int64_t)L.n * P, BLK)), dim3(BLK), 0, stream, L.n, L.pptr.p, L.pcol.p,
                               L.pval.p, (const float*)amg[l + 1]->x2.p, (const float*)L.x.p, L.x.p);
        });
        PA_LAUNCH_CHECK();
        float* out = l == 0 ? cg_z.p : L.x2.p;
        // level 0 emits r.z partials, so it runs on the partial-sum grid
        with_lpr(L.lpr_a, [&](auto c) {
            constexpr int P = decltype(c)::value;
            const bool small = l == 0 ? small_rows(n, a_lpr) : small_rows(L.n, P);
            const int grid = l == 0 ? nb : grid_for((int64_t)L.n * P, small ? SBLK : PBLK);
            hipLaunchKernelGGL((small                     ? k_amg_post<P, false, SBLK>
                                : multi_pass(L.n, grid, P) ? k_amg_post<P, true, PBLK>
                                                           : k_amg_post<P, false, PBLK>),
                               dim3(grid), dim3(small ? SBLK : PBLK), 0, stream,
                               L.n, L.aptr.p, L.acol.p, L.aval.p, L.dinv.p, L.omega,
                               bl, (const float*)L.x.p, out, l == 0 ? cg_part.p : (double*)nullptr);
        });
        PA_LAUNCH_CHECK();
    }
}

// Mixed-precision refinement: each pass computes the FP64 residual
// r_0 = b - A x of the FP32 iterate, solves A d = r_0 with preconditioned FP32
// CG until |r_k| <= tol |r_0| per column (the recursive residual), and adds d.
// A later pass runs only while the FP64 residual exceeds 1e-12 |b|.  Iterations are
// launched in chunks between convergence read-backs; the first chunk is sized
// by the previous solve's count (consecutive ADMM iterations need similar
// counts).  Returns the PCG iterations summed over passes.
// One PCG iteration `it` (state slot it & 1).  Fused AMG path: k_cg_dir_spmv,
// k_cg_update_pre and the rest of the V-cycle, with the p and r ping-pong
// buffers selected by pc / rc (toggled here).  Plain path: SpMV, update,
// preconditioner, direction.
void Backend::pcg_iteration(int it, bool fused, int& pc, int& rc) {
    const int nb = cg_blocks;
    const int slot = it & 1;
    float* pbuf[2] = {cg_p.p, cg_p2.p};
    float* rbuf[2] = {cg_r.p, cg_r2.p};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const bool mark = (profiling & 1) && !capturing;
    if (mark) {
        e0 = next_event();
        e1 = next_event();
        PA_HIP(hipEventRecord(e0, stream));
    }
    if (fused) {
        with_lpr(a_lpr, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL((small_rows(n, a_lpr)     ? k_cg_dir_spmv<P, false, SBLK>
                                : multi_pass(n, nb, P) ? k_cg_dir_spmv<P, true, PBLK>
                                                       : k_cg_dir_spmv<P, false, PBLK>),
                               dim3(nb), dim3(small_rows(n, a_lpr) ? SBLK : PBLK), 0, stream,
                               n, it == 0 ? 1 : 0, slot ^ 1, nb, cg_state.p, a_ptr.p,
                               a_col.p, a_val.p, a_diag.p, (const float*)cg_z.p, (const float*)pbuf[pc], pbuf[pc ^ 1], cg_q.p,
                               cg_part.p);
        });
        pc ^= 1;
    } else {
        with_lpr(a_lpr, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL(k_cg_spmv<P>, dim3(nb), dim3(PBLK), 0, stream, n, a_ptr.p, a_col.p, a_val.p, a_diag.p,
                               (const float*)cg_p.p, cg_q.p, cg_part.p);
        });
    }
    PA_LAUNCH_CHECK();
    if (mark) {
        PA_HIP(hipEventRecord(e1, stream));
        spmv_marks.push_back({e0, e1});
    }
    if (fused) {
        DevLevel& L0 = *amg[0];
        with_lpr(L0.lpr_a, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL((small_rows(n, a_lpr)     ? k_cg_update_pre<P, false, SBLK>
                                : multi_pass(n, nb, P) ? k_cg_update_pre<P, true, PBLK>
                                                       : k_cg_update_pre<P, false, PBLK>),
                               dim3(nb), dim3(small_rows(n, a_lpr) ? SBLK : PBLK), 0, stream, n, slot, nb, cg_state.p, L0.aptr.p, L0.acol.p,
                               L0.aval.p, L0.dinv.p, L0.omega, (const float*)pbuf[pc], (const float*)cg_q.p, cg_d.p,
                               (const float*)rbuf[rc], rbuf[rc ^ 1], L0.x.p, L0.r.p, cg_part.p);
        });
        PA_LAUNCH_CHECK();
        rc ^= 1;
        precondition(rbuf[rc], true);
    } else {
        hipLaunchKernelGGL(k_cg_update, dim3(nb), dim3(PBLK), 0, stream, n, slot, nb, cg_state.p, cg_p.p, cg_q.p, cg_d.p, cg_r.p,
                           cg_part.p);
        PA_LAUNCH_CHECK();
        precondition(cg_r.p);
        hipLaunchKernelGGL(k_cg_dir, dim3(nb), dim3(PBLK), 0, stream, n, slot, nb, cg_state.p, cg_z.p, cg_p.p, cg_part.p);
        PA_LAUNCH_CHECK();
    }
}

// Two fused iterations (it, it + 1 with it even, so the state slots and the
// ping-pong buffers return to where they started) captured once as a HIP
// graph: index 1 holds the first pair of a solve (it = 0, direction = z),
// index 0 every later pair.  One graph launch replaces twenty kernel
// launches, which the host cannot issue as fast as these short kernels run.
// The captured arguments are the backend's persistent buffers, so the graphs
// stay valid for the backend's lifetime.
hipGraphExec_t Backend::pcg_pair_graph(bool first_pair) {
    hipGraphExec_t& g = pcg_graph[first_pair ? 1 : 0];
    if (g) return g;
    hipGraph_t graph = nullptr;
    PA_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    capturing = true;
    try {
        int pc = 0, rc = 0;
        pcg_iteration(first_pair ? 0 : 2, true, pc, rc);
        pcg_iteration(first_pair ? 1 : 3, true, pc, rc);
    } catch (...) {
        capturing = false;
        hipGraph_t tmp = nullptr;
        (void)hipStreamEndCapture(stream, &tmp);
        if (tmp) (void)hipGraphDestroy(tmp);
        throw;
    }
    capturing = false;
    PA_HIP(hipStreamEndCapture(stream, &graph));
    const hipError_t e = hipGraphInstantiate(&g, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
        g = nullptr;
        PA_HIP(e);
    }
    return g;
}

// Mixed-precision refinement: each pass computes the FP64 residual
// r_0 = b - A x of the FP32 iterate, solves A d = r_0 with preconditioned FP32
// CG until |r_k| <= tol |r_0| per column (the recursive residual), and adds d.
// A later pass runs only while the FP64 residual exceeds 1e-12 |b|.
// Iterations are launched in chunks between convergence read-backs (the first
// chunk sized by the previous solve's count); on the fused path a chunk is a
// sequence of graph-launched iteration pairs.  Returns the PCG iterations
// summed over passes.
// Batched scenes on the global AMG-PCG: per-scene |r|^2 (one workgroup per
// scene).  k_scene_norms keeps them as the pass's initial residuals;
// k_scene_check counts the scenes with a column above tol^2 |r0|^2 and records,
// per scene, the iteration at which it first met its tolerance.
__global__ void __launch_bounds__(BLK) k_scene_norms(const int32_t* __restrict__ off, const float* __restrict__ r,
                                                      double* __restrict__ out) {
    const int s = blockIdx.x;
    double acc[3] = {0, 0, 0};
    for (int i = off[s] + threadIdx.x; i < off[s + 1]; i += BLK) {
        const float3 ri = ld3(r, i);
        acc[0] += (double)ri.x * ri.x;
        acc[1] += (double)ri.y * ri.y;
        acc[2] += (double)ri.z * ri.z;
    }
    block_sum_write<3>(acc, out, 3, 0);
}

__global__ void __launch_bounds__(BLK) k_scene_check(const int32_t* __restrict__ off, const float* __restrict__ r,
                                                      const double* __restrict__ r0, double tol2, int it, int32_t* __restrict__ first_it,
                                                      uint32_t* __restrict__ open) {
    __shared__ double sh[3][BLK / 64];
    const int s = blockIdx.x;
    double acc[3] = {0, 0, 0};
    for (int i = off[s] + threadIdx.x; i < off[s + 1]; i += BLK) {
        const float3 ri = ld3(r, i);
        acc[0] += (double)ri.x * ri.x;
        acc[1] += (double)ri.y * ri.y;
        acc[2] += (double)ri.z * ri.z;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < 3; k++) {
        double v = acc[k];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) sh[k][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        bool ok = true;
        for (int k = 0; k < 3; k++) {
            double v = 0;
            for (int w = 0; w < BLK / 64; w++) v += sh[k][w];
            ok = ok && v <= tol2 * r0[3 * s + k];
        }
        if (!ok) atomicAdd(open, 1u);
        else if (first_it[s] < 0) first_it[s] = it;
    }
}

// iters[s] += the iteration at which scene s met its tolerance (all of them if it did not)
__global__ void k_scene_accum(int nscene, const int32_t* __restrict__ first, int total, int32_t* __restrict__ iters) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nscene) iters[s] += first[s] >= 0 ? first[s] : total;
}

void Backend::chol_setup(const std::vector<int32_t>& aptr, const std::vector<int32_t>& acol, const std::vector<double>& aval,
                         const double* x0h) {
    const auto t0 = std::chrono::steady_clock::now();
    HostCsr Ah;
    Ah.rows = Ah.cols = n;
    Ah.ptr = aptr;
    Ah.col = acol;
    Ah.val = aval;
    SupernodalFactor F;
    try {
        F = chol_factor(Ah, x0h, n <= CHOL_BIG_LEAF_N ? 160 : 64, CHOL_TOP_MAX);
    } catch (const std::exception& e) {
        throw Error(PA_ERR_NOT_SPD, std::string("direct solve set-up: ") + e.what());
    }
    const int ns = F.nsuper;
    PA_CHECK(F.below.size() < ((size_t)1 << 31), PA_ERR_INVALID, "direct solve: too many rows below the diagonal blocks");
    // supernodes below the dense tops by height
    chol_levels = F.lower_levels;
    std::vector<int32_t> lvl_ptr(chol_levels + 1, 0);
    for (int k = 0; k < ns; k++)
        if (!F.is_top[k]) lvl_ptr[F.height[k] + 1]++;
    for (int h = 0; h < chol_levels; h++) lvl_ptr[h + 1] += lvl_ptr[h];
    std::vector<int32_t> lvl_sup(lvl_ptr[chol_levels]);
    {
        std::vector<int32_t> fill(lvl_ptr.begin(), lvl_ptr.end() - 1);
        for (int k = 0; k < ns; k++)
            if (!F.is_top[k]) lvl_sup[fill[F.height[k]]++] = k;
    }
    // panels [D; -W], column-major, both blocks' rows padded to whole float4s
    auto pad4 = [](int64_t v) { return (v + 3) & ~(int64_t)3; };
    std::vector<int64_t> panel_off(ns + 1, 0);
    for (int k = 0; k < ns; k++) panel_off[k + 1] = panel_off[k] + (F.is_top[k] ? 0 : (pad4(F.width(k)) + pad4(F.nbelow(k))) * F.width(k));
    std::vector<float> panels(std::max<int64_t>(4, panel_off[ns]), 0.f);
    {
        std::atomic<int> next{0};
        auto work = [&, max_nb = (size_t)F.max_rows]() noexcept {
            std::unique_ptr<double[]> col(new (std::nothrow) double[max_nb + 1]);
            if (!col) return; // the other workers, or the check below, take the rest
            for (int k; (k = next.fetch_add(1)) < ns;) {
                if (F.is_top[k]) continue;
                const int64_t w = F.width(k), nb = F.nbelow(k), nr = w + nb, wp = pad4(w), ld = wp + pad4(nb);
                const double* L21 = F.panel.data() + F.panel_off[k] + w;
                const double* Li = F.linv.data() + F.inv_off[k];
                for (int64_t i = 0; i < w; i++) {
                    float* o = panels.data() + panel_off[k] + i * ld;
                    for (int64_t j = 0; j < w; j++) { // D = L11^-T L11^-1
                        double acc = 0;
                        for (int64_t q = std::max(i, j); q < w; q++) acc += Li[i * w + q] * Li[j * w + q];
                        o[j] = (float)acc;
                    }
                    std::fill_n(col.get(), nb, 0.0); // column i of W = L21 L11^-1
                    for (int64_t q = i; q < w; q++) {
                        const double l = Li[i * w + q];
                        const double* c = L21 + q * nr;
                        for (int64_t j = 0; j < nb; j++) col[j] += c[j] * l;
                    }
                    for (int64_t j = 0; j < nb; j++) o[wp + j] = (float)-col[j];
                }
            }
        };
        std::vector<std::thread> pool;
        const unsigned nt = std::max(1u, std::min({16u, std::thread::hardware_concurrency(), (unsigned)std::max(1, ns / 8)}));
        try {
            pool.reserve(nt);
            for (unsigned q = 1; q < nt; q++) pool.emplace_back(work);
        } catch (const std::exception&) { // fewer workers
        }
        work();
        for (std::thread& q : pool) q.join();
        PA_CHECK(next.load() >= ns, PA_ERR_INVALID, "direct solve set-up: out of memory");
    }
    // where the rows of every front come from: the children's update-vector entries
    std::vector<int32_t> gat_off(ns, 0), gat_rows;
    for (int k = 0; k < ns; k++) {
        const int kids = F.child_ptr[k + 1] - F.child_ptr[k];
        if (F.is_top[k] || kids == 0) continue;
        PA_CHECK(gat_rows.size() < ((size_t)1 << 30), PA_ERR_INVALID, "direct solve: front tables too large");
        gat_off[k] = (int32_t)gat_rows.size();
        gat_rows.resize(gat_rows.size() + (size_t)kids * (F.width(k) + F.nbelow(k)), -1);
        for (int q = 0; q < kids; q++) {
            const int c = F.child[F.child_ptr[k] + q];
            for (int64_t e = F.below_ptr[c]; e < F.below_ptr[c + 1]; e++) gat_rows[gat_off[k] + (size_t)F.rel[e] * kids + q] = (int32_t)e;
        }
    }
    if (gat_rows.empty()) gat_rows.push_back(-1);
    // tiles of every level.  The tile size is the largest that still gives the
    // level CHOL_TILES_MIN workgroups (one per CU): narrow levels of large
    // fronts spread over the chip, wide ones gather each front fewer times
    // (256x256 cloth step: 13.7 ms at 2048, 13.0 at 1024, 12.5 at 256, 12.4 at 128).
    constexpr int CHOL_TILES_MIN = 256;
    std::vector<CholTile> up, down;
    chol_up_ptr.assign(chol_levels + 1, 0);
    chol_down_ptr.assign(chol_levels + 1, 0);
    chol_rg.assign(chol_levels, 16);
    chol_lp.assign(chol_levels, 8);
    chol_up_lds.assign(chol_levels, 0);
    chol_down_lds.assign(chol_levels, 0);
    for (int h = 0; h < chol_levels; h++) {
        auto count = [&](bool rows, int size) {
            int64_t c = 0;
            for (int q = lvl_ptr[h]; q < lvl_ptr[h + 1]; q++) {
                const int v = rows ? F.nbelow(lvl_sup[q]) : F.width(lvl_sup[q]);
                c += std::max(1, (v + size - 1) / size);
            }
            return c;
        };
        while (chol_rg[h] > 4 && count(true, 4 * chol_rg[h]) < CHOL_TILES_MIN) chol_rg[h] /= 2;
        while (chol_lp[h] < 32 && count(false, CHOL_BLK / chol_lp[h]) < CHOL_TILES_MIN) chol_lp[h] *= 2;
        for (int q = lvl_ptr[h]; q < lvl_ptr[h + 1]; q++) {
            const int k = lvl_sup[q], w = F.width(k), nb = F.nbelow(k);
            PA_CHECK(w <= 4096 && nb <= 4096, PA_ERR_INVALID, "direct solve: a supernode is too large (use precond 1)");
            CholTile T{panel_off[k], F.col0[k], w, nb, 0, (int32_t)F.below_ptr[k], gat_off[k], F.child_ptr[k + 1] - F.child_ptr[k], 0};
            for (T.first = 0; T.first < std::max(1, nb); T.first += 4 * chol_rg[h]) up.push_back(T);
            for (T.first = 0; T.first < w; T.first += CHOL_BLK / chol_lp[h]) down.push_back(T);
            chol_up_lds[h] = std::max(chol_up_lds[h], (int)sizeof(float4) * std::max(1, w));
            chol_down_lds[h] = std::max<int>(chol_down_lds[h], (int)sizeof(float) * 3 * (pad4(w) + pad4(nb)));
        }
        PA_CHECK(chol_up_lds[h] <= 65536 - 4096 && chol_down_lds[h] <= 65536, PA_ERR_INVALID,
                 "direct solve: a front is too large for one workgroup's LDS (use precond 1)");
        chol_up_ptr[h + 1] = (int32_t)up.size();
        chol_down_ptr[h + 1] = (int32_t)down.size();
    }
    // dense tops: workgroup tiles, LDS, and S^-1 with padded rows
    std::vector<int2> tiles;
    int max_m = 0;
    std::vector<int64_t> sinv_off(F.sinv_off.size(), 0);
    for (size_t blk = 0; blk + 1 < F.top_ptr.size(); blk++) {
        const int m = (int)(F.top_ptr[blk + 1] - F.top_ptr[blk]);
        max_m = std::max(max_m, m);
        for (int r0 = 0; r0 < m; r0 += CHOL_TOP_ROWS) tiles.push_back(make_int2((int)blk, r0));
        if (blk + 1 < sinv_off.size()) sinv_off[blk + 1] = sinv_off[blk] + (int64_t)m * pad4(m);
    }
    PA_CHECK(max_m <= CHOL_TOP_MAX, PA_ERR_INVALID, "direct solve: a dense top is too large");
    std::vector<float> sinv;
    for (size_t blk = 0; blk + 1 < F.top_ptr.size(); blk++) {
        const int64_t m = F.top_ptr[blk + 1] - F.top_ptr[blk], mp = pad4(m);
        sinv.resize(sinv_off[blk] + m * mp, 0.f);
        const double* S = F.sinv.data() + F.sinv_off[blk];
        for (int64_t i = 0; i < m; i++)
            for (int64_t j = 0; j < m; j++) sinv[sinv_off[blk] + i * mp + j] = (float)S[i * m + j];
    }
    if (sinv.empty()) sinv.push_back(0.f);
    chol_top_tiles = (int)tiles.size();
    chol_top_nv = 1;
    while (256 * chol_top_nv < max_m) chol_top_nv *= 2;
    chol_top_lds = (int)sizeof(float) * 3 * (int)pad4(std::max(max_m, 4));
    // per top entry a fixed-width list of the update-vector entries it gathers (-1: none)
    const size_t ntop = F.top_pos.size();
    chol_gmax = 1;
    for (size_t q = 0; q < ntop; q++) chol_gmax = std::max<int>(chol_gmax, (int)(F.gat_ptr[q + 1] - F.gat_ptr[q]));
    PA_CHECK(chol_gmax <= CHOL_TOP_GMAX, PA_ERR_INVALID, "direct solve: a dense-top entry gathers too many update vectors");
    std::vector<int64_t> gat_fix(std::max<size_t>(1, ntop) * chol_gmax, -1);
    for (size_t q = 0; q < ntop; q++)
        for (int64_t e = F.gat_ptr[q]; e < F.gat_ptr[q + 1]; e++) gat_fix[q * chol_gmax + (e - F.gat_ptr[q])] = F.gat[e];
    auto nonempty = [](std::vector<int32_t> v) {
        if (v.empty()) v.push_back(0);
        return v;
    };
    if (up.empty()) up.push_back(CholTile{});
    if (down.empty()) down.push_back(CholTile{});
    if (tiles.empty()) tiles.push_back(make_int2(0, 0));
    chol_up_tiles.reserve(up.size() * sizeof(CholTile));
    chol_up_tiles.upload(reinterpret_cast<const uint8_t*>(up.data()), up.size() * sizeof(CholTile), stream);
    chol_down_tiles.reserve(down.size() * sizeof(CholTile));
    chol_down_tiles.upload(reinterpret_cast<const uint8_t*>(down.data()), down.size() * sizeof(CholTile), stream);
    chol_panels.upload(panels, stream);
    chol_gat_rows.upload(gat_rows, stream);
    chol_ipos.upload(F.iperm, stream);
    chol_below.upload(nonempty(F.below), stream);
    chol_top_ptr.upload(F.top_ptr, stream);
    chol_top_pos.upload(nonempty(F.top_pos), stream);
    chol_gat.upload(gat_fix, stream);
    chol_sinv_off.upload(sinv_off, stream);
    chol_sinv.upload(sinv, stream);
    chol_tiles.upload(tiles, stream);
    chol_f.alloc(3 * (size_t)n);
    chol_x.alloc(3 * (size_t)n);
    chol_u.alloc(3 * std::max<size_t>(1, F.below.size()));
    chol_ftop.alloc(3 * std::max<size_t>(1, ntop));
    chol_entries = panel_off[ns] + (int64_t)sinv.size();
    chol_top_cols = (int64_t)F.top_pos.size();
    chol_top_sq = (int64_t)F.sinv.size();
    use_chol = true;
    chol_setup_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

// The dense-top product; r: the residual in elimination order, which is the
// right-hand side itself where there is no level below the tops.
void Backend::chol_top_launch(const float* r) {
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(chol_top_tiles), dim3(CHOL_TOP_BLK), chol_top_lds, stream, (const int2*)chol_tiles.p,
                           (const int64_t*)chol_top_ptr.p, (const int32_t*)chol_top_pos.p, (const int64_t*)chol_sinv_off.p,
                           (const float*)chol_sinv.p, chol_levels > 0 ? (const float*)chol_ftop.p : r,
                           chol_levels > 0 ? (const int32_t*)nullptr : (const int32_t*)chol_top_pos.p, chol_x.p);
    };
    switch (chol_top_nv) {
    case 1: go(k_chol_top<1>); break;
    case 2: go(k_chol_top<2>); break;
    case 4: go(k_chol_top<4>); break;
    case 8: go(k_chol_top<8>); break;
    default: go(k_chol_top<16>); break;
    }
    PA_LAUNCH_CHECK();
}

// chol_x = A^-1 r, both in elimination order (3 interleaved columns, FP32).
void Backend::chol_solve(const float* r) {
    const CholTile* up = reinterpret_cast<const CholTile*>(chol_up_tiles.p);
    const CholTile* down = reinterpret_cast<const CholTile*>(chol_down_tiles.p);
    for (int h = 0; h < chol_levels; h++) {
        const int nt = chol_up_ptr[h + 1] - chol_up_ptr[h];
        if (nt == 0) continue;
        hipLaunchKernelGGL((chol_rg[h] == 16 ? k_chol_up<16> : chol_rg[h] == 8 ? k_chol_up<8> : k_chol_up<4>), dim3(nt), dim3(CHOL_BLK),
                           chol_up_lds[h], stream, up + chol_up_ptr[h], (const float*)chol_panels.p, (const int32_t*)chol_gat_rows.p, r,
                           chol_f.p, chol_u.p);
        PA_LAUNCH_CHECK();
    }
    if (chol_top_tiles > 0) {
        if (chol_levels > 0) {
            hipLaunchKernelGGL(k_chol_top_f, dim3(grid_for(chol_top_cols, BLK)), dim3(BLK), 0, stream, (int)chol_top_cols,
                               (const int32_t*)chol_top_pos.p, (const int64_t*)chol_gat.p, chol_gmax, r, (const float*)chol_u.p, chol_ftop.p);
            PA_LAUNCH_CHECK();
        }
        hipEvent_t e0 = nullptr, e1 = nullptr;
        const bool mark = (profiling & 1) && !capturing;
        if (mark) {
            e0 = next_event();
            e1 = next_event();
            PA_HIP(hipEventRecord(e0, stream));
        }
        chol_top_launch(r);
        if (mark) {
            PA_HIP(hipEventRecord(e1, stream));
            spmv_marks.push_back({e0, e1});
        }
    }
    for (int h = chol_levels - 1; h >= 0; h--) {
        const int nt = chol_down_ptr[h + 1] - chol_down_ptr[h];
        if (nt == 0) continue;
        hipLaunchKernelGGL((chol_lp[h] == 8 ? k_chol_down<8> : chol_lp[h] == 16 ? k_chol_down<16> : k_chol_down<32>), dim3(nt),
                           dim3(CHOL_BLK), chol_down_lds[h], stream, down + chol_down_ptr[h], (const float*)chol_panels.p,
                           (const int32_t*)chol_below.p, (const float*)chol_f.p, chol_x.p);
        PA_LAUNCH_CHECK();
    }
}

int Backend::global_solve(int max_iter, double tol, bool defer_last, bool resid_ready) {
    const int nb = cg_blocks;
    const int passes = std::max(1, cfg.global_refine);
    // the fused iteration needs a real level 0 (nl >= 2); a one-level
    // hierarchy is an exact coarse solve and keeps the plain sequence
    const bool fused = use_amg && amg.size() >= 2;
    const bool graphs = fused && use_graphs && !(profiling & 1);
    int total_iters = 0;
    double hs[24];
    // Batched scenes: the stop test is per scene (each scene's own |r| against
    // its own |r0|), so the whole-system thresholds are off (zero).
    const bool per_scene = nscene > 0;
    uint32_t open_scenes = 0;
    auto scene_check = [&](const float* rcur, int it) {
        fill<uint32_t>(scene_open.p, 0u, 1, stream);
        hipLaunchKernelGGL(k_scene_check, dim3(nscene), dim3(BLK), 0, stream, (const int32_t*)scene_off.p, rcur, (const double*)scene_r0.p,
                           tol * tol, it, scene_first.p, scene_open.p);
        PA_LAUNCH_CHECK();
        PA_HIP(hipMemcpyAsync(&open_scenes, scene_open.p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    };
    if (use_chol) { // direct solve: each pass applies the factor to the FP64 residual, no read-back
        for (int pass = 0; pass < passes; pass++) {
            if (pass > 0 || !resid_ready) {
                with_lpr(a_lpr, [&](auto c) {
                    constexpr int P = decltype(c)::value;
                    hipLaunchKernelGGL(k_cg_resid64<P>, dim3(nb), dim3(PBLK), 0, stream, n, a_ptr.p, a_col.p, a_val.p, a_val_lo.p,
                                       a_diag.p, a_diag_lo.p, b.p, x.p, cg_r.p, cg_d.p, cg_part.p, (const int32_t*)chol_ipos.p);
                });
                PA_LAUNCH_CHECK();
            }
            chol_solve(cg_r.p);
            if (defer_last && pass == passes - 1) { // x += d is applied by the next dual update
                dx_pending = true;
                break;
            }
            hipLaunchKernelGGL(k_axpy_d, dim3(grid_for(3 * (int64_t)n, BLK)), dim3(BLK), 0, stream, n, (const float*)chol_x.p,
                               (const int32_t*)chol_ipos.p, x.p, (const int32_t*)stop_guard);
            PA_LAUNCH_CHECK();
        }
        return passes;
    }
    for (int pass = 0; pass < passes; pass++) {
        with_lpr(a_lpr, [&](auto c) {
            constexpr int P = decltype(c)::value;
            hipLaunchKernelGGL(k_cg_resid64<P>, dim3(nb), dim3(PBLK), 0, stream, n, a_ptr.p, a_col.p, a_val.p, a_val_lo.p, a_diag.p,
                               a_diag_lo.p, b.p, x.p, cg_r.p, cg_d.p, cg_part.p, (const int32_t*)nullptr);
        });
        PA_LAUNCH_CHECK();
        if (per_scene) {
            hipLaunchKernelGGL(k_scene_norms, dim3(nscene), dim3(BLK), 0, stream, (const int32_t*)scene_off.p, (const float*)cg_r.p,
                               scene_r0.p);
            PA_LAUNCH_CHECK();
            fill<int32_t>(scene_first.p, -1, nscene, stream);
        }
        precondition(cg_r.p);
        hipLaunchKernelGGL(k_cg_init_state, dim3(1), dim3(PBLK), 0, stream, cg_part.p, nb, per_scene ? 0.0 : tol * tol, cg_state.p);
        PA_LAUNCH_CHECK();
        if (!fused) {
            hipLaunchKernelGGL(k_copy, dim3(grid_for(3 * (int64_t)n, BLK)), dim3(BLK), 0, stream, 3 * (int64_t)n, cg_z.p, cg_p.p);
            PA_LAUNCH_CHECK();
        }
        if (pass > 0) {
            PA_HIP(hipMemcpyAsync(hs, cg_state.p, sizeof(hs), hipMemcpyDeviceToHost, stream));
            PA_HIP(hipStreamSynchronize(stream));
            if (hs[3] != 0 && hs[4] != 0 && hs[5] != 0) break;
        }
        int pc = 0, rc = 0;
        int chunk = std::max(2, pass == 0 ? last_pcg_iters : 2);
        if (graphs) chunk += chunk & 1;
        int it = 0;
        while (it < max_iter) {
            const int stop = std::min(max_iter, it + chunk);
            chunk = 2;
            while (it < stop) {
                if (graphs && it + 2 <= stop && (it & 1) == 0 && pc == 0 && rc == 0) {
                    PA_HIP(hipGraphLaunch(pcg_pair_graph(it == 0), stream));
                    it += 2;
                } else {
                    pcg_iteration(it, fused, pc, rc);
                    it++;
                }
            }
            if (fused) { // the state slot of iteration `it`, which k_cg_dir_spmv would compute next
                hipLaunchKernelGGL(k_cg_state, dim3(1), dim3(PBLK), 0, stream, (it - 1) & 1, nb, cg_state.p, (const double*)cg_part.p);
                PA_LAUNCH_CHECK();
            }
            PA_HIP(hipMemcpyAsync(hs, cg_state.p, sizeof(hs), hipMemcpyDeviceToHost, stream));
            if (per_scene) scene_check(fused ? (const float*)(rc ? cg_r2.p : cg_r.p) : (const float*)cg_r.p, it);
            PA_HIP(hipStreamSynchronize(stream));
            const double* sl = hs + (it & 1) * 8;
            if (sl[3] != 0 && sl[4] != 0 && sl[5] != 0) break;
            if (per_scene && open_scenes == 0) break;
        }
        if (pass == 0) last_pcg_iters = (int)hs[19];
        total_iters += (int)hs[19];
        if (per_scene) {
            hipLaunchKernelGGL(k_scene_accum, dim3(grid_for(nscene, BLK)), dim3(BLK), 0, stream, nscene, (const int32_t*)scene_first.p,
                               (int)hs[19], scene_iters.p);
            PA_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_axpy_d, dim3(grid_for(3 * (int64_t)n, BLK)), dim3(BLK), 0, stream, n, (const float*)cg_d.p,
                           (const int32_t*)nullptr, x.p, (const int32_t*)stop_guard);
        PA_LAUNCH_CHECK();
    }
    return total_iters;
}

// Blocks of the three kernels that write the residual partials (k_elem,
// k_dual_vert, k_rhs), as launched by elem_update, dual_vertices and rhs.
int3 Backend::resid_blocks() {
    ElemArgs a = make_elem_args(*this);
    return make_int3(elem_grid(a, hc.n_pin), grid_for(n, BLK), grid_for((int64_t)n * rhs_lpr, BLK));
}

void Backend::residual_read(double* rp, double* rd) {
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(BLK), 0, stream, res_part.p, resid_blocks(), res_sum.p, 0.0, (int32_t*)nullptr);
    PA_LAUNCH_CHECK();
    PA_HIP(hipMemcpyAsync(chk_host, res_sum.p, 8 * sizeof(double), hipMemcpyDeviceToHost, stream));
    PA_HIP(hipStreamSynchronize(stream));
    *rp = chk_host[6];
    *rd = chk_host[7];
}

// Enqueues the residual check of iteration `it` with the device stop test
// (see k_resid_final) and its copy into pinned slot it & 1, marked by
// ev_chk[it & 1]; read_check reads it back after that event.
void Backend::residual_enqueue(int it) {
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(BLK), 0, stream, res_part.p, resid_blocks(), res_sum.p, cfg.residual_tol, stop_ctl.p);
    PA_LAUNCH_CHECK();
    PA_HIP(hipMemcpyAsync(chk_host + 8 * (it & 1), res_sum.p, 8 * sizeof(double), hipMemcpyDeviceToHost, stream));
    PA_HIP(hipEventRecord(ev_chk[it & 1], stream));
}

void Backend::read_check(int it, double* rp, double* rd) {
    PA_HIP(hipEventSynchronize(ev_chk[it & 1]));
    *rp = chk_host[8 * (it & 1) + 6];
    *rd = chk_host[8 * (it & 1) + 7];
}

// Phase ranges are also roctx ranges (pa.detection, pa.local, ...), visible
// to rocprofv3 --marker-trace; without a tracer attached they cost a call.
static const char* const kPhaseNames[6] = {"pa.detection", "pa.local", "pa.contact", "pa.rhs", "pa.global", "pa.other"};

void Backend::mark_begin(int phase, hipEvent_t* e0) {
    roctxRangePushA(kPhaseNames[phase]);
    *e0 = nullptr;
    if (!(profiling & 2)) return;
    *e0 = next_event();
    PA_HIP(hipEventRecord(*e0, stream));
}

void Backend::mark_end(int phase, hipEvent_t e0) {
    roctxRangePop();
    if (!(profiling & 2)) return;
    hipEvent_t e1 = next_event();
    PA_HIP(hipEventRecord(e1, stream));
    ev_marks.push_back({phase, {e0, e1}});
}

void Backend::collect_phase_times() {
    if (!profiling) return;
    PA_HIP(hipStreamSynchronize(stream));
    for (int k = 0; k < 6; k++) phase_ms[k] = 0;
    for (auto& m : ev_marks) {
        float ms = 0;
        PA_HIP(hipEventElapsedTime(&ms, m.second.first, m.second.second));
        phase_ms[m.first] += ms;
    }
    for (auto& m : spmv_marks) {
        float ms = 0;
        PA_HIP(hipEventElapsedTime(&ms, m.first, m.second));
        spmv_ms_sum += ms;
        spmv_launches++;
    }
    ev_marks.clear();
    spmv_marks.clear();
    ev_next = 0;
}

void Backend::set_warm_start(const pa_warm_start& w) {
    PA_CHECK(w.mode >= 0 && w.mode <= 2, PA_ERR_INVALID, "warm start mode must be 0, 1 or 2");
    PA_CHECK(w.mode != 1 || w.params, PA_ERR_INVALID, "warm start mode 1 needs the network parameters");
    PA_CHECK(w.patience >= 0 && w.stall_ratio >= 0 && w.clamp >= 0, PA_ERR_INVALID, "negative warm start setting");
    std::vector<float> consts(22);
    for (int k = 0; k < 10; k++) {
        consts[k] = w.in_shift[k];
        consts[10 + k] = w.in_scale[k];
    }
    consts[20] = w.out_scale[0];
    consts[21] = w.out_scale[1];
    for (float c : consts) PA_CHECK(std::isfinite(c), PA_ERR_INVALID, "non-finite warm start normalisation");
    if (w.mode == 1) {
        if (!ws_mlp) ws_mlp = std::make_unique<Mlp>(stream);
        ws_mlp->set_params(w.params);
    }
    ws_consts.reserve(consts.size());
    ws_consts.upload(consts.data(), consts.size(), stream);
    ws = w;
    ws.params = nullptr;
    if (ws.patience == 0) ws.patience = 2;
    if (ws.stall_ratio == 0) ws.stall_ratio = 1e3;
    if (ws.clamp == 0) ws.clamp = 50;
    ws_bad = 0;
}

// Judge of a seeded window (once per window): its seeds against its final
// duals.  A window with sum |r_final - seed|^2 > 4 sum |r_final|^2 (the seeds
// miss by more than twice what zero would) counts as bad, and `patience` bad
// windows in a row abandon the attempt.
void Backend::ws_judge() {
    if (!ws_window || !ws_window_seeded || ws_judged || ws_nc == 0) return;
    ws_judged = true;
    const int c = ws_nc;
    const int blocks = std::min(grid_for(c, BLK), 1024);
    ws_err.reserve(2 * (size_t)blocks);
    hipLaunchKernelGGL(k_ws_judge, dim3(blocks), dim3(BLK), 0, stream, c, (const float4*)rc.p, (const float4*)ws_seed.p, ws_err.p);
    PA_LAUNCH_CHECK();
    std::vector<double> h(2 * (size_t)blocks);
    ws_err.download(h.data(), h.size(), stream);
    PA_HIP(hipStreamSynchronize(stream));
    double e_seed = 0, e_zero = 0;
    for (int k = 0; k < blocks; k++) {
        e_seed += h[2 * (size_t)k];
        e_zero += h[2 * (size_t)k + 1];
    }
    const bool bad = e_seed > 4.0 * e_zero;
    ws_bad = bad ? ws_bad + 1 : 0;
    ws_bad_windows += bad ? 1 : 0;
    if (ws_bad >= ws.patience) ws_restart = true;
}

// End of a detection window (before the next detection replaces the list):
// judge the seeds against the window's final duals, log the window, and keep
// its keys and duals for matching in the next window.
void Backend::ws_window_end() {
    const bool want = ws.mode != 0 || log_cap > 0;
    if (!want || !ws_window || ws_nc == 0 || !det || det->n_contacts != ws_nc) {
        ws_forget();
        return;
    }
    const int c = ws_nc;
    const float sc = (float)(cfg.dt / cfg.thickness);
    ws_judge();
    if (log_cap > 0 && log_rows < log_cap) {
        const int take = (int)std::min<int64_t>(c, log_cap - log_rows);
        hipLaunchKernelGGL(k_ws_log, dim3(grid_for(take, BLK)), dim3(BLK), 0, stream, take, sc, (const float*)ws_feat.p,
                           (const float4*)rc.p, (const float4*)det->c.nrm.p, (const float4*)ws_tan.p, log_buf.p + (size_t)log_rows * 12);
        PA_LAUNCH_CHECK();
        log_rows += take;
    }
    prev_type.reserve(c);
    prev_p0.reserve(c);
    prev_p1.reserve(c);
    prev_rc.reserve(c);
    PA_HIP(hipMemcpyAsync(prev_type.p, det->c.type.p, sizeof(int32_t) * c, hipMemcpyDeviceToDevice, stream));
    PA_HIP(hipMemcpyAsync(prev_p0.p, det->c.prim0.p, sizeof(int32_t) * c, hipMemcpyDeviceToDevice, stream));
    PA_HIP(hipMemcpyAsync(prev_p1.p, det->c.prim1.p, sizeof(int32_t) * c, hipMemcpyDeviceToDevice, stream));
    PA_HIP(hipMemcpyAsync(prev_rc.p, rc.p, sizeof(float4) * c, hipMemcpyDeviceToDevice, stream));
    nc_prev = c;
    ws_window = false;
}

// Start of a detection window (after contact_setup zeroed r_c): features, and
// in a warm-started attempt the seeds.
void Backend::ws_window_begin() {
    ws_nc = nc;
    ws_window = false;
    ws_window_seeded = false;
    ws_judged = false;
    const bool want = ws.mode != 0 || log_cap > 0;
    if (want && nc > 0) {
        const bool use_mlp = ws_active && ws.mode == 1;
        ws_feat.reserve(10 * (size_t)nc);
        ws_tan.reserve(nc);
        ws_match.reserve(nc);
        ws_seed.reserve(nc);
        if (use_mlp) ws_norm.reserve(10 * (size_t)nc);
        hipLaunchKernelGGL(k_ws_features, dim3(grid_for(nc, BLK)), dim3(BLK), 0, stream, nc, n, nc_prev, (float)cfg.dt,
                           (float)cfg.thickness, (const int32_t*)det->c.type.p, (const int32_t*)det->c.prim0.p,
                           (const int32_t*)det->c.prim1.p, (const int4*)det->c.v.p, (const float4*)det->c.bary.p,
                           (const float4*)det->c.nrm.p, (const float4*)kc.p, (const double*)x.p, (const double*)x0.p, (const float*)Uc.p,
                           (const float*)p.p, (const double*)v.p, (const int32_t*)prev_type.p, (const int32_t*)prev_p0.p,
                           (const int32_t*)prev_p1.p, (const float4*)prev_rc.p, use_mlp ? 1 : 0, (const float*)ws_consts.p, ws_feat.p,
                           ws_norm.p, ws_tan.p, ws_match.p);
        PA_LAUNCH_CHECK();
        ws_window = true;
        if (ws_active) {
            if (use_mlp) {
                const int rows = Mlp::pad_rows(nc);
                ws_mlp->infer(ws_norm.p, 10, nc, rows, ws_mlp->outputs(rows));
            }
            hipLaunchKernelGGL(k_ws_seed, dim3(grid_for(nc, BLK)), dim3(BLK), 0, stream, nc, ws.mode, (float)(cfg.thickness / cfg.dt),
                               (float)ws.clamp, use_mlp ? (const float*)ws_mlp->Y.p : nullptr, (const float*)ws_consts.p,
                               (const float4*)det->c.nrm.p, (const float4*)ws_tan.p, (const int32_t*)ws_match.p,
                               (const float4*)prev_rc.p, rc.p, ws_seed.p);
            PA_LAUNCH_CHECK();
            ws_window_seeded = true;
            ws_seeded_count++;
        }
    }
    if (seed_log) {
        std::vector<float> h;
        if (ws_window_seeded) {
            std::vector<float4> q(nc);
            ws_seed.download(q.data(), nc, stream);
            PA_HIP(hipStreamSynchronize(stream));
            h.resize(3 * (size_t)nc);
            for (int c = 0; c < nc; c++) {
                h[3 * (size_t)c] = q[c].x;
                h[3 * (size_t)c + 1] = q[c].y;
                h[3 * (size_t)c + 2] = q[c].z;
            }
        }
        seed_log_h.push_back(std::move(h));
    }
}

bool Backend::state_nonfinite() {
    fill<uint32_t>(bad_flag.p, 0u, 1, stream);
    hipLaunchKernelGGL(k_nonfinite, dim3(grid_for(3 * (int64_t)n_all, BLK)), dim3(BLK), 0, stream, 3 * (int64_t)n_all, (const double*)x.p,
                       (const double*)v.p, bad_flag.p);
    PA_LAUNCH_CHECK();
    uint32_t bad = 0;
    PA_HIP(hipMemcpyAsync(&bad, bad_flag.p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    PA_HIP(hipStreamSynchronize(stream));
    return bad != 0;
}

template <class T> static void copy_dev(DBuf<T>& dst, const DBuf<T>& src, size_t count, hipStream_t s, bool grow) {
    if (grow) dst.reserve(count);
    if (count) PA_HIP(hipMemcpyAsync(dst.p, src.p, sizeof(T) * count, hipMemcpyDeviceToDevice, s));
}

// The last good state (x, v, Ue, Uc and the rigid tracks' frame counters):
// kept at init, reset, after every step whose state is finite, and at the
// start of a step whose state was set from the host; a failed step returns
// to it.
void Backend::save_good_state() {
    copy_dev(good_x, x, 3 * (size_t)n_all, stream, true);
    copy_dev(good_v, v, 3 * (size_t)n_all, stream, true);
    copy_dev(good_ue, Ue, 3 * (size_t)m, stream, true);
    copy_dev(good_uc, Uc, 3 * (size_t)n, stream, true);
    good_track_frames.resize(tracks.size());
    for (size_t k = 0; k < tracks.size(); k++) good_track_frames[k] = tracks[k]->cur;
}

void Backend::restore_good_state() {
    copy_dev(x, good_x, 3 * (size_t)n_all, stream, false);
    copy_dev(v, good_v, 3 * (size_t)n_all, stream, false);
    copy_dev(Ue, good_ue, 3 * (size_t)m, stream, false);
    copy_dev(Uc, good_uc, 3 * (size_t)n, stream, false);
    // the tracks go back to their frames, with the last placed positions
    // re-placed so the next step's static velocities are an uninterrupted run's
    if (!tracks.empty() && good_track_frames.size() == tracks.size())
        set_track_frames(good_track_frames.data(), (int)tracks.size());
    ws_forget();
    PA_HIP(hipStreamSynchronize(stream));
    if (sync_to_host) get_state(x_host.data(), v_host.data());
}

// A step that fails (contact overflow, non-finite state, a failed check)
// leaves the state as it was at the start of the step: positions,
// velocities, duals and track frames.  After a HIP error the device state is
// not touched.
void Backend::step(pa_step_stats* st) {
    PA_CHECK(initialized, PA_ERR_INVALID, "step before init");
    PA_CHECK(!cfg.enable_contact || det, PA_ERR_INVALID, "contact enabled but no detector attached");
    if (state_dirty) { // state set from the host since the last step: check it before detection uses it
        state_dirty = false;
        if (state_nonfinite()) {
            restore_good_state();
            if (st) std::memset(st, 0, sizeof(*st));
            throw Error(PA_ERR_NUMERICAL, "non-finite positions or velocities given to the step; state rolled back to the last good step");
        }
        save_good_state(); // the step's start is the state to return to
    }
    try {
        step_impl(st);
    } catch (const Error& err) {
        if (err.code != PA_ERR_HIP) restore_good_state();
        if (st) {
            std::memset(st, 0, sizeof(*st));
            st->overflow = err.code == PA_ERR_OVERFLOW ? 1 : 0;
        }
        throw;
    }
}

void Backend::step_impl(pa_step_stats* st) {
    const bool contact = cfg.enable_contact != 0;
    auto t0 = std::chrono::steady_clock::now();
    pa_step_stats S{};
    if (!tracks.empty()) animate_tracks(false);
    const double hd = cfg.dt;
    const float eps = (float)(1.0 / (hd * hd * cfg.kappa + hd * cfg.beta));
    const float gam_ = (float)(hd * cfg.kappa / (hd * cfg.kappa + cfg.beta));
    const float hinv = (float)(1.0 / hd);
    ev_next = 0;
    ev_marks.clear();
    spmv_marks.clear();
    // A warm-started attempt can be abandoned (ws_restart): the step then
    // re-runs cold from this snapshot, exactly as a plain step would.
    const bool can_warm = contact && ws.mode != 0;
    if (can_warm) {
        copy_dev(snap_x, x, 3 * (size_t)n_all, stream, true);
        copy_dev(snap_v, v, 3 * (size_t)n_all, stream, true);
        copy_dev(snap_ue, Ue, 3 * (size_t)m, stream, true);
        copy_dev(snap_uc, Uc, 3 * (size_t)n, stream, true);
    }
    if (nscene) { // per-scene solve statistics of this step
        fill<int32_t>(scene_iters.p, 0, nscene, stream);
        fill<unsigned long long>(scene_ticks.p, 0ull, nscene, stream);
    }
    ws_bad = 0;
    ws_bad_windows = 0;
    ws_restart = false;
    ws_seeded_count = 0;
    if (seed_log) seed_log_h.clear();
    int it = 0;
    for (int attempt = 0;; attempt++) {
        ws_active = can_warm && attempt == 0;
        hipEvent_t e;
        mark_begin(5, &e);
        if (!cfg.warmstart_ue) fill<float>(Ue.p, 0.f, 3 * (int64_t)m, stream);
        if (!cfg.warmstart_uc) fill<float>(Uc.p, 0.f, 3 * (int64_t)n, stream);
        hipLaunchKernelGGL(k_begin_step, dim3(grid_for(n_all, BLK)), dim3(BLK), 0, stream, n_all, n, hd, hinv, cfg.g, pinned.p, x.p, v.p, x0.p,
                           p.p, bconst.p, mass.p, (const double*)bpin.p, (const float*)Uc.p);
        PA_LAUNCH_CHECK();
        if (nnz_dm > 0) {
            hipLaunchKernelGGL(k_spmv_add, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, n, dm_ptr.p, dm_col.p, dm_val.p, x0.p, bconst.p);
            PA_LAUNCH_CHECK();
        }
        mark_end(5, e);
        it = admm_loop(S, eps, gam_, hinv);
        if (!ws_restart) break;
        S.ws_fallback = 1;
        S.ws_wasted_iters += it;
        S.detections = S.global_iters = S.converged = S.n_contacts_max = 0;
        S.r_primal = S.r_dual = 0;
        copy_dev(x, snap_x, 3 * (size_t)n_all, stream, false);
        copy_dev(v, snap_v, 3 * (size_t)n_all, stream, false);
        copy_dev(Ue, snap_ue, 3 * (size_t)m, stream, false);
        copy_dev(Uc, snap_uc, 3 * (size_t)n, stream, false);
        ws_forget();
        ws_restart = false;
        ws_seeded_count = 0;
        if (seed_log) seed_log_h.clear();
    }
    ws_active = false;
    hipEvent_t e;
    mark_begin(5, &e);
    hipLaunchKernelGGL(k_end_step, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, n, hd, (const double*)x.p, (const double*)x0.p, v.p);
    PA_LAUNCH_CHECK();
    mark_end(5, e);
    // non-finite positions or velocities: step() goes back to the last good state
    if (state_nonfinite())
        throw Error(PA_ERR_NUMERICAL, "non-finite positions or velocities after the step; state rolled back to the last good step");
    save_good_state();
    if (sync_to_host) {
        x.download(x_host.data(), x_host.size(), stream);
        v.download(v_host.data(), v_host.size(), stream);
        PA_HIP(hipStreamSynchronize(stream));
    } else {
        PA_HIP(hipStreamSynchronize(stream));
    }
    collect_phase_times();
    if (nscene && !use_chol) { // the critical path: the most PCG iterations of any scene (the direct solve counts passes)
        std::vector<int32_t> its(nscene);
        batch_stats(its.data(), nullptr);
        S.global_iters = *std::max_element(its.begin(), its.end());
    }
    S.iterations = it;
    S.n_contacts = nc;
    S.ws_seeded = ws_seeded_count;
    S.ws_bad_windows = ws_bad_windows;
    S.step_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (st) *st = S;
}

// The ADMM iterations of one attempt (after the step prologue); returns the
// iterations run.  Stops early at residual_tol, or when the warm start is
// abandoned (ws_restart).
int Backend::admm_loop(pa_step_stats& S, float eps, float gam_, float hinv) {
    const bool contact = cfg.enable_contact != 0;
    hipEvent_t e;
    nc = 0;
    dx_pending = false;
    res_log.clear(); // this attempt's checks
    double best = std::numeric_limits<double>::infinity();
    int it = 0;
    auto checked = [&](int q) { return cfg.residual_tol > 0 && (q + 1) % cfg.residual_interval == 0; };
    // Stop test on the device (direct solve, no learned warm start): the
    // check of iteration q is read back once iteration q + 1 is enqueued, or
    // before a detection, so the queue does not drain at every check.  An
    // iteration enqueued past the converged one runs with its state writers
    // stopped (stop_guard: x, Ue, Uc, r_c keep the converged values) and is
    // not counted.  The warm-start attempt compares each check with the best
    // so far and reads it at once.
    const bool lagged = use_chol && !ws_active && cfg.residual_tol > 0;
    struct GuardReset {
        const int32_t*& g;
        ~GuardReset() { g = nullptr; }
    } guard_reset{stop_guard};
    stop_guard = lagged ? stop_ctl.p : nullptr;
    if (lagged) fill<int32_t>(stop_ctl.p, 0, 1, stream);
    int pending = -1; // iteration whose check is enqueued and not read yet
    auto take_check = [&](int q) {
        double rp, rd;
        read_check(q, &rp, &rd);
        S.r_primal = rp;
        S.r_dual = rd;
        res_log.push_back(rp);
        res_log.push_back(rd);
        return std::max(rp, rd) <= cfg.residual_tol;
    };
    for (; it < cfg.admm_max_iter; it++) {
        if (lagged && pending >= 0 && contact && it % cfg.dcd_interval == 0) { // no detection past the stop
            const int q = pending;
            pending = -1;
            if (take_check(q)) {
                S.converged = 1;
                break; // it == q + 1
            }
        }
        if (it == 0) {
            mark_begin(1, &e);
            local_step();
            mark_end(1, e);
        }
        if (contact && it % cfg.dcd_interval == 0) {
            mark_begin(0, &e);
            ws_window_end();
            if (ws_restart) {
                mark_end(0, e);
                break;
            }
            // rebuild at the step's first detection, refit later ones
            det->detect(x.p, it > 0, VertexCount{vcnt.p, vloc.p, n_all});
            contact_setup(eps, gam_, hinv, true);
            ws_window_begin();
            S.detections++;
            S.n_contacts_max = std::max(S.n_contacts_max, nc);
            mark_end(0, e);
        }
        if (contact) {
            mark_begin(2, &e);
            contact_project(it == 0);
            mark_end(2, e);
        }
        const bool check = checked(it);
        mark_begin(3, &e);
        rhs(check, it == 0);
        mark_end(3, e);
        mark_begin(4, &e);
        const int gi = (nscene && !use_amg && !use_chol) ? batch_solve(cfg.global_max_iter, cfg.global_tol)
                                                         : global_solve(cfg.global_max_iter, cfg.global_tol, true, use_chol);
        S.global_iters += gi;
        mark_end(4, e);
        mark_begin(1, &e);
        dual_vertices(check);
        elem_update(check, it + 1 >= cfg.admm_max_iter, checked(it + 1));
        mark_end(1, e);
        if (lagged) {
            if (check) residual_enqueue(it);
            if (pending >= 0) {
                const int q = pending;
                pending = -1;
                if (take_check(q)) { // this iteration ran past the stop
                    S.converged = 1;
                    S.global_iters -= gi;
                    break; // it == q + 1
                }
            }
            if (check) pending = it;
        } else if (check) {
            double rp, rd;
            residual_read(&rp, &rd);
            S.r_primal = rp;
            S.r_dual = rd;
            res_log.push_back(rp);
            res_log.push_back(rd);
            const double r = std::max(rp, rd);
            if (ws_active) {
                if (!std::isfinite(r) || r > ws.stall_ratio * best) {
                    ws_restart = true;
                    it++;
                    break;
                }
                best = std::min(best, r);
            }
            if (r <= cfg.residual_tol) {
                S.converged = 1;
                it++;
                break;
            }
        }
    }
    if (lagged && pending >= 0 && take_check(pending)) S.converged = 1; // the last iteration's check
    if (ws_active && !ws_restart) ws_judge(); // the last window of the attempt
    return it;
}

// Reference ADMMImplCPUBase::reset (admm_impl_cpu.cpp:71-88), reached from
// ADMMImplGPU::reset (admm_impl_gpu.cu:151-155): positions from the caller,
// zero velocities and duals, contact history dropped, tracks back at frame 0.
void Backend::reset(const double* x0h) {
    PA_CHECK(initialized, PA_ERR_INVALID, "reset before init");
    x.upload(x0h, 3 * (size_t)n_all, stream);
    x0.upload(x0h, 3 * (size_t)n_all, stream);
    fill<double>(v.p, 0.0, 3 * (int64_t)n_all, stream);
    fill<float>(Ue.p, 0.f, 3 * (int64_t)m, stream);
    fill<float>(Uc.p, 0.f, 3 * (int64_t)n, stream);
    ws_forget();
    state_dirty = false;
    if (!tracks.empty()) animate_tracks(true);
    save_good_state(); // after the tracks are placed at frame 0
    PA_HIP(hipStreamSynchronize(stream));
    x.download(x_host.data(), x_host.size(), stream);
    std::fill(v_host.begin(), v_host.end(), 0.0);
    PA_HIP(hipStreamSynchronize(stream));
}

void Backend::get_state(double* xo, double* vo) {
    PA_CHECK(initialized, PA_ERR_INVALID, "get_state before init");
    if (xo) x.download(xo, 3 * (size_t)n_all, stream);
    if (vo) v.download(vo, 3 * (size_t)n_all, stream);
    PA_HIP(hipStreamSynchronize(stream));
}

void Backend::set_state(const double* xi, const double* vi) {
    PA_CHECK(initialized, PA_ERR_INVALID, "set_state before init");
    state_dirty = true;
    if (xi) x.upload(xi, 3 * (size_t)n_all, stream);
    if (vi) v.upload(vi, 3 * (size_t)n_all, stream);
}

void Backend::get_duals(double* ue, double* uc) {
    PA_CHECK(initialized, PA_ERR_INVALID, "get_duals before init");
    std::vector<float> a(3 * (size_t)m), c(3 * (size_t)n);
    Ue.download(a.data(), a.size(), stream);
    Uc.download(c.data(), c.size(), stream);
    PA_HIP(hipStreamSynchronize(stream));
    if (ue)
        for (size_t i = 0; i < a.size(); i++) ue[i] = a[i];
    if (uc)
        for (size_t i = 0; i < c.size(); i++) uc[i] = c[i];
}

void Backend::set_duals(const double* ue, const double* uc) {
    state_dirty = true;
    PA_CHECK(initialized, PA_ERR_INVALID, "set_duals before init");
    if (ue) {
        std::vector<float> a(ue, ue + 3 * (size_t)m);
        Ue.upload(a.data(), a.size(), stream);
        PA_HIP(hipStreamSynchronize(stream));
    }
    if (uc) {
        std::vector<float> c(uc, uc + 3 * (size_t)n);
        Uc.upload(c.data(), c.size(), stream);
        PA_HIP(hipStreamSynchronize(stream));
    }
}

// Friction coefficient per vertex (default: pa_admm_config.mu everywhere).  A
// contact takes the coefficient of its first vertex: the query vertex of a
// point-triangle pair, the first endpoint of edge i of an edge-edge pair; in
// a merged batch every vertex of a scene carries that scene's coefficient.
void Backend::set_vertex_mu(const double* mu) {
    PA_CHECK(initialized, PA_ERR_INVALID, "set_vertex_mu before init");
    std::vector<float> f(n_all);
    for (int i = 0; i < n_all; i++) {
        PA_CHECK(std::isfinite(mu[i]) && mu[i] >= 0, PA_ERR_INVALID, "friction coefficients must be finite and non-negative");
        f[i] = (float)mu[i];
    }
    mu_v.upload(f.data(), f.size(), stream);
}

void Backend::set_static_state(const double* xs, const double* vs) {
    PA_CHECK(initialized, PA_ERR_INVALID, "set_static_state before init");
    state_dirty = true;
    const size_t ns = 3 * (size_t)(n_all - n);
    if (ns == 0) return;
    if (xs) PA_HIP(hipMemcpyAsync(x.p + 3 * (size_t)n, xs, ns * sizeof(double), hipMemcpyHostToDevice, stream));
    if (vs) PA_HIP(hipMemcpyAsync(v.p + 3 * (size_t)n, vs, ns * sizeof(double), hipMemcpyHostToDevice, stream));
    PA_HIP(hipStreamSynchronize(stream));
}

} // namespace pa
