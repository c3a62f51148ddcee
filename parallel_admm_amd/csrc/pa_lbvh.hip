// LBVH proximity detection on gfx950.
//
// Per detection: primitive boxes -> scene box -> 30-bit Morton codes ->
// stable LDS radix sort -> Karras radix tree (T. Karras, "Maximizing
// Parallelism in the Construction of BVHs, Octrees, and k-d Trees", HPG 2012)
// -> node boxes from leaf ranges -> 128-byte wide node records (the boxes,
// ids and last sorted leaf of a node's up to four grandchildren, a leaf child
// standing in for its own pair, so a traversal step descends two levels with
// one dependent load; the stack top's record is loaded ahead, so a pop needs
// none) -> one traversal per query with the FP64 predicate,
// accepted pairs appended to a staging list with their segment.
//
// Point-triangle: one lane per surface vertex; its pairs form the vertex's
// segment.  Edge-edge: one lane per sorted leaf k, visiting only leaves after
// k, so each unordered pair is tested once; the pair belongs to the segment of
// its smaller edge id.  Segment counts -> exclusive scan -> partner ids into
// their segments -> every pair to its rank in its segment: the list comes out
// in canonical order, bit-identical on every run, with no global sort.
//
// Segmented mode (merged scenes): keys carry the scene id above a 21-bit
// Morton code, so every scene is one subtree and queries start at their own
// scene's subtree root.
//
// Reference: lbvh_f/lbvh_e::Construct (src/contact/lbvh/lbvh.cu:1468-1540),
// _dcd_vf/_dcd_ee (:1694-1813); acceptance follows ProximalQuery
// (src/contact/narrow_phase.cpp:192-245, 313-469) rather than the reference
// GPU's interior-only test, so the GPU set equals the CPU set.
#include "pa_detector.hpp"
#include "pa_geom.hpp"

#include <algorithm>
#include <type_traits>
#include <vector>

#pragma clang fp contract(off)

namespace pa {
namespace {

constexpr int BLK = 256;
constexpr int QBLK = 128;
constexpr int STACK = 64;

__device__ inline float4 fmin4(float4 a, float4 b) { return make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z), 0.f); }
__device__ inline float4 fmax4(float4 a, float4 b) { return make_float4(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z), 0.f); }

// FP32 box of FP64 position v, rounded outward (the boxes only cull, so
// they must contain the exact positions the FP64 predicate sees).
__device__ inline float4 pos_lo(const double* __restrict__ x, int v) {
    return make_float4(__double2float_rd(x[3 * v]), __double2float_rd(x[3 * v + 1]), __double2float_rd(x[3 * v + 2]), 0.f);
}
__device__ inline float4 pos_hi(const double* __restrict__ x, int v) {
    return make_float4(__double2float_ru(x[3 * v]), __double2float_ru(x[3 * v + 1]), __double2float_ru(x[3 * v + 2]), 0.f);
}

// Boxes of triangles (k = 3) or edges (k = 2).
__global__ void k_prim_boxes(const double* __restrict__ x, const int32_t* __restrict__ prims, int k, int n,
                             float4* __restrict__ box) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    for (int q = 0; q < k; q++) {
        int v = prims[k * i + q];
        lo = fmin4(lo, pos_lo(x, v));
        hi = fmax4(hi, pos_hi(x, v));
    }
    box[2 * i] = lo;
    box[2 * i + 1] = hi;
}

__device__ inline float4 wave_min4(float4 v) {
    for (int o = 32; o > 0; o >>= 1) {
        v.x = fminf(v.x, __shfl_xor(v.x, o, 64));
        v.y = fminf(v.y, __shfl_xor(v.y, o, 64));
        v.z = fminf(v.z, __shfl_xor(v.z, o, 64));
    }
    return v;
}
__device__ inline float4 wave_max4(float4 v) {
    for (int o = 32; o > 0; o >>= 1) {
        v.x = fmaxf(v.x, __shfl_xor(v.x, o, 64));
        v.y = fmaxf(v.y, __shfl_xor(v.y, o, 64));
        v.z = fmaxf(v.z, __shfl_xor(v.z, o, 64));
    }
    return v;
}

// Union of n boxes (2 float4 each) per block -> out[2 * blockIdx].
__global__ void __launch_bounds__(BLK) k_box_union(const float4* __restrict__ box, int n, float4* __restrict__ out) {
    __shared__ float4 slo[BLK / 64], shi[BLK / 64];
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        lo = fmin4(lo, box[2 * i]);
        hi = fmax4(hi, box[2 * i + 1]);
    }
    lo = wave_min4(lo);
    hi = wave_max4(hi);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        slo[wave] = lo;
        shi[wave] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLK / 64; w++) {
            lo = fmin4(lo, slo[w]);
            hi = fmax4(hi, shi[w]);
        }
        out[2 * blockIdx.x] = lo;
        out[2 * blockIdx.x + 1] = hi;
    }
}

__device__ inline uint32_t spread10(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ inline uint32_t quant10(float u) {
    float q = fminf(fmaxf(u * 1024.0f, 0.0f), 1023.0f);
    return (uint32_t)q;
}

__global__ void k_morton(const float4* __restrict__ box, int n, const float4* __restrict__ scene, uint32_t* __restrict__ keys,
                         uint32_t* __restrict__ ids) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 slo = scene[0], shi = scene[1];
    float4 lo = box[2 * i], hi = box[2 * i + 1];
    float ex = shi.x - slo.x, ey = shi.y - slo.y, ez = shi.z - slo.z;
    float cx = 0.5f * (lo.x + hi.x) - slo.x, cy = 0.5f * (lo.y + hi.y) - slo.y, cz = 0.5f * (lo.z + hi.z) - slo.z;
    uint32_t qx = quant10(ex > 0.f ? cx / ex : 0.f);
    uint32_t qy = quant10(ey > 0.f ? cy / ey : 0.f);
    uint32_t qz = quant10(ez > 0.f ? cz / ez : 0.f);
    keys[i] = (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz);
    ids[i] = (uint32_t)i;
}

// Segmented keys: segment id in the top 11 bits, then a 21-bit Morton code
// (7 bits per axis) of the box centre in the box of all segments.
__global__ void k_morton_seg(const float4* __restrict__ box, const int32_t* __restrict__ prims, int k, int n,
                             const int32_t* __restrict__ vseg, const float4* __restrict__ scene, uint32_t* __restrict__ keys,
                             uint32_t* __restrict__ ids) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 slo = scene[0], shi = scene[1];
    float4 lo = box[2 * i], hi = box[2 * i + 1];
    float ex = shi.x - slo.x, ey = shi.y - slo.y, ez = shi.z - slo.z;
    float cx = 0.5f * (lo.x + hi.x) - slo.x, cy = 0.5f * (lo.y + hi.y) - slo.y, cz = 0.5f * (lo.z + hi.z) - slo.z;
    auto q7 = [](float u) { return (uint32_t)fminf(fmaxf(u * 128.0f, 0.0f), 127.0f); };
    const uint32_t qx = q7(ex > 0.f ? cx / ex : 0.f), qy = q7(ey > 0.f ? cy / ey : 0.f), qz = q7(ez > 0.f ? cz / ez : 0.f);
    const uint32_t m = (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz); // 21 bits
    keys[i] = ((uint32_t)vseg[prims[k * i]] << 21) | m;
    ids[i] = (uint32_t)i;
}

// First and last sorted leaf of every segment (segments with no primitive keep -1).
__global__ void k_seg_bounds(const uint32_t* __restrict__ keys, int n, int32_t* __restrict__ first, int32_t* __restrict__ last) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t s = keys[k] >> 21;
    if (k == 0 || (keys[k - 1] >> 21) != s) first[s] = k;
    if (k == n - 1 || (keys[k + 1] >> 21) != s) last[s] = k;
}

// The subtree root of each segment: the internal node whose leaf range is the
// segment's range (it exists: the segment id is a key prefix), or the leaf
// itself for a one-primitive segment.
__global__ void k_seg_roots(int n, const int2* __restrict__ range, const uint32_t* __restrict__ keys, const int32_t* __restrict__ first,
                            const int32_t* __restrict__ last, int32_t* __restrict__ root) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n - 1) {
        const int2 r = range[i];
        const uint32_t s = keys[r.x] >> 21;
        if (first[s] == r.x && last[s] == r.y) root[s] = i;
    }
    if (i < n) {
        const uint32_t s = keys[i] >> 21;
        if (first[s] == i && last[s] == i) root[s] = (n - 1) + i;
    }
}

__device__ inline int kdelta(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ ids, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = ((uint64_t)keys[i] << 32) | ids[i];
    uint64_t b = ((uint64_t)keys[j] << 32) | ids[j];
    return __clzll(a ^ b);
}

// Karras construction of internal node i over sorted unique 64-bit keys.
__global__ void k_karras(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ ids, int n, int32_t* __restrict__ child,
                         int2* __restrict__ range) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (kdelta(keys, ids, n, i, i + 1) - kdelta(keys, ids, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = kdelta(keys, ids, n, i, i - d);
    int lmax = 2;
    while (kdelta(keys, ids, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (kdelta(keys, ids, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = kdelta(keys, ids, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (kdelta(keys, ids, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int g = i + s * d + (d < 0 ? d : 0);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const int left = (lo == g) ? (n - 1) + g : g;
    const int right = (hi == g + 1) ? (n - 1) + g + 1 : g + 1;
    child[2 * i] = left;
    child[2 * i + 1] = right;
    range[i] = make_int2(lo, hi);
}

// Node boxes without cross-block synchronisation: an internal node covers
// the contiguous sorted-leaf range [lo, hi] (Karras), so its box is the union
// of that range, taken from the leaf boxes at the ends and from precomputed
// unions of aligned 64- and 4096-leaf chunks in the middle.  (A bottom-up
// climb with atomic visit flags needs device-scope fences, which write back
// and invalidate the per-XCD L2 on this part.)
// Leaf data of a tree over K-vertex primitives (K = 2 edges, 3 triangles):
// per double2 slots of leaf_stride<K>, first the primitive's FP64 vertex
// positions (3K doubles, a zero pads triangles to 10), then an int4 of its
// primitive id and vertex ids (-1 for none).  A traversal tests a leaf with
// this one load instead of the chain sorted id -> vertex ids -> positions.
template <int K> constexpr int leaf_stride() { return (3 * K + 1) / 2 + 1; }

// Wide node record i (8 float4): four slots, slot j = (lo, node id) at
// 2j and (hi, last sorted leaf under the node) at 2j + 1, ids and leaf
// positions as int bits in w.  Slots 0-1 come from the left child, 2-3 from
// the right: an internal child gives its two children, a leaf child itself
// (slot 0 or 2), and an unused slot holds id -1 and an empty box.
//
// Every node's box is written straight into the slots that hold it: an
// internal node sits in one slot (its grandparent's record; none for the
// root and its children), a leaf in up to two (its parent's record when the
// parent keeps it as slot 0 or 2, and its grandparent's).  The positions
// (float4 index of the slot's lo) are found once per build by
// k_record_slots; a refit only rewrites the boxes.
__device__ inline void put_slot(float4* __restrict__ rec, int p, float4 lo, float4 hi, int id, int last) {
    rec[p] = make_float4(lo.x, lo.y, lo.z, __int_as_float(id));
    rec[p + 1] = make_float4(hi.x, hi.y, hi.z, __int_as_float(last));
}

// Leaf k (sorted order): its box (into leaf_box and its record slots) and
// its leaf data.  The box is the primitive box of k_prim_boxes
// (outward-rounded FP32 of the FP64 positions), so a refit needs no
// primitive boxes.
template <int K>
__global__ void k_leaf_data(const double* __restrict__ x, const int32_t* __restrict__ prims, const uint32_t* __restrict__ ids, int n,
                            float4* __restrict__ leaf_box, double2* __restrict__ leafd, const int2* __restrict__ lpos,
                            float4* __restrict__ rec) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int pid = (int)ids[k];
    int v[K];
    double p[3 * K + 1];
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
#pragma unroll
    for (int q = 0; q < K; q++) {
        v[q] = prims[K * pid + q];
        p[3 * q] = x[3 * v[q]];
        p[3 * q + 1] = x[3 * v[q] + 1];
        p[3 * q + 2] = x[3 * v[q] + 2];
        lo = fmin4(lo, pos_lo(x, v[q]));
        hi = fmax4(hi, pos_hi(x, v[q]));
    }
    p[3 * K] = 0.0;
    leaf_box[2 * k] = lo;
    leaf_box[2 * k + 1] = hi;
    if (n > 1) {
        const int2 lp = lpos[k];
        if (lp.x >= 0) put_slot(rec, lp.x, lo, hi, (n - 1) + k, k);
        if (lp.y >= 0) put_slot(rec, lp.y, lo, hi, (n - 1) + k, k);
    }
    constexpr int NP = leaf_stride<K>() - 1;
    double2* o = leafd + (size_t)leaf_stride<K>() * k;
#pragma unroll
    for (int j = 0; j < NP; j++) o[j] = make_double2(p[2 * j], p[2 * j + 1]);
    *reinterpret_cast<int4*>(o + NP) = make_int4(pid, v[0], v[1], K == 3 ? v[K - 1] : -1);
}

// Block b's place in the query order.  Workgroups go round-robin to the 8
// XCDs (block b to XCD b mod 8); the query order is dealt to them in chunks
// of XCD_CHUNK consecutive blocks, chunk c to XCD c mod 8, so spatially close
// queries (consecutive in Morton order) share one L2 for the records and
// leaf data they visit, while the chunks of a dense region still spread over
// all XCDs.  The grid is padded to a multiple of 8 XCD_CHUNK blocks
// (query_grid), which makes the map a permutation of the blocks.
constexpr int XCD_CHUNK = 16;
__device__ inline int xcd_block(int b) {
    const int j = b >> 3; // the j-th block this XCD receives
    return ((j / XCD_CHUNK) * 8 + (b & 7)) * XCD_CHUNK + j % XCD_CHUNK;
}
inline int query_grid(int n) {
    constexpr int m = 8 * XCD_CHUNK;
    return (grid_for(n, QBLK) + m - 1) / m * m;
}

// out[c] = union of in[c*64 .. c*64+63] (clamped to n), one wave per chunk.
__global__ void __launch_bounds__(BLK) k_chunk_union(const float4* __restrict__ in, int n, float4* __restrict__ out, int nchunks) {
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (wave >= nchunks) return;
    const int e = wave * 64 + lane;
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (e < n) {
        lo = in[2 * e];
        hi = in[2 * e + 1];
    }
    lo = wave_min4(lo);
    hi = wave_max4(hi);
    if (lane == 0) {
        out[2 * wave] = lo;
        out[2 * wave + 1] = hi;
    }
}

// Box of internal node i (the union of the leaf boxes of its range [a, b))
// into its record slot.  Levels: leaves, then unions of 64 leaves, of 4096,
// and (c256k non-null) of 262144; at each level the range's ends up to the
// next level's boundaries, the whole chunks between them at the next level.
__global__ void k_node_boxes(int n, const int2* __restrict__ range, const int32_t* __restrict__ ipos, const float4* __restrict__ leaf_box,
                             const float4* __restrict__ c64, const float4* __restrict__ c4k, const float4* __restrict__ c256k,
                             float4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int p = ipos[i];
    if (p < 0) return; // the root and its children sit in no slot
    const int2 rg = range[i];
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    // union of arr's boxes [u, v), eight loads in flight (a clamped index
    // repeats a box of the range, which leaves the union unchanged)
    auto take = [&](const float4* arr, int u, int v) {
        for (; u < v; u += 8) {
            float4 l[8], h[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int k = min(u + t, v - 1);
                l[t] = arr[2 * k];
                h[t] = arr[2 * k + 1];
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                lo = fmin4(lo, l[t]);
                hi = fmax4(hi, h[t]);
            }
        }
    };
    const float4* lv[4] = {leaf_box, c64, c4k, c256k};
    int a = rg.x, b = rg.y + 1;
#pragma unroll
    for (int L = 0; L < 3; L++) {
        if (L == 2 && !c256k) break;
        const int a2 = min((a + 63) & ~63, b), b2 = max(b & ~63, a2);
        take(lv[L], a, a2);
        take(lv[L], b2, b);
        a = a2 >> 6;
        b = b2 >> 6;
    }
    take(c256k ? c256k : c4k, a, b);
    put_slot(rec, p, lo, hi, i, rg.y);
}

// Record slots (build only): empty slots get their constant, and every node
// that sits in a slot gets the slot's position (ipos for internal nodes;
// lpos.x for a leaf kept by its parent, lpos.y in its grandparent's record),
// each written by exactly one thread.
__global__ void k_record_slots(int n, const int32_t* __restrict__ child, float4* __restrict__ rec, int32_t* __restrict__ ipos,
                               int32_t* __restrict__ lpos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int l = child[2 * i], r = child[2 * i + 1];
    const bool li = l < n - 1, ri = r < n - 1;
    const int sl[4] = {li ? child[2 * l] : l, li ? child[2 * l + 1] : -1, ri ? child[2 * r] : r, ri ? child[2 * r + 1] : -1};
    const bool inner[4] = {li, li, ri, ri}; // slot holds a grandchild (not the child itself)
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int p = 8 * i + 2 * j, c = sl[j];
        if (c < 0) {
            rec[p] = make_float4(3e38f, 3e38f, 3e38f, __int_as_float(-1));
            rec[p + 1] = make_float4(-3e38f, -3e38f, -3e38f, __int_as_float(-1));
        } else if (c < n - 1) {
            ipos[c] = p;
        } else {
            lpos[2 * (c - (n - 1)) + (inner[j] ? 1 : 0)] = p;
        }
    }
}

// Slot j's id from the four slot ids (j is wave-divergent; selects, no
// dynamically indexed array).
__device__ inline int pick4(int j, int c0, int c1, int c2, int c3) { return j == 0 ? c0 : j == 1 ? c1 : j == 2 ? c2 : c3; }

__device__ inline bool box_far(float4 nlo, float4 nhi, float4 qlo, float4 qhi, float gap) {
    return (nlo.x - qhi.x > gap) || (qlo.x - nhi.x > gap) || (nlo.y - qhi.y > gap) || (qlo.y - nhi.y > gap) ||
           (nlo.z - qhi.z > gap) || (qlo.z - nhi.z > gap);
}

__device__ inline dv3 ldd(const double* x, int v) { return dmk(x[3 * v], x[3 * v + 1], x[3 * v + 2]); }

struct QueryOut {
    int32_t* type;
    int32_t* prim0;
    int32_t* prim1;
    int4* v;
    float4* bary;
    float4* nrm;
    double* dist;
    int cap;
};

__device__ inline void write_contact(const QueryOut& o, int idx, int type, int p0, int p1, int4 vv, const ContactFields& f,
                                     double dist) {
    o.type[idx] = type;
    o.prim0[idx] = p0;
    o.prim1[idx] = p1;
    o.v[idx] = vv;
    o.bary[idx] = make_float4((float)f.bary[0], (float)f.bary[1], (float)f.bary[2], (float)f.bary[3]);
    o.nrm[idx] = make_float4((float)f.n.x, (float)f.n.y, (float)f.n.z, (float)f.h_cN);
    o.dist[idx] = dist;
}

// Slot in the staging list for every lane of the wave that reaches this call
// together (one atomic per wave and call site; lanes that diverged away are
// not counted).
__device__ inline int stage_slot(uint32_t* __restrict__ counter) {
    const unsigned long long m = __ballot(1);
    const int lane = __lane_id();
    const int leader = __ffsll(m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    return (int)(base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)));
}

// Wide-record traversal for one query box from internal node `start`: calls
// leaf(node) for every leaf slot within `gap` of the box whose last sorted
// leaf is after `after` (-1: every used slot), in a fixed order.  The stack
// (SK entries per lane, in LDS) overflowing sets bit 0 of flags[1].
template <int SK, class Leaf>
__device__ inline void traverse(const float4* __restrict__ rec, int start, int leaf0, float4 qlo, float4 qhi, float gap, int after,
                                int32_t (*stack)[QBLK], uint32_t* __restrict__ flags, Leaf&& leaf) {
    int sp = 0, node = start;
    float4 s[8], t[8]; // the current node's record; the stack top's, loaded ahead
    int top = -1;      // the node whose record t holds
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = rec[8 * (size_t)node + j];
    while (true) {
        // The next pop takes the stack top: its record is loaded while this
        // node is processed, so a pop costs no dependent load.
        const int st_top = sp > 0 ? stack[sp - 1][threadIdx.x] : -1;
        if (st_top >= 0 && st_top != top) {
            top = st_top;
#pragma unroll
            for (int j = 0; j < 8; j++) t[j] = rec[8 * (size_t)top + j];
        }
        int c[4];
        unsigned leaves = 0, inner = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            c[j] = __float_as_int(s[2 * j].w);
            // an unused slot has id -1 and last leaf -1
            const bool hit = __float_as_int(s[2 * j + 1].w) > after && !box_far(s[2 * j], s[2 * j + 1], qlo, qhi, gap);
            if (hit) (c[j] >= leaf0 ? leaves : inner) |= 1u << j;
        }
        while (leaves) {
            const int j = __ffs(leaves) - 1;
            leaves &= leaves - 1;
            leaf(pick4(j, c[0], c[1], c[2], c[3]));
        }
        if (inner) {
            const int j = __ffs(inner) - 1;
            inner &= inner - 1;
            node = pick4(j, c[0], c[1], c[2], c[3]);
            while (inner) {
                const int u = __ffs(inner) - 1;
                inner &= inner - 1;
                if (sp < SK) stack[sp++][threadIdx.x] = pick4(u, c[0], c[1], c[2], c[3]);
                else atomicOr(&flags[1], 1u);
            }
#pragma unroll
            for (int q = 0; q < 8; q++) s[q] = rec[8 * (size_t)node + q];
        } else {
            if (sp == 0) break;
            node = stack[--sp][threadIdx.x];
            if (node == top) {
#pragma unroll
                for (int q = 0; q < 8; q++) s[q] = t[q];
                top = -1;
            } else {
#pragma unroll
                for (int q = 0; q < 8; q++) s[q] = rec[8 * (size_t)node + q];
            }
        }
    }
}

// Queries run in two passes.  Collect (MODE 0): the traversal alone, on a
// short stack (SHORT_STACK entries); the sorted index of each leaf it reaches
// goes to the query's slab (the first CAND hits, strided by the query count:
// cand[h * nq + q]) or, past CAND, to a shared overflow list of (query, leaf)
// pairs (capacity nq, filled in per-lane chunks); ccount[q] = hits.  Test
// (MODE 1): lane (q, y) runs the exact FP64 predicate on slab rows y, y + R,
// ... of query q (R = gridDim.y, test_rows: up to CAND rows for few queries,
// one for millions), and lane (i, 0) also tests overflow entry i: no
// traversal and few tests per lane, so a query with many close leaves no
// longer holds its wave through a long serial chain.  Every reached
// leaf is tested once, so the accepted set is that of the single pass
// (MODE 2: traversal and test together, on a STACK-entry stack), which runs
// instead when the short stack or the overflow list was too small (bits 0
// and 1 of flags[1]).
constexpr int CAND = 16;
constexpr int SHORT_STACK = 32;
// Slab rows spread over the test pass's grid: CAND (one test per lane) for up
// to 2^18 queries, fewer as the query count grows, 1 from 2^22 queries on.
inline int test_rows(int nq) { return std::max(1, std::min(CAND, (1 << 22) / std::max(nq, 1))); }

// Point-triangle candidate: query vertex v (FP64 position p, segment q)
// against the triangle at sorted leaf lf; an accepted pair goes to the
// staging list and qcount[q] counts it.
__device__ inline void pt_candidate(int q, int v, dv3 p, int lf, const double2* __restrict__ leafd, int n_dyn, double dhat,
                                    uint32_t* __restrict__ qcount, const QueryOut& st, int2* __restrict__ st_seg,
                                    uint32_t* __restrict__ counter) {
    const double2* L = leafd + (size_t)leaf_stride<3>() * lf;
    const double2 u0 = L[0], u1 = L[1], u2 = L[2], u3 = L[3], u4 = L[4];
    const int4 m = *reinterpret_cast<const int4*>(L + 5);
    const int f = m.x, a = m.y, b = m.z, c = m.w;
    if (v == a || v == b || v == c || (v >= n_dyn && a >= n_dyn)) return;
    const dv3 t0 = dmk(u0.x, u0.y, u1.x), t1 = dmk(u1.y, u2.x, u2.y), t2 = dmk(u3.x, u3.y, u4.x);
    const PTOut r = point_triangle(p, t0, t1, t2);
    if (!pt_accept(r, dhat)) return;
    const uint32_t place = atomicAdd(&qcount[q], 1u);
    const int idx = stage_slot(counter);
    if (idx < st.cap) {
        write_contact(st, idx, 0, v, f, make_int4(v, a, b, c), pt_fields(p, t0, t1, t2, r, dhat), r.dist);
        st_seg[idx] = make_int2(q, (int)place);
    }
}

// Hits of the collect pass: the first CAND in the query's slab, the rest in
// the overflow list, where a lane reserves OVF_CHUNK entries at a time (one
// atomic per chunk) and pads the unused end of its last chunk with query -1.
// A reservation beyond the list's capacity sets bit 1 of flags[1].
constexpr int OVF_CHUNK = 16;
struct HitSink {
    int hits = 0;
    int chunk = -1; // start of the lane's current overflow chunk (-2: list full)
    int fill = 0;   // entries used in it
    __device__ inline void add(int q, int nq, int lf, int32_t* __restrict__ cand, int2* __restrict__ ovf, uint32_t* __restrict__ ovf_count,
                               uint32_t* __restrict__ flags) {
        if (hits < CAND) {
            cand[(size_t)hits * nq + q] = lf;
        } else if (chunk != -2) {
            if (chunk < 0 || fill == OVF_CHUNK) {
                const uint32_t b = atomicAdd(ovf_count, (uint32_t)OVF_CHUNK);
                if (b + OVF_CHUNK > (uint32_t)nq) {
                    atomicOr(&flags[1], 2u);
                    chunk = -2;
                } else {
                    chunk = (int)b;
                    fill = 0;
                }
            }
            if (chunk >= 0) ovf[chunk + fill++] = make_int2(q, lf);
        }
        hits++;
    }
    __device__ inline void finish(int2* __restrict__ ovf) {
        if (chunk >= 0)
            for (int i = fill; i < OVF_CHUNK; i++) ovf[chunk + i] = make_int2(-1, -1);
    }
};

// Point-triangle queries: one lane per surface vertex q.  Accepted pairs go
// to the staging list (any order) with segment q, counted in qcount[q]
// (zeroed beforehand).
template <int MODE, int SK>
__global__ void __launch_bounds__(QBLK) k_query_pt(const double* __restrict__ x, const int32_t* __restrict__ surf_verts, int nv,
                                                   int n_dyn, int nf, const float4* __restrict__ rec,
                                                   const double2* __restrict__ leafd, double dhat, float gap, uint32_t* __restrict__ qcount,
                                                   QueryOut st, int2* __restrict__ st_seg, uint32_t* __restrict__ counter,
                                                   uint32_t* __restrict__ flags, const int32_t* __restrict__ vseg,
                                                   const int32_t* __restrict__ roots, int32_t* __restrict__ cand,
                                                   uint32_t* __restrict__ ccount, int2* __restrict__ ovf, uint32_t* __restrict__ ovf_count) {
    __shared__ int32_t stack[MODE == 1 ? 1 : SK][QBLK];
    const int leaf0 = nf - 1;
    if (MODE == 1) { // lane (q, blockIdx.y): slab rows blockIdx.y + i gridDim.y of query q; row 0 also overflow entry q
        const int q = blockIdx.x * blockDim.x + threadIdx.x;
        if (q >= nv || nf == 0) return;
        const int nh = (int)min(ccount[q], (uint32_t)CAND);
        if ((int)blockIdx.y < nh) {
            const int v = surf_verts[q];
            const dv3 p = ldd(x, v);
            for (int h = blockIdx.y; h < nh; h += gridDim.y)
                pt_candidate(q, v, p, cand[(size_t)h * nv + q], leafd, n_dyn, dhat, qcount, st, st_seg, counter);
        }
        if (blockIdx.y == 0 && !(flags[1] & 2u) && (uint32_t)q < min(*ovf_count, (uint32_t)nv)) { // a full list reruns as a single pass
            const int2 o = ovf[q];
            if (o.x >= 0) {
                const int v = surf_verts[o.x];
                pt_candidate(o.x, v, ldd(x, v), o.y, leafd, n_dyn, dhat, qcount, st, st_seg, counter);
            }
        }
        return;
    }
    const int q = xcd_block(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= nv) return;
    if (nf == 0) {
        if (MODE == 0) ccount[q] = 0;
        return;
    }
    const int v = surf_verts[q];
    const dv3 p = ldd(x, v);
    HitSink sink;
    auto leaf = [&](int node) {
        if (MODE == 0) sink.add(q, nv, node - leaf0, cand, ovf, ovf_count, flags);
        else pt_candidate(q, v, p, node - leaf0, leafd, n_dyn, dhat, qcount, st, st_seg, counter);
    };
    // start node: the root, or in segmented mode the vertex's segment subtree
    const int start = roots ? roots[vseg[v]] : 0;
    if (start < 0) {
        // no triangle in this segment
    } else if (start >= leaf0) {
        leaf(start);
    } else {
        traverse<SK>(rec, start, leaf0, pos_lo(x, v), pos_hi(x, v), gap, -1, stack, flags, leaf);
    }
    if (MODE == 0) {
        sink.finish(ovf);
        ccount[q] = (uint32_t)sink.hits;
    }
}

// Edge-edge candidate: query edge e (vertices a0, a1, FP64 endpoints A0, A1)
// against the edge at sorted leaf lf.  A pair (i, j), i < j, is evaluated
// with edge i first, as the canonical definition does, and belongs to segment
// i: it goes to the staging list with segment seg0 + i and qcount[i] counts it.
__device__ inline void ee_candidate(int e, int a0, int a1, dv3 A0, dv3 A1, int lf, const double2* __restrict__ leafd, int n_dyn,
                                    double dhat, uint32_t* __restrict__ qcount, int seg0, const QueryOut& st,
                                    int2* __restrict__ st_seg, uint32_t* __restrict__ counter) {
    const double2* L = leafd + (size_t)leaf_stride<2>() * lf;
    const double2 u0 = L[0], u1 = L[1], u2 = L[2];
    const int4 m = *reinterpret_cast<const int4*>(L + 3);
    const int f = m.x, b0 = m.y, b1 = m.z;
    if (a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1 || (a0 >= n_dyn && b0 >= n_dyn)) return;
    const dv3 B0 = dmk(u0.x, u0.y, u1.x), B1 = dmk(u1.y, u2.x, u2.y);
    const bool first = e < f;
    const int i = first ? e : f, j = first ? f : e;
    const int i0 = first ? a0 : b0, i1 = first ? a1 : b1, j0 = first ? b0 : a0, j1 = first ? b1 : a1;
    const dv3 P0 = first ? A0 : B0, P1 = first ? A1 : B1, Q0 = first ? B0 : A0, Q1 = first ? B1 : A1;
    const EEOut r = segment_segment(P0, P1, Q0, Q1);
    if (!ee_accept(r, dhat)) return;
    const uint32_t place = atomicAdd(&qcount[i], 1u);
    const int idx = stage_slot(counter);
    if (idx < st.cap) {
        write_contact(st, idx, 1, i, j, make_int4(i0, i1, j0, j1), ee_fields(P0, P1, Q0, Q1, r, dhat), r.dist);
        st_seg[idx] = make_int2(seg0 + i, (int)place);
    }
}

// The query edge at sorted leaf k: id, vertices and FP64 endpoints.
struct EEQuery {
    int e, a0, a1;
    dv3 A0, A1;
};
__device__ inline EEQuery ee_query(const double2* __restrict__ leafd, int k) {
    const double2* Lk = leafd + (size_t)leaf_stride<2>() * k;
    const double2 w0 = Lk[0], w1 = Lk[1], w2 = Lk[2];
    const int4 mk = *reinterpret_cast<const int4*>(Lk + 3);
    return EEQuery{mk.x, mk.y, mk.z, dmk(w0.x, w0.y, w1.x), dmk(w1.y, w2.x, w2.y)};
}

// Edge-edge queries: lane k takes the edge at sorted leaf k and reaches only
// leaves after k, so each unordered pair is tested once (qcount zeroed
// beforehand).
template <int MODE, int SK>
__global__ void __launch_bounds__(QBLK) k_query_ee(int ne, int n_dyn, const float4* __restrict__ rec,
                                                   const double2* __restrict__ leafd, double dhat,
                                                   float gap, uint32_t* __restrict__ qcount, int seg0, QueryOut st,
                                                   int2* __restrict__ st_seg, uint32_t* __restrict__ counter,
                                                   uint32_t* __restrict__ flags, const int32_t* __restrict__ vseg,
                                                   const int32_t* __restrict__ roots, int32_t* __restrict__ cand,
                                                   uint32_t* __restrict__ ccount, int2* __restrict__ ovf, uint32_t* __restrict__ ovf_count) {
    __shared__ int32_t stack[MODE == 1 ? 1 : SK][QBLK];
    if (ne < 2) return;
    const int leaf0 = ne - 1;
    if (MODE == 1) { // lane (k, blockIdx.y): slab rows blockIdx.y + i gridDim.y of query k; row 0 also overflow entry k
        const int k = blockIdx.x * blockDim.x + threadIdx.x;
        if (k >= ne) return;
        const int nh = (int)min(ccount[k], (uint32_t)CAND);
        if ((int)blockIdx.y < nh) {
            const EEQuery Q = ee_query(leafd, k);
            for (int h = blockIdx.y; h < nh; h += gridDim.y)
                ee_candidate(Q.e, Q.a0, Q.a1, Q.A0, Q.A1, cand[(size_t)h * ne + k], leafd, n_dyn, dhat, qcount, seg0, st, st_seg, counter);
        }
        if (blockIdx.y == 0 && !(flags[1] & 2u) && (uint32_t)k < min(*ovf_count, (uint32_t)ne)) { // a full list reruns as a single pass
            const int2 o = ovf[k];
            if (o.x >= 0) {
                const EEQuery Q = ee_query(leafd, o.x);
                ee_candidate(Q.e, Q.a0, Q.a1, Q.A0, Q.A1, o.y, leafd, n_dyn, dhat, qcount, seg0, st, st_seg, counter);
            }
        }
        return;
    }
    const int k = xcd_block(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= ne) return;
    // the query edge is leaf k itself
    const EEQuery Q = ee_query(leafd, k);
    HitSink sink;
    auto leaf = [&](int node) {
        if (MODE == 0) sink.add(k, ne, node - leaf0, cand, ovf, ovf_count, flags);
        else ee_candidate(Q.e, Q.a0, Q.a1, Q.A0, Q.A1, node - leaf0, leafd, n_dyn, dhat, qcount, seg0, st, st_seg, counter);
    };
    // start node: the root, or in segmented mode the edge's segment subtree
    // (a segment with one edge has no pair)
    const int start = roots ? roots[vseg[Q.a0]] : 0;
    if (start >= 0 && start < leaf0) {
        const float4 qlo = make_float4(__double2float_rd(fmin(Q.A0.x, Q.A1.x)), __double2float_rd(fmin(Q.A0.y, Q.A1.y)),
                                       __double2float_rd(fmin(Q.A0.z, Q.A1.z)), 0.f);
        const float4 qhi = make_float4(__double2float_ru(fmax(Q.A0.x, Q.A1.x)), __double2float_ru(fmax(Q.A0.y, Q.A1.y)),
                                       __double2float_ru(fmax(Q.A0.z, Q.A1.z)), 0.f);
        traverse<SK>(rec, start, leaf0, qlo, qhi, gap, k, stack, flags, leaf);
    }
    if (MODE == 0) {
        sink.finish(ovf);
        ccount[k] = (uint32_t)sink.hits;
    }
}

// Canonical order of the staged contacts: segment by segment, sorted by
// partner id inside a segment.  The partner ids go to their segments first
// (in the order the test pass met them), then every staged contact counts the
// smaller ids of its segment (a pair occurs once, so ids are distinct) and
// moves straight to its final place.  The counts are independent loads over
// one lane per contact; an insertion sort by one lane per segment moved each
// 68-byte record several times in a dependent chain (13-30 us per detection
// for segments of 10 to 30).
__global__ void k_segment_keys(int n, const int2* __restrict__ st_seg, const int32_t* __restrict__ prim1,
                               const uint32_t* __restrict__ qoffset, int32_t* __restrict__ seg_key) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const int2 sg = st_seg[c];
    seg_key[qoffset[sg.x] + sg.y] = prim1[c];
}

__global__ void k_place_contacts(int n, const int2* __restrict__ st_seg, QueryOut st, const uint32_t* __restrict__ qoffset,
                                 const uint32_t* __restrict__ qcount, const int32_t* __restrict__ seg_key, QueryOut o, VertexCount vc) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const int sg = st_seg[c].x;
    const int begin = (int)qoffset[sg], cnt = (int)qcount[sg];
    const int key = st.prim1[c];
    const int4 v = st.v[c];
    int rank = 0;
    for (int q = 0; q < cnt; q += 8) {
        int k[8];
#pragma unroll
        for (int u = 0; u < 8; u++) k[u] = seg_key[begin + min(q + u, cnt - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++) rank += q + u < cnt && k[u] < key ? 1 : 0;
    }
    const int idx = begin + rank;
    o.type[idx] = st.type[c];
    o.prim0[idx] = st.prim0[c];
    o.prim1[idx] = key;
    o.v[idx] = v;
    o.bary[idx] = st.bary[c];
    o.nrm[idx] = st.nrm[c];
    o.dist[idx] = st.dist[c];
    if (vc.cnt) {
        int4 l;
        l.x = (int)atomicAdd(&vc.cnt[v.x], 1u);
        l.y = (int)atomicAdd(&vc.cnt[v.y], 1u);
        l.z = (int)atomicAdd(&vc.cnt[v.z], 1u);
        l.w = (int)atomicAdd(&vc.cnt[v.w], 1u);
        vc.loc[idx] = l;
    }
}

} // namespace

Detector::Detector(int n_all_, int n_dyn_, int nv_, const int32_t* sv, int nf_, const int32_t* t, int ne_, const int32_t* e,
                   int cap, double dhat_, hipStream_t s)
    : stream(s), n_all(n_all_), n_dyn(n_dyn_), nv(nv_), nf(nf_), ne(ne_), dhat(dhat_) {
    PA_CHECK(cap > 0, PA_ERR_INVALID, "detector capacity must be positive");
    PA_CHECK(dhat > 0, PA_ERR_INVALID, "thickness must be positive");
    if (!stream) {
        PA_HIP(hipStreamCreateWithFlags(&own_stream, hipStreamNonBlocking));
        stream = own_stream;
    }
    PA_HIP(hipStreamCreateWithFlags(&side, hipStreamNonBlocking)); // default priority
    PA_HIP(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming));
    PA_HIP(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming));
    for (int i = 0; i < nv; i++) PA_CHECK(sv[i] >= 0 && sv[i] < n_all, PA_ERR_INVALID, "surface vertex out of range");
    for (int i = 0; i < 3 * nf; i++) PA_CHECK(t[i] >= 0 && t[i] < n_all, PA_ERR_INVALID, "surface triangle index out of range");
    for (int i = 0; i < 2 * ne; i++) PA_CHECK(e[i] >= 0 && e[i] < n_all, PA_ERR_INVALID, "surface edge index out of range");
    surf_verts.alloc(nv);
    surf_verts.upload(sv, nv, stream);
    tris.alloc(3 * (size_t)nf);
    tris.upload(t, 3 * (size_t)nf, stream);
    edges.alloc(2 * (size_t)ne);
    edges.upload(e, 2 * (size_t)ne, stream);
    edges_h.assign(e, e + 2 * (size_t)ne);
    auto init_tree = [&](Tree& T, int n, int stride) {
        T.n = n;
        T.leaf_stride = stride;
        if (n == 0) return;
        T.prim_box.alloc(2 * (size_t)n);
        T.leaf_box.alloc(2 * (size_t)n);
        T.leafd.alloc((size_t)T.leaf_stride * n);
        T.ipos.alloc(std::max(n - 1, 1));
        T.lpos.alloc(2 * (size_t)n);
        T.keys.alloc(n);
        T.ids.alloc(n);
        T.child.alloc(2 * (size_t)std::max(n - 1, 1));
        T.range.alloc(std::max(n - 1, 1));
        T.rec.alloc(8 * (size_t)std::max(n - 1, 1));
        T.chunk64.alloc(2 * (size_t)((n + 63) / 64));
        T.chunk4k.alloc(2 * (size_t)((n + 4095) / 4096));
        T.chunk256k.alloc(2 * (size_t)((n + 262143) / 262144));
        T.scene.alloc(2);
        T.partial.alloc(2 * 256);
    };
    init_tree(ft, nf, leaf_stride<3>());
    init_tree(et, ne, leaf_stride<2>());
    c.cap = cap;
    c.type.alloc(cap);
    c.prim0.alloc(cap);
    c.prim1.alloc(cap);
    c.v.alloc(cap);
    c.bary.alloc(cap);
    c.nrm.alloc(cap);
    c.dist.alloc(cap);
    counts.alloc((size_t)nv + ne + 8);
    total = counts.p;
    ovf_count = counts.p + 3;
    qcount = counts.p + 8; // 16-byte aligned for the scan
    qoffset.alloc((size_t)nv + ne + 1);
    PA_HIP(hipHostMalloc((void**)&total_host, 3 * sizeof(uint32_t), hipHostMallocDefault));
    stg.cap = cap;
    stg.type.alloc(cap);
    stg.prim0.alloc(cap);
    stg.prim1.alloc(cap);
    stg.v.alloc(cap);
    stg.bary.alloc(cap);
    stg.nrm.alloc(cap);
    stg.dist.alloc(cap);
    st_seg.alloc(cap);
    seg_key.alloc(cap);
    cand_pt.alloc((size_t)CAND * std::max(nv, 1));
    cand_ee.alloc((size_t)CAND * std::max(ne, 1));
    ccount_pt.alloc(std::max(nv, 1));
    ccount_ee.alloc(std::max(ne, 1));
    ovf_pt.alloc(std::max(nv, 1));
    ovf_ee.alloc(std::max(ne, 1));
    PA_HIP(hipStreamSynchronize(stream));
}

Detector::~Detector() {
    if (side) {
        (void)hipStreamSynchronize(side);
        (void)hipStreamDestroy(side);
    }
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    if (ev_join) (void)hipEventDestroy(ev_join);
    if (total_host) (void)hipHostFree(total_host); // every scan that writes it is waited for in detect()
    if (own_stream) {
        (void)hipStreamSynchronize(own_stream);
        (void)hipStreamDestroy(own_stream);
    }
}

void Detector::build_tree(Tree& T, const double* x, bool faces, hipStream_t stream, PrimScratch& scratch, bool refit) {
    const int n = T.n;
    if (n == 0) return;
    auto leaf_data = [&]() {
        if (faces)
            hipLaunchKernelGGL(k_leaf_data<3>, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, x, (const int32_t*)tris.p,
                               (const uint32_t*)T.ids.p, n, T.leaf_box.p, T.leafd.p, (const int2*)T.lpos.p, T.rec.p);
        else
            hipLaunchKernelGGL(k_leaf_data<2>, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, x, (const int32_t*)edges.p,
                               (const uint32_t*)T.ids.p, n, T.leaf_box.p, T.leafd.p, (const int2*)T.lpos.p, T.rec.p);
        PA_LAUNCH_CHECK();
    };
    if (refit) { // same sorted order and Karras topology, new boxes and leaf data
        leaf_data();
        if (n > 1) node_boxes(T, stream);
        return;
    }
    hipLaunchKernelGGL(k_prim_boxes, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, x, faces ? tris.p : edges.p, faces ? 3 : 2, n,
                       T.prim_box.p);
    PA_LAUNCH_CHECK();
    const int nb = std::min(256, grid_for(n, BLK));
    hipLaunchKernelGGL(k_box_union, dim3(nb), dim3(BLK), 0, stream, T.prim_box.p, n, T.partial.p);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_box_union, dim3(1), dim3(BLK), 0, stream, T.partial.p, nb, T.scene.p);
    PA_LAUNCH_CHECK();
    if (nseg > 0) {
        hipLaunchKernelGGL(k_morton_seg, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, T.prim_box.p, faces ? tris.p : edges.p,
                           faces ? 3 : 2, n, (const int32_t*)vseg.p, T.scene.p, T.keys.p, T.ids.p);
        PA_LAUNCH_CHECK();
        radix_sort_pairs(T.keys.p, T.ids.p, n, 32, scratch, stream);
    } else {
        hipLaunchKernelGGL(k_morton, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, T.prim_box.p, n, T.scene.p, T.keys.p, T.ids.p);
        PA_LAUNCH_CHECK();
        radix_sort_pairs(T.keys.p, T.ids.p, n, 30, scratch, stream);
    }
    if (n > 1) {
        hipLaunchKernelGGL(k_karras, dim3(grid_for(n - 1, BLK)), dim3(BLK), 0, stream, T.keys.p, T.ids.p, n, T.child.p, T.range.p);
        PA_LAUNCH_CHECK();
        fill<int32_t>(T.ipos.p, -1, n - 1, stream);
        fill<int32_t>(T.lpos.p, -1, 2 * (int64_t)n, stream);
        hipLaunchKernelGGL(k_record_slots, dim3(grid_for(n - 1, BLK)), dim3(BLK), 0, stream, n, (const int32_t*)T.child.p, T.rec.p,
                           T.ipos.p, T.lpos.p);
        PA_LAUNCH_CHECK();
    }
    leaf_data();
    if (n > 1) node_boxes(T, stream);
    if (nseg > 0) {
        fill<int32_t>(T.seg_first.p, -1, nseg, stream);
        fill<int32_t>(T.seg_last.p, -1, nseg, stream);
        fill<int32_t>(T.seg_root.p, -1, nseg, stream);
        hipLaunchKernelGGL(k_seg_bounds, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, (const uint32_t*)T.keys.p, n, T.seg_first.p,
                           T.seg_last.p);
        PA_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_seg_roots, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, n, (const int2*)T.range.p, (const uint32_t*)T.keys.p,
                           (const int32_t*)T.seg_first.p, (const int32_t*)T.seg_last.p, T.seg_root.p);
        PA_LAUNCH_CHECK();
    }
}

// Internal node boxes from the leaf boxes (chunk unions, range unions),
// written into their record slots (the leaves' slots are written with the
// leaf data).  The 262144-leaf level is built only where a range can hold
// more than 64 of the 4096-leaf chunks.
void Detector::node_boxes(Tree& T, hipStream_t stream) {
    const int n = T.n;
    const int n64 = (n + 63) / 64, n4k = (n + 4095) / 4096, n256k = (n + 262143) / 262144;
    hipLaunchKernelGGL(k_chunk_union, dim3(grid_for((int64_t)n64 * 64, BLK)), dim3(BLK), 0, stream, (const float4*)T.leaf_box.p, n,
                       T.chunk64.p, n64);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_chunk_union, dim3(grid_for((int64_t)n4k * 64, BLK)), dim3(BLK), 0, stream, (const float4*)T.chunk64.p, n64,
                       T.chunk4k.p, n4k);
    PA_LAUNCH_CHECK();
    const bool top = n4k > 64;
    if (top) {
        hipLaunchKernelGGL(k_chunk_union, dim3(grid_for((int64_t)n256k * 64, BLK)), dim3(BLK), 0, stream, (const float4*)T.chunk4k.p,
                           n4k, T.chunk256k.p, n256k);
        PA_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_node_boxes, dim3(grid_for(n - 1, BLK)), dim3(BLK), 0, stream, n, (const int2*)T.range.p, (const int32_t*)T.ipos.p,
                       (const float4*)T.leaf_box.p, (const float4*)T.chunk64.p, (const float4*)T.chunk4k.p,
                       top ? (const float4*)T.chunk256k.p : nullptr, T.rec.p);
    PA_LAUNCH_CHECK();
}

void Detector::set_segments(const int32_t* vs, int count) {
    PA_CHECK(count >= 1 && count <= 2048, PA_ERR_INVALID, "segment count must be in [1, 2048]");
    for (int i = 0; i < n_all; i++) PA_CHECK(vs[i] >= 0 && vs[i] < count, PA_ERR_INVALID, "vertex segment out of range");
    // a primitive's vertices must share one segment (its key takes the first vertex's)
    std::vector<int32_t> t(3 * (size_t)nf), e(2 * (size_t)ne);
    tris.download(t.data(), t.size(), stream);
    edges.download(e.data(), e.size(), stream);
    PA_HIP(hipStreamSynchronize(stream));
    for (int f = 0; f < nf; f++)
        PA_CHECK(vs[t[3 * f]] == vs[t[3 * f + 1]] && vs[t[3 * f]] == vs[t[3 * f + 2]], PA_ERR_INVALID, "triangle spans two segments");
    for (int k = 0; k < ne; k++) PA_CHECK(vs[e[2 * k]] == vs[e[2 * k + 1]], PA_ERR_INVALID, "edge spans two segments");
    vseg.alloc(n_all);
    vseg.upload(vs, n_all, stream);
    nseg = count;
    built = false; // keys change: the next detection rebuilds
    for (Tree* T : {&ft, &et}) {
        T->seg_first.alloc(count);
        T->seg_last.alloc(count);
        T->seg_root.alloc(count);
    }
}

int Detector::detect(const double* x, bool refit, VertexCount vc) {
    refit = refit && built;
    // the edge tree (build, query) runs on the side stream beside the triangle tree
    fill2<uint32_t>(counts.p, 8 + (int64_t)nv + ne, vc.cnt, vc.cnt ? vc.n : 0, 0u, stream);
    PA_HIP(hipEventRecord(ev_fork, stream));
    PA_HIP(hipStreamWaitEvent(side, ev_fork, 0));
    const float gap = (float)(dhat * 1.001);
    QueryOut o{c.type.p, c.prim0.p, c.prim1.p, c.v.p, c.bary.p, c.nrm.p, c.dist.p, c.cap};
    QueryOut st{stg.type.p, stg.prim0.p, stg.prim1.p, stg.v.p, stg.bary.p, stg.nrm.p, stg.dist.p, stg.cap};
    const int32_t* ee_roots = nseg > 0 ? (const int32_t*)et.seg_root.p : nullptr;
    const int32_t* pt_roots = nseg > 0 ? (const int32_t*)ft.seg_root.p : nullptr;
    // Per query a collect pass (traversal, leaf hits to the slab or the
    // overflow list) and a test pass (FP64 predicate): pairs to the staging
    // list (total[2] counts them, atomically from both streams), per-segment
    // counts to qcount.  The edge tree and its queries, the longer chain, are
    // enqueued first so the side stream starts while the host still enqueues
    // the triangle tree.
    auto ee_pass = [&](auto mode, auto sk, hipStream_t s, dim3 grid) {
        hipLaunchKernelGGL((k_query_ee<decltype(mode)::value, decltype(sk)::value>), grid, dim3(QBLK), 0, s, ne, n_dyn,
                           (const float4*)et.rec.p, (const double2*)et.leafd.p, dhat, gap, qcount + nv, nv, st, st_seg.p, total + 2,
                           total, (const int32_t*)vseg.p, ee_roots, cand_ee.p, ccount_ee.p, ovf_ee.p, ovf_count + 1);
        PA_LAUNCH_CHECK();
    };
    auto pt_pass = [&](auto mode, auto sk, hipStream_t s, dim3 grid) {
        hipLaunchKernelGGL((k_query_pt<decltype(mode)::value, decltype(sk)::value>), grid, dim3(QBLK), 0, s, x, surf_verts.p, nv,
                           n_dyn, nf, (const float4*)ft.rec.p, (const double2*)ft.leafd.p, dhat, gap, qcount, st, st_seg.p,
                           total + 2, total, (const int32_t*)vseg.p, pt_roots, cand_pt.p, ccount_pt.p, ovf_pt.p, ovf_count);
        PA_LAUNCH_CHECK();
    };
    using M0 = std::integral_constant<int, 0>;
    using M1 = std::integral_constant<int, 1>;
    using M2 = std::integral_constant<int, 2>;
    using SS = std::integral_constant<int, SHORT_STACK>;
    using LS = std::integral_constant<int, STACK>;
    const bool two = !force_single_pass;
    build_tree(et, x, false, side, scratch_side, refit);
    if (ne > 0 && two) {
        ee_pass(M0{}, SS{}, side, dim3(query_grid(ne)));
        ee_pass(M1{}, SS{}, side, dim3(grid_for(ne, QBLK), test_rows(ne)));
    }
    build_tree(ft, x, true, stream, scratch, refit);
    built = true;
    if (nv > 0 && two) {
        pt_pass(M0{}, SS{}, stream, dim3(query_grid(nv)));
        pt_pass(M1{}, SS{}, stream, dim3(grid_for(nv, QBLK), test_rows(nv)));
    }
    PA_HIP(hipEventRecord(ev_join, side));
    PA_HIP(hipStreamWaitEvent(stream, ev_join, 0));
    uint32_t h[3] = {0u, 0u, 0u};
    auto count_found = [&](uint32_t* o) { // segment offsets; the totals reach the host with the scan's last launch
        scan_exclusive(qcount, qoffset.p, (int64_t)nv + ne, total, scratch, stream, total_host);
        PA_HIP(hipStreamSynchronize(stream));
        for (int k = 0; k < 3; k++) o[k] = total_host[k];
    };
    if (two) {
        count_found(h);
    }
    if (!two || h[1] != 0) {
        // the short stack or an overflow list was too small: the single pass
        // (traversal and test together, full stack) for both queries
        fill<uint32_t>(counts.p, 0u, 8 + (int64_t)nv + ne, stream);
        if (ne > 0) ee_pass(M2{}, LS{}, stream, dim3(query_grid(ne)));
        if (nv > 0) pt_pass(M2{}, LS{}, stream, dim3(query_grid(nv)));
        count_found(h);
        if (two) single_pass_fallbacks++;
    }
    found_total = h[0];
    stack_overflow = h[1] != 0;
    PA_CHECK(!stack_overflow, PA_ERR_INVALID, "LBVH traversal stack overflow");
    PA_CHECK(h[2] == h[0], PA_ERR_INVALID, "contact staging count differs from the segment counts");
    if (found_total > c.cap) {
        n_contacts = 0;
        throw Error(PA_ERR_OVERFLOW, "contact capacity exceeded: found " + std::to_string(found_total) + " > " + std::to_string(c.cap));
    }
    n_contacts = (int)found_total;
    peak = std::max(peak, n_contacts);
    if (n_contacts > 0) {
        // canonical order: segments in query order (PT by vertex, EE by the
        // smaller edge id), each sorted by partner id
        hipLaunchKernelGGL(k_segment_keys, dim3(grid_for(n_contacts, BLK)), dim3(BLK), 0, stream, n_contacts, (const int2*)st_seg.p,
                           (const int32_t*)stg.prim1.p, (const uint32_t*)qoffset.p, seg_key.p);
        PA_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_place_contacts, dim3(grid_for(n_contacts, BLK)), dim3(BLK), 0, stream, n_contacts, (const int2*)st_seg.p, st,
                           (const uint32_t*)qoffset.p, (const uint32_t*)qcount, (const int32_t*)seg_key.p, o, vc);
        PA_LAUNCH_CHECK();
    }
    return n_contacts;
}

} // namespace pa
