// LBVH proximity detection on gfx950.
//
// Per detection: primitive boxes -> scene box -> 30-bit Morton codes ->
// stable LDS radix sort -> Karras radix tree (T. Karras, "Maximizing
// Parallelism in the Construction of BVHs, Octrees, and k-d Trees", HPG 2012)
// -> node boxes from leaf ranges -> 128-byte wide node records (the boxes,
// ids and last sorted leaf of a node's up to four grandchildren, a leaf child
// standing in for its own pair, so a traversal step descends two levels with
// one dependent load) -> a traversal by waves that share a stack, collecting close
// leaves, then the FP64 predicate on them, accepted pairs marked and counted
// per segment.
//
// Point-triangle: one query per surface vertex; its pairs form the vertex's
// segment.  Edge-edge: one query per sorted leaf k, visiting only leaves after
// k, so each unordered pair is tested once; the pair belongs to the segment of
// its smaller edge id.  Segment counts -> exclusive scan -> partner ids into
// their segments -> every pair's fields to its rank in its segment: the list comes out
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
constexpr int STACK = 64;          // single pass: stack entries per lane
constexpr int CAND = 16;           // collected hits per query before the overflow list
constexpr int CBLK = 256;          // collect block (four waves)
constexpr int CSTACK = 1024, CSTACK_HIGH = 768; // collect: stack entries per wave, and the depth-first threshold
constexpr int COLLECT_BITS = 26;   // collect: node and leaf indices in a packed entry
constexpr uint32_t COLLECT_MASK = (1u << COLLECT_BITS) - 1u;
constexpr int TBLK = 256, TQ = 64; // test block and its queries

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

__device__ inline uint32_t morton_key(float4 lo, float4 hi, float4 slo, float4 shi, float cells, float last) {
    const float ex = shi.x - slo.x, ey = shi.y - slo.y, ez = shi.z - slo.z;
    const float cx = 0.5f * (lo.x + hi.x) - slo.x, cy = 0.5f * (lo.y + hi.y) - slo.y, cz = 0.5f * (lo.z + hi.z) - slo.z;
    auto cell = [&](float u) { return (uint32_t)fminf(fmaxf(u * cells, 0.0f), last); };
    return (spread10(cell(ex > 0.f ? cx / ex : 0.f)) << 2) | (spread10(cell(ey > 0.f ? cy / ey : 0.f)) << 1) | spread10(cell(ez > 0.f ? cz / ez : 0.f));
}

__global__ void k_morton(const float4* __restrict__ box, int n, const float4* __restrict__ scene, uint32_t* __restrict__ keys,
                         uint32_t* __restrict__ ids) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = morton_key(box[2 * i], box[2 * i + 1], scene[0], scene[1], 1024.0f, 1023.0f);
    ids[i] = (uint32_t)i;
}

// Segmented keys: segment id in the top 11 bits, then a 21-bit Morton code
// (7 bits per axis) of the box centre in the box of all segments.
__global__ void k_morton_seg(const float4* __restrict__ box, const int32_t* __restrict__ prims, int k, int n,
                             const int32_t* __restrict__ vseg, const float4* __restrict__ scene, uint32_t* __restrict__ keys,
                             uint32_t* __restrict__ ids) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = ((uint32_t)vseg[prims[k * i]] << 21) | morton_key(box[2 * i], box[2 * i + 1], scene[0], scene[1], 128.0f, 127.0f); // 21 bits
    ids[i] = (uint32_t)i;
}

// Sorted leaves of a tree of up to SMALL_BUILD primitives in one workgroup:
// primitive boxes, scene box, keys, the radix sort (the elements of a pass in
// registers, written back to LDS in their new order) and the leaf ids, with the
// results of the kernels above and radix_sort_pairs.  Those take 17 launches
// and about 110 us for a tree of 5000 primitives, little of it work; this takes
// 34-47 us on one CU, and both trees run side by side.  SMALL_BUILD is what LDS
// holds, and it wins up to there: a detection of a cloth over its sphere takes
// 0.12 ms with it against 0.20-0.23 with the launches at 2,625 edges, 0.16
// against 0.21-0.24 at 6,800, 0.19 against 0.21-0.24 at 13,953 and 0.20-0.21
// against 0.21-0.24 at 16,341 (ranges over two processes).
constexpr int SMALL_BUILD = 16384, SB_BLK = 1024, SB_ITEMS = SMALL_BUILD / SB_BLK, SB_WAVES = SB_BLK / 64;
struct SmallTree {
    const int32_t* prims;
    int k, n; // vertices per primitive, primitives
    uint32_t* keys;
    uint32_t* ids;
    int4* leafid;
};
__global__ void __launch_bounds__(SB_BLK) k_build_small(const double* __restrict__ x, const int32_t* __restrict__ vseg, SmallTree E, SmallTree F) {
    __shared__ uint32_t lk[SMALL_BUILD], li[SMALL_BUILD / 2]; // keys; ids fit 14 bits, two to a word
    __shared__ uint32_t cnt[SB_WAVES][256];
    __shared__ float4 slo[SB_WAVES], shi[SB_WAVES];
    const SmallTree& T = blockIdx.x == 0 ? E : F;
    const int n = T.n;
    if (n == 0) return;
    uint16_t* const lid = reinterpret_cast<uint16_t*>(li);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // a wave owns consecutive elements, so that equal digits keep their order
    const int items = (n + SB_BLK - 1) / SB_BLK, e0 = wave * 64 * items + lane;
    float4 lo[SB_ITEMS], hi[SB_ITEMS], blo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), bhi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    uint32_t key[SB_ITEMS], id[SB_ITEMS];
#pragma unroll
    for (int j = 0; j < SB_ITEMS; j++) {
        const int e = e0 + 64 * j;
        lo[j] = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
        hi[j] = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
        if (j < items && e < n)
            for (int q = 0; q < T.k; q++) {
                const int v = T.prims[T.k * e + q];
                lo[j] = fmin4(lo[j], pos_lo(x, v));
                hi[j] = fmax4(hi[j], pos_hi(x, v));
            }
        blo = fmin4(blo, lo[j]);
        bhi = fmax4(bhi, hi[j]);
    }
    blo = wave_min4(blo);
    bhi = wave_max4(bhi);
    if (lane == 0) {
        slo[wave] = blo;
        shi[wave] = bhi;
    }
    __syncthreads();
    for (int w = 0; w < SB_WAVES; w++) {
        blo = fmin4(blo, slo[w]);
        bhi = fmax4(bhi, shi[w]);
    }
#pragma unroll
    for (int j = 0; j < SB_ITEMS; j++) {
        const int e = e0 + 64 * j;
        key[j] = 0u;
        id[j] = (uint32_t)e;
        if (j < items && e < n)
            key[j] = vseg ? (uint32_t)vseg[T.prims[T.k * e]] << 21 | morton_key(lo[j], hi[j], blo, bhi, 128.0f, 127.0f)
                          : morton_key(lo[j], hi[j], blo, bhi, 1024.0f, 1023.0f);
    }
    for (int shift = 0; shift < 32; shift += 8) {
        for (int c = t; c < SB_WAVES * 256; c += SB_BLK) cnt[c >> 8][c & 255] = 0;
        __syncthreads();
        uint32_t pos[SB_ITEMS];
#pragma unroll
        for (int j = 0; j < SB_ITEMS; j++)
            pos[j] = j < items ? rs_rank((key[j] >> shift) & 255u, e0 + 64 * j < n, cnt[wave]) : 0u;
        __syncthreads();
        // digit d's start: the smaller digits' totals, then the waves before
        uint32_t tot = 0;
        if (t < 256)
            for (int w = 0; w < SB_WAVES; w++) tot += cnt[w][t];
        uint32_t inc = tot;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(inc, o, 64);
            if (lane >= o) inc += y;
        }
        if (t < 256 && lane == 63) lk[wave] = inc; // lk is free here: the elements are in registers
        __syncthreads();
        if (t < 256) {
            uint32_t run = inc - tot;
            for (int w = 0; w < wave; w++) run += lk[w];
            for (int w = 0; w < SB_WAVES; w++) {
                const uint32_t c = cnt[w][t];
                cnt[w][t] = run;
                run += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SB_ITEMS; j++)
            if (j < items && e0 + 64 * j < n) {
                const uint32_t p = cnt[wave][(key[j] >> shift) & 255u] + pos[j];
                lk[p] = key[j];
                lid[p] = (uint16_t)id[j];
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SB_ITEMS; j++)
            if (j < items && e0 + 64 * j < n) {
                key[j] = lk[e0 + 64 * j];
                id[j] = lid[e0 + 64 * j];
            }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < SB_ITEMS; j++) {
        const int e = e0 + 64 * j;
        if (j < items && e < n) {
            T.keys[e] = key[j];
            T.ids[e] = id[j];
            const int32_t* p = T.prims + T.k * (int)id[j];
            T.leafid[e] = make_int4((int)id[j], p[0], p[1], T.k == 3 ? p[2] : -1);
        }
    }
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

// What the build of a tree's topology reads and writes.  Both trees share a
// launch, as in a refit.
struct TopoArgs {
    int n;
    const uint32_t* keys;
    const uint32_t* ids;
    int32_t* child;
    int2* range;
    int32_t* ipos;
    int32_t* lpos;
    float4* rec;
};

// Karras construction of internal node i over sorted unique 64-bit keys; also
// clears the slot positions that k_record_slots then fills (-1: none).
__global__ void k_karras(TopoArgs E, TopoArgs F, int e_blocks) {
    const bool edges = (int)blockIdx.x < e_blocks;
    const TopoArgs& T = edges ? E : F;
    const uint32_t *__restrict__ keys = T.keys, *__restrict__ ids = T.ids;
    int32_t* __restrict__ child = T.child;
    int2* __restrict__ range = T.range;
    const int n = T.n;
    int i = (edges ? (int)blockIdx.x : (int)blockIdx.x - e_blocks) * (int)blockDim.x + (int)threadIdx.x;
    if (i < n) reinterpret_cast<int2*>(T.lpos)[i] = make_int2(-1, -1);
    if (i >= n - 1) return;
    T.ipos[i] = -1;
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
// of that range (k_refit, k_cross_boxes).  (A bottom-up climb with atomic visit
// flags needs device-scope fences, which write back and invalidate the per-XCD
// L2 on this part.)
// Leaf ids of a tree: per sorted leaf its primitive id and vertex ids (-1 for
// none), written once per build, so a query tests a leaf's vertices with one
// load instead of the chain sorted id -> vertex ids.
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

// Refit of RB consecutive sorted leaves: their boxes from x (a box is the
// primitive box of k_prim_boxes, the outward-rounded FP32 of the FP64
// positions) into their record slots, the box of every internal node whose
// leaf range lies inside the block, and the block's own box (blk_box).
// Node i's range begins or ends at leaf i (Karras), so node i of this block
// is the only kind that can.  Its box is the union of two overlapping windows
// of a power of two leaves (a union may count a leaf twice), read from a table
// of all such windows that the block builds in LDS in log2(RB) steps: a node
// costs two reads whatever its range.  Unions straight from the leaf boxes and
// from chunks of them in memory are a chain of up to 30 dependent loads per node
// (edges of a 160-scene batch: 632 us in three launches, against 233 for this
// and 93 for k_cross_boxes).  Blocks of 128 and 64 leaves leave two and four
// times the crossing nodes and were slower in sum (edges of the 256x256 cloth:
// 19 + 12 and 17 + 21 us, 16 + 9 with 256).  Both trees of that cloth: 20 + 15
// us; 512 scenes: 679 + 287 us, where the 55 KB of LDS that leave a CU two
// blocks bound it.
//
// Both trees share a launch here and in the kernels below: first the blocks of
// the edge tree, the longer chain, then those of the triangle tree.  Two
// streams cost a small scene's host more than its GPU gains, and a large
// scene's launches fill the chip by themselves.
constexpr int RB = 256, RB_LEVELS = 9;
struct TreeArgs {
    int n; // leaves
    const int4* leafid;
    float4* leaf_box;
    const int2* lpos;
    const int2* range;
    const int32_t* ipos;
    float4* blk_box;
    float4* rec;
};
template <int K>
__device__ inline void refit_block(const TreeArgs& T, int block, const double* __restrict__ x, float (&win)[RB_LEVELS][6][RB]) {
    const int n = T.n;
    const int4* __restrict__ leafid = T.leafid;
    const int2 *__restrict__ lpos = T.lpos, *__restrict__ range = T.range;
    const int32_t* __restrict__ ipos = T.ipos;
    float4 *__restrict__ leaf_box = T.leaf_box, *__restrict__ blk_box = T.blk_box, *__restrict__ rec = T.rec;
    const int t = threadIdx.x, b0 = block * RB, k = b0 + t;
    const bool node = k < n - 1;
    const int p = node ? ipos[k] : -1; // the root and its children sit in no slot
    const int2 rg = node ? range[k] : make_int2(0, 0);
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (k < n) {
        const int2 lp = n > 1 ? lpos[k] : make_int2(-1, -1);
        const int4 id = leafid[k];
        const int v[3] = {id.y, id.z, id.w};
#pragma unroll
        for (int j = 0; j < K; j++) {
            lo = fmin4(lo, pos_lo(x, v[j]));
            hi = fmax4(hi, pos_hi(x, v[j]));
        }
        leaf_box[2 * k] = lo;
        leaf_box[2 * k + 1] = hi;
        if (lp.x >= 0) put_slot(rec, lp.x, lo, hi, (n - 1) + k, k);
        if (lp.y >= 0) put_slot(rec, lp.y, lo, hi, (n - 1) + k, k);
    }
    auto put = [&](int l) {
        win[l][0][t] = lo.x;
        win[l][1][t] = lo.y;
        win[l][2][t] = lo.z;
        win[l][3][t] = hi.x;
        win[l][4][t] = hi.y;
        win[l][5][t] = hi.z;
    };
    auto get_lo = [&](int l, int a) { return make_float4(win[l][0][a], win[l][1][a], win[l][2][a], 0.f); };
    auto get_hi = [&](int l, int a) { return make_float4(win[l][3][a], win[l][4][a], win[l][5][a], 0.f); };
    put(0);
#pragma unroll
    for (int l = 1; l < RB_LEVELS; l++) {
        __syncthreads();
        const int a = t + (1 << (l - 1)); // a window past the block's end is cut there
        if (a < RB) {
            lo = fmin4(lo, get_lo(l - 1, a));
            hi = fmax4(hi, get_hi(l - 1, a));
        }
        put(l);
    }
    if (t == 0) {
        blk_box[2 * block] = lo;
        blk_box[2 * block + 1] = hi;
    }
    __syncthreads();
    if (p < 0 || rg.x < b0 || rg.y >= b0 + RB) return; // the others: k_cross_boxes
    const int len = rg.y - rg.x + 1, l = 31 - __clz(len), a = rg.x - b0, b = a + len - (1 << l);
    put_slot(rec, p, fmin4(get_lo(l, a), get_lo(l, b)), fmax4(get_hi(l, a), get_hi(l, b)), k, rg.y);
}

__global__ void __launch_bounds__(RB) k_refit(TreeArgs E, TreeArgs F, int e_blocks, const double* __restrict__ x) {
    __shared__ float win[RB_LEVELS][6][RB]; // win[l][.][a]: box of leaves [a, a + 2^l) of the block
    if ((int)blockIdx.x < e_blocks) refit_block<2>(E, blockIdx.x, x, win);
    else refit_block<3>(F, (int)blockIdx.x - e_blocks, x, win);
}

// Boxes of the internal nodes whose range crosses a block boundary of k_refit:
// the leaves of the first and the last block that a node covers in part, and the
// boxes of the blocks between them, all loads independent.  A wave looks at
// `per` nodes and works on its few crossing ones (most have none) with all
// lanes, one after the other: 16 nodes up to CROSS_SMALL leaves, where the
// longest wave is the launch (6.2 us against 8.3 with 64 on 3000 leaves), 64
// above (14 us against 18 on 330,000, 110 against 148 on 2.5 million).  A list of
// the crossing nodes, made once per build, spreads them evenly but costs more
// than it gives: appending to it takes 10-20 ns per wave on one counter (37 us
// of the 256x256 cloth's build, 440 of a batch's).
constexpr int CROSS_SMALL = 1 << 16;
__global__ void __launch_bounds__(BLK) k_cross_boxes(TreeArgs E, TreeArgs F, int e_blocks, int per) {
    const bool edges = (int)blockIdx.x < e_blocks;
    const TreeArgs& T = edges ? E : F;
    const float4 *__restrict__ leaf_box = T.leaf_box, *__restrict__ blk_box = T.blk_box;
    const int lane = threadIdx.x & 63;
    const int i = (edges ? (int)blockIdx.x : (int)blockIdx.x - e_blocks) * (per * (BLK / 64)) + (int)(threadIdx.x >> 6) * per + lane;
    const bool node = lane < per && i < T.n - 1;
    const int2 r = node ? T.range[i] : make_int2(0, 0);
    const int slot = node ? T.ipos[i] : -1; // none for the root and its children
    for (unsigned long long todo = __ballot(slot >= 0 && r.x / RB != r.y / RB); todo; todo &= todo - 1) {
        const int from = __ffsll(todo) - 1, p = __shfl(slot, from, 64), id = i - lane + from;
        const int2 rg = make_int2(__shfl(r.x, from, 64), __shfl(r.y, from, 64));
        const int A = rg.x / RB, B = rg.y / RB;
        float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
        auto take = [&](const float4* arr, int u, int v) { // boxes [u, v): lane u + lane, .. + 64, ..., four in flight
            for (int e = u + lane; e < v; e += 256) {
                float4 l[4], h[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int c = e + 64 * q < v ? e + 64 * q : e; // a repeated box leaves the union unchanged
                    l[q] = arr[2 * c];
                    h[q] = arr[2 * c + 1];
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    lo = fmin4(lo, l[q]);
                    hi = fmax4(hi, h[q]);
                }
            }
        };
        take(leaf_box, rg.x, (A + 1) * RB);
        take(leaf_box, B * RB, rg.y + 1);
        take(blk_box, A + 1, B);
        lo = wave_min4(lo);
        hi = wave_max4(hi);
        if (lane == 0) put_slot(T.rec, p, lo, hi, id, rg.y);
    }
}

// Block b's place in the query order.  Workgroups go round-robin to the 8
// XCDs (block b to XCD b mod 8); the query order is dealt to them in chunks
// of `chunk` consecutive blocks, chunk c to XCD c mod 8, so spatially close
// queries (consecutive in Morton order) share one L2 for the records they
// visit, while the chunks of a dense region still spread over all XCDs.  The
// grid is padded to a multiple of 8 chunks (query_grid), which makes the map a
// permutation of the blocks.
__device__ inline int xcd_block(int b, int chunk) {
    const int j = b >> 3; // the j-th block this XCD receives
    return ((j / chunk) * 8 + (b & 7)) * chunk + j % chunk;
}
// Chunks of up to 2048 queries; fewer where the launch is small, so that every
// XCD gets at least four.
inline int query_chunk(int n, int per_block) { return std::max(1, std::min(2048 / per_block, grid_for(n, per_block) / 32)); }
inline int query_grid(int n, int per_block) {
    const int m = 8 * query_chunk(n, per_block);
    return (grid_for(n, per_block) + m - 1) / m * m;
}
// Queries per wave: a power of two from 4 to 64 that leaves COLLECT_WAVES waves
// where there are enough queries.
constexpr int COLLECT_WAVES = 4096;
inline int collect_qw(int n) {
    int qw = 4;
    while (qw < 64 && n / (2 * qw) >= COLLECT_WAVES) qw *= 2;
    return qw;
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

template <int K>
__global__ void k_leaf_ids(const int32_t* __restrict__ prims, const uint32_t* __restrict__ ids, int n, int4* __restrict__ leafid) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int pid = (int)ids[k];
    leafid[k] = make_int4(pid, prims[K * pid], prims[K * pid + 1], K == 3 ? prims[K * pid + K - 1] : -1);
}

// Record slots (build only): empty slots get their constant, and every node
// that sits in a slot gets the slot's position (ipos for internal nodes;
// lpos.x for a leaf kept by its parent, lpos.y in its grandparent's record),
// each written by exactly one thread.
__global__ void k_record_slots(TopoArgs E, TopoArgs F, int e_blocks) {
    const bool edges = (int)blockIdx.x < e_blocks;
    const TopoArgs& T = edges ? E : F;
    const int n = T.n, i = (edges ? (int)blockIdx.x : (int)blockIdx.x - e_blocks) * (int)blockDim.x + (int)threadIdx.x;
    if (i >= n - 1) return;
    const int32_t* __restrict__ child = T.child;
    float4* __restrict__ rec = T.rec;
    int32_t *__restrict__ ipos = T.ipos, *__restrict__ lpos = T.lpos;
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

// Queries run in two passes.
//
// Collect: a wave takes QW queries and one stack of (query, node) pairs in LDS.
// A step pops up to 16 pairs, four lanes each: every lane tests one child slot
// of its node against its query's box; children that pass go back on the stack
// and leaves to the wave's hit buffer, both packed by ballots.  With one lane
// per query and a stack each (the single pass), a launch takes as long as its
// longest chain of dependent loads (40 visits of 0.9 us on a 16 x 16 cloth, 130
// at the fold of a 256 x 256 one), the lanes that are done idle, and a visit
// reads its 128-byte record in eight 16-byte pieces per lane.  Here a wave's
// lanes are busy until its last query is done, four of them read a record
// together, and a query's nodes are visited many at a time.  Few queries give
// few waves, so QW falls with their number (collect_qw) until a wave has four.
// Hits are filtered 64 at a time by their vertex ids (pairs that share a vertex
// or are both static, most of the hits in a cloth at rest) before they go to
// the query's slab (the first CAND, strided by the query count:
// cand[h * nq + q]) or, past CAND, to a shared overflow list of (query, leaf)
// pairs (capacity nq); ccount[q] counts them.
//
// Test: a block takes TQ queries and spreads their slab entries over its lanes;
// each runs the exact FP64 predicate on its pair, and a lane of the launch also
// tests one overflow entry.  Every kept hit is tested once, so the accepted set
// is that of the single pass (k_single: one lane per query, traversal and test
// together, on a STACK-entry stack), which runs instead when the shared stack
// or the overflow list was too small (bits 0 and 1 of flags[1]).  Then what the
// collect pass finds is of no use, so a wave that meets a limit stops and the
// test pass does nothing: going on costs one atomic on one counter per 64 hits
// (8 sheets of 120 x 120 vertices within the contact distance, 5 million
// contacts: 19.1 ms a detection that way, 9.5 with the stop).
//
// Both kinds in one launch, 256 x 256 cloth: collect 72 us, test 12; by a lane
// per query the two collects took 82 and 46 us. 512 scenes: 1417 and 281 us. On
// a 16 x 16 cloth the collects of the two kinds took 9.4 and 9.0 us in launches
// of their own, by a lane per query 38 and 28.  A batch's collect gains nothing
// (160 scenes 530 + 267 us, by a lane per query 505 + 230): its instructions and
// loads bound it, not its chains.
struct ListOut {
    int32_t* cand;
    uint32_t* ccount;
    int2* ovf;
    uint32_t* ovf_count;
    uint32_t* flags;
};

// The two kinds of query.  Point-triangle: query q is surface vertex q.
// Edge-edge: query k is the edge at sorted leaf k, which reaches only leaves
// after k, so each unordered pair is tested once; a pair (i, j), i < j, is
// evaluated with edge i first, as the canonical definition does.
struct PTQuery {
    const double* x;
    const int32_t* surf_verts;
    const int4* leafid; // of the triangle tree
    const int32_t* vseg;
    const int32_t* roots;
    int nq, nleaf, n_dyn;
    struct Q {
        int v;
        dv3 p;
    };
    __device__ inline Q query(int q) const {
        const int v = surf_verts[q];
        return Q{v, ldd(x, v)};
    }
    // start node: the root, or in segmented mode the vertex's segment subtree
    __device__ inline int start(const Q& Q) const { return nleaf == 0 ? -1 : roots ? roots[vseg[Q.v]] : 0; }
    __device__ inline void box(const Q& Q, float4* lo, float4* hi) const {
        *lo = pos_lo(x, Q.v);
        *hi = pos_hi(x, Q.v);
    }
    __device__ inline int after(int) const { return -1; }
    __device__ inline int2 verts(const Q& Q) const { return make_int2(Q.v, -1); }
    __device__ inline bool keep(int2 v, int lf) const {
        const int4 m = leafid[lf];
        return !(v.x == m.y || v.x == m.z || v.x == m.w || (v.x >= n_dyn && m.y >= n_dyn));
    }
    __device__ inline bool accept(const Q& Q, int lf, double dhat) const {
        const int4 m = leafid[lf];
        return pt_accept(point_triangle(Q.p, ldd(x, m.y), ldd(x, m.z), ldd(x, m.w)), dhat);
    }
    __device__ inline int2 segment(int q, const Q&, int lf) const { return make_int2(q, leafid[lf].x); } // (segment, partner)
    __device__ inline int4 write(const Q& Q, int lf, double dhat, const QueryOut& o, int idx) const {
        const int4 m = leafid[lf], vv = make_int4(Q.v, m.y, m.z, m.w);
        const dv3 t0 = ldd(x, m.y), t1 = ldd(x, m.z), t2 = ldd(x, m.w);
        const PTOut r = point_triangle(Q.p, t0, t1, t2);
        write_contact(o, idx, 0, Q.v, m.x, vv, pt_fields(Q.p, t0, t1, t2, r, dhat), r.dist);
        return vv;
    }
};

struct EEQuery {
    const double* x;
    const int4* leafid; // of the edge tree
    const int32_t* vseg;
    const int32_t* roots;
    int nq, nleaf, n_dyn, seg0; // segments seg0 + edge id
    struct Q {
        int e, a0, a1;
        dv3 A0, A1;
    };
    __device__ inline Q query(int k) const {
        const int4 m = leafid[k];
        return Q{m.x, m.y, m.z, ldd(x, m.y), ldd(x, m.z)};
    }
    // a lone edge, of the tree or of its segment, has no partner (start is a leaf then)
    __device__ inline int start(const Q& Q) const {
        const int s = nleaf < 2 ? -1 : roots ? roots[vseg[Q.a0]] : 0;
        return s >= nleaf - 1 ? -1 : s;
    }
    __device__ inline void box(const Q& Q, float4* lo, float4* hi) const {
        *lo = make_float4(__double2float_rd(fmin(Q.A0.x, Q.A1.x)), __double2float_rd(fmin(Q.A0.y, Q.A1.y)),
                          __double2float_rd(fmin(Q.A0.z, Q.A1.z)), 0.f);
        *hi = make_float4(__double2float_ru(fmax(Q.A0.x, Q.A1.x)), __double2float_ru(fmax(Q.A0.y, Q.A1.y)),
                          __double2float_ru(fmax(Q.A0.z, Q.A1.z)), 0.f);
    }
    __device__ inline int after(int k) const { return k; }
    __device__ inline int2 verts(const Q& Q) const { return make_int2(Q.a0, Q.a1); }
    __device__ inline bool keep(int2 v, int lf) const {
        const int4 m = leafid[lf];
        return !(v.x == m.y || v.x == m.z || v.y == m.y || v.y == m.z || (v.x >= n_dyn && m.y >= n_dyn));
    }
    // the pair's edges in canonical order: i < j
    struct Pair {
        int i, j;
        int4 v;
        dv3 P0, P1, Q0, Q1;
    };
    __device__ inline Pair pair(const Q& Q, int lf) const {
        const int4 m = leafid[lf];
        const dv3 B0 = ldd(x, m.y), B1 = ldd(x, m.z);
        return Q.e < m.x ? Pair{Q.e, m.x, make_int4(Q.a0, Q.a1, m.y, m.z), Q.A0, Q.A1, B0, B1}
                         : Pair{m.x, Q.e, make_int4(m.y, m.z, Q.a0, Q.a1), B0, B1, Q.A0, Q.A1};
    }
    __device__ inline bool accept(const Q& Q, int lf, double dhat) const {
        const Pair p = pair(Q, lf);
        return ee_accept(segment_segment(p.P0, p.P1, p.Q0, p.Q1), dhat);
    }
    __device__ inline int2 segment(int, const Q& Q, int lf) const { // (segment, partner)
        const int f = leafid[lf].x;
        return make_int2(seg0 + min(Q.e, f), max(Q.e, f));
    }
    __device__ inline int4 write(const Q& Q, int lf, double dhat, const QueryOut& o, int idx) const {
        const Pair p = pair(Q, lf);
        const EEOut r = segment_segment(p.P0, p.P1, p.Q0, p.Q1);
        write_contact(o, idx, 1, p.i, p.j, p.v, ee_fields(p.P0, p.P1, p.Q0, p.Q1, r, dhat), r.dist);
        return p.v;
    }
};

// Compiler barrier between LDS accesses of lanes of one wave (the hardware
// keeps a wave's LDS accesses in order).
__device__ inline void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

template <int QW> struct CollectWave {
    uint32_t stack[CSTACK];  // (query of the wave << COLLECT_BITS) | node
    uint32_t hit[128];       // (query << COLLECT_BITS) | sorted leaf
    float4 blo[QW], bhi[QW]; // query boxes grown by gap; w: the query's vertex ids
    int cnt[QW];
};
template <class QK, int QW>
__device__ inline void collect_wave(const QK& K, int block, const float4* __restrict__ rec, float gap, const ListOut& out, CollectWave<QW>& sh) {
    const int lane = threadIdx.x & 63;
    uint32_t* const stack = sh.stack;
    uint32_t* const hit = sh.hit;
    float4 *const blo = sh.blo, *const bhi = sh.bhi;
    int* const cnt = sh.cnt;
    const int q0 = (block * (CBLK / 64) + (int)(threadIdx.x >> 6)) * QW;
    const int leaf0 = K.nleaf - 1;
    auto rank = [&](unsigned long long m) { return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u)); };
    int sp = 0, nh = 0; // entries of stack and hit, the same in all lanes
    bool full = false;  // this wave met a limit (the same in all lanes)
    {
        int start = -1;
        if (lane < QW) {
            cnt[lane] = 0;
            if (q0 + lane < K.nq) {
                const auto Q = K.query(q0 + lane);
                start = K.start(Q);
                float4 lo, hi;
                K.box(Q, &lo, &hi);
                const int2 v = K.verts(Q);
                blo[lane] = make_float4(__double2float_rd((double)lo.x - gap), __double2float_rd((double)lo.y - gap), __double2float_rd((double)lo.z - gap),
                                         __int_as_float(v.x));
                bhi[lane] = make_float4(__double2float_ru((double)hi.x + gap), __double2float_ru((double)hi.y + gap), __double2float_ru((double)hi.z + gap),
                                         __int_as_float(v.y));
            }
        }
        const bool node = start >= 0 && start < leaf0, leaf = start >= 0 && start >= leaf0; // a leaf: a one-leaf tree or segment
        const unsigned long long mn = __ballot(node), ml = __ballot(leaf);
        if (node) stack[rank(mn)] = (uint32_t)lane << COLLECT_BITS | (uint32_t)start;
        if (leaf) hit[rank(ml)] = (uint32_t)lane << COLLECT_BITS | (uint32_t)(start - leaf0);
        sp = __popcll(mn);
        nh = __popcll(ml);
    }
    wave_lds_order();
    // filters the last (up to) 64 buffered hits
    auto flush = [&]() {
        const int k = min(nh, 64);
        bool over = false;
        int q = 0, lf = 0;
        if (lane < k) {
            const uint32_t e = hit[nh - k + lane];
            const int ql = (int)(e >> COLLECT_BITS);
            q = q0 + ql;
            lf = (int)(e & COLLECT_MASK);
            if (K.keep(make_int2(__float_as_int(blo[ql].w), __float_as_int(bhi[ql].w)), lf)) {
                const int pos = atomicAdd(&cnt[ql], 1);
                if (pos < CAND) out.cand[(size_t)pos * K.nq + q] = lf;
                else over = true;
            }
        }
        const unsigned long long mo = __ballot(over);
        if (mo) {
            const int leader = __ffsll(mo) - 1, need = __popcll(mo);
            uint32_t b = 0;
            if (lane == leader) b = atomicAdd(out.ovf_count, (uint32_t)need);
            b = __shfl(b, leader, 64);
            if (b + need > (uint32_t)K.nq) {
                if (lane == leader) atomicOr(&out.flags[1], 2u);
                full = true;
            } else if (over) {
                out.ovf[b + rank(mo)] = make_int2(q, lf);
            }
        }
        nh -= k;
        wave_lds_order();
    };
    while (sp > 0) {
        // a nearly full stack is worked off one node at a time, depth first,
        // which adds at most three entries per tree level
        const int take = sp > CSTACK_HIGH ? 1 : min(16, sp), slot = lane >> 2;
        const bool on = slot < take;
        const uint32_t e = on ? stack[sp - 1 - slot] : 0u;
        const int ql = (int)(e >> COLLECT_BITS);
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        if (on) {
            const float4* r = rec + 8 * (size_t)(e & COLLECT_MASK) + 2 * (lane & 3);
            lo = r[0];
            hi = r[1];
        }
        const float4 ql4 = blo[ql], qh4 = bhi[ql];
        sp -= take;
        const int id = __float_as_int(lo.w);
        // an unused slot has id -1 and last leaf -1
        const bool in = on && __float_as_int(hi.w) > K.after(q0 + ql) && !(lo.x > qh4.x || lo.y > qh4.y || lo.z > qh4.z || ql4.x > hi.x ||
                                                                         ql4.y > hi.y || ql4.z > hi.z);
        const bool leaf = id >= leaf0;
        const unsigned long long mn = __ballot(in && !leaf), ml = __ballot(in && leaf);
        wave_lds_order();
        const uint32_t tag = (uint32_t)ql << COLLECT_BITS;
        if (in && !leaf) {
            const int at = sp + rank(mn);
            if (at < CSTACK) stack[at] = tag | (uint32_t)id;
        }
        if (in && leaf) hit[nh + rank(ml)] = tag | (uint32_t)(id - leaf0);
        sp += __popcll(mn);
        nh += __popcll(ml);
        if (sp > CSTACK) {
            if (lane == 0) atomicOr(&out.flags[1], 1u);
            full = true;
        }
        wave_lds_order();
        if (nh >= 64) flush(); // at most 63 stay, and a step adds at most 64
        if (full) return;
    }
    while (nh > 0 && !full) flush();
    if (lane < QW && q0 + lane < K.nq) out.ccount[q0 + lane] = (uint32_t)cnt[lane];
}

template <int QW>
__global__ void __launch_bounds__(CBLK) k_collect(EEQuery EE, const float4* __restrict__ erec, ListOut el, int e_grid, int e_chunk, PTQuery PT,
                                                  const float4* __restrict__ frec, ListOut pl, int p_chunk, float gap) {
    __shared__ CollectWave<QW> sh[CBLK / 64];
    if ((int)blockIdx.x < e_grid) // a multiple of 8 blocks: the XCD of a block of either part is its index mod 8
        collect_wave<EEQuery, QW>(EE, xcd_block(blockIdx.x, e_chunk), erec, gap, el, sh[threadIdx.x >> 6]);
    else
        collect_wave<PTQuery, QW>(PT, xcd_block((int)blockIdx.x - e_grid, p_chunk), frec, gap, pl, sh[threadIdx.x >> 6]);
}

// Exclusive prefix sums of the slab entries of queries q0 .. q0 + TQ into pre
// (TQ + 1 values); returns their number.
__device__ inline int slab_prefix(const uint32_t* __restrict__ ccount, int q0, int nq, int* pre) {
    const int t = threadIdx.x;
    if (t < TQ) { // one wave
        int s = q0 + t < nq ? (int)min(ccount[q0 + t], (uint32_t)CAND) : 0;
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(s, d, 64);
            if (t >= d) s += y;
        }
        pre[t + 1] = s;
        if (t == 0) pre[0] = 0;
    }
    __syncthreads();
    return pre[TQ];
}
// The query (0 .. TQ - 1) whose entries hold entry i.
__device__ inline int slab_query(const int* pre, int i) {
    int lo = 0;
#pragma unroll
    for (int s = TQ / 2; s > 0; s >>= 1)
        if (pre[lo + s] <= i) lo += s;
    return lo;
}
__device__ inline int ovf_entries(const ListOut& l, int nq) { return (int)min(*l.ovf_count, (uint32_t)nq); }

// Accepted entries keep a mark in the leaf index's sign bit, and their segment
// counts them; nothing is appended to a common list: one counter that every
// wave with a contact adds to costs 10 to 20 ns a wave (the two kinds of test of
// a 160-scene batch 322 and 329 us with it, 68 and 73 without).
constexpr int ACCEPTED = (int)0x80000000;

template <class QK>
__device__ inline void test_block(const QK& K, const ListOut& l, int block, double dhat, uint32_t* __restrict__ qcount, int* pre) {
    const uint32_t limits = l.flags[1];
    const int q0 = block * TQ, total = slab_prefix(l.ccount, q0, K.nq, pre);
    if (limits) return; // counts and entries are incomplete, and the detection reruns
    auto test = [&](int q, int32_t* entry) {
        const auto Q = K.query(q);
        const int lf = *entry;
        if (!K.accept(Q, lf, dhat)) return;
        *entry = lf | ACCEPTED;
        atomicAdd(&qcount[K.segment(q, Q, lf).x], 1u);
    };
    for (int i = threadIdx.x; i < total; i += TBLK) {
        const int s = slab_query(pre, i);
        test(q0 + s, &l.cand[(size_t)(i - pre[s]) * K.nq + q0 + s]);
    }
    const int i = block * TBLK + threadIdx.x; // the launch has at least nq lanes
    if (i < ovf_entries(l, K.nq)) test(l.ovf[i].x, &l.ovf[i].y);
}

__global__ void __launch_bounds__(TBLK) k_test(EEQuery EE, ListOut el, int e_blocks, PTQuery PT, ListOut pl, double dhat,
                                               uint32_t* __restrict__ qcount) {
    __shared__ int pre[TQ + 1];
    if ((int)blockIdx.x < e_blocks) test_block(EE, el, blockIdx.x, dhat, qcount, pre);
    else test_block(PT, pl, (int)blockIdx.x - e_blocks, dhat, qcount, pre);
}

// Canonical order of the accepted pairs: segment by segment (PT by vertex, EE
// by the smaller edge id), sorted by partner id inside a segment.  PASS 0 puts
// the partner ids into their segments (any order inside one).  PASS 1: every
// pair counts the smaller ids of its segment (a pair occurs once, so they are
// distinct), evaluates its contact and writes it to its final place.  The
// counts are independent loads over one lane per contact, where an insertion
// sort by one lane per segment moves each 68-byte record several times in a
// dependent chain (13-30 us per detection for segments of 10 to 30, and 1.2 ms
// for those of 8 sheets of 60 x 60 vertices, whose pairs this places in 0.25).
struct PlaceArgs {
    const uint32_t* qoffset;
    const uint32_t* qcount;
    uint32_t* qfill;
    int32_t* seg_key;
    double dhat;
    QueryOut o;
    VertexCount vc;
};

template <int PASS, class QK>
__device__ inline void place_pair(const QK& K, int q, int lf, const PlaceArgs& a) {
    const auto Q = K.query(q);
    const int2 sp = K.segment(q, Q, lf);
    const int begin = (int)a.qoffset[sp.x];
    if (PASS == 0) {
        a.seg_key[begin + (int)atomicAdd(&a.qfill[sp.x], 1u)] = sp.y;
        return;
    }
    const int cnt = (int)a.qcount[sp.x];
    int rank = 0;
    for (int e = 0; e < cnt; e += 8) {
        int k[8];
#pragma unroll
        for (int u = 0; u < 8; u++) k[u] = a.seg_key[begin + min(e + u, cnt - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++) rank += e + u < cnt && k[u] < sp.y ? 1 : 0;
    }
    const int idx = begin + rank;
    const int4 v = K.write(Q, lf, a.dhat, a.o, idx);
    if (a.vc.cnt) {
        int4 c;
        c.x = (int)atomicAdd(&a.vc.cnt[v.x], 1u);
        c.y = (int)atomicAdd(&a.vc.cnt[v.y], 1u);
        c.z = (int)atomicAdd(&a.vc.cnt[v.z], 1u);
        c.w = (int)atomicAdd(&a.vc.cnt[v.w], 1u);
        a.vc.loc[idx] = c;
    }
}

// The accepted slab entries of TQ queries, gathered in LDS so that full waves
// work on them, and the overflow entries.
template <int PASS, class QK>
__device__ inline void place_block(const QK& K, const ListOut& l, int block, const PlaceArgs& a, int* pre, uint16_t* list, int* count) {
    const int t = threadIdx.x, q0 = block * TQ;
    if (t == 0) *count = 0;
    const int total = slab_prefix(l.ccount, q0, K.nq, pre); // its barrier also covers count
    for (int i = t; i < total; i += TBLK) {
        const int s = slab_query(pre, i), h = i - pre[s];
        if (l.cand[(size_t)h * K.nq + q0 + s] & ACCEPTED) list[atomicAdd(count, 1)] = (uint16_t)(s * CAND + h);
    }
    __syncthreads();
    for (int j = t; j < *count; j += TBLK) {
        const int q = q0 + list[j] / CAND;
        place_pair<PASS>(K, q, l.cand[(size_t)(list[j] % CAND) * K.nq + q] & ~ACCEPTED, a);
    }
    const int i = block * TBLK + t;
    if (i < ovf_entries(l, K.nq) && (l.ovf[i].y & ACCEPTED)) place_pair<PASS>(K, l.ovf[i].x, l.ovf[i].y & ~ACCEPTED, a);
}

template <int PASS>
__global__ void __launch_bounds__(TBLK) k_place(PTQuery PT, ListOut pl, int pt_blocks, EEQuery EE, ListOut el, PlaceArgs a) {
    __shared__ int pre[TQ + 1];
    __shared__ uint16_t list[TQ * CAND];
    __shared__ int count;
    if ((int)blockIdx.x < pt_blocks) place_block<PASS>(PT, pl, blockIdx.x, a, pre, list, &count);
    else place_block<PASS>(EE, el, (int)blockIdx.x - pt_blocks, a, pre, list, &count);
}

// The single pass: accepted pairs to a list of (query, leaf) of capacity cap, EE
// queries with the sign bit set; k_place_single then places them.
template <class QK>
__global__ void __launch_bounds__(QBLK) k_single(QK K, int mark, const float4* __restrict__ rec, float gap, double dhat,
                                                 uint32_t* __restrict__ qcount, int2* __restrict__ pairs, int cap,
                                                 uint32_t* __restrict__ counter, uint32_t* __restrict__ flags) {
    __shared__ int32_t stack[STACK][QBLK];
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= K.nq) return;
    const int leaf0 = K.nleaf - 1;
    const typename QK::Q Q = K.query(q);
    const int start = K.start(Q);
    if (start < 0) return;
    auto leaf = [&](int node) {
        const int lf = node - leaf0;
        if (!K.keep(K.verts(Q), lf) || !K.accept(Q, lf, dhat)) return;
        atomicAdd(&qcount[K.segment(q, Q, lf).x], 1u);
        const int idx = stage_slot(counter);
        if (idx < cap) pairs[idx] = make_int2(q | mark, lf);
    };
    if (start >= leaf0) {
        leaf(start);
    } else {
        float4 lo, hi;
        K.box(Q, &lo, &hi);
        traverse<STACK>(rec, start, leaf0, lo, hi, gap, K.after(q), stack, flags, leaf);
    }
}

template <int PASS>
__global__ void __launch_bounds__(TBLK) k_place_single(PTQuery PT, EEQuery EE, const int2* __restrict__ pairs, int n, PlaceArgs a) {
    const int i = blockIdx.x * TBLK + threadIdx.x;
    if (i >= n) return;
    const int2 e = pairs[i];
    if (e.x & ACCEPTED) place_pair<PASS>(EE, e.x & ~ACCEPTED, e.y, a);
    else place_pair<PASS>(PT, e.x, e.y, a);
}

} // namespace

Detector::Detector(int n_all_, int n_dyn_, int nv_, const int32_t* sv, int nf_, const int32_t* t, int ne_, const int32_t* e,
                   int cap, double dhat_, hipStream_t s)
    : Detector() {
    stream = s;
    n_all = n_all_;
    n_dyn = n_dyn_;
    nv = nv_;
    nf = nf_;
    ne = ne_;
    dhat = dhat_;
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
    auto init_tree = [&](Tree& T, int n) {
        T.n = n;
        if (n == 0) return;
        T.prim_box.alloc(2 * (size_t)n);
        T.leaf_box.alloc(2 * (size_t)n);
        T.leafid.alloc(n);
        T.ipos.alloc(std::max(n - 1, 1));
        T.lpos.alloc(2 * (size_t)n);
        T.keys.alloc(n);
        T.ids.alloc(n);
        T.child.alloc(2 * (size_t)std::max(n - 1, 1));
        T.range.alloc(std::max(n - 1, 1));
        T.rec.alloc(8 * (size_t)std::max(n - 1, 1));
        T.blk_box.alloc(2 * (size_t)grid_for(n, RB));
        T.scene.alloc(2);
        T.partial.alloc(2 * 256);
    };
    init_tree(ft, nf);
    init_tree(et, ne);
    c.cap = cap;
    c.type.alloc(cap);
    c.prim0.alloc(cap);
    c.prim1.alloc(cap);
    c.v.alloc(cap);
    c.bary.alloc(cap);
    c.nrm.alloc(cap);
    c.dist.alloc(cap);
    const size_t segs = ((size_t)nv + ne + 3) & ~(size_t)3;
    counts.alloc(8 + 2 * segs);
    total = counts.p;
    ovf_count = counts.p + 3;
    qcount = counts.p + 8; // 16-byte aligned for the scan
    qfill = qcount + segs;
    qoffset.alloc((size_t)nv + ne + 1);
    PA_HIP(hipHostMalloc((void**)&total_host, 3 * sizeof(uint32_t), hipHostMallocDefault));
    seg_key.alloc(cap);
    single_pairs.alloc(cap); // here, not on the first fallback: an allocation that fails inside a step would cost its rollback
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

// Sorted leaves of one tree: keys, ids and leaf ids.
void Detector::sort_leaves(Tree& T, const double* x, bool faces, hipStream_t stream, PrimScratch& scratch) {
    const int n = T.n;
    if (n == 0) return;
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
    if (faces)
        hipLaunchKernelGGL(k_leaf_ids<3>, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, (const int32_t*)tris.p, (const uint32_t*)T.ids.p, n,
                           T.leafid.p);
    else
        hipLaunchKernelGGL(k_leaf_ids<2>, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, (const int32_t*)edges.p, (const uint32_t*)T.ids.p, n,
                           T.leafid.p);
    PA_LAUNCH_CHECK();
}

// Topology, record slots and segment roots of both trees over their sorted
// leaves; the boxes follow in refit_trees.
void Detector::build_topology() {
    auto args = [](const Tree& T) {
        return TopoArgs{T.n, T.keys.p, T.ids.p, T.child.p, T.range.p, T.ipos.p, T.lpos.p, T.rec.p};
    };
    const TopoArgs E = args(et), F = args(ft);
    const int eb = et.n > 1 ? grid_for(et.n, BLK) : 0, fb = ft.n > 1 ? grid_for(ft.n, BLK) : 0;
    if (eb + fb > 0) {
        hipLaunchKernelGGL(k_karras, dim3(eb + fb), dim3(BLK), 0, stream, E, F, eb);
        PA_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_record_slots, dim3(eb + fb), dim3(BLK), 0, stream, E, F, eb);
        PA_LAUNCH_CHECK();
    }
    if (nseg > 0) {
        segment_roots(et);
        segment_roots(ft);
    }
}

void Detector::segment_roots(Tree& T) {
    const int n = T.n;
    if (n == 0) return;
    fill<int32_t>(T.seg_first.p, -1, nseg, stream);
    fill<int32_t>(T.seg_last.p, -1, nseg, stream);
    fill<int32_t>(T.seg_root.p, -1, nseg, stream);
    hipLaunchKernelGGL(k_seg_bounds, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, (const uint32_t*)T.keys.p, n, T.seg_first.p, T.seg_last.p);
    PA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_seg_roots, dim3(grid_for(n, BLK)), dim3(BLK), 0, stream, n, (const int2*)T.range.p, (const uint32_t*)T.keys.p,
                       (const int32_t*)T.seg_first.p, (const int32_t*)T.seg_last.p, T.seg_root.p);
    PA_LAUNCH_CHECK();
}

// Boxes of both trees from x.
void Detector::refit_trees(const double* x) {
    auto args = [](const Tree& T) {
        return TreeArgs{T.n, T.leafid.p, T.leaf_box.p, (const int2*)T.lpos.p, T.range.p, T.ipos.p, T.blk_box.p, T.rec.p};
    };
    const TreeArgs E = args(et), F = args(ft);
    const int eb = grid_for(et.n, RB), fb = grid_for(ft.n, RB);
    if (eb + fb == 0) return;
    hipLaunchKernelGGL(k_refit, dim3(eb + fb), dim3(RB), 0, stream, E, F, eb, x);
    PA_LAUNCH_CHECK();
    const int per = et.n + ft.n <= CROSS_SMALL ? 16 : 64, block = per * (BLK / 64); // nodes per wave and per block
    const int ec = et.n > RB ? grid_for(et.n, block) : 0, fc = ft.n > RB ? grid_for(ft.n, block) : 0;
    if (ec + fc == 0) return;
    hipLaunchKernelGGL(k_cross_boxes, dim3(ec + fc), dim3(BLK), 0, stream, E, F, ec, per);
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
    // all of it first: if an allocation fails, the detector stays as it was
    DBuf<int32_t> seg(n_all), first[2], last[2], root[2];
    seg.upload(vs, n_all, stream);
    for (int k = 0; k < 2; k++) {
        first[k].alloc(count);
        last[k].alloc(count);
        root[k].alloc(count);
    }
    vseg = std::move(seg);
    Tree* const trees[2] = {&ft, &et};
    for (int k = 0; k < 2; k++) {
        trees[k]->seg_first = std::move(first[k]);
        trees[k]->seg_last = std::move(last[k]);
        trees[k]->seg_root = std::move(root[k]);
    }
    nseg = count;
    built = false; // keys change: the next detection rebuilds
}

int Detector::detect(const double* x, bool refit, VertexCount vc) {
    refit = refit && built;
    fill2<uint32_t>(counts.p, (int64_t)counts.n, vc.cnt, vc.cnt ? vc.n : 0, 0u, stream);
    if (!refit) {
        if (std::max(et.n, ft.n) <= SMALL_BUILD) {
            const SmallTree E{edges.p, 2, et.n, et.keys.p, et.ids.p, et.leafid.p};
            const SmallTree F{tris.p, 3, ft.n, ft.keys.p, ft.ids.p, ft.leafid.p};
            hipLaunchKernelGGL(k_build_small, dim3(2), dim3(SB_BLK), 0, stream, x, nseg > 0 ? (const int32_t*)vseg.p : nullptr, E, F);
            PA_LAUNCH_CHECK();
        } else { // the edge tree is sorted on the side stream beside the triangle tree
            PA_HIP(hipEventRecord(ev_fork, stream));
            PA_HIP(hipStreamWaitEvent(side, ev_fork, 0));
            sort_leaves(et, x, false, side, scratch_side);
            sort_leaves(ft, x, true, stream, scratch);
            PA_HIP(hipEventRecord(ev_join, side));
            PA_HIP(hipStreamWaitEvent(stream, ev_join, 0));
        }
        build_topology();
        built = true;
    }
    refit_trees(x); // a refit keeps the sorted order and the Karras topology
    const float gap = (float)(dhat * 1.001);
    QueryOut o{c.type.p, c.prim0.p, c.prim1.p, c.v.p, c.bary.p, c.nrm.p, c.dist.p, c.cap};
    // A collect pass and a test pass, which marks the accepted pairs and counts
    // them per segment.
    const EEQuery EE{x, et.leafid.p, vseg.p, nseg > 0 ? (const int32_t*)et.seg_root.p : nullptr, ne, ne, n_dyn, nv};
    const PTQuery PT{x, surf_verts.p, ft.leafid.p, vseg.p, nseg > 0 ? (const int32_t*)ft.seg_root.p : nullptr, nv, nf, n_dyn};
    const ListOut el{cand_ee.p, ccount_ee.p, ovf_ee.p, ovf_count + 1, total}, pl{cand_pt.p, ccount_pt.p, ovf_pt.p, ovf_count, total};
    auto single_pass = [&](auto K, int mark, const Tree& T) {
        using QK = decltype(K);
        hipLaunchKernelGGL(k_single<QK>, dim3(grid_for(K.nq, QBLK)), dim3(QBLK), 0, stream, K, mark, (const float4*)T.rec.p, gap, dhat, qcount,
                           single_pairs.p, c.cap, total + 2, total);
        PA_LAUNCH_CHECK();
    };
    const bool two = !force_single_pass && std::max(nf, ne) <= (int)COLLECT_MASK;
    if (two && nv + ne > 0) {
        const int qw = collect_qw(nv + ne), per = qw * (CBLK / 64); // queries per wave and per block
        const int eg = ne > 0 ? query_grid(ne, per) : 0, pg = nv > 0 ? query_grid(nv, per) : 0;
        hipLaunchKernelGGL((qw == 4 ? k_collect<4> : qw == 8 ? k_collect<8> : qw == 16 ? k_collect<16> : qw == 32 ? k_collect<32> : k_collect<64>),
                           dim3(eg + pg), dim3(CBLK), 0, stream, EE, (const float4*)et.rec.p, el, eg, query_chunk(ne, per), PT,
                           (const float4*)ft.rec.p, pl, query_chunk(nv, per), gap);
        PA_LAUNCH_CHECK();
        const int eb = grid_for(ne, TQ);
        hipLaunchKernelGGL(k_test, dim3(eb + grid_for(nv, TQ)), dim3(TBLK), 0, stream, EE, el, eb, PT, pl, dhat, qcount);
        PA_LAUNCH_CHECK();
    }
    uint32_t h[3] = {0u, 0u, 0u};
    auto count_found = [&](uint32_t* o) { // segment offsets; the totals reach the host with the scan's last launch
        scan_exclusive(qcount, qoffset.p, (int64_t)nv + ne, total, scratch, stream, total_host);
        PA_HIP(hipStreamSynchronize(stream));
        for (int k = 0; k < 3; k++) o[k] = total_host[k];
    };
    if (two) {
        count_found(h);
    }
    const bool single = !two || h[1] != 0;
    if (single) {
        // a wave's shared stack or an overflow list was too small: the single pass
        // (traversal and test by one lane per query) for both queries
        fill<uint32_t>(counts.p, 0u, (int64_t)counts.n, stream);
        if (ne > 0) single_pass(EE, ACCEPTED, et);
        if (nv > 0) single_pass(PT, 0, ft);
        count_found(h);
        if (two) single_pass_fallbacks++;
    }
    found_total = h[0];
    stack_overflow = h[1] != 0;
    PA_CHECK(!stack_overflow, PA_ERR_INVALID, "LBVH traversal stack overflow");
    PA_CHECK(!single || h[2] == h[0], PA_ERR_INVALID, "contact list length differs from the segment counts");
    if (found_total > c.cap) {
        n_contacts = 0;
        throw Error(PA_ERR_OVERFLOW, "contact capacity exceeded: found " + std::to_string(found_total) + " > " + std::to_string(c.cap));
    }
    n_contacts = (int)found_total;
    peak = std::max(peak, n_contacts);
    if (n_contacts > 0) {
        const PlaceArgs pa{qoffset.p, qcount, qfill, seg_key.p, dhat, o, vc};
        if (single) {
            const dim3 g(grid_for(n_contacts, TBLK));
            hipLaunchKernelGGL(k_place_single<0>, g, dim3(TBLK), 0, stream, PT, EE, (const int2*)single_pairs.p, n_contacts, pa);
            PA_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_place_single<1>, g, dim3(TBLK), 0, stream, PT, EE, (const int2*)single_pairs.p, n_contacts, pa);
            PA_LAUNCH_CHECK();
        } else {
            const int pt_blocks = grid_for(nv, TQ);
            const dim3 g(pt_blocks + grid_for(ne, TQ));
            hipLaunchKernelGGL(k_place<0>, g, dim3(TBLK), 0, stream, PT, pl, pt_blocks, EE, el, pa);
            PA_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_place<1>, g, dim3(TBLK), 0, stream, PT, pl, pt_blocks, EE, el, pa);
            PA_LAUNCH_CHECK();
        }
    }
    return n_contacts;
}

} // namespace pa
