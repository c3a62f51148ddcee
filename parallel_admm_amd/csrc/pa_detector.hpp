// LBVH proximity detector (replaces BVH_GPU + lbvh_f/lbvh_e,
// src/contact/collision_detection_cuda.*, src/contact/lbvh/lbvh.cu).
#pragma once

#include "pa_common.hpp"
#include "pa_prims.hpp"

namespace pa {

// One Karras radix tree over N primitives: internal nodes [0, N-1),
// leaves [N-1, 2N-1); boxes as (lo, hi) float4 pairs.
struct Tree {
    int n = 0;
    DBuf<float4> prim_box;   // 2 per primitive (lo, hi)
    DBuf<float4> leaf_box;   // 2 per sorted leaf (lo, hi)
    DBuf<int4> leafid;       // per sorted leaf: primitive id and vertex ids
    DBuf<uint32_t> keys, ids; // sorted Morton codes and primitive ids
    DBuf<int32_t> child;     // 2 per internal node
    DBuf<int2> range;        // per internal node: first and last sorted leaf it covers
    DBuf<float4> rec;        // 8 per internal node: boxes, ids and last leaf of its up to four grandchildren
    DBuf<float4> blk_box;    // 2 per block of sorted leaves that the refit takes together
    DBuf<int32_t> ipos;      // per internal node: float4 index of its record slot (-1: none)
    DBuf<int32_t> lpos;      // 2 per leaf: its slot in the parent's record, in the grandparent's (-1: none)
    DBuf<float4> scene;      // 2: scene box
    DBuf<float4> partial;    // 2 per reduction block
    DBuf<int32_t> seg_first, seg_last, seg_root; // per segment: sorted leaf range and subtree root (segmented mode)
};

// Contact list in canonical order (PT by (vertex, face), then EE by (edge i, edge j)).
struct ContactBuffers {
    int cap = 0;
    DBuf<int32_t> type, prim0, prim1;
    DBuf<int4> v;        // vertex ids
    DBuf<float4> bary;   // 4 signed weights
    DBuf<float4> nrm;    // normal xyz, h_cN in w
    DBuf<double> dist;
};

// Per-vertex contact counts wanted by the caller of Detector::detect: cnt[v]
// (n entries, cleared by the detection) counts the contacts of vertex v, and
// loc[c] holds, for each vertex of contact c, its place among them (any order).
struct VertexCount {
    uint32_t* cnt = nullptr;
    int4* loc = nullptr;
    int64_t n = 0;
};

struct Detector {
    hipStream_t stream = nullptr;     // stream work is issued on (the backend's once attached)
    hipStream_t own_stream = nullptr; // created here when none was given; destroyed here
    int n_all = 0, n_dyn = 0, nv = 0, nf = 0, ne = 0;
    double dhat = 0;
    DBuf<int32_t> surf_verts, tris, edges;
    std::vector<int32_t> edges_h; // surface edges (host copy, for the set-up check of edge lengths)
    DBuf<double> x_own; // positions uploaded through detect(host x)
    Tree ft, et;
    ContactBuffers c;   // canonical list
    DBuf<int2> single_pairs; // single pass: accepted (query, leaf) pairs
    DBuf<int32_t> seg_key;  // partner ids in segment order, unsorted inside a segment
    // one buffer, cleared by one launch per detection: total[0] contacts found
    // (segment counts), [1] limit flags, [2] pairs of the single pass;
    // ovf_count[0..1]; qcount: nv + ne segment counts (PT per query vertex, EE
    // per smaller edge id); qfill: partner ids written per segment
    DBuf<uint32_t> counts;
    uint32_t* total = nullptr;
    uint32_t* ovf_count = nullptr;
    uint32_t* qcount = nullptr;
    uint32_t* qfill = nullptr;
    DBuf<uint32_t> qoffset;       // nv + ne segment offsets
    uint32_t* total_host = nullptr; // pinned: total[0..2] after the scan
    // Leaf hits of the collect pass: per query a slab of up to 16 sorted leaf
    // indices (strided by the query count) and the number of hits; hits past
    // the slab as (query, leaf) pairs in an overflow list of one entry per
    // query ([0] PT, [1] EE counts).
    DBuf<int32_t> cand_pt, cand_ee;
    DBuf<uint32_t> ccount_pt, ccount_ee;
    DBuf<int2> ovf_pt, ovf_ee;
    int64_t single_pass_fallbacks = 0; // detections that reran as a single pass (shared stack or overflow list too small)
    bool force_single_pass = false;    // every detection runs the single pass
    PrimScratch scratch;
    // A large edge tree is sorted on a second stream, concurrently with the
    // triangle tree (own sort scratch; joined before the topology).
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    PrimScratch scratch_side;
    // Segmented mode (batched scenes): vertex v belongs to segment vseg[v];
    // pairs are only sought inside a segment.  Keys are (segment << 21 |
    // 21-bit Morton code), so each segment's leaves form one subtree of the
    // Karras tree, and every query starts at its own segment's subtree root.
    int nseg = 0;
    DBuf<int32_t> vseg;
    int n_contacts = 0, peak = 0;
    int64_t found_total = 0; // contacts found by the last detection (may exceed cap)
    bool stack_overflow = false;

    Detector(int n_all, int n_dyn, int nv, const int32_t* sv, int nf, const int32_t* t, int ne, const int32_t* e, int cap,
             double dhat, hipStream_t s);
    ~Detector();
    // Runs detection on device positions x (3 n_all doubles, on this->stream).
    // With refit the trees keep the sorted order and topology of the last
    // build and only their boxes are recomputed from x; the contact list does
    // not depend on the tree, only the traversal's cost does.
    // Returns the number of contacts; the sorted list is complete once the
    // work queued on this->stream has run (the last kernels are queued after
    // the host reads the count).  Sets found_total and throws PA_ERR_OVERFLOW
    // (list unspecified) if more than `cap` contacts were found.
    // With vc, also counts the contacts of every vertex.
    int detect(const double* x, bool refit = false, VertexCount vc = VertexCount());
    // Enables segmented mode: vseg (n_all host ints) in [0, nseg), nseg <= 2048.
    void set_segments(const int32_t* vseg_host, int nseg);
    void set_stream(hipStream_t s) { stream = s; }

  private:
    Detector() = default; // the public constructor delegates: one that fails half-way is destroyed
    void sort_leaves(Tree& T, const double* x, bool faces, hipStream_t s, PrimScratch& scr);
    void build_topology();
    void segment_roots(Tree& T);
    void refit_trees(const double* x);
    bool built = false; // trees built at least once (a refit needs their order and topology)
};

} // namespace pa
