// ADMM backend state on one gfx950 device (replaces ADMMImplGPU,
// src/solver/backend_gpu/admm_impl_gpu.{h,cu}, and the kernels of
// src/solver/{jacobi_solver,contact_solver,compact_sparse_matrix_util}.cu
// and src/constraint/*_device.cu).
#pragma once

#include <memory>
#include <string>
#include <vector>

#include "pa_common.hpp"
#include "pa_detector.hpp"
#include "pa_prims.hpp"
#include "pa_amg.hpp"
#include "pa_mlp.hpp"

namespace pa {

// Contact sets of at most this many contacts run every Jacobi sweep of a
// projection in one workgroup (k_contact_sweeps_wg).
constexpr int CONTACT_WG_MAX = 2048;

struct HostConstraints {
    int n_tri = 0, n_tet = 0, n_bend = 0, n_pin = 0;
    int tri_row0 = 0, tet_row0 = 0, bend_row0 = 0, pin_row0 = 0;
    std::vector<int32_t> tri_inds, tet_inds, bend_ptr, bend_inds, pin_inds;
    std::vector<double> tri_binv, tri_w, tet_binv, tet_w, bend_coef, bend_w, pin_pos, pin_w;
    int rows() const { return 2 * n_tri + 3 * n_tet + n_bend + n_pin; }
};

int batch_variant_index(int threads, int lanes); // -1 if not a variant of the batched solve

struct PhaseTimer {
    bool enabled = false;
    hipEvent_t ev[2] = {nullptr, nullptr};
};

struct Backend {
    int device = 0;
    int verbose = 0;
    hipStream_t stream = nullptr;
    std::string last_error;

    pa_admm_config cfg{};
    bool have_cfg = false;
    HostConstraints hc;
    bool have_constraints = false;
    int m_declared = -1;
    bool finalized = false;
    bool initialized = false;
    bool sync_to_host = true;

    int n_all = 0, n = 0, m = 0;
    std::vector<double> mass_h;
    std::vector<uint8_t> surface_h, pinned_h;
    std::vector<double> x_host, v_host; // host mirror (sync_to_host)

    // state: positions and velocities in FP64 (x, x0, v over n_all); the
    // ADMM variables in FP32 (p over n_all, Ue/z/zprev over m rows, Uc over n)
    DBuf<double> x, x0, v;
    DBuf<float> p, Ue, Uc, z, zprev;
    DBuf<double> b, bconst; // right-hand side in FP64
    DBuf<double> bpin;      // per dynamic vertex: sum over its pins of h^2 w^2 pin position (pin rows are kept relative)
    // per vertex: lumped mass and h^2 w_c in FP64 (they multiply absolute
    // positions in the right-hand side, so they must equal the matrix's
    // FP64 coefficients exactly); w_c and 1/w_c in FP32 for the contact
    // projection (wc* over n_all)
    DBuf<double> mass, wch2;
    DBuf<float> wc, wc_inv;
    DBuf<float> mu_v; // friction coefficient per vertex (n_all)
    DBuf<uint8_t> pinned;
    // constraints
    DBuf<int4> tri_v, tet_v;
    DBuf<float4> tri_binv;
    DBuf<double> pin_pos;  // 3 per pin
    DBuf<double> bend_sum; // per bending row: FP64 sum of its coefficients
    DBuf<float> tet_binv, tri_w, tet_w, bend_w, pin_w, bend_coef;
    DBuf<int32_t> bend_ptr, bend_idx, pin_v;
    // D^T We^2 h^2 gather (per dynamic vertex)
    DBuf<int32_t> dt_ptr, dt_row;
    DBuf<float> dt_coef;
    // system matrix (off-diagonal CSR + diagonal) and damping matrix (full CSR)
    DBuf<int32_t> a_ptr, a_col, dm_ptr, dm_col;
    DBuf<float> a_val, a_diag, a_dinv;
    DBuf<double> dm_val; // damping matrix in FP64: Damp x0 multiplies absolute positions
    DBuf<float> a_val_lo, a_diag_lo; // A = hi + lo to ~2^-48 for the FP64 residual
    int64_t nnz_a_off = 0, nnz_dm = 0;
    // PCG
    DBuf<float> cg_r, cg_z, cg_p, cg_q, cg_d;
    DBuf<float> cg_r2, cg_p2; // ping-pong partners of cg_r and cg_p for the fused AMG iteration
    DBuf<double> cg_part;  // per block partial sums
    DBuf<double> cg_state; // two slots of (rz[3], done[3]); [16..18] threshold, [19] iterations, [20..22] |b|^2
    int cg_blocks = 0;     // grid of every kernel that writes cg_part (grid-stride over rows)
    int a_lpr = 2;         // lanes per row for SpMVs with A
    int rhs_lpr = 2;       // lanes per vertex for the D^T gather of the right-hand side
    int last_pcg_iters = 0; // iterations of the previous solve's first pass (sizes the first launch chunk)
    // AMG preconditioner (device copy of the hierarchy built at init)
    struct DevLevel {
        int n = 0, nnext = 0;
        float omega = 0.f; // weight of the V-cycle's Jacobi sweeps (AmgLevel::omega_smooth)
        int lpr_a = 2, lpr_p = 2, lpr_r = 2; // lanes per row for A, P and R
        DBuf<int32_t> aptr, acol, pptr, pcol, rptr, rcol;
        DBuf<float> aval, dinv, pval, rval;
        DBuf<float> b, x, x2, r; // 3 n each
    };
    std::vector<std::unique_ptr<DevLevel>> amg;
    DBuf<float> amg_cinv;
    int amg_nc = 0, amg_ncp = 0; // coarsest size and its row stride (multiple of 4)
    bool use_amg = false;
    std::vector<int> amg_sizes;
    // direct global solve (precond 2): the supernodal Cholesky factor built at
    // init (pa_chol.hpp), FP32 copies in the layouts the level kernels read
    bool use_chol = false;
    int chol_levels = 0;                  // levels below the dense tops
    // per level: ranges in the tile arrays, lanes along rows (up) or per column
    // (down), LDS bytes
    std::vector<int32_t> chol_up_ptr, chol_down_ptr;
    std::vector<int> chol_rg, chol_lp, chol_up_lds, chol_down_lds;
    DBuf<uint8_t> chol_up_tiles, chol_down_tiles; // CholTile descriptors (pa_solver.hip)
    DBuf<float> chol_panels;              // [D; -W] per supernode, column-major
    DBuf<int32_t> chol_gat_rows;          // per front row: the children's update-vector entries added there
    DBuf<int32_t> chol_ipos, chol_below;  // place of each unknown in elimination order; rows below of each supernode
    int chol_top_tiles = 0, chol_top_lds = 0, chol_top_nv = 1;
    DBuf<int32_t> chol_top_pos;
    DBuf<int64_t> chol_top_ptr, chol_gat, chol_sinv_off;
    int chol_gmax = 1;                    // width of the dense tops' gather table chol_gat (entries -1: none)
    DBuf<int2> chol_tiles;                // (top block, first row) of each workgroup of the dense-top launch
    DBuf<float> chol_sinv;                // dense tops: S^-1, row-major, rows padded to whole float4s
    DBuf<float> chol_f, chol_x, chol_u;   // fronts' column right-hand sides and solution (elimination order), update vectors
    DBuf<float> chol_ftop;                // right-hand side of every dense-top entry (3 per entry)
    int64_t chol_entries = 0;             // stored factor entries (panels, S^-1)
    int64_t chol_top_cols = 0, chol_top_sq = 0; // dense tops: sum of m and of m^2
    double chol_setup_ms = 0;
    void chol_setup(const std::vector<int32_t>& aptr, const std::vector<int32_t>& acol, const std::vector<double>& aval,
                    const double* x0h);
    void chol_solve(const float* r); // chol_x = A^-1 r
    void chol_top_launch(const float* r);
    // scripted animation of static vertex ranges (ScriptAnimator rigid and
    // point-sequence scripts)
    struct RigidTrack {
        int first = 0, count = 0, fps = 1, cur = 0, frames = 0;
        bool points = false;             // a point sequence (pts) instead of a rigid motion (trans, quat)
        std::vector<double> trans, quat; // 3 and 4 (w, x, y, z) per frame
        DBuf<double> rest, prev;         // 3 count each: rest positions, last placed positions
        DBuf<double> pts;                // point sequence: frames x count x 3 positions
    };
    std::vector<std::unique_ptr<RigidTrack>> tracks;
    std::vector<double> x_init_h; // positions given to init (rest positions of the tracks)
    // contacts
    Detector* det = nullptr;
    std::unique_ptr<Detector> own_det;
    int nc = 0;
    DBuf<float4> gam, kc, rc;
    DBuf<int32_t> cslot;  // per contact: entry slot of each of its 4 vertices (-1: static)
    DBuf<float4> gdu;     // per vertex entry: Gamma_k du of the last sweep
    DBuf<uint32_t> vcnt, vptr, vent; // contacts per vertex; entries per dynamic vertex (offsets, sorted entries 4 c + k)
    DBuf<int4> vloc;                 // per contact: its place among each vertex's contacts, any order
    DBuf<uint32_t> vraw;             // entries in their runs, unsorted
    DBuf<int2> erun;      // per vertex entry: (vertex, end of its entries) on its first entry, else (-1, 0)
    int contact_wg_max = CONTACT_WG_MAX; // contact sets up to this size sweep in one workgroup
    PrimScratch scratch;
    // warm start of the contact duals at each detection (pa_warm_start)
    pa_warm_start ws{};             // params pointer cleared; weights live in ws_mlp
    std::unique_ptr<Mlp> ws_mlp;
    bool ws_active = false;         // seeding in the current attempt of the step
    bool ws_restart = false;        // the seeded-window check or the stall check abandoned the attempt
    int ws_bad = 0;                 // consecutive windows judged worse than a zero seed
    int ws_nc = 0;                  // contacts of the current window
    bool ws_window = false;         // the current window has features (and maybe seeds)
    bool ws_window_seeded = false;
    bool ws_judged = false;         // the current window's seeds were judged
    int ws_seeded_count = 0;
    int ws_bad_windows = 0;         // windows judged bad during the step (all attempts)
    DBuf<float> ws_feat, ws_norm;   // 10 raw / normalised features per contact
    DBuf<float4> ws_tan, ws_seed;   // tangent of the feature frame; seeded dual
    DBuf<int32_t> ws_match;         // index of the same contact in the previous window, or -1
    DBuf<int32_t> prev_type, prev_p0, prev_p1;
    DBuf<float4> prev_rc;
    int nc_prev = 0;
    DBuf<double> ws_err;            // judge partial sums
    DBuf<float> ws_consts;          // in_shift[10], in_scale[10], out_scale[2]
    DBuf<double> snap_x, snap_v, good_x, good_v;  // step-start state for a cold re-run; last good state
    DBuf<float> snap_ue, snap_uc, good_ue, good_uc; // (init, reset, every finite step)
    std::vector<int32_t> good_track_frames;        // the tracks' frame counters with the last good state
    DBuf<uint32_t> bad_flag;
    bool state_dirty = false; // set_state / set_duals / set_static_state since the last step
    bool state_nonfinite();
    void save_good_state();
    void restore_good_state();
    int64_t log_cap = 0, log_rows = 0;
    DBuf<float> log_buf;
    bool seed_log = false;
    std::vector<std::vector<float>> seed_log_h;
    // batched scenes (a merged, block-diagonal scene): the global solve runs
    // as one persistent launch with a workgroup per scene (pa_batch.hip)
    int nscene = 0; // 0: one scene
    std::vector<int32_t> scene_dyn_off, scene_stat_off;
    DBuf<int32_t> scene_off, scene_order;    // dynamic row ranges; launch order (largest first)
    DBuf<int32_t> scene_iters;               // PCG iterations per scene (to its own tolerance), summed over the step
    DBuf<unsigned long long> scene_ticks;    // wall-clock ticks per scene in the solve, summed over the step
    int wall_khz = 100000;
    int tune_variant = -1;                   // chosen (threads, lanes per row) variant; -1: tune at the next solve
    std::vector<double> tune_ms;             // the autotuner's timing of every variant (ms)
    DBuf<double> tune_x;
    DBuf<double> scene_r0;                   // AMG-PCG on a batch: per-scene |r0|^2 (3 per scene)
    DBuf<uint32_t> scene_open;               // scenes not yet at tolerance
    DBuf<int32_t> scene_first;               // iteration at which each scene met its tolerance in this pass
    void setup_batch(const std::vector<int32_t>& dyn_off, const std::vector<int32_t>& stat_off);
    void set_batch_tuning(int threads, int lanes);
    int batch_solve(int max_iter, double tol);
    void batch_stats(int32_t* iters, double* ms);
    // residual partial sums; (r_primal, r_dual) of every check of the last step
    DBuf<double> res_part, res_sum;
    std::vector<double> res_log;
    // Device stop test (direct solve, no learned warm start): k_resid_final
    // sets stop_ctl[0] when an iteration meets residual_tol, and the state
    // writers of later iterations read it through stop_guard (null: no
    // test).  Each check is copied into a pinned slot (chk_host, two of 8
    // doubles) marked by an event, so the host reads it one iteration late
    // without draining the queue.
    DBuf<int32_t> stop_ctl;
    const int32_t* stop_guard = nullptr;
    double* chk_host = nullptr;
    hipEvent_t ev_chk[2] = {nullptr, nullptr};
    int res_blocks = 0;
    // timing
    int profiling = 0; // bit 0: PCG SpMV launch events, bit 1: phase events
    double phase_ms[6] = {0, 0, 0, 0, 0, 0};
    std::vector<hipEvent_t> ev_pool;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev_marks;
    size_t ev_next = 0;
    double spmv_ms_sum = 0;
    int64_t spmv_launches = 0;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> spmv_marks;

    Backend() = default; // no device work; the constructor below delegates: one that fails half-way is destroyed
    explicit Backend(const pa_device_opts* o);
    ~Backend();

    void apply_config(const pa_admm_config& c);
    void set_constraints(const pa_constraint_soa& c);
    void set_constraint_dim(int m_rows) { m_declared = m_rows; }
    void finalize_constraints();
    void init(const double* x0, const double* mass, int n_all, int n_dyn, const uint8_t* surface, int n_pins, const int32_t* pins);
    void attach_detector(Detector* d);
    void detach_detector(const Detector* d); // the detector is going away: forget it (no-op if another is attached)
    void step(pa_step_stats* st);
    void step_impl(pa_step_stats* st);
    void reset(const double* x0);
    void get_state(double* x, double* v);
    void set_state(const double* x, const double* v);
    void get_duals(double* ue, double* uc);
    void set_duals(const double* ue, const double* uc);
    void set_static_state(const double* xs, const double* vs);
    void set_vertex_mu(const double* mu);

    // sub-phases (also used by step)
    void local_step();
    void contact_setup(float eps, float gamma, float hinv, bool counted = false);
    void contact_project(bool first_iter);
    void contact_sweep_once();
    void rhs(bool want_residual, bool first_iter);
    double spmv_time_ms(int reps);
    // Rigid track for static vertices [first, first + count): frame k places
    // them at trans_k + R(q_k) rest; see pa_backend_add_rigid_track.
    void add_rigid_track(int first, int count, int frames, const double* pos, const double* quat_xyzw, int fps);
    void add_point_track(int first, int count, int frames, const double* points, int fps);
    void animate_tracks(bool place_first_frame);
    void get_track_frames(int32_t* frames) const;
    void set_track_frames(const int32_t* frames, int count);
    // defer_last (direct solve): the last pass leaves x += d to the next
    // dual update (dx_pending), which applies it before reading x.
    // resid_ready (direct solve): cg_r holds b - A x already (left by rhs)
    int global_solve(int max_iter, double tol, bool defer_last = false, bool resid_ready = false);
    bool dx_pending = false;
    void pcg_iteration(int it, bool fused, int& pc, int& rc);
    hipGraphExec_t pcg_pair_graph(bool first_pair);
    hipGraphExec_t pcg_graph[2] = {nullptr, nullptr}; // [0] later pairs, [1] the first pair of a solve
    bool capturing = false;                           // inside a stream capture: no event records
    bool use_graphs = true;
    // cg_z = M^-1 r, partial r.z into cg_part[*, 6..8]; with skip_pre0 the
    // level-0 pre-smoothing was already done by k_cg_update_pre.
    void precondition(const float* r, bool skip_pre0 = false);
    void dual_vertices(bool want_residual);
    void elem_update(bool want_residual, bool last, bool next_check);
    void residual_read(double* rp, double* rd);
    void residual_enqueue(int it);
    int3 resid_blocks();
    void read_check(int it, double* rp, double* rd);
    // warm start: configuration, window end (judge, log, keep the duals for
    // matching) and window start (features, seeds); see pa_warm_start
    void set_warm_start(const pa_warm_start& w);
    void ws_judge();
    void ws_window_end();
    void ws_window_begin();
    void ws_forget() {
        ws_window = false;
        nc_prev = 0;
    }
    int admm_loop(pa_step_stats& S, float eps, float gam, float hinv);

  private:
    void assemble_and_upload(const double* x0);
    hipEvent_t next_event();
    void mark_begin(int phase, hipEvent_t* e0);
    void mark_end(int phase, hipEvent_t e0);
    void collect_phase_times();
};

} // namespace pa
