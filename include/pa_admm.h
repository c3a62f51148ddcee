/*
 * pa_admm.h - C ABI of the MI355X (gfx950) ADMM frictional-contact backend.
 *
 * A drop-in for the GPU path of OkifuZ/parallel_admm:
 *   pa_backend_*   replaces ADMMBackendGPU behind ADU::IADMMBackend
 *                  (src/solver/core/admm_backend.h:15-41; implementation
 *                  src/solver/backend_gpu/admm_impl_gpu.cu)
 *   pa_detector_*  replaces BVH_GPU behind ADU::ICollisionDetector
 *                  (src/contact/icollision_detector.h:19-47,
 *                  src/contact/collision_detection_cuda.h:45-105)
 *   pa_scene_*     host-side setup that the reference does in MeshData +
 *                  Mesh2Constraint + the constraint constructors
 *                  (src/mesh/mesh_container.h:232-472,
 *                  src/constraint/mesh_to_constraint.h:29-153)
 *
 * Conventions: plain pointers and sizes only; every call returns pa_status
 * (0 = success) and never exits the process (the reference prints and calls
 * exit(), src/mutils/cuda_tools.cuh:37-46).  Positions are xyz-interleaved
 * row-major (n x 3), y-up, gravity along -y, as in the reference.  Host
 * buffers belong to the caller and are copied in or out; device memory
 * belongs to the handle.  One handle is used from one host thread at a time;
 * distinct handles are independent (the reference allows one backend per
 * process because of function-local statics, admm_impl_gpu.cu:69-82).
 */
#ifndef PA_ADMM_H
#define PA_ADMM_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef int32_t pa_status;
enum {
    PA_OK = 0,
    PA_ERR_INVALID = 1,   /* bad argument or call order */
    PA_ERR_HIP = 2,       /* HIP runtime error */
    PA_ERR_NO_DEVICE = 3, /* no GPU visible */
    PA_ERR_OVERFLOW = 4,  /* contact capacity exceeded (contacts were not truncated silently) */
    PA_ERR_NOT_SPD = 5,   /* system matrix not positive definite */
    PA_ERR_GEOMETRY = 6,  /* degenerate or inverted rest geometry */
    PA_ERR_NUMERICAL = 7  /* a step produced non-finite positions or velocities; the state was rolled back
                             to the end of the last good step (or init / reset) */
};

/* ---------------------------------------------------------------------------
 * Solver configuration.  Mirrors ADU::ADMMSolverConfig
 * (src/solver/core/admm_config.h:13-55) and the scene keys that feed it
 * (src/solver/solver_config_applier.cpp:5-53), plus the convergence controls
 * this backend adds (the reference computes no residual).
 * ------------------------------------------------------------------------- */
typedef struct pa_admm_config {
    double dt;              /* time step h */
    double g;               /* gravity magnitude along -y */
    int32_t admm_max_iter;  /* admm_max_iter */
    int32_t dcd_interval;   /* DCD_interval: detection every k ADMM iterations */
    int32_t gs_max_iter;    /* GS_max_iter: contact projection sweeps per iteration */
    int32_t warmstart_ue;   /* admm.warmstart_Ue */
    int32_t warmstart_uc;   /* admm.warmstart_Uc */
    int32_t enable_contact; /* contact.enable */
    double mu;              /* contact.mu */
    double kappa;           /* contact.kappa */
    double beta;            /* contact.beta */
    double thickness;       /* narrow.thickness (d-hat) */
    double damp_kl;         /* damp.kl */
    double damp_km;         /* damp.km */
    double w_scale;         /* contact.w_scale: w_c = m / h^2 * w_scale */
    double residual_tol;    /* stop when max(r_primal, r_dual) <= tol; 0 = run admm_max_iter */
    int32_t residual_interval; /* check the residual every k iterations */
    int32_t global_max_iter;   /* cap on PCG iterations per refinement pass (Global_Jacobi_iter) */
    double global_tol;         /* PCG stop per pass and column: |r_k| <= global_tol |r_0|, r_0 = b - A x in FP64; default 5e-4 */
    int32_t max_contacts;      /* narrow.max_collision: contact capacity */
    int32_t global_refine;     /* refinement passes per global solve (FP64 residual, FP32 correction) */
    int32_t precond;           /* global solve: PCG with 0 Jacobi or 1 smoothed-aggregation AMG V-cycle
                                * preconditioner; 2 direct (supernodal Cholesky factored once at init,
                                * level-scheduled FP32 triangular solves, global_refine passes) */
    int32_t graphs;            /* 1: replay PCG iteration pairs as HIP graphs; 0: launch every kernel (default) */
    /* contact.use_heu_wc / wc_sigma / wc_beta (solver_config_applier.cpp:38-42):
     * heuristic contact weights of the GPU precompute (admm_impl_gpu.cu:205-218),
     * w_c,i = max(sigma a_ii, min(beta m_i, a_ii)) * 10 / h^2 with a_ii the
     * diagonal of M + h^2 D^T We^2 D + Damp, instead of m_i / h^2 * w_scale */
    int32_t use_heu_wc;
    double wc_sigma;           /* default 0.001 */
    double wc_beta;            /* default 25 */
} pa_admm_config;

/* Fills the reference's ADMMSolverConfig defaults (admm_config.h:20-53). */
void pa_admm_config_default(pa_admm_config* cfg);

/* ---------------------------------------------------------------------------
 * Scene: mesh + topology + elastic constraints + lumped mass.
 * Vertex order: dynamic vertices [0, n_dyn) then static obstacle vertices
 * [n_dyn, n_all) (static_vert_begin, src/config/mesh_from_config.h:63-82).
 * Constraint rows: triangles (2 rows), tets (3), bending (1), pins (1), in
 * that order (mesh_to_constraint.h + app_initializer.cpp:145-172).
 * ------------------------------------------------------------------------- */
typedef struct pa_scene pa_scene;

typedef struct pa_mesh_desc {
    int32_t n_all, n_dyn;
    const double* x;           /* 3 n_all */
    const double* density;     /* n_all (static vertices: 1e12) */
    int32_t n_tri;
    const int32_t* tris;       /* 3 n_tri: dynamic cloth faces first, then static faces */
    const double* tri_k;       /* n_tri stretch stiffness (ignored for static faces) */
    const double* bend_k;      /* n_all bending stiffness per vertex */
    int32_t n_tet;
    const int32_t* tets;       /* 4 n_tet */
    const double* tet_k;       /* n_tet */
    int32_t n_tet_boundary;
    const int32_t* tet_boundary; /* 3 n_tet_boundary: surface facets of the tet meshes */
    int32_t n_pins;
    const int32_t* pins;
} pa_mesh_desc;

/* Build topology, constraints and lumped mass from a raw mesh
 * (MeshData::precompute_geometry_info + Mesh2Constraint + get_mass). */
pa_status pa_scene_create(const pa_mesh_desc* mesh, pa_scene** out);

/* Generators for the benchmark scenes (parameters in the implementation):
 *   kind 1: 32x32 cloth (1 cm) over a level-3 icosphere (r 0.2 m), two pinned corners
 *   kind 2: 20x20x20-cell 5-tet box (0.2 m) with a seeded random rotation over a ground quad
 *   kind 3: 256x256 cloth (2 mm) over a sphere (r 0.15 m) and a cylinder (r 0.05 m)
 *   kind 4: one cloth of side `side` (16..96) over a sphere of radius `radius` at drop height `drop`
 * `side`, `seed`, `radius` and `drop` are used where the kind needs them (0 = default). */
pa_status pa_scene_generate(int32_t kind, int32_t side, uint64_t seed, double radius, double drop, pa_scene** out);
void pa_scene_destroy(pa_scene* s);

typedef struct pa_scene_info {
    int32_t n_all, n_dyn, m_rows;
    int32_t n_tri, n_tet, n_tet_boundary, n_pins;
    int32_t n_tri_c, n_tet_c, n_bend_c, n_pin_c; /* constraints per type */
    int32_t n_surf_verts, n_surf_tris, n_surf_edges;
    int64_t nnz_d, bend_entries;
} pa_scene_info;
pa_status pa_scene_get_info(const pa_scene* s, pa_scene_info* out);

/* Copies of the raw mesh (arrays sized as in pa_scene_info; NULL skips). */
pa_status pa_scene_get_mesh(const pa_scene* s, double* x, double* density, int32_t* tris, double* tri_k, double* bend_k,
                            int32_t* tets, double* tet_k, int32_t* tet_boundary, int32_t* pins);
/* Surface topology: sorted surface vertices, surface triangles, surface edges (min,max). */
pa_status pa_scene_get_topology(const pa_scene* s, int32_t* surf_verts, int32_t* surf_tris, int32_t* surf_edges);
pa_status pa_scene_get_mass(const pa_scene* s, double* mass);

/* Flattened constraints (≙ the Constraint objects passed to add_constraints,
 * solver.h:96; tri/tet Binv row-major, bending ring + coefficients). */
typedef struct pa_constraint_soa {
    int32_t n_tri, n_tet, n_bend, n_pin;
    int32_t tri_row0, tet_row0, bend_row0, pin_row0; /* first row of each block; rows contiguous within a type */
    const int32_t* tri_inds;  /* 3 n_tri */
    const double* tri_binv;   /* 4 n_tri */
    const double* tri_w;      /* n_tri */
    const int32_t* tet_inds;  /* 4 n_tet */
    const double* tet_binv;   /* 9 n_tet */
    const double* tet_w;      /* n_tet */
    const int32_t* bend_ptr;  /* n_bend + 1 */
    const int32_t* bend_inds; /* middle vertex then ring, bend_ptr[n_bend] entries */
    const double* bend_coef;  /* one per bend_inds entry */
    const double* bend_w;     /* n_bend */
    const int32_t* pin_inds;  /* n_pin */
    const double* pin_pos;    /* 3 n_pin */
    const double* pin_w;      /* n_pin */
} pa_constraint_soa;

/* Writable views into the scene's own constraint arrays (valid while the scene lives). */
pa_status pa_scene_get_constraints(const pa_scene* s, pa_constraint_soa* out);

/* ---------------------------------------------------------------------------
 * Collision detector (≙ ICollisionDetector / BVH_GPU): LBVH over the surface
 * triangles and edges, canonical sorted contact list.
 * ------------------------------------------------------------------------- */
typedef struct pa_detector pa_detector;

typedef struct pa_surface {
    int32_t n_all, n_dyn;
    int32_t n_surf_verts, n_surf_tris, n_surf_edges;
    const int32_t* surf_verts; /* sorted */
    const int32_t* surf_tris;  /* 3 n_surf_tris */
    const int32_t* surf_edges; /* 2 n_surf_edges, (min, max) */
} pa_surface;

/* ≙ BVH_GPU::init(max_collision) (collision_detection_cuda.cpp:39-83). */
pa_status pa_detector_create(const pa_surface* surf, int32_t capacity, double thickness, pa_detector** out);
void pa_detector_destroy(pa_detector* d);
/* ≙ ICollisionDetector::detect(pos): positions from the host (3 n_all doubles,
 * rounded to FP32 on upload). */
pa_status pa_detector_detect(pa_detector* d, const double* x_host, int32_t* n_contacts);
/* Canonical contact list of the last detection: ints = 7 per contact
 * (type 0=PT/1=EE, prim0, prim1, v0..v3); reals = 9 per contact (bary[4],
 * normal[3], h_cN, distance).  Order: PT by (vertex, face), then EE by
 * (edge i, edge j), i < j. */
pa_status pa_detector_get_contacts(pa_detector* d, int32_t* ints, double* reals, int32_t cap, int32_t* n_contacts);
/* contact_count / max_slots / peak_contact_count (icollision_detector.h:30-36). */
pa_status pa_detector_counts(const pa_detector* d, int32_t* count, int32_t* max_slots, int32_t* peak);
/* points() / normals() (icollision_detector.h:38-44): exactly max_slots
 * entries each, unused slots zero-filled. */
pa_status pa_detector_points(pa_detector* d, float* points3);
pa_status pa_detector_normals(pa_detector* d, float* normals3);
/* clear() */
pa_status pa_detector_clear(pa_detector* d);

/* ---------------------------------------------------------------------------
 * Backend (≙ IADMMBackend + the Solver::init/reset/getVertices entry points
 * reached through as_solver(), core/admm_solver.cpp:5-17, solver.h:66-137).
 * Call order (app_initializer.cpp:109-224): create -> apply_config ->
 * set_constraints -> set_constraint_dim -> finalize_constraints -> init ->
 * set_sync_to_host -> attach_detector; then step() per sub-step.
 * ------------------------------------------------------------------------- */
typedef struct pa_backend pa_backend;

typedef struct pa_device_opts {
    int32_t device;  /* HIP device ordinal */
    int32_t verbose; /* 0: silent */
} pa_device_opts;

typedef struct pa_step_stats {
    int32_t iterations;    /* ADMM iterations run */
    int32_t n_contacts;    /* contacts of the last detection */
    int32_t converged;     /* residual reached residual_tol */
    int32_t overflow;      /* contact capacity exceeded */
    int32_t global_iters;  /* PCG iterations summed over the step */
    int32_t detections;
    double r_primal, r_dual; /* last residual check */
    double step_ms;          /* host wall time of the step */
    int32_t ws_seeded;       /* detections whose contact duals were warm-started (kept attempt) */
    int32_t ws_fallback;     /* 1: the warm-started attempt was abandoned and the step re-run cold */
    int32_t ws_wasted_iters; /* ADMM iterations of the abandoned attempt */
    int32_t ws_bad_windows;  /* seeded windows judged bad (see pa_warm_start.patience) */
    int32_t n_contacts_max;  /* most contacts of any detection of the step */
    int32_t reserved;
} pa_step_stats;

pa_status pa_backend_create(const pa_device_opts* opts, pa_backend** out);
void pa_backend_destroy(pa_backend* b);
const char* pa_backend_last_error(const pa_backend* b);

/* ≙ IADMMBackend::apply_config (before init). */
pa_status pa_backend_apply_config(pa_backend* b, const pa_admm_config* cfg);
/* ≙ Solver::add_constraints + addPins: constraint data (copied). */
pa_status pa_backend_set_constraints(pa_backend* b, const pa_constraint_soa* c);
/* ≙ IADMMBackend::set_constraint_dim(m_nCDim). */
pa_status pa_backend_set_constraint_dim(pa_backend* b, int32_t m_rows);
/* ≙ IADMMBackend::finalize_constraints: checks rows, packs device SoA. */
pa_status pa_backend_finalize_constraints(pa_backend* b);
/* ≙ Solver::init(verts, mass, dt) + ADMMImplGPU::init/precompute: assembles
 * M, D, We, Damp, Wc and A, uploads them and the state.  surface_flags marks
 * surface vertices (vinds_surf_set), pins lists the pinned vertices. */
pa_status pa_backend_init(pa_backend* b, const double* x0, const double* mass, int32_t n_all, int32_t n_dyn,
                          const uint8_t* surface_flags, int32_t n_pins, const int32_t* pins);
/* ≙ set_sync_to_host: copy x, v back to host after each step. */
pa_status pa_backend_set_sync_to_host(pa_backend* b, int32_t enabled);
/* ≙ Solver::bvh pointer: the detector runs on the backend's device positions
 * and stream.  The detector must outlive the backend's use of it. */
pa_status pa_backend_attach_detector(pa_backend* b, pa_detector* d);
/* ≙ IADMMBackend::step. */
pa_status pa_backend_step(pa_backend* b, pa_step_stats* out);
/* ≙ Solver::reset(ini_verts): state <- x0, v <- 0, duals <- 0. */
pa_status pa_backend_reset(pa_backend* b, const double* x0);
/* ≙ getVertices / getVelocities (explicit copy-out, 3 n_all each; NULL skips). */
pa_status pa_backend_get_state(pa_backend* b, double* x, double* v);
pa_status pa_backend_set_state(pa_backend* b, const double* x, const double* v);
/* Dual variables Ue (3 m) and Uc (3 n_dyn). */
pa_status pa_backend_get_duals(pa_backend* b, double* ue, double* uc);
pa_status pa_backend_set_duals(pa_backend* b, const double* ue, const double* uc);
/* Static obstacle motion for the next step (≙ ScriptAnimator::animate_all,
 * src/solver/animator.cpp:199-205): positions and velocities of [n_dyn, n_all). */
pa_status pa_backend_set_static_state(pa_backend* b, const double* x_static, const double* v_static);
/* Friction coefficient per vertex (n_all values, finite and >= 0; default
 * pa_admm_config.mu everywhere).  A contact takes the coefficient of its
 * first vertex: the query vertex of a point-triangle pair, the first endpoint
 * of edge i of an edge-edge pair (i < j).  The reference holds one scalar mu
 * (ADMMSolverConfig::mu, admm_config.h:35; get_delta_u_kernel,
 * contact_solver.cu:337); per-vertex values let a merged batch of scenes give
 * each scene its own friction, every vertex of a scene carrying that scene's. */
pa_status pa_backend_set_vertex_mu(pa_backend* b, const double* mu, int32_t n_all);

/* Rigid track for the static vertices [first, first + count) (≙ a rigid
 * ScriptAnimator script attached to a static mesh, src/solver/animator.cpp:9-39,
 * 83-130): frame k places them at pos[k] + q[k] (x) rest, rest = the positions
 * given to pa_backend_init, q[k] = quat_xyzw[4k..4k+3] in the npz order
 * (x, y, z, w) (normalised).  Registration places frame 0 with zero velocity;
 * each step first advances the frame counter by frames_per_step (the reference
 * advances it once in animate_all and once per rigid mesh in animate_rigid, so
 * one rigid mesh moves 2 frames per step) and sets the static velocity to
 * (x - x_prev) / h; past the last frame the vertices stay there with zero
 * velocity.  Needs n_frames >= 3; tracks may not overlap; reset() re-places
 * frame 0.  Call after pa_backend_init. */
pa_status pa_backend_add_rigid_track(pa_backend* b, int32_t first, int32_t count, int32_t n_frames, const double* pos,
                                     const double* quat_xyzw, int32_t frames_per_step);

/* Point-sequence track for the static vertices [first, first + count) (≙ a
 * ScriptAnimator script whose npz holds per-frame points,
 * src/solver/animator.cpp:41-61,132-178): frame k places them at
 * points[k][i] (n_frames x count x 3, world positions, i.e. the mesh's
 * translate + rotate (scale p) already applied).  Registration places frame 0
 * with zero velocity; each step advances frames_per_step frames and sets the
 * static velocity to (x - x_prev) / h; once the counter passes the last frame
 * the vertices stay there with zero velocity (the point script reads the
 * shared counter before the rigid scripts advance it, so it shows its last
 * frame one step longer than a rigid track would).  Shares the frame-counter
 * entry points below with the rigid tracks. */
pa_status pa_backend_add_point_track(pa_backend* b, int32_t first, int32_t count, int32_t n_frames, const double* points,
                                     int32_t frames_per_step);

/* Frame counters of the rigid tracks in registration order (*count = number
 * of tracks; frames may be NULL).  Setting them (for resuming a checkpoint,
 * after pa_backend_set_state has restored the positions) also re-places each
 * track's last-placed positions at that frame, so the next step's static
 * velocities equal an uninterrupted run's. */
pa_status pa_backend_get_track_frames(pa_backend* b, int32_t* frames, int32_t* count);
pa_status pa_backend_set_track_frames(pa_backend* b, const int32_t* frames, int32_t count);

/* Convenience: runs the whole call order above for a scene (creates and
 * attaches its own detector when contact is enabled). */
pa_status pa_backend_create_from_scene(const pa_scene* s, const pa_admm_config* cfg, const pa_device_opts* opts,
                                       pa_backend** out);

/* ---------------------------------------------------------------------------
 * Sub-step entry points for parity tests and profiling.  Each runs one
 * device phase on the backend's current device state.
 * ------------------------------------------------------------------------- */
/* Local step: z = prox(D x + Ue) for host x (3 n_all) and Ue (3 m); writes z (3 m). */
pa_status pa_backend_project_elastic(pa_backend* b, const double* x, const double* ue, double* z);
/* Contact projection with the attached detector's current contacts: p
 * (3 n_all) in/out; r_c out for the first min(n_contacts, rc_cap) contacts
 * (3 each; rc may be null when rc_cap is 0); *n_contacts = the contact count.
 * Runs the Scc setup and gs_max_iter Jacobi sweeps. */
pa_status pa_backend_project_contacts(pa_backend* b, double* p, double* rc, int32_t rc_cap, int32_t* n_contacts);
/* Global solve A x = rhs (3 n_dyn) to global_tol, from x_init (3 n_dyn); returns PCG iterations. */
pa_status pa_backend_global_solve(pa_backend* b, const double* rhs, const double* x_init, double* x, int32_t* iters);
/* hipEvent timing (adds event records to the stream; off by default):
 * mode bit 0 times every PCG SpMV launch, bit 1 times the step phases. */
pa_status pa_backend_set_profiling(pa_backend* b, int32_t mode);
/* Device timing of the last step by phase (ms): detection, local, contact, rhs, global, other. */
pa_status pa_backend_phase_times(pa_backend* b, double* ms6);
/* The ADMM residuals of the last step at every check (residual_tol > 0, every
 * residual_interval iterations): pairs (r_primal, r_dual) in check order, at
 * most cap pairs written to out; *count = the number of checks.  A
 * warm-started step that fell back to a cold re-run reports the re-run's.
 * (The reference declares residual slots but never fills them,
 * src/solver/backend_cpu/admm_impl_cpu.h:126,154,167; the definition is this
 * library's, stated beside pa_admm_config.residual_tol.) */
pa_status pa_backend_residual_log(pa_backend* b, double* out, int32_t cap, int32_t* count);
/* Sizes: [n_all, n_dyn, m_rows, nnz of the off-diagonal system matrix,
 * nnz of the damping matrix, nnz of the D^T gather, contacts of the last
 * detection, and for the direct solve (precond 2; zeros otherwise): stored
 * factor entries, dense-top columns (sum of m), dense-top entries (sum of m^2)]. */
pa_status pa_backend_get_sizes(pa_backend* b, int64_t* out10);
/* The global solve's measured kernel: the fused PCG SpMV (k_cg_dir_spmv,
 * precond 0 and 1) or the dense-top product of the direct solve (k_chol_top,
 * precond 2).
 * which = 0: per-launch average (ms) of HIP event pairs around every launch
 * of it on the backend's stream during the steps since the last call with
 * reset = 1 (each pair also holds the launch's dispatch latency), and the
 * launch count.
 * which = 1: launches it *launches (in) times back-to-back on the current
 * device state between two events and returns the average per launch (ms);
 * call between steps (it writes only solver scratch). */
pa_status pa_backend_kernel_time(pa_backend* b, int32_t which, int32_t reset, double* avg_ms, int64_t* launches);

/* ---------------------------------------------------------------------------
 * Learned warm start of the contact duals.  No counterpart in the reference:
 * there the contact duals r_c restart from zero at every detection
 * (src/solver/contact_solver.cu:243; CPU src/contact/contact_info.h:46).
 * At each detection a small MLP (10 -> 128 -> 128 -> 128 -> 2, SiLU, BF16
 * weights, FP32 accumulation on MFMA) maps per-contact features to an initial
 * dual; plain cold start stays as the fallback.
 *
 * Features of a contact at the start of its detection window (raw units; h =
 * time step, dhat = contact distance, s = h / dhat, n = contact normal, p0 =
 * (x - x0 + Uc) / h on dynamic and the static velocity on static vertices,
 * u0 = sum_k b_k p0_k + K_c, v = velocities at the step start, t = unit
 * tangential part of u0 (any unit vector normal to n when it vanishes),
 * lambda_prev = the dual of the same contact (same type and primitives) at
 * the end of the previous window):
 *   0 h_cN / dhat          1 s (u0.n)              2 s |u0 - (u0.n) n|
 *   3 s (v_rel.n)          4 s |v_rel - (v_rel.n) n|  (v_rel = sum_k b_k v_k)
 *   5 mu                   6 type (0 PT, 1 EE)      7 1 if lambda_prev exists
 *   8 s (lambda_prev.n)    9 s (lambda_prev.t)
 * Outputs: s (lambda.n), s (lambda.t); the seeded dual is lambda.
 * ------------------------------------------------------------------------- */
#define PA_MLP_FEATURES 10
#define PA_MLP_OUTPUTS 2
#define PA_MLP_PARAMS 34690 /* W1[128][10] b1[128] W2[128][128] b2 W3[128][128] b3 W4[2][128] b4[2] */

typedef struct pa_warm_start {
    int32_t mode;        /* 0 cold start, 1 learned MLP, 2 the previous window's dual of the same contact */
    int32_t patience;    /* seeded windows in a row judged bad, sum |r_final - seed|^2 > 4 sum |r_final|^2
                            (the seeds miss the window's final duals by more than twice what zero would),
                            before the step is re-run cold; 0 = 2 */
    double stall_ratio;  /* a residual check above stall_ratio x the step's best so far, or non-finite,
                            re-runs the step cold; 0 = 1000 (the residual jumps by 10x and more after a
                            detection brings new contacts, in plain steps too) */
    double clamp;        /* |seed component| <= clamp in units of dhat / h; 0 = 50 */
    const float* params; /* mode 1: PA_MLP_PARAMS weights in the flat layout above (copied) */
    float in_shift[PA_MLP_FEATURES], in_scale[PA_MLP_FEATURES]; /* network input = (feature - shift) * scale */
    float out_scale[PA_MLP_OUTPUTS];                              /* s lambda = network output * out_scale */
} pa_warm_start;

/* Re-running cold replays the step from its starting state, so a fallback step
 * is bit-identical to a plain step. */
pa_status pa_backend_set_warm_start(pa_backend* b, const pa_warm_start* ws);
/* Contact-state log (training data): at the end of each detection window one
 * row of 12 floats per contact, the 10 features at the window's start and the
 * window's final dual as s (lambda.n), s (lambda.t).  capacity 0 disables;
 * rows beyond the capacity are dropped. */
pa_status pa_backend_set_contact_log(pa_backend* b, int64_t capacity_rows);
/* Copies up to cap_rows rows and empties the log; *rows = rows copied. */
pa_status pa_backend_read_contact_log(pa_backend* b, float* out, int64_t cap_rows, int64_t* rows);
/* Seed log of the last step: per detection of the kept attempt, the 3 n_c
 * seeded duals in contact order (counts[k] = 0 when detection k was not seeded). */
pa_status pa_backend_set_seed_log(pa_backend* b, int32_t enabled);
pa_status pa_backend_read_seed_log(pa_backend* b, float* out, int64_t cap_floats, int32_t* counts, int32_t max_detections,
                                   int32_t* n_detections);
/* Current contact duals r_c (3 n_contacts, contact order). */
pa_status pa_backend_get_contact_duals(pa_backend* b, double* rc);

/* MLP handle for training on the device (forward, backward and Adam on MFMA). */
typedef struct pa_mlp pa_mlp;
/* Weights and biases ~ U(-1/sqrt(fan_in), 1/sqrt(fan_in)) from `seed`. */
pa_status pa_mlp_create(uint64_t seed, pa_mlp** out);
void pa_mlp_destroy(pa_mlp* m);
pa_status pa_mlp_get_params(pa_mlp* m, float* params);
/* Also resets the Adam state. */
pa_status pa_mlp_set_params(pa_mlp* m, const float* params);
/* y[n][2] = MLP(x[n][10]). */
pa_status pa_mlp_forward(pa_mlp* m, const float* x, int32_t n, float* y);
/* The same y[n][2] = MLP(x[n][10]) without allocating or freeing any device
 * memory.  No counterpart in the reference; it is for callers that cannot
 * allocate (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  Input and output are staged in one file-scope device array
 * per GPU of PA_MLP_NOALLOC_SCRATCH_BYTES (0.8 MB, held until the process
 * ends); n is at most PA_MLP_NOALLOC_MAX_ROWS per call (more is refused with
 * PA_ERR_INVALID).  Calls that overlap on one GPU share that array and race:
 * serialise them. */
#define PA_MLP_NOALLOC_MAX_ROWS 16384
#define PA_MLP_NOALLOC_SCRATCH_BYTES 786432
pa_status pa_mlp_forward_noalloc(pa_mlp* m, const float* x, int32_t n, float* y);
/* Gradient of L = 1/(2n) sum |MLP(x) - t|^2 (t[n][2]) in the flat layout; *loss = L. */
pa_status pa_mlp_gradients(pa_mlp* m, const float* x, const float* t, int32_t n, float* grad, double* loss);
/* One Adam step (beta1 0.9, beta2 0.999, eps 1e-8) on that loss; *loss = L before the step. */
pa_status pa_mlp_adam_step(pa_mlp* m, const float* x, const float* t, int32_t n, double lr, double* loss);
/* Adam over `epochs` shuffled passes (seeded) of samples[n][12] (10 inputs, 2
 * targets) in batches of `batch` (a multiple of 32); epoch_loss[e] = mean L. */
pa_status pa_mlp_train(pa_mlp* m, const float* samples, int64_t n, int32_t epochs, int32_t batch, double lr, uint64_t seed,
                       double* epoch_loss);
/* Average ms per forward (which 0) or forward + backward + Adam (which 1) of
 * `rows` rows over `reps` back-to-back runs (weights kept, Adam state reset). */
pa_status pa_mlp_time(pa_mlp* m, int32_t which, int32_t rows, int32_t reps, double* ms);

/* ---------------------------------------------------------------------------
 * Batched scenes.  No counterpart in the reference, which runs one scene per
 * process (its solver keeps function-static state).  Scenes merged into one
 * block-diagonal scene step together in one backend: one detection over all
 * of them (each scene's primitives in their own LBVH subtree, so no pair spans
 * two scenes), one pass of every per-element kernel over all rows, and the
 * global solve as one persistent launch with a workgroup per scene
 * (Jacobi-preconditioned CG, per-scene convergence; the workgroup shape is
 * autotuned on the batch's own system at the first solve, or pinned).
 * pa_backend_create_from_scene on a merged scene builds this batched backend.
 * The ADMM stop test (residual_tol) is over the whole batch.
 * ------------------------------------------------------------------------- */
/* Merges 1..2048 scenes: the dynamic vertices of all scenes first (scene
 * order), then their static vertices; elements keep their scene order. */
pa_status pa_scene_merge(const pa_scene* const* scenes, int32_t count, pa_scene** out);
/* Segmented detection for a merged scene: seg[v] (n_all) is the scene of
 * vertex v (count scenes); pairs are only sought inside a scene.  Keys become
 * (scene << 21 | 21-bit Morton code), so each scene's primitives form one
 * subtree, and every query starts at its own scene's subtree root. */
pa_status pa_detector_set_segments(pa_detector* d, const int32_t* seg, int32_t count);
/* Query passes: 0 (default) a collect pass (traversal only, leaf hits to
 * per-query slabs and an overflow list) then a test pass (the FP64 predicate
 * on the hits), rerun as the single pass when the shared traversal stack or the
 * overflow list was too small; 1 the single pass (traversal and predicate
 * together) always.  Both give the same list.  No counterpart in the
 * reference: a diagnostic for checking that they do. */
pa_status pa_detector_set_single_pass(pa_detector* d, int32_t on);
/* Scene of every vertex (n_all), and per scene the first dynamic and first
 * static vertex (count + 1 entries each); any pointer may be NULL.  *count is
 * 1 for a scene that was not merged. */
pa_status pa_scene_get_segments(const pa_scene* s, int32_t* seg, int32_t* dyn_off, int32_t* stat_off, int32_t* count);
/* Per scene of a batched backend: PCG iterations and device time (ms) of its
 * workgroup in the global solves of the last step. */
pa_status pa_backend_batch_stats(pa_backend* b, int32_t* iters, double* solve_ms);
/* Contact sets of at most max_contacts contacts (0..2048, default 2048) run
 * every Jacobi sweep of a contact projection in one workgroup, one launch per
 * projection; larger sets launch two kernels per sweep.  Both give the same
 * bits.  No counterpart in the reference (contact_solver.cu:316-400 launches
 * per sweep); a diagnostic for comparing the two paths. */
pa_status pa_backend_set_contact_sweep_wg(pa_backend* b, int32_t max_contacts);
/* Pins the batched solve's workgroup size (256, 512 or 1024) and lanes per CSR
 * row (1 or 4); 0, 0 re-tunes at the next solve.  Results depend on the
 * variant at the rounding level (reduction order), so pin it for bit-exact
 * reruns. */
pa_status pa_backend_set_batch_tuning(pa_backend* b, int32_t threads, int32_t lanes);
/* The variant in use (0, 0 before tuning) and the autotuner's time of each of
 * the 6 variants (ms; zeros when pinned). */
pa_status pa_backend_get_batch_tuning(pa_backend* b, int32_t* threads, int32_t* lanes, double* ms6);

/* Message of the last failed call on this host thread (any handle). */
const char* pa_last_error_message(void);

#ifdef __cplusplus
}
#endif

#endif /* PA_ADMM_H */
