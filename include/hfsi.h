/*
 * hfsi.h -- C ABI of the MI355X (gfx950) pressure-projection and MPM library
 * (libhfsi.so).
 *
 * Conventions
 *   - Device buffers are owned by the caller and passed as plain pointers.
 *     Cell arrays are row-major [i][j][k] with k fastest (nx*ny*nz elements);
 *     velocity is [i][j][k][3] float32 where component d is the normal flux on
 *     the LOW d-face of the cell.
 *   - Every call takes the HIP stream (hipStream_t, passed as void*) it
 *     enqueues on and returns an int status: 0 ok, < 0 usage/runtime error
 *     (message from hfsi_last_error()).
 *   - A handle may be used from one host thread / one stream at a time.
 *     Calls are asynchronous unless they say they synchronise.
 *
 * The Python facade (easyfsi_amd.simulation_core) maps these calls onto the
 * reference's CartesianFluidSolver / NeoHookeanMpmState methods; each entry
 * point names the reference function it replaces.
 */
#ifndef HFSI_H
#define HFSI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define HFSI_OK 0
#define HFSI_ERR_ARG (-1)
#define HFSI_ERR_HIP (-2)
#define HFSI_ERR_STATE (-3)

/* Solve precision modes (bit values; hfsi_fluid_create takes a mask). */
#define HFSI_PREC_REF64 1 /* float64 CG vectors and level-0 V-cycle, float32 coarse levels */
#define HFSI_PREC_FP32 2  /* float32 CG vectors and V-cycle, float64 solution and dots      */
#define HFSI_PREC_MIXED 4 /* fp16-stored V-cycle, float32 CG, float64 solution and dots     */

/* Preconditioners (simulation_core/fluid.py:16 CG_PRECONDITIONER_CHOICES). */
#define HFSI_PRECOND_AUTO 0
#define HFSI_PRECOND_JACOBI 1
#define HFSI_PRECOND_MG 2       /* "fv_multigrid": 2 pre / 24 coarse / 2 post          */
#define HFSI_PRECOND_MG_LIGHT 3 /* "fv_multigrid_light": 1 / 12 / 1                     */

/* Breakdown kinds reported in hfsi_cg_stats.breakdown_kind
 * (messages of simulation_core/fluid.py:6668-6797). */
#define HFSI_BREAKDOWN_NONE 0
#define HFSI_BREAKDOWN_INITIAL_DOT 1   /* "initial residual/preconditioner dot is not positive finite"   */
#define HFSI_BREAKDOWN_DEVICE_SCALAR 2 /* "device-side CG scalar update failed"                          */
#define HFSI_BREAKDOWN_RESTART_DOT 3   /* "restarted residual/preconditioner dot is not positive finite" */
#define HFSI_BREAKDOWN_BICGSTAB_SHADOW 4        /* "BiCGSTAB shadow residual dot is not finite" */
#define HFSI_BREAKDOWN_BICGSTAB_RECURRENCE 5    /* "BiCGSTAB recurrence scalar is not finite"   */
#define HFSI_BREAKDOWN_BICGSTAB_BETA 6          /* "BiCGSTAB beta is not finite"                */
#define HFSI_BREAKDOWN_BICGSTAB_ALPHA_DEN 7     /* "BiCGSTAB alpha denominator is not finite"   */
#define HFSI_BREAKDOWN_BICGSTAB_ALPHA 8         /* "BiCGSTAB alpha is not finite"               */
#define HFSI_BREAKDOWN_BICGSTAB_OMEGA_DEN 9     /* "BiCGSTAB omega denominator is not finite"   */
#define HFSI_BREAKDOWN_BICGSTAB_OMEGA 10        /* "BiCGSTAB omega is not finite"               */
#define HFSI_BREAKDOWN_BICGSTAB_NOT_CONVERGED 11 /* "BiCGSTAB fallback did not converge"        */

typedef struct hfsi_fluid hfsi_fluid;

/* Per-solve statistics (the reference's last_cg_* host mirrors,
 * simulation_core/fluid.py:1079-1091). */
typedef struct hfsi_cg_stats {
  int32_t iterations;
  int32_t converged;
  int32_t breakdown_code; /* device code: 1 non-positive dAd, 2 beta breakdown */
  int32_t breakdown_kind; /* HFSI_BREAKDOWN_* */
  int32_t host_residual_checks;
  int32_t mean_projection_count;
  int32_t restart_count;
  int32_t used_multigrid;
  int32_t true_residual_replacements;
  int32_t vcycles;
  double b_norm;
  double initial_relative_residual;
  double relative_residual;      /* of the residual the convergence test used      */
  double breakdown_dAd;
  double true_relative_residual; /* ||b - A x||_V / ||b||_V in float64 at exit, or -1 */
} hfsi_cg_stats;

/* Solve options for hfsi_fluid_solve_cg. */
typedef struct hfsi_cg_options {
  int32_t precision;          /* one HFSI_PREC_* bit the handle was created with          */
  int32_t preconditioner;     /* HFSI_PRECOND_*                                           */
  int32_t max_iterations;     /* >= 1                                                     */
  int32_t remove_mean;        /* project the closed-domain null space (V-weighted mean)   */
  int32_t outlet_zmin;        /* Dirichlet p = 0 ghost below k = 0                        */
  int32_t interface_active;   /* pressure-interface matrix terms present: no MG          */
  int32_t check_interval;     /* residual check interval (reference: 16)                  */
  int32_t restart_interval;   /* exact-residual restart interval (reference: 512)         */
  int32_t true_residual;      /* 1: every check recomputes r = b - A x in float64        */
  int32_t true_residual_at_exit;
  int32_t monitor_lag;        /* MIXED only, L > 0: every iteration computes the float64 true
                                 residual norm of x (not stored) into a host-mapped ring; at
                                 the end of iteration it, with its V-cycle queued, the host
                                 reads iteration it - L + 1.  L = 1 stops at the first iterate
                                 that meets the tolerance; L > 1 checks one iteration after a
                                 hit.  0: checks every check_interval iterations only        */
  double tolerance;           /* relative, on ||r||_V / ||b||_V                            */
  double rhs_scale;           /* rho / dt                                                 */
} hfsi_cg_options;

/* ---- library ------------------------------------------------------------ */

int hfsi_version(void);
const char* hfsi_last_error(void);
/* 1 if a gfx950 device is visible and the code objects load, else 0 (synchronises). */
int hfsi_device_ok(void);

/* ---- fluid grid handle ---------------------------------------------------- */

/* Grid + multigrid hierarchy + solver workspaces for the requested precision
 * modes.  Replaces CartesianFluidSolver.__init__'s field allocation and metric
 * upload (simulation_core/fluid.py:736-1199): level shapes halve while every
 * axis is above 3 (fluid.py:692-701), coarse widths are pairwise sums
 * (fluid.py:704-708), metrics are stored as float32 like the reference's
 * fields.  Allocates device memory: after it, the only handle calls that allocate are
 * hfsi_fluid_set_interface_couplings when it compiles more couplings than reserved
 * (hfsi_fluid_reserve_couplings) and hfsi_fluid_reserve_couplings itself; the HIBM marker calls
 * (force scatter, surface feedback, stress sampling, force aggregation, no-slip residual) draw
 * their workspaces from a per-device memory pool. */
int hfsi_fluid_create(hfsi_fluid** out, int32_t nx, int32_t ny, int32_t nz, const double* widths_x,
                      const double* widths_y, const double* widths_z, const double* origin3,
                      int32_t precision_mask, void* stream);
int hfsi_fluid_destroy(hfsi_fluid* h);
int32_t hfsi_fluid_num_levels(const hfsi_fluid* h);
/* Level shape (3 ints) of level `level`. */
int hfsi_fluid_level_shape(const hfsi_fluid* h, int32_t level, int32_t* shape3);
/* Device bytes held by the handle. */
size_t hfsi_fluid_device_bytes(const hfsi_fluid* h);

/* Derive the per-level open-face masks, coarse obstacle / velocity-Dirichlet
 * flags and V-averaged interface diagonals from the caller's fields
 * (restriction rules of _mg_restrict_residual_kernel, fluid.py:5309-5388).
 * vd_active / vd_weight / iface_diag may be NULL (all zero). */
int hfsi_fluid_set_masks(hfsi_fluid* h, const int32_t* obstacle, const int32_t* vd_active,
                         const float* vd_weight, const double* iface_diag, void* stream);

/* div = sum_d (u_d[c+e_d] - u_d[c]) / w_d[c] over open faces
 * (_compute_divergence_kernel, fluid.py:3450-3486).  Uses the masks of the
 * last hfsi_fluid_set_masks. */
int hfsi_fluid_divergence(hfsi_fluid* h, const float* velocity, float* divergence, int32_t outlet_zmin,
                          void* stream);

/* q = A p (_fv_laplacian_apply_kernel, fluid.py:4311-4340, plain path). */
int hfsi_fluid_apply(hfsi_fluid* h, const double* p, double* q, int32_t outlet_zmin, void* stream);

/* Jacobi diagonal (_fv_diagonal_kernel, fluid.py:4280-4309). */
int hfsi_fluid_diagonal(hfsi_fluid* h, double* diag, int32_t outlet_zmin, void* stream);

/* sum over free cells of V a b (_weighted_dot_kernel, fluid.py:4533-4544);
 * synchronises and writes the result to *out. */
int hfsi_fluid_weighted_dot(hfsi_fluid* h, const double* a, const double* b, double* out, void* stream);

/* One V-cycle z = M^-1 r (_apply_fv_multigrid_preconditioner, fluid.py:6085-6262)
 * at the given precision; r and z are float64 level-0 arrays.  With
 * HFSI_PREC_MIXED, coarse = 0 solves the coarsest level directly in float64
 * (levels of at most 512 cells; 8 RB sweeps otherwise). */
int hfsi_fluid_vcycle(hfsi_fluid* h, const double* r, double* z, int32_t precision, int32_t pre,
                      int32_t coarse, int32_t post, int32_t outlet_zmin, void* stream);

/* Flexible PCG on A p = -(rhs0 - mean) with rhs0 = f32(rhs_scale)*(div - source)
 * - iface_rhs (_solve_pressure_poisson_fv_cg, fluid.py:6535-6811).  pressure is
 * the float64 warm start and result.  source / iface_rhs may be NULL.
 * Synchronises at residual checks; stats may be NULL. */
int hfsi_fluid_solve_cg(hfsi_fluid* h, const float* divergence, const float* source, const double* iface_rhs,
                        double* pressure, const hfsi_cg_options* opt, hfsi_cg_stats* stats, void* stream);

/* Standalone solvers on the same operator: `iterations` damped Jacobi sweeps
 * (fv_jacobi, fluid.py:5977-5990) and Jacobi V-cycles 3/36/3 (+ final sweeps on
 * graded grids) (fv_multigrid, fluid.py:5992-6083).  pressure is in/out. */
int hfsi_fluid_solve_fv_jacobi(hfsi_fluid* h, const float* divergence, const float* source,
                               const double* iface_rhs, double* pressure, double rhs_scale, int32_t iterations,
                               int32_t outlet_zmin, void* stream);
int hfsi_fluid_solve_fv_multigrid(hfsi_fluid* h, const float* divergence, const float* source,
                                  const double* iface_rhs, double* pressure, double rhs_scale, int32_t iterations,
                                  int32_t cycles, int32_t outlet_zmin, void* stream);

/* Compact uniform-grid Jacobi, the reference project() default
 * (_pressure_jacobi_kernel + copy, fluid.py:3996-4053, 5842-5860). */
int hfsi_fluid_solve_legacy_jacobi(hfsi_fluid* h, const float* divergence, const float* source,
                                   const int32_t* obstacle, double* pressure, double rhs_scale, double inv_dx2,
                                   double inv_dy2, double inv_dz2, int32_t iterations, int32_t outlet_zmin,
                                   void* stream);

/* u_d -= (dt/rho) w (p_c - p_{c-e_d}) / d_d[c] (_subtract_pressure_gradient_kernel,
 * fluid.py:5538-5582).  vd_* may be NULL. */
int hfsi_fluid_subtract_gradient(hfsi_fluid* h, float* velocity, const double* pressure, const int32_t* vd_active,
                                 const float* vd_weight, const float* vd_value, float dt_over_rho,
                                 int32_t outlet_zmin, void* stream);

/* Zero the normal flux of the low wall faces
 * (_apply_closed_boundary_no_normal_flow_kernel, fluid.py:5528-5536). */
int hfsi_fluid_wall_clamp(hfsi_fluid* h, float* velocity, int32_t outlet_zmin, void* stream);

/* Divergence report reductions (_divergence_stats_kernel,
 * _divergence_residual_stats_kernel, _divergence_final_report_kernel,
 * fluid.py:3493-3663): 18 slots x (max, sum of squares, count) written to
 * out54 (float64, host memory); synchronises.  Slots 0/1 all free cells
 * (raw/residual), 2/3 interior, 4/5 stencil touching a velocity-Dirichlet
 * row, 6/7 the rest, 8/9 pressure-correctable, 10/11 fixed, 12-15 their
 * interior parts, 16/17 unused here (HIBM unreached set).  vd_active and
 * source and iface_div may be NULL. */
int hfsi_fluid_divergence_report(hfsi_fluid* h, const float* divergence, const float* source,
                                 const double* iface_div, const int32_t* vd_active, int32_t outlet_zmin,
                                 double* out54, void* stream);

/* _mark_sphere_kernel (simulation_core/fluid.py:2828-2858): obstacle[i][j][k] = 1 where
 * (cx[i]-c0)^2 + (cy[j]-c1)^2 + (cz[k]-c2)^2 <= radius^2 in float32 (that order, no
 * contraction), else 0.  center_x/y/z: the float32 cell-centre arrays (device); centre3 (host). */
int hfsi_fluid_mark_sphere(hfsi_fluid* h, const float* center_x, const float* center_y, const float* center_z,
                           const float* centre3, float radius, int32_t* obstacle, void* stream);

/* ---- velocity rows -------------------------------------------------------------------------
 * Per-cell arithmetic in float32 in the order of the reference kernels (no contraction); the
 * reports are float64 sums over the per-cell float32 values, written to host memory (the call
 * then synchronises).  velocity is [n][3] float32, the widths those of the handle. */

/* _apply_velocity_dirichlet_boundary_rows_kernel (simulation_core/fluid.py:2549-2594): free cells
 * with vd_active != 0 take vd_value [n][3].  report6 (host, may be NULL): active cells,
 * sum |dv|, max |dv|, momentum change rho dv V (3). */
int hfsi_fluid_apply_velocity_rows(hfsi_fluid* h, float* velocity, const int32_t* obstacle,
                                   const int32_t* vd_active, const float* vd_value, float rho, double* report6,
                                   void* stream);

/* The constraint fields of simulation_core/fluid.py:897-902 ([n][3] sums, [n] weights). */
typedef struct hfsi_velocity_constraints {
  const float* sum;
  const float* weight;
  const float* primary_sum;
  const float* primary_weight;
  const float* secondary_sum;
  const float* secondary_weight;
} hfsi_velocity_constraints;

/* _apply_velocity_constraints_kernel (simulation_core/fluid.py:2629-2700): free cells with
 * weight > 0 move by s (sum / weight - u), s = blend / (1 + solid_mobility_ratio) in float32.
 * primary_impulse3 / secondary_impulse3 (device float64, accumulated on every call) gain the
 * momentum change of the primary / secondary parts, (s (part_sum - u part_weight) / weight)
 * rho V.  report12 (host, may be NULL): active cells, sum |dv|, max |dv|, momentum change (3),
 * primary (3), secondary (3). */
int hfsi_fluid_apply_velocity_constraints(hfsi_fluid* h, float* velocity, const int32_t* obstacle,
                                          const hfsi_velocity_constraints* c, float blend,
                                          float solid_mobility_ratio, float rho, double* primary_impulse3,
                                          double* secondary_impulse3, double* report12, void* stream);

/* One sweep of _local_divergence_cleanup_kernel (simulation_core/fluid.py:5766-5836), uniform
 * grids only: every free cell relaxes its divergence - source over the faces it shares with a
 * free neighbour that carry no velocity-Dirichlet row.  Deterministic (each face gathers its two
 * contributions).  source and vd_active may be NULL. */
int hfsi_fluid_local_divergence_cleanup(hfsi_fluid* h, float* velocity, const float* divergence,
                                        const float* source, const int32_t* obstacle, const int32_t* vd_active,
                                        float dx, float dy, float dz, float relaxation, void* stream);

/* ---- learned initial guess (no reference counterpart) ----------------------
 * The network grid is the solve grid coarsened 2:1 per axis (coarsen = 1, even dimensions) or the
 * solve grid itself.  hfsi_guess_features writes the network input [n_net][5] float32: the
 * divergence of a network cell's free children averaged over their volume and divided by its
 * volume-weighted RMS over the network grid, the solid volume fraction, log2(width /
 * net_min_width) per axis.  hfsi_guess_pressure takes the network output (network grid, units of
 * -p kappa / ((rho/dt) RMS)), interpolates it trilinearly to the solve grid (half-cell centres,
 * clamped at the walls), zeroes cells that are not free, removes the volume-weighted mean on a
 * closed domain (outlet_zmin = 0), and scales it by the energy-optimal factor
 * gamma = <p, b>_V / <p, A p>_V with b = -(rho/dt)(divergence - source); the result goes to
 * pressure (float64, the PCG start).  The RMS, mean and factor stay on the device; gamma_out
 * (host, may be NULL) synchronises and returns the factor.  A p is the operator without
 * interface couplings.  Both use the handle's float64 scratch vector. */
int hfsi_guess_features(hfsi_fluid* h, const float* divergence, int32_t coarsen, double net_min_width,
                        float* features, void* stream);
int hfsi_guess_pressure(hfsi_fluid* h, const float* net_out, const float* divergence, const float* source,
                        double rho_over_dt, double net_kappa, int32_t coarsen, int32_t outlet_zmin, double* pressure,
                        double* gamma_out, void* stream);

/* ---- neo-Hookean MPM ------------------------------------------------------ */

typedef struct hfsi_mpm hfsi_mpm;

/* Particle arrays (caller-owned device memory, float32 unless noted):
 * x, v, rest_x, external_force, normal, rest_normal: [P][3];  C, F: [P][3][3]
 * row-major;  mass, volume, area, rest_area: [P];  fixed, region: int32 [P].
 * fixed, region, external_force may be NULL (all zero); the four surface
 * arrays are all NULL or all set. */
typedef struct hfsi_mpm_particles {
  float* x;
  float* v;
  float* C;
  float* F;
  const float* mass;
  const float* volume;
  const float* rest_x;
  const int32_t* fixed;
  const int32_t* region;
  const float* external_force;
  float* normal;
  const float* rest_normal;
  float* area;
  const float* rest_area;
} hfsi_mpm_particles;

/* Background grid (caller-owned): mass [n], velocity / momentum [n][3],
 * force [n][3], n = nx*ny*nz nodes, k fastest. */
typedef struct hfsi_mpm_grid {
  float* mass;
  float* velocity;
  float* force;
} hfsi_mpm_grid;

/* Uniform background grid: dx_a = (max_a - min_a) / n_a
 * (NeoHookeanMpmState.__init__, simulation_core/neo_hookean_mpm.py:57-142).
 * Allocates the reduction workspace. */
int hfsi_mpm_create(hfsi_mpm** out, int32_t particle_capacity, const double* bounds_min3, const double* bounds_max3,
                    const int32_t* grid_nodes3, void* stream);
int hfsi_mpm_destroy(hfsi_mpm* h);

/* P2G scatter: HFSI_MPM_P2G_BINNED (default) buckets particles by block of
 * 4^3 nodes (states of up to 2^19 particles) or 8^3 nodes and accumulates each block in an LDS tile; the tiles are stored
 * whole and the grid update sums, for every node, the (up to 8) tiles that
 * cover it in a fixed order (grids of more than 65536 blocks of 8^3 nodes add each tile
 * to the grid with global atomics instead).  HFSI_MPM_P2G_ATOMIC scatters
 * every particle's 27 node contributions with global float atomics.  Same
 * arithmetic per particle; float summation order differs. */
#define HFSI_MPM_P2G_BINNED 0
#define HFSI_MPM_P2G_ATOMIC 1
int hfsi_mpm_set_p2g_mode(hfsi_mpm* h, int32_t mode);

/* The grid arrays are outputs of hfsi_mpm_step.  With the tile path
 * (HFSI_MPM_P2G_BINNED, at most 65536 blocks) a step rewrites every node of
 * the blocks its particles reach and zeroes the blocks the previous step
 * wrote that it does not reach, instead of clearing the whole grid (the
 * reference clears it, neo_hookean_mpm.py:706-709): the result is the same
 * as long as nobody else writes the grid arrays between steps.  A step with
 * other grid arrays than the previous one, the first step and the first step
 * after this call (or after a change of P2G mode) clear the whole grid.  Call
 * it after writing the grid arrays outside hfsi_mpm_step.  No reference
 * counterpart. */
int hfsi_mpm_invalidate_grid(hfsi_mpm* h);

/* One step: grid clear (see hfsi_mpm_invalidate_grid), P2G with the SVD clamp and neo-Hookean stress, grid
 * update with damping, G2P / APIC / F update, surface update and the report
 * reductions (NeoHookeanMpmState._step_kernel, neo_hookean_mpm.py:695-959).
 * When report34 (host) is not NULL the call synchronises and writes the 28
 * values + 6 counts of the reference's packed snapshot (neo_hookean_mpm.py:909-959). */
int hfsi_mpm_step(hfsi_mpm* h, const hfsi_mpm_particles* particles, int32_t count, const hfsi_mpm_grid* grid,
                  float dt_s, float mu_pa, float lambda_pa, float velocity_damping, int32_t primary_region_id,
                  int32_t secondary_region_id, double* report34, void* stream);

/* Particle set-up and loads.  Every particle array of hfsi_mpm_particles must be given
 * (the init call writes the const ones too). */

/* NeoHookeanMpmState._initialize_layered_tri_surface_kernel
 * (simulation_core/neo_hookean_mpm.py:231-294): face_count * layer_count particles, particle
 * face * layer_count + layer at centroid + normal * (((layer + 0.5) / layer_count - 0.5) *
 * thickness), area / layer_count of the face's area, volume area * thickness, mass density *
 * volume; region of its face; faces of fixed_region_id (>= 0) take the primary thickness and fix
 * their particles.  centroid / normal [faces][3], area [faces] float32, face_region int32
 * (device).  The primary and secondary region masses are kept in the handle (float32). */
int hfsi_mpm_init_layered(hfsi_mpm* h, const hfsi_mpm_particles* particles, const float* centroid,
                          const float* normal, const float* area, const int32_t* face_region, int32_t face_count,
                          int32_t layer_count, int32_t primary_region_id, int32_t secondary_region_id,
                          int32_t fixed_region_id, float density, float primary_thickness,
                          float secondary_thickness, void* stream);
/* The region masses of the last hfsi_mpm_init_layered (primary, secondary; host, synchronises). */
int hfsi_mpm_region_masses(hfsi_mpm* h, float* out2, void* stream);

/* Region loads on the external force (neo_hookean_mpm.py:422-508), for particles p < count:
 * SET_PRESSURE f = -pressure * area * normal in region_id, 0 elsewhere
 * (_set_region_normal_pressure_kernel); ADD_PRESSURE f += -pressure * area * normal in region_id
 * (_add_region_normal_pressure_kernel); ADD_AREA f += load3 * area in region_id
 * (_add_region_area_load_kernel; load3 host, N/m^2). */
#define HFSI_MPM_LOAD_SET_PRESSURE 0
#define HFSI_MPM_LOAD_ADD_PRESSURE 1
#define HFSI_MPM_LOAD_ADD_AREA 2
#define HFSI_MPM_LOAD_LAYERED 3
int hfsi_mpm_region_load(hfsi_mpm* h, const hfsi_mpm_particles* particles, int32_t count, int32_t mode,
                         int32_t region_id, float pressure, const float* load3, void* stream);
/* _set_layered_region_loads_kernel (neo_hookean_mpm.py:357-391): f = primary_area_load * area +
 * primary_reaction * mass / max(primary mass, 1e-12) in the primary region, secondary_reaction *
 * mass / max(secondary mass, 1e-12) in the secondary region, 0 elsewhere (masses of the last
 * hfsi_mpm_init_layered; vectors host, float32). */
int hfsi_mpm_layered_region_loads(hfsi_mpm* h, const hfsi_mpm_particles* particles, int32_t count,
                                  int32_t primary_region_id, int32_t secondary_region_id,
                                  const float* primary_area_load3, const float* primary_reaction3,
                                  const float* secondary_reaction3, void* stream);
/* _enforce_rest_x_plane_kernel / _enforce_rest_z_plane_kernel (neo_hookean_mpm.py:540-573),
 * axis 0 (x) or 2 (z): x_axis = rest_x_axis, v_axis = 0, the axis row and column of C zero and of F
 * the identity's, then the surface normal and area from F. */
int hfsi_mpm_enforce_rest_plane(hfsi_mpm* h, const hfsi_mpm_particles* particles, int32_t count, int32_t axis,
                                void* stream);

/* ---- mixed-precision V-cycle (HFSI_PREC_MIXED; no reference counterpart) ---
 * The MIXED solve keeps the reference's flexible PCG driver with float32
 * vectors and float64 solution, SpMV arithmetic, dots and true residual, and
 * replaces its V-cycle by a red-black Gauss-Seidel V-cycle on a
 * semi-coarsened hierarchy (cells merge along an axis while the merged width
 * is <= 2.5x the level's nominal width), trilinear graded prolongation, a
 * float64 direct solve of the coarsest level, and fp16 storage on the levels
 * with at least half_min_cells cells (default 2^20).  Grids with
 * velocity-Dirichlet rows or an interface diagonal fall back to the FP32
 * V-cycle (hfsi_cg_stats.used_multigrid = 1; 2 when the mixed V-cycle ran).
 * hfsi_fluid_vcycle with HFSI_PREC_MIXED applies it to r (scale from r). */
/* Number of mixed levels (0 without HFSI_PREC_MIXED); *half_levels gets the
 * number stored in fp16. */
int hfsi_fluid_mixed_levels(const hfsi_fluid* h, int32_t* half_levels);
int hfsi_fluid_mixed_level_shape(const hfsi_fluid* h, int32_t level, int32_t* shape3);
int hfsi_fluid_mixed_set_half_min_cells(hfsi_fluid* h, int64_t min_cells);
/* Fused sweeps: both colour passes of a red-black sweep in one marching pass
 * over memory, on grid-launched levels with nz even and at least min_cells
 * cells (default 2^21); other levels run one launch per colour pass.  Both
 * forms give identical results. */
int hfsi_fluid_mixed_set_fused_min_cells(hfsi_fluid* h, int64_t min_cells);
/* Target number of workgroups of a fused sweep (default 1280, the number
 * resident at once: 5 per CU on 256 CUs): a workgroup marches a chunk of
 * nx * tiles / workgroups planes (a multiple of 4, 4 .. 64), and every chunk
 * recomputes 3 planes of its neighbour, so fewer workgroups do less redundant
 * work and keep fewer waves in flight.  Results do not depend on it. */
int hfsi_fluid_mixed_set_sweep_workgroups(hfsi_fluid* h, int64_t workgroups);

/* ---- learned pressure initial guess (no reference counterpart) -----------
 * A 3-level 3D U-Net (3x3x3 convolutions, channels 16 / 32 / 64, two per
 * level, 2x2x2 average pooling, nearest upsampling with skip concatenation,
 * ReLU, 1x1 output) in bf16 on MFMA with float32 accumulation, trained with
 * these entry points.  A handle is built for one grid shape (multiples of 4).
 * Input: 5 float channels per cell, channels-last [n][5]; output: 1 float per
 * cell.  Parameters (float32 masters), in order for each of the ten 3x3x3
 * layers E1A E1B E2A E2B B3A B3B D2A D2B D1A D1B: W[cout][27][cin] (tap =
 * (dz+1)*9 + (dy+1)*3 + (dx+1), E1A's cin padded 5 -> 16), b[cout]; then the
 * output layer w[16], b[1]. */
typedef struct hfsi_unet hfsi_unet;
int hfsi_unet_create(hfsi_unet** out, int32_t nx, int32_t ny, int32_t nz, int32_t train, uint64_t seed,
                     void* stream);
int hfsi_unet_destroy(hfsi_unet* h);
int64_t hfsi_unet_num_params(const hfsi_unet* h);
/* host <-> device parameter and gradient copies (synchronise) */
int hfsi_unet_get_params(hfsi_unet* h, float* host, void* stream);
int hfsi_unet_set_params(hfsi_unet* h, const float* host, void* stream);
int hfsi_unet_get_grads(hfsi_unet* h, float* host, void* stream);
int hfsi_unet_zero_grads(hfsi_unet* h, void* stream);
/* out[n] = net(in5[n][5]) (device pointers); keeps the activations for backward */
int hfsi_unet_forward(hfsi_unet* h, const float* in5, float* out, void* stream);
/* accumulate d(loss)/d(params) for d(loss)/d(out) = dout (after forward; train handles only) */
int hfsi_unet_backward(hfsi_unet* h, const float* dout, void* stream);
/* loss = sum_m (out - target)^2 / sum_m target^2 over mask != 0 (all cells if mask is NULL),
 * dout = its gradient; *loss (host, may be NULL: no synchronisation) */
int hfsi_unet_loss(hfsi_unet* h, const float* out, const float* target, const uint8_t* mask, float* dout,
                   double* loss, void* stream);
int hfsi_unet_adam_step(hfsi_unet* h, float lr, float beta1, float beta2, float eps, float weight_decay,
                        void* stream);

/* ---------------------------------------------------------------------------
 * Sharp-interface pressure couplings
 * ------------------------------------------------------------------------- */

#define HFSI_INTERFACE_SLOTS 16 /* primary + 15 extra slots per owner cell */

/* The solver's pressure-interface coupling fields (simulation_core/fluid.py:772-811),
 * device pointers: per-owner slots (count, first neighbour [n][3] and coefficient
 * [n], extra neighbours [n][15][3] and coefficients [n][15]; slot_active may be NULL
 * for none, the two extra arrays NULL together for all-zero extra slots) and the row list (owner and neighbour [rows][3], transmissibility
 * [rows]), which replaces the slots when row_count > 0 (at most n rows are read). */
typedef struct hfsi_interface_fields {
  const int32_t* slot_active;
  const int32_t* slot_neighbor;
  const double* slot_coefficient;
  const int32_t* extra_neighbor;
  const double* extra_coefficient;
  const int32_t* row_owner;
  const int32_t* row_neighbor;
  const double* row_transmissibility;
  int32_t row_count;
} hfsi_interface_fields;

/* Capacity of the compiled coupling list (couplings, 24 B each): hfsi_fluid_set_interface_couplings
 * reallocates the list only when it compiles more than this.  Synchronises the device; callers that
 * cannot allocate at set-up time reserve here.  No reference counterpart. */
int hfsi_fluid_reserve_couplings(hfsi_fluid* h, int64_t capacity);

/* Compile the off-diagonal interface terms of the operator
 * (_fv_laplacian_apply_kernel, fluid.py:4346-4456): every valid row or slot joins
 * fluid cells a and b as (A p)[a] -= T/V_a p[b], (A p)[b] -= T/V_b p[a].  From then
 * on hfsi_fluid_apply and the CG solves include them (the mixed V-cycle path is not
 * used while couplings exist).  Call again after the fields or the obstacle change;
 * a call with no rows and slot_active NULL removes them.  Also fills, when not NULL,
 * row_diagonal_density [n] (device; sum of T/V over report-valid rows) and
 * report[6] (host): report-valid rows, invalid rows, overflow rows, sum of 2T,
 * max T, couplings applied -- the row part of
 * _pressure_interface_matrix_terms_report_kernel (fluid.py:2864-3078).
 * Synchronises the stream. */
int hfsi_fluid_set_interface_couplings(hfsi_fluid* h, const int32_t* obstacle, const hfsi_interface_fields* f,
                                       double* row_diagonal_density, double* report, void* stream);
/* out += scale * (C p) with C the compiled couplings: the coupling part of
 * _update_pressure_interface_projection_divergence_kernel (fluid.py:5625-5693) with
 * scale = dt/rho.  p and out are [n] float64. */
int hfsi_fluid_interface_apply(hfsi_fluid* h, const double* p, double* out, double scale, void* stream);

/* Jacobi-preconditioned BiCGSTAB continuing from `pressure` on A p = rhs
 * (_continue_pressure_poisson_fv_bicgstab, fluid.py:6264-6533): the fallback after a
 * PCG solve with interface rows stops unconverged.  rhs is the float64 right-hand side
 * (NULL: that of the last hfsi_fluid_solve_cg on this handle), b_norm its V-norm; the
 * operator includes the interface couplings.  stats is updated in place: iterations
 * (start_iteration + the BiCGSTAB iteration of the last check), relative_residual,
 * converged, breakdown_kind (HFSI_BREAKDOWN_BICGSTAB_*), and the restart, residual
 * check and mean projection counters are incremented.  Synchronises at every scalar. */
int hfsi_fluid_solve_bicgstab(hfsi_fluid* h, const double* rhs, double* pressure, int32_t start_iteration,
                              int32_t max_iterations, double b_norm, int32_t outlet_zmin, double tolerance,
                              int32_t remove_mean, hfsi_cg_stats* stats, void* stream);

/* ---------------------------------------------------------------------------
 * Velocity predictor
 * ------------------------------------------------------------------------- */

/* Float32 metric arrays of the grid, as the solver's 1D fields hold them
 * (simulation_core/fluid.py:1013-1024): per axis a, faces[a] has n_a + 1
 * entries, centers[a] and widths[a] n_a, center_distances[a] n_a (entry d > 0
 * is centre d minus centre d - 1).  Device pointers. */
typedef struct hfsi_axis_metrics {
  const float* faces[3];
  const float* centers[3];
  const float* widths[3];
  const float* center_distances[3];
} hfsi_axis_metrics;

#define HFSI_ADVECT_EULER 0
#define HFSI_ADVECT_RK2 1

/* velocity = predictor(velocity_prev): semi-Lagrangian advection (Euler or RK2
 * backtrace, obstacle-aware trilinear sampling) plus explicit FV diffusion
 * dt * nu * lap(u), obstacle == 1 cells zeroed.  Replaces
 * CartesianFluidSolver._predict_kernel (simulation_core/fluid.py:2447-2513)
 * as launched by predict() (fluid.py:2515-2527), whose velocity -> velocity_prev
 * copy is the caller's (the Python host swaps the two buffers instead).
 * velocity_prev and velocity are [n][3] float32 and must not overlap;
 * obstacle is [n] int32.  Float32 arithmetic in the reference's operation
 * order without contraction.  Needs at least 2 cells per axis, dt_s > 0. */
int hfsi_fluid_predict(hfsi_fluid* h, const float* velocity_prev, const int32_t* obstacle, float* velocity,
                       const hfsi_axis_metrics* metrics, float dt_s, float nu_m2_s, int32_t scheme, void* stream);

/* ---------------------------------------------------------------------------
 * HIBM: marker -> MPM particle force scatter
 * ------------------------------------------------------------------------- */

typedef struct hfsi_marker_scatter_report {
  int32_t active_marker_count;   /* markers whose force was spread                        */
  int32_t invalid_marker_count;  /* non-finite markers and markers with weight sum <= 1e-12 */
  int64_t active_particle_count; /* (marker, particle) pairs with a positive weight        */
  double total_marker_force[3];  /* sum of the spread marker forces                       */
  double total_external_force[3];/* sum of the float32 contributions added to particles   */
} hfsi_marker_scatter_report;

/* external_force[p] += sum over markers m of float32(F_m * (w_mp / sum_q w_mq)) with the
 * tent weight w = prod_axis max(1 - |x_m - x_p| / support_radius, 0) in float32, over
 * markers with finite position and force and a weight sum above 1e-12 and particles with
 * finite positions.  Replaces
 * HibmMpmSurfaceMarkers._scatter_marker_forces_to_mpm_particles_kernel
 * (simulation_core/hibm_mpm.py:4899-4960); the particles are binned into cells of edge
 * >= support_radius so each marker visits the cells within its reach (at most 4 per axis)
 * instead of every particle.  Its bin and reduction workspaces come from a per-device
 * stream-ordered memory pool that keeps its memory between calls (the first call, and a call
 * with more particles or markers than any before, allocates from the device).
 * marker_position [M][3] float32, marker_force [M][3] float64, particle_position and
 * external_force [P][3] float32 (device).  report (host) may be NULL.  Synchronises. */
int hfsi_scatter_marker_forces(const float* marker_position, const double* marker_force, int32_t marker_count,
                               const float* particle_position, float* external_force, int32_t particle_count,
                               float support_radius, hfsi_marker_scatter_report* report, void* stream);

/* hfsi_scatter_marker_forces without allocation: the same kernels and results, with the
 * bins and the reduction workspace in one file-scope device array of the library (about
 * 25 MB per device, held until the process ends) instead of the memory pool.  At most
 * 1048576 particles and 262144 markers per call (larger calls return HFSI_ERR_ARG and run
 * nothing).  Every call on a device uses that device's array: calls that overlap on one
 * device race.  Synchronises.  No reference counterpart: for callers that cannot allocate
 * device memory (code under stream capture, serving loops, harnesses that forbid it). */
int hfsi_scatter_marker_forces_static(const float* marker_position, const double* marker_force, int32_t marker_count,
                                      const float* particle_position, float* external_force, int32_t particle_count,
                                      float support_radius, hfsi_marker_scatter_report* report, void* stream);

typedef struct hfsi_marker_feedback_report {
  int32_t updated_marker_count;   /* markers with a weight sum above 1e-12 */
  int32_t invalid_marker_count;   /* the others (left unchanged)           */
  double max_marker_displacement; /* max |x_new - x_old| (float32 norm)     */
  double max_marker_speed;        /* max |v_new|                           */
} hfsi_marker_feedback_report;

/* Marker surface feedback: each marker with particles inside its support takes the
 * tent-weighted average velocity of those particles (float32) and moves by dt times it;
 * the others are left unchanged.  Replaces
 * HibmMpmSurfaceMarkers._update_surface_feedback_from_mpm_particles_kernel
 * (simulation_core/hibm_mpm.py:5013-5054), binned like hfsi_scatter_marker_forces (same pool).
 * marker_position [M][3] float32 (in/out), marker_velocity [M][3] float32 (out),
 * particle_position / particle_velocity [P][3] float32 (device).  Synchronises. */
int hfsi_marker_feedback(float* marker_position, float* marker_velocity, int32_t marker_count,
                         const float* particle_position, const float* particle_velocity, int32_t particle_count,
                         float support_radius, float dt, hfsi_marker_feedback_report* report, void* stream);

typedef struct hfsi_marker_geometry_report {
  int32_t geometry_updated_marker_count; /* moved markers that took a new normal and area       */
  int32_t geometry_invalid_marker_count; /* the rest (unmoved markers included)                 */
  double max_marker_normal_change;       /* max |n_new - n_old| (float32 norm)                   */
  double max_marker_area_change;         /* max |A_new - A_old|                                  */
} hfsi_marker_geometry_report;

/* hfsi_marker_feedback for surface particles: as there, and a moved marker whose support
 * holds particles with a surface normal of norm above 1e-12 and a positive area also takes
 * their weighted normal (normalised: the reciprocal of the norm times the sum) and their
 * weighted mean area, when the geometry weight sum and the summed normal's norm exceed 1e-12.
 * Replaces HibmMpmSurfaceMarkers._update_surface_feedback_from_mpm_surface_particles_kernel
 * (simulation_core/hibm_mpm.py:5098-5180).  marker_normal [M][3] and marker_area [M] float32
 * (in/out), particle_normal [P][3] and particle_area [P] float32.  Synchronises. */
int hfsi_marker_surface_feedback(float* marker_position, float* marker_velocity, float* marker_normal,
                                 float* marker_area, int32_t marker_count, const float* particle_position,
                                 const float* particle_velocity, const float* particle_normal,
                                 const float* particle_area, int32_t particle_count, float support_radius, float dt,
                                 hfsi_marker_feedback_report* report, hfsi_marker_geometry_report* geometry_report,
                                 void* stream);

/* Bin grid of the marker / particle calls above for particle bounds [lo3, hi3] (finite,
 * lo <= hi): cells of edge support_radius * 2^k for the smallest k with at most max_cells
 * cells, every axis holding floor(extent / edge) + 1 cells (extents in double).  Host only, no
 * device work.  No reference counterpart (exposed so that the sizing is testable on its own). */
int hfsi_hibm_bin_grid(const float* lo3, const float* hi3, float support_radius, int32_t max_cells, int32_t* dims3,
                       float* cell_edge);

/* ---- Fluid stress sampled at the surface markers ----------------------------------------------
 * HibmMpmSurfaceMarkers.sample_fluid_stress_to_marker_tractions (simulation_core/hibm_mpm.py:
 * 3710-4100).  The fields are the fluid solver's (cell-centred, k fastest). */
typedef struct hfsi_stress_fluid {
  int32_t nx, ny, nz;                /* >= 2 each                                               */
  const double* pressure;            /* [nx][ny][nz] float64                                    */
  const float* velocity;             /* [nx][ny][nz][3] float32 (read when viscosity > 0)      */
  const int32_t* obstacle;           /* [nx][ny][nz] int32, the projection obstacle            */
  const int32_t* sampling_obstacle;  /* NULL, or the obstacle view the samplers read instead   */
  const float* cell_face[3];         /* [n + 1] float32 per axis                               */
  const float* cell_center[3];       /* [n] float32 per axis                                   */
  const float* cell_width[3];        /* [n] float32 per axis                                   */
} hfsi_stress_fluid;

typedef struct hfsi_stress_markers {
  int32_t marker_count;
  const float* position;   /* [M][3] float32 (x_gamma_m)                         */
  const float* normal;     /* [M][3] float32 (n_gamma, unit)                      */
  const int32_t* region_id;/* [M]                                                 */
  double* traction;        /* [M][3] float64 out (t_gamma_pa)                    */
  int32_t* pressure_valid; /* [M] out: 1 where the marker's traction is valid     */
  int32_t* viscous_mode;   /* [M] out: 0 pressure only, 1 one-sided, 2 two-sided,
                              3 / 4 far-pressure closure with water on -n / +n,
                              5 / 6 one-sided region with water on -n / +n       */
} hfsi_stress_markers;

typedef struct hfsi_stress_options {
  double viscosity;                      /* Pa s, finite >= 0 (used as float32)            */
  int32_t two_sided_pressure;
  int32_t far_pressure_region_id;        /* -1: none                                       */
  float two_sided_probe_max_multiplier;  /* >= 3                                           */
  int32_t one_sided_pressure_region_id;  /* -1: none                                       */
  float one_sided_reference_pressure;    /* Pa                                             */
  float one_sided_probe_max_multiplier;  /* >= 3                                           */
  int32_t use_pressure_anchor_fallback;
  int32_t node_anchor_given;             /* the caller passed a node anchor field           */
  float far_pressure;                    /* Pa, the dry side of a closure-region marker     */
  float far_pressure_side_normal_sign;   /* -1, 0 or 1                                     */
  float far_pressure_inside_probe_max_multiplier; /* >= 3                                   */
} hfsi_stress_options;

typedef struct hfsi_stress_report {
  int32_t valid_marker_count;
  int32_t invalid_marker_count;
  double max_abs_traction;
  int32_t two_sided_pressure_marker_count;
  int32_t viscous_gradient_invalid_marker_count;
  int32_t two_sided_extended_marker_count;
  int32_t one_sided_pressure_marker_count;
  int32_t one_sided_extended_marker_count;
  int32_t one_sided_gradient_missing_marker_count;
  int32_t far_pressure_closed_marker_count;
  int32_t far_pressure_closed_extended_marker_count;
  int32_t far_pressure_outside_suppressed_marker_count;
  int32_t closure_gradient_missing_marker_count;
} hfsi_stress_report;

/* Marker tractions from the fluid stress, one thread per marker, with the reference's three
 * dispatches (hibm_mpm.py:3806-4062):
 *  - zero viscosity, no far-pressure region (id < 0), no anchors, no sampling view: the
 *    pressure-only kernel (2253-2433), t = -p n from the obstacle-masked trilinear pressure,
 *    or with two_sided_pressure the first fluid samples at 1, 2, 3 normal spacings on either
 *    side (t = (p_in - p_out) n, a one-sided region against its reference pressure);
 *  - two_sided_pressure off: the general kernel's one-sided branch (1305-1339, 2205-2251),
 *    t = -p n + mu (G + G^T) n with G the velocity gradient of 1043-1152, invalid when its
 *    stencil misses fluid;
 *  - two_sided_pressure on: the general kernel's two-sided walk (1340-1560), the extended
 *    inside walk of a far-pressure closure marker (1564-1640), the extended walk of the others
 *    when a probe maximum exceeds 3 (1669-1808) and the decision chain (1816-1946), then, when
 *    the viscosity is positive, the split viscous pass (3316-3708) adding mu (G + G^T) n from
 *    the gradients found along the walks.  The pressure-anchor fallback of this dispatch
 *    (1946-2190, which reads the anchors of the pressure-Neumann row assembly) is not built:
 *    a call with use_pressure_anchor_fallback returns HFSI_ERR_ARG ("not available") and runs
 *    nothing.
 * Float32 samplers without contraction, float64 pressure sums and tractions.  Synchronises
 * (the report is read back). */
int hfsi_sample_fluid_stress(const hfsi_stress_fluid* fluid, const hfsi_stress_markers* markers,
                             const hfsi_stress_options* options, hfsi_stress_report* report, void* stream);

/* force[m] = traction[m] * area[m] (float64 [M][3] times float32 [M]).  Replaces
 * HibmMpmSurfaceMarkers._compute_marker_forces_kernel (simulation_core/hibm_mpm.py:903-906). */
int hfsi_marker_compute_forces(const double* traction, const float* area, double* force, int32_t marker_count,
                               void* stream);

typedef struct hfsi_marker_force_report {
  double total_force[3], primary_force[3], secondary_force[3];
  double total_force_norm_sum, primary_force_norm_sum, secondary_force_norm_sum;
  double total_force_norm_max, primary_force_norm_max, secondary_force_norm_max;
  int32_t total_marker_count, primary_marker_count, secondary_marker_count;
  int32_t primary_stress_valid_marker_count, primary_stress_invalid_marker_count;
  int32_t secondary_stress_valid_marker_count, secondary_stress_invalid_marker_count;
} hfsi_marker_force_report;

/* Sums, norm sums and norm maxima of the marker forces over all markers and over the markers
 * of the primary / secondary region, with their counts and stress-valid counts.  Replaces
 * HibmMpmSurfaceMarkers._aggregate_region_forces_kernel (simulation_core/hibm_mpm.py:
 * 5240-5289); the sums are reduced in a fixed order (the reference adds with atomics).
 * force [M][3] float64, region_id and pressure_valid [M] int32.  Synchronises. */
int hfsi_marker_aggregate_forces(const double* force, const int32_t* region_id, const int32_t* pressure_valid,
                                 int32_t marker_count, int32_t primary_region_id, int32_t secondary_region_id,
                                 hfsi_marker_force_report* report, void* stream);

typedef struct hfsi_no_slip_report {
  int32_t valid_marker_count;   /* markers where the trilinear velocity sees fluid */
  int32_t invalid_marker_count;
  double max_residual;          /* max |u_fluid - v_marker| (float32 norm)          */
  double sum_residual2;         /* sum of the float32 squared residual norms        */
} hfsi_no_slip_report;

/* No-slip residual at the markers: the obstacle-masked trilinear fluid velocity at each
 * marker against the marker velocity.  Replaces
 * HibmMpmSurfaceMarkers._sample_no_slip_residual_kernel (simulation_core/hibm_mpm.py:
 * 4737-4792); reads fluid->velocity, obstacle, cell_face and cell_center only.
 * marker_position / marker_velocity [M][3] float32.  Synchronises. */
int hfsi_marker_no_slip_residual(const hfsi_stress_fluid* fluid, const float* marker_position,
                                 const float* marker_velocity, int32_t marker_count, hfsi_no_slip_report* report,
                                 void* stream);

/* ---- Mooney-Rivlin membrane shell MPM on a triangle mesh ------------------------------------
 * TriMooneyShellMpmState (simulation_core/mooney_shell_mpm.py:105-1392).  The handle holds the
 * mesh (faces, face regions, unique edges, the vertex -> incident-face table) and its
 * workspaces; the particle and grid arrays are the caller's.  Per-face corner forces are summed
 * per vertex in face order (deterministic); P2G adds into the grid with float atomics as the
 * reference does; every report value is a float64 sum or max. */
typedef struct hfsi_shell hfsi_shell;

/* The state arrays, device memory: particle [n][3] float32 x, rest_x, u, v, surface_normal,
 * internal_force, external_force; [n] float32 mass and area_weight, int32 vertex_region and
 * fixed; grid [nx][ny][nz] float32 grid_mass and [..][3] grid_velocity,
 * grid_velocity_before_force, grid_force; report_snapshot [37] float64, the packed report of
 * the last step (mooney_shell_mpm.py:337-392 layout: 32 values, then 5 counts). */
typedef struct hfsi_shell_state {
  float* x;
  const float* rest_x;
  float* u;
  float* v;
  float* mass;
  float* area_weight;
  float* surface_normal;
  float* internal_force;
  float* external_force;
  int32_t* vertex_region;
  int32_t* fixed;
  float* grid_mass;
  float* grid_velocity;
  float* grid_velocity_before_force;
  float* grid_force;
  double* report_snapshot;
} hfsi_shell_state;

/* Mooney constants (c1 > 0, c2 >= 0), the membrane force scale and the thicknesses. */
typedef struct hfsi_shell_material {
  float c1;
  float c2;
  float membrane_force_scale;
  float thickness;
  float primary_thickness;
  float secondary_thickness;
} hfsi_shell_material;

/* One step.  region_mode 0: _step_kernel (mooney_shell_mpm.py:860-1003), every face at
 * `thickness` with the internal pressure `pressure`.  region_mode 1: _step_region_kernel
 * (1005-1177): region thicknesses, the area load (per unit rest area) on faces of
 * area_load_region and the interface reactions spread over the primary / secondary faces by
 * rest area (region_area2: device float32 primary / secondary rest area), keeping the existing
 * external forces when preserve_external is set.  The report's region means use
 * report_primary_region / report_secondary_region.  uv_variant: the rules of
 * UvMooneyShellMpmState._step_kernel (mooney_shell_mpm.py:1948-2068) -- no clamp of C, determinant
 * floor 1e-12, no force cap, and a particle joins the centre sums when it was inside the grid
 * before its update. */
typedef struct hfsi_shell_step_args {
  float dt;
  float velocity_damping;
  float flip_blend;
  float body_acceleration[3];
  int32_t region_mode;
  float pressure;
  int32_t primary_region;
  int32_t secondary_region;
  int32_t area_load_region;
  float area_load[3];
  float primary_reaction[3];
  float secondary_reaction[3];
  int32_t preserve_external;
  const float* region_area2;
  int32_t report_primary_region;
  int32_t report_secondary_region;
  int32_t uv_variant;      /* UvMooneyShellMpmState's rules (below) */
  double* edge_count_out;  /* device, may be NULL: edges with both lengths above 1e-12 */
} hfsi_shell_step_args;

/* Mesh upload (host arrays: face_indices [faces][3], face_region [faces] or NULL for 0,
 * edge_indices [edges][2]) and the grid: nodes at bounds_min + i dx, float32.  Allocates. */
int hfsi_shell_create(hfsi_shell** out, int32_t particles, int32_t faces, const int32_t* face_indices,
                      const int32_t* face_region, int32_t edges, const int32_t* edge_indices, const int32_t* grid_nodes3,
                      const float* bounds_min3, const float* dx3, void* stream);
int hfsi_shell_destroy(hfsi_shell* h);
/* _init_mass_kernel (mooney_shell_mpm.py:480-541): particle mass and region from the incident
 * faces' rest areas, fixed flags, zero u / v / forces, the surface normals; region_area_mass4
 * (device float32): primary area, secondary area, primary mass, secondary mass.
 * mass_from_total_area: mass = density thickness (sum of the rest shares), the UV-sphere
 * variant's _init_kernel (1524-1553). */
int hfsi_shell_init_mass(hfsi_shell* h, const hfsi_shell_state* state, float thickness, float density,
                         int32_t primary_region, int32_t secondary_region, int32_t fixed_region,
                         float primary_thickness, float secondary_thickness, int32_t mass_from_total_area,
                         float* region_area_mass4, void* stream);
/* _update_particle_surface_normals (mooney_shell_mpm.py:437-462) from the current positions. */
int hfsi_shell_update_normals(hfsi_shell* h, const hfsi_shell_state* state, void* stream);
/* _add_region_area_load_kernel (mooney_shell_mpm.py:710-728): external force += load * rest area / 3
 * at each corner of the region's faces (load3 on the host). */
int hfsi_shell_add_region_area_load(hfsi_shell* h, const hfsi_shell_state* state, int32_t region, const float* load3,
                                    void* stream);
int hfsi_shell_step(hfsi_shell* h, const hfsi_shell_state* state, const hfsi_shell_material* material,
                    const hfsi_shell_step_args* args, void* stream);

/* ---- HIBM immersed-boundary node search ------------------------------------------------- */

/* The surface the nodes are searched against: marker positions and normals [M][3] float32 and
 * the projection triangles [T][3] (marker indices; NULL and 0 to search the markers
 * themselves), all device memory.  A triangle with an index outside [0, M) is skipped. */
typedef struct hfsi_ib_markers {
  const float* positions;
  const float* normals;
  const int32_t* triangles;
  int32_t marker_count;
  int32_t triangle_count;
} hfsi_ib_markers;

/* The per-node fields of HibmMpmIbNodeSearch (simulation_core/hibm_mpm.py:5420-5441), device
 * memory over the [nx][ny][nz] node grid: kind (0 none, 1 external IB, 2 internal), nearest
 * marker, signed distance, boundary point [3], interior fluid point [3], projection marker
 * indices [3] and weights [3]. */
typedef struct hfsi_ib_nodes {
  int32_t* kind;
  int32_t* nearest_marker;
  float* signed_distance;
  float* boundary_point;
  float* interior_point;
  int32_t* projection_indices;
  float* projection_weights;
} hfsi_ib_nodes;

/* _search_and_classify_kernel (center_x/y/z NULL: node (i, j, k) at bounds_min + (i + 0.5)
 * spacing, both host float3) and _search_and_classify_grid_fields_kernel (nodes at the device
 * cell-centre arrays) of simulation_core/hibm_mpm.py:5601-6058, same results and the same
 * float32 arithmetic, without the full node x triangle loop: each 4 x 8 x 8 node tile tests
 * only the triangles whose box, grown by the search radius, reaches the tile, and with
 * classify_far_internal_nodes only nodes without a near candidate walk every triangle,
 * stopping at the first that has them on its positive side.  report4 (device int32, written
 * on the stream): near-boundary, external IB, internal and invalid-projection node counts. */
int hfsi_ib_node_search(int32_t nx, int32_t ny, int32_t nz, const float* bounds_min3, const float* spacing3,
                        const float* center_x, const float* center_y, const float* center_z,
                        const hfsi_ib_markers* markers, float search_radius, float interior_probe_distance,
                        float sign_tolerance, int32_t classify_far_internal_nodes, const hfsi_ib_nodes* out,
                        int32_t* report4, void* stream);

/* Live kernel timing (no reference counterpart; measurement support):
 * while enabled, HIP events are recorded on the launch stream around every
 * launch of the selected level-0 kernel and their elapsed times summed.
 * kernel_id 0 disables. */
#define HFSI_TIMER_OFF 0
#define HFSI_TIMER_L0_SWEEP 1         /* level-0 weighted-Jacobi sweep (not the first, not the prolongating one) */
#define HFSI_TIMER_SPMV_DOT 2         /* q = A d with <d, q>_V                                                   */
#define HFSI_TIMER_L0_RESTRICT 3      /* level-0 residual + restriction                                          */
#define HFSI_TIMER_L0_PROLONG_SWEEP 4 /* level-0 prolongation fused into the first post-smoothing sweep          */
#define HFSI_TIMER_MIX_RB 5           /* mixed V-cycle: level-0 red-black colour pass (not the first from zero)  */
#define HFSI_TIMER_CG_UPDATE 6        /* mixed solve: x += alpha d, r -= alpha q with <r,r>_V                    */
#define HFSI_TIMER_PREDICT 7          /* velocity predictor (hfsi_fluid_predict)                                 */
int hfsi_fluid_kernel_timer(hfsi_fluid* h, int32_t kernel_id);
/* Synchronises on the recorded events; totals since the last enable. */
int hfsi_fluid_kernel_timer_read(hfsi_fluid* h, int64_t* launches, double* total_ms);

#ifdef __cplusplus
}
#endif
#endif /* HFSI_H */
