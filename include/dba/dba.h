/*
 * dba.h - C ABI of the MI355X dynamic-block-activation (DBA) time step.
 *
 * This is the only way into the HIP path. It carries no HIP or torch types:
 * plain pointers, sizes and POD structs, so the C++ drop-in drivers, ctypes,
 * cgo or JNI can bind it unchanged.
 *
 * What each entry point replaces in the reference (zhangruoyao68/DBA):
 *
 *   dba_init / dba_finalize
 *       cudaSetDevice + the per-run setup of main()
 *       (example_Dendritic_growth/kernel.cu:881-896,
 *        example_Reactive_ModelB/kernel.cu:1012-1029,
 *        example_Kelvin_Helmholtz/KH_DBA.cu:1329-1346).
 *   dba_instance_create / dba_instance_destroy
 *       ReadInput's derived constants + Allocate + FreeMemory
 *       (example_Dendritic_growth/kernel.cu:67-135, 866-879;
 *        example_Reactive_ModelB/kernel.cu:90-170;
 *        example_Kelvin_Helmholtz/KH_DBA.cu:88-221).
 *       All tiles start awake, as Initialize does
 *       (example_Dendritic_growth/kernel.cu:149-161).
 *   dba_upload
 *       the field writes of the Initialize kernels
 *       (example_Dendritic_growth/kernel.cu:138-178,
 *        example_Reactive_ModelB/kernel.cu:173-238,
 *        example_Kelvin_Helmholtz/KH_DBA.cu:1047-1130 + getConserved :335-372).
 *       Initial conditions are generated by the caller and uploaded.
 *   dba_step
 *       one iteration of the time loop, repeated n_steps times:
 *       dendrite  Evolve_p_wakeup/Evolve_T_wakeup/Wakeup_Next/Wakeup_Neighbor
 *                 (example_Dendritic_growth/kernel.cu:946-987, regular :916-945);
 *       Model B   Calc_mu_wakeup/Update_wakeup/Swap_wakeup/Wakeup_Next/Wakeup_Neighbor
 *                 (example_Reactive_ModelB/kernel.cu:1091-1132, regular :1060-1090);
 *       Model B conserved adds the change sums and Conservation
 *                 (example_Reactive_ModelB/Conserved/kernel.cu:1128-1187);
 *       KH        getPrimitive_wakeup/extrap_in_time_wakeup/calc_flux_wakeup/
 *                 apply_flux_wakeup/Wakeup_Next/Wakeup_Neighbor
 *                 (example_Kelvin_Helmholtz/KH_DBA.cu:1436-1500, regular :1387-1435);
 *       KH conserved (example_Kelvin_Helmholtz/Conserved/KH_DBA.cu:1553-1575).
 *       Several ids in one call are stepped together over one merged worklist.
 *   dba_download
 *       the host reads of managed memory after cudaDeviceSynchronize that feed
 *       the VTK writers and diagnostics (example_Dendritic_growth/kernel.cu:990-1010,
 *       example_Reactive_ModelB/kernel.cu:1140-1159).
 *   dba_active_tiles / dba_active_history
 *       the wake-up flag arrays read by Calc_RealTime_Values and Output_wakeup
 *       (example_Dendritic_growth/kernel.cu:840-852, 711-757).
 *   dba_last_error
 *       CUDACHECK / CheckLastCudaError, which print and exit(1)/exit(2)
 *       (example_Dendritic_growth/kernel.cu:12-29). Here errors are returned;
 *       the drop-in drivers map DBA_ERR_HIP to exit code 1 and DBA_ERR_LAUNCH to 2.
 *
 * Threading: a dba_ctx is owned by one host thread. Calls are asynchronous
 * until dba_download / dba_sync / dba_active_* (which synchronise).
 */
#ifndef DBA_DBA_H
#define DBA_DBA_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct dba_ctx dba_ctx;
typedef int32_t dba_status;

/* Status codes. */
#define DBA_OK             0
#define DBA_ERR_INVALID   -1  /* bad argument or parameter combination */
#define DBA_ERR_HIP       -2  /* HIP API error (reference exit code 1) */
#define DBA_ERR_LAUNCH    -3  /* kernel launch error (reference exit code 2) */
#define DBA_ERR_NOMEM     -4  /* device allocation failed */
#define DBA_ERR_NOTFOUND  -5  /* unknown instance id */
#define DBA_ERR_NUMERIC   -6  /* non-finite value detected by dba_check_finite */

/* Models. */
#define DBA_MODEL_DENDRITE_K94  1  /* reference 3D Kobayashi-94 dendrite, example_Dendritic_growth/kernel.cu:181-293 */
#define DBA_MODEL_DENDRITE_K93  2  /* 2D Kobayashi-93 anisotropic dendrite with latent heat K */
#define DBA_MODEL_MODELB        3  /* reference ternary Flory-Huggins + reaction, example_Reactive_ModelB/kernel.cu:349-437 */
#define DBA_MODEL_CH            4  /* 2D Cahn-Hilliard + linear reaction (reactive Model B) */
#define DBA_MODEL_KH            5  /* 2D compressible Euler, MUSCL-Hancock + Rusanov, example_Kelvin_Helmholtz/KH_DBA.cu:335-923 */

/* Modes. */
#define DBA_MODE_REGULAR    0  /* every tile every step (reference mode 0) */
#define DBA_MODE_DBA        1  /* dynamic block activation (reference mode 1) */
#define DBA_MODE_CONSERVED  2  /* DBA + uniform mean correction (reference Conserved/ variants) */

/* Boundary conditions, per axis. */
#define DBA_BC_PERIODIC  0  /* wrap (reference default) */
#define DBA_BC_NOFLUX    1  /* mirror about the boundary face: f(-1-k) = f(k) */
#define DBA_BC_WALL      2  /* KH reflective wall: mirror, normal velocity negated */

/* KH time-step and detector choices. */
#define DBA_DT_FIXED  0
#define DBA_DT_CFL    1
#define DBA_KH_METRIC_ALLGRAD 0  /* sum of the 8 |gradients| (example_Kelvin_Helmholtz/KH_DBA.cu:614-617) */
#define DBA_KH_METRIC_DENSITY 1  /* |rho_x| + |rho_y| (example_Kelvin_Helmholtz/KH_DBA.cu:618) */

/* Field ids for dba_upload / dba_download. */
#define DBA_F_PHI   0  /* dendrite p (phase field) */
#define DBA_F_T     1  /* dendrite T */
#define DBA_F_C     0  /* CH concentration c */
#define DBA_F_X     0  /* Model B x, y, z, phi */
#define DBA_F_Y     1
#define DBA_F_Z     2
#define DBA_F_MBPHI 3
#define DBA_F_MASS  0  /* KH conserved Mass, Momx, Momy, Energy (cell integrals, vol = dx*dy) */
#define DBA_F_MOMX  1
#define DBA_F_MOMY  2
#define DBA_F_ENERGY 3

/* Activation sets. */
#define DBA_SET_MAIN 0  /* p (dendrite), c, x/y/z, U */
#define DBA_SET_T    1  /* dendrite T set */

/*
 * One simulation instance. Fields that a model does not use are ignored.
 * Constants follow the reference's names (InputPara in each example).
 */
typedef struct dba_params {
    int32_t model;
    int32_t mode;
    int32_t nx, ny, nz;
    int32_t tile_x, tile_y, tile_z;   /* activation block; reference: 4x4x4 (D, M), 8x8x1 (K) */
    int32_t bc_x, bc_y, bc_z;
    int32_t stencil;                  /* CH Laplacian: 5 or 9 points */
    int32_t aniso_j;                  /* K93 anisotropy mode j */
    int32_t dt_mode;                  /* KH: DBA_DT_FIXED or DBA_DT_CFL */
    int32_t metric_kind;              /* KH detector */
    int32_t threads;                  /* workgroup size 64/128/256 (CH, K93 also 512/1024), 0 = default
                                         (single-launch K93 16x16: 512, 256 or 128 by grid size) */
    int32_t history_cap;              /* steps of per-step active counts kept on device */
    int32_t reserved_i;
    double dx, dy, dz, dt;
    double thresh_a;                  /* dendrite Metric_p; Model B / CH / KH Metric_eps */
    double thresh_b;                  /* dendrite Metric_T */
    /* dendrite: K94 uses delta, tau, eps_bar(=epsilon), alpha, gamma;
       K93 adds theta0, latent_k (K), t_eq. */
    double tau, eps_bar, delta, alpha, gamma, theta0, latent_k, t_eq;
    /* CH: dc/dt = M lap(c^3 - c - kappa lap c) - react_gamma (c - cbar) */
    double mobility, kappa, react_gamma, cbar;
    /* Model B ternary (example_Reactive_ModelB/kernel.cu:52-62) */
    double chi_xy, chi_xz, chi_yz, chi_xb, chi_yb, chi_zb;
    double v_x, v_y, v_z, r_x, r_y, r_z, n_exp, m_exp;
    double epsx_sq, epsy_sq, epsz_sq, epsphi_sq;
    double mob_x, mob_y, mob_z, mob_phi;
    double k_eq, z_crit, p_gel, k_0;
    /* KH */
    double gas_gamma, cfl;
} dba_params;

/* Per-instance state summary. */
typedef struct dba_info {
    int64_t steps_done;
    int32_t ntiles;            /* tiles in the activation grid */
    int32_t ntiles_x, ntiles_y, ntiles_z;
    double  sim_time;          /* accumulated time (KH: sum of dt) */
    double  last_dt;
    double  cons_offset;       /* conserved: cumulative mean correction applied */
    int64_t footprint_bytes;   /* device bytes held by this instance */
    int64_t cell_updates;      /* active cell-updates performed so far (device count):
                                  field_updates / number of field sets */
    int32_t single_launch;     /* 1: stepped alone, the instance takes single-launch steps */
    int32_t reserved;
    int64_t field_updates;     /* cells x field sets advanced: per step, the cells of the
                                  tiles that ran set 0 (all fields of CH, Model B, KH;
                                  dendrite phi) plus, for the dendrite, the cells of the
                                  tiles that ran either set (T is written in p-awake
                                  tiles, example_Dendritic_growth/kernel.cu:479-490) */
} dba_info;

/* Context. */
dba_status dba_init(int32_t device, dba_ctx** out);
dba_status dba_finalize(dba_ctx* ctx);
const char* dba_last_error(void);

/* Device bytes an instance with these parameters would hold (admission control). */
dba_status dba_footprint(const dba_params* p, int64_t* bytes);

/* Free and total device memory of the context's GPU (hipMemGetInfo), for
   admission against HBM capacity. No reference counterpart: the reference runs
   one simulation per process; callers are batching and serving loops. */
dba_status dba_device_memory(dba_ctx* ctx, int64_t* free_bytes, int64_t* total_bytes);

/* Instances. */
dba_status dba_instance_create(dba_ctx* ctx, const dba_params* p, int32_t* id);
dba_status dba_instance_destroy(dba_ctx* ctx, int32_t id);
dba_status dba_instance_info(dba_ctx* ctx, int32_t id, dba_info* out);

/* Field transfer. n must equal nx*ny*nz. Upload resets nothing else; all
   tiles are awake after create. Download synchronises. */
dba_status dba_upload(dba_ctx* ctx, int32_t id, int32_t field, const double* host, size_t n);
dba_status dba_download(dba_ctx* ctx, int32_t id, int32_t field, double* host, size_t n);

/* Advance instances n_steps. Instances in one call share one merged worklist
   per model and one launch per step; they must be distinct. */
dba_status dba_step(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, int32_t n_steps);

/* Same, but replayed from a captured hipGraph of `chunk` steps (chunk >= 1). */
dba_status dba_step_graph(dba_ctx* ctx, const int32_t* ids, int32_t n_ids, int32_t n_steps, int32_t chunk);

dba_status dba_sync(dba_ctx* ctx);

/* Single-launch steps. A group whose instances all have a single-launch kernel
 * (reactive CH and the Kobayashi-93 dendrite, regular or DBA mode; conserved DBA
 * for one CH instance of at most 1024 tiles, whose workgroups each recompute the
 * previous step's mean shift in the finalize's order) steps with one launch per
 * step instead of the step kernel plus the finalize
 * of the reference's Wakeup_Next / Wakeup_Neighbor pair
 * (example_Reactive_ModelB/kernel.cu:1094-1131): one workgroup per tile of every
 * instance derives its awake bit and buffer parity from the previous step's
 * per-tile bytes, and a canonicalising kernel (two for several instances or more
 * than 1024 tiles) at the end of each dba_step / graph chunk restores the
 * bitmaps, counters and time. Sleeping tiles still take a workgroup each, so a
 * sparse batch can run faster on the worklist path.
 * A call of 12 steps or more for one reactive CH or K93 instance (threads 0, no timing) whose
 * tiles fit the GPU at once, by a context alone on its device in this process, takes
 * resident steps in modes 1 and 2: all its steps in one cooperative launch that keeps
 * the fields on chip. (A context that is not finalised counts as one on its device.)
 * One process at a time has the GPU's queue for such launches; a context of another one
 * is refused its first and keeps to the other paths.
 * Such a launch needs all its workgroups on the GPU together. Where something else, such
 * as another process, keeps some of them off it, the others wait for about a second
 * (dba_set_resident_wait) and then give the launch up, which leaves the instance as it
 * was; the next call that waits for the GPU has its steps made on the other paths, and
 * the context keeps to those until dba_set_resident.
 * mode 0: worklist path for every group; 1 (default): single-launch steps for
 * groups of one instance; 2: also for batches. Results are bit-identical in every
 * mode. DBA_ERR_INVALID for another mode. */
dba_status dba_set_single_launch(dba_ctx* ctx, int32_t mode);

/* Resident steps of this context: 0 keeps it on the paths that launch every step,
 * not 0 (the default) takes resident steps where dba_set_single_launch's text says.
 * Results are bit-identical. */
dba_status dba_set_resident(dba_ctx* ctx, int32_t enable);

/* How often a workgroup of a resident step looks for a word of another one (each look
 * is a trip to memory, about a microsecond) before it gives the wait up; 0: the default. */
dba_status dba_set_resident_wait(dba_ctx* ctx, int32_t polls);

/* How many dba_step / dba_step_graph calls of this context took resident steps, and how
 * many of their steps were given up and made again on the other paths. */
dba_status dba_resident_calls(dba_ctx* ctx, int64_t* taken);
dba_status dba_resident_redone(dba_ctx* ctx, int64_t* steps);

/* Active tiles of a set for the NEXT step (after dilation). mask (optional)
   receives ntiles bytes, 1 = awake. Synchronises. */
dba_status dba_active_tiles(dba_ctx* ctx, int32_t id, int32_t set, int32_t* count, uint8_t* mask);

/* Compacted worklist of the next step for one instance, ascending tile ids
   (the order std::copy_if over tile indices gives). Synchronises. */
dba_status dba_worklist(dba_ctx* ctx, int32_t id, int32_t* tiles, int32_t cap, int32_t* count);

/* Active-tile count per executed step (set 0 and, dendrite, set 1), as recorded
   on device; counts[2*i + set]. Synchronises. */
dba_status dba_active_history(dba_ctx* ctx, int32_t id, int32_t* counts, int32_t max_steps, int32_t* n_steps);

/* Kernel timing: when enabled, every step kernel launch is bracketed by
   hipEvents on the library stream; query returns the summed milliseconds
   and launch count of the stencil (step) kernels since enable. */
dba_status dba_timing_enable(dba_ctx* ctx, int32_t enable);
dba_status dba_timing_query(dba_ctx* ctx, double* step_kernel_ms, int64_t* step_kernel_launches,
                            double* compact_kernel_ms, int64_t* compact_kernel_launches);

/* Wall time of the stream between two markers (hipEvents on the library stream). */
dba_status dba_marker(dba_ctx* ctx, int32_t slot);
dba_status dba_marker_elapsed(dba_ctx* ctx, int32_t slot_a, int32_t slot_b, double* ms);

/* Returns DBA_ERR_NUMERIC if any current field value of the instance is not finite. */
dba_status dba_check_finite(dba_ctx* ctx, int32_t id);

/* Diagnostics on the device (no field download); each synchronises.
   Sum of a field's current values over all cells, in a fixed order
   (replaces Integral, example_Reactive_ModelB/kernel.cu:989-1009 and
   example_Kelvin_Helmholtz/KH_DBA.cu:1273-1288, host loops over managed memory). */
dba_status dba_field_sum(dba_ctx* ctx, int32_t id, int32_t field, double* sum);

/* Dendrite growth front at columns xs[0..n), n <= 64: scanning up from Ny/2 at
   z = Nz/2, the first phi < 0.5 interpolated with the cell below, minus Ny/2;
   0 if none (growth_front / tip_curvature, example_Dendritic_growth/kernel.cu:760-790). */
dba_status dba_growth_front(dba_ctx* ctx, int32_t id, const int32_t* xs, int32_t n, double* front);

/* KH growth-mode amplitude of vy (Calc_Vy_mode, example_Kelvin_Helmholtz/KH_DBA.cu:1291-1326). */
dba_status dba_kh_vy_mode(dba_ctx* ctx, int32_t id, double* amplitude);

/* Droplet (coarsening) analysis of a field on the device, the rule of
 * example_Reactive_ModelB/coarsening_analysis.cpp:48-170 (which reads a 256^3 VTK
 * file on the host): threshold avg = (max(0.5, max v) + min(0.5, min v)) / 2;
 * a droplet is a periodic face-connected component (6 neighbours in 3D, 4 in 2D)
 * of cells with !(v < avg) that holds a cell with v > avg; volume = cells with
 * v > avg. Writes the droplet count and, when cap > 0, the first cap droplet
 * sizes in the reference's order (by each droplet's first cell v > avg in index
 * order, x fastest). The mean radius is cbrt(3 volume / (4 pi n)) in 3D and
 * sqrt(volume / (pi n)) in 2D (coarsening_analysis.cpp:170). Grids below 2^31
 * cells; allocates 13 bytes per cell of device scratch for the call. */
dba_status dba_droplets(dba_ctx* ctx, int32_t id, int32_t field, double* avg, int64_t* volume,
                        int64_t* n_droplets, int64_t* sizes, int64_t cap);

/* dba_droplets without any allocation: no counterpart in the reference; for
 * callers that cannot allocate device memory (tight serving loops, harnesses
 * that forbid hipMalloc). Same arguments and results as dba_droplets; every
 * buffer lives in a static device array of 13 * 2^22 + 64 KiB bytes per GPU
 * (held from the library's load until the process ends), so grids of at most
 * 4,194,304 cells (2048^2, 161^3) are accepted and larger ones fail with
 * DBA_ERR_INVALID. The host side allocates nothing either: the droplet order
 * is built on the device. All calls on one GPU share the array: calls that
 * overlap on one GPU (two contexts, two threads) race. Synchronises. */
dba_status dba_droplets_noalloc(dba_ctx* ctx, int32_t id, int32_t field, double* avg, int64_t* volume,
                                int64_t* n_droplets, int64_t* sizes, int64_t cap);

#ifdef __cplusplus
}
#endif
#endif /* DBA_DBA_H */
