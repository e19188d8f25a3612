/*
 * imexlb.h -- C ABI of the MI355X lattice Boltzmann time step.
 *
 * The reference (IMEXLB-1.0) exposes this path as argument-less Fortran
 * module procedures acting on module variables (lbm.f90, initialization.f90,
 * cart_mpi.f90).  Each entry point below replaces one of them; the Fortran
 * module shims in imexlb-1.0_amd/fortran bind these with ISO_C_BINDING so the
 * reference's main.f90 call sequence drives the GPU unchanged.
 *
 * Conventions
 *  - Every function returns IMEXLB_OK (0) or a negative IMEXLB_E_* code;
 *    imexlb_strerror() describes it and imexlb_last_error() gives details.
 *  - Inputs are copied; the caller keeps ownership of every pointer.
 *  - A context owns all of its device memory and one HIP stream.  It is not
 *    thread-safe.  Calls enqueue work asynchronously; imexlb_monitor and the
 *    download functions synchronise.
 *  - "Reference layout" (IMEXLB_LAYOUT_REF) is the reference's own host
 *    layout: a flat array over array_size = prod(n_d+7) cells with a
 *    3-wide ghost shell, cell id = (x+3) + dy*(y+3) [+ dz*(z+3)],
 *    dy = nx+7, dz = (nx+7)*(ny+7); populations AoS f[id*nq+q]
 *    (lbm.f90:44), velocity AoS u[id*dim+d] (lbm.f90:34).
 *    "Interior layout" (IMEXLB_LAYOUT_INTERIOR) is structure-of-arrays over
 *    the (nx+1)(ny+1)[(nz+1)] interior nodes, x fastest: f[q][z][y][x],
 *    p[z][y][x], u[d][z][y][x].
 *  - Lattice numbering is the reference's (initialization.f90:112-123;
 *    initialization_3d.f90:108-122): D2Q9 q=(ex+1)*3+(ey+1),
 *    D3Q27 q=(ez+1)*9+(ex+1)*3+(ey+1); the opposite of q is nq-1-q.
 */
#ifndef IMEXLB_H
#define IMEXLB_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct imexlb_ctx imexlb_ctx;

/* status codes */
#define IMEXLB_OK 0
#define IMEXLB_E_ARG (-1)    /* invalid argument or size                      */
#define IMEXLB_E_HIP (-2)    /* HIP runtime error                             */
#define IMEXLB_E_OOM (-3)    /* device or host allocation failed              */
#define IMEXLB_E_STATE (-4)  /* call out of the Collision..PostProcessing order */
#define IMEXLB_E_UB (-5)     /* the reference's result depends on a read past
                                the end of its arrays (undefined there)       */
#define IMEXLB_E_NODEV (-6)  /* compute call on a host-only context (device<0) */
#define IMEXLB_E_NAN (-7)    /* Monitor found a non-finite velocity: the
                                lattice has diverged                          */

/* storage / arithmetic forms */
#define IMEXLB_F64 0       /* FP64 storage and arithmetic in the reference's
                              operation order: results equal the reference's */
#define IMEXLB_F32 1       /* FP32 storage, FP32 arithmetic                  */
#define IMEXLB_F16_F32 2   /* FP16 storage of f, FP32 arithmetic              */
#define IMEXLB_BF16_F32 3  /* BF16 storage of f, FP32 arithmetic              */
#define IMEXLB_BF16SR_F32 4 /* BF16 storage of f with stochastic rounding (no
                               rounding bias, more noise), FP32 arithmetic;
                               deterministic: runs repeat bit for bit        */

#define IMEXLB_LAYOUT_REF 0
#define IMEXLB_LAYOUT_INTERIOR 1

#define IMEXLB_PDF_F 0   /* post-propagation populations  (array f)  */
#define IMEXLB_PDF_FB 1  /* post-collision populations    (array fb) */

/* list identifiers for imexlb_geometry_size / imexlb_geometry_list, in the
 * reference's names (initialization.f90:44-50; initialization_3d.f90:44-50) */
#define IMEXLB_LIST_FLUID 0
#define IMEXLB_LIST_BL 1
#define IMEXLB_LIST_BR 2
#define IMEXLB_LIST_BU 3
#define IMEXLB_LIST_BD 4
#define IMEXLB_LIST_BF 5
#define IMEXLB_LIST_BB 6
#define IMEXLB_LIST_USER 7

const char *imexlb_strerror(int code);
/* text of the most recent error raised on this thread */
const char *imexlb_last_error(void);

/* omp_get_num_devices() as main.f90:31 uses it: number of visible GPUs. */
int imexlb_device_count(int *n);

/* MPISetup + InitLattice + AllocateArrays at one rank
 * (cart_mpi.f90:47-138, initialization.f90:112-144; _3d counterparts).
 * dim 2 (D2Q9, nz ignored) or 3 (D3Q27); n* are the largest node indices
 * (nodes per axis = n+1, cart_mpi.f90:63-64).  device >= 0 selects the GPU
 * (omp_set_default_device, main.f90:32); device = -1 makes a host-only
 * context on which only the geometry functions work. */
int imexlb_create(imexlb_ctx **ctx, int dim, int nx, int ny, int nz, int device, int precision);
/* DeAllocateArrays + TARGET EXIT DATA (initialization.f90:148-163, main.f90:75) */
int imexlb_destroy(imexlb_ctx *ctx);

/* Scalars DataInput derives and the kernels use (initialization.f90:59-81):
 * relaxation parameter ome, density rho0, inlet velocity scale uu. */
int imexlb_set_params(imexlb_ctx *ctx, double ome, double rho0, double uu);

/* SetGeometry (initialization.f90:167-255; initialization_3d.f90:170-279):
 * cylinder/sphere mask centred at (pos, ny/2[, nz/2]), boundary lists,
 * PassInt(geo), the body list b_user, and the device boundary tables. */
int imexlb_set_geometry(imexlb_ctx *ctx, double pos, double radius);
/* SetGeometry with an elliptic body (2D; no counterpart in the reference,
 * for the warm-start study): the ellipse of the same area as the circle of
 * `radius`, axis ratio `aspect` (semi-axes radius*sqrt(aspect) along its
 * axis and radius/sqrt(aspect) across), axis turned by angle_deg from x.
 * aspect 1, angle 0 is imexlb_set_geometry.  Everything after the mask
 * (lists, body scan, tables) follows the reference's rules unchanged. */
int imexlb_set_geometry_shape(imexlb_ctx *ctx, double pos, double radius, double aspect, double angle_deg);
/* Sizes / contents of the lists SetGeometry builds, as 0-based reference
 * cell ids (int32, like the reference's integer arrays). */
int imexlb_geometry_size(imexlb_ctx *ctx, int list, int64_t *n);
int imexlb_geometry_list(imexlb_ctx *ctx, int list, int32_t *out, int64_t cap);
/* geo over array_size cells (reference layout, ghost shell included) */
int imexlb_geometry_geo(imexlb_ctx *ctx, int32_t *geo, int64_t cap);
/* Resolved boundary table: for every (cell, q) slot that a fluid node
 * pulls from a ghost cell or a body cell, the reference slot id*nq+q and
 * the interior fluid slot its value comes from after PassF and the five
 * boundary phases (-1: the slot holds 0).  stats: [0] slots, [1] reads
 * that depend on the order inside one boundary phase. */
int imexlb_bc_table(imexlb_ctx *ctx, int64_t *slot, int64_t *src, int64_t cap, int64_t stats[2]);

/* InitUP (initialization.f90:259-282; initialization_3d.f90:282-308) with
 * the caller's 100 random numbers (the reference's r_vec(0:99)). */
int imexlb_init_up(imexlb_ctx *ctx, const double *r_vec);
/* Warm start: replace p and u (layout IMEXLB_LAYOUT_*), e.g. with a
 * predicted field; follow with imexlb_init_pdf (lbm.f90:24-48). */
int imexlb_upload_fields(imexlb_ctx *ctx, const double *p, const double *u, int layout);
/* Warm start of a 2D lattice from device memory (no counterpart in the
 * reference; for callers whose predicted fields are already on the GPU):
 * fields is a device FP32 stack [3][H][W] of p, u_x, u_y at node rows
 * y < H and columns x < W (nodes beyond take the last row and column);
 * p = p_scale f0, u_x = u_scale f1 r, u_y = u_scale f2, 0 on body nodes,
 * with r InitUP's perturbation factor 1 + 0.4 (r_vec[id mod 100] - 0.5)
 * (initialization.f90:273) when r_vec is given (NULL: r = 1).  Follow
 * with imexlb_init_pdf.  The stack must be complete: the call does not wait
 * for work on other streams. */
int imexlb_init_fields_f32(imexlb_ctx *ctx, const float *fields, int H, int W, double p_scale, double u_scale,
                           const double *r_vec);
/* Body mask of a 2D lattice into device memory (no counterpart in the
 * reference; the input of a field predictor): out[y W + x] = 1 on body
 * nodes, 0 on fluid nodes, for node rows y < H <= ny+1 and columns
 * x < W <= nx+1.  Asynchronous on the context's stream (imexlb_synchronize
 * before other streams read it). */
int imexlb_body_mask_f32(imexlb_ctx *ctx, float *out, int H, int W);
/* InitPDF (lbm.f90:24-48): f = feq(p, u) on fluid nodes. */
int imexlb_init_pdf(imexlb_ctx *ctx);

/* The four phases of one time step, main.f90:57-61.  In fused mode, on a
 * lattice whose step writes its own boundary copies, the step's kernel is
 * queued rather than launched by PostProcessing: queued steps run together
 * once 7 to 19 are pending (by size) and before any other call that launches work
 * or reads device state (so results are the same; an error of such a launch
 * is returned by the call that runs it).  set_params after a fused step
 * relaxes the next Collision with the new parameters, as the reference. */
int imexlb_collision(imexlb_ctx *ctx);           /* Collision          lbm.f90:52-76   */
int imexlb_boundary_condition(imexlb_ctx *ctx);  /* BoundaryCondition  lbm.f90:96-155,
                                                    incl. PassF        cart_mpi.f90:240 */
int imexlb_propagation(imexlb_ctx *ctx);         /* Propagation        lbm.f90:80-92   */
int imexlb_post_processing(imexlb_ctx *ctx);     /* PostProcessing     lbm.f90:159-201 */

/* Choose how the four phases execute: fused = 1 (default) runs
 * Propagation+PostProcessing+next Collision as one pull kernel and
 * materialises f/p/u only when read; fused = 0 runs one kernel per phase.
 * Both give identical results. */
int imexlb_set_fused(imexlb_ctx *ctx, int fused);

/* nsteps complete iterations (Collision, BoundaryCondition, Propagation,
 * PostProcessing), i.e. nsteps trips of the loop body at main.f90:48-63
 * without the Monitor call. */
int imexlb_advance(imexlb_ctx *ctx, int64_t nsteps);

/* Monitor's local maximum (lbm.f90:205-217): max over fluid entries 1..F-1
 * of sqrt(ux^2+uy^2).  Synchronises.  If any of those entries has a
 * non-finite ux^2+uy^2 (NaN or infinity: the lattice has diverged), *um is
 * set to NaN and the call returns IMEXLB_E_NAN, with the number of such
 * nodes in imexlb_last_error(); the reference's max() would instead print
 * whatever its NaN handling gives (lbm.f90:214). */
int imexlb_monitor(imexlb_ctx *ctx, double *um);

/* Force on the body by momentum exchange, in lattice units, for the most
 * recent BoundaryCondition: sum over fluid nodes x and directions q with an
 * interior solid neighbour x+e_q of e_q (fb(x,q) + fb(x+e_q, nq-1-q)).
 * F[0] is the drag (along the inlet flow), F[1] (and F[2] in 3D) the lift.
 * No counterpart in the reference, whose Monitor (lbm.f90:205-227) logs
 * only the maximum speed; FP64 accumulation, deterministic order.
 * Synchronises. */
int imexlb_forces(imexlb_ctx *ctx, double F[3]);

/* Mass check: sum over fluid nodes of sum_q f_q of the current populations
 * f (the density deviation; the reference's p is that sum over 3,
 * lbm.f90:178), accumulated in FP64 from every storage form, in an order
 * that depends on the lattice only.  No counterpart in the reference.
 * Synchronises. */
int imexlb_mass(imexlb_ctx *ctx, double *m);

/* TARGET UPDATE from(u,p) (lbm.f90:244): p and u of the current state. */
int imexlb_download_fields(imexlb_ctx *ctx, double *p, double *u, int layout);
/* f (IMEXLB_PDF_F) or fb (IMEXLB_PDF_FB) of the current state, as FP64.
 * Reference layout writes interior cells only; fb ghost values are the
 * resolved ones where a fluid node reads them. */
int imexlb_download_pdf(imexlb_ctx *ctx, int which, double *out, int layout);

/* Wait for all work queued on the context's stream. */
int imexlb_synchronize(imexlb_ctx *ctx);

/* Kernel timing with HIP events on the context stream.  While enabled,
 * every launch is bracketed by events; imexlb_profile_read returns, for
 * kernel class k (0 fused step, 1 boundary fill, 2 other), the launch count
 * and the summed milliseconds since the last reset.  A pass that makes several
 * steps counts as so many launches. */
int imexlb_profile(imexlb_ctx *ctx, int enable);
int imexlb_profile_read(imexlb_ctx *ctx, int64_t launches[3], double ms[3]);

/* Sizes: [0] interior nodes, [1] fluid nodes, [2] bytes of one population
 * array on the device, [3] device bytes allocated, [4] storage bytes per
 * population value, [5] boundary-table entries. */
int imexlb_info(imexlb_ctx *ctx, int64_t out[6]);

/* How the fused steps of imexlb_advance and of the queued phase calls run on
 * this lattice, as SetGeometry chose (results do not depend on it): [0] the
 * most steps one pass over the lattice makes (1; 2; 3 to 9: several per
 * launch, in windows), [1], [2] a window's cells along x and y (0 without
 * windows), [3] cells of a padded row. */
int imexlb_step_form(imexlb_ctx *ctx, int32_t out[4]);

/* ---------------------------------------------------------------------
 * Batched ensemble.  No counterpart in the reference, which runs one
 * lattice per process: ncase independent D2Q9 lattices, each with its own
 * size and parameters, advanced together, several steps per launch where every
 * case suits that, else by one step launch per time step (pairs of steps
 * replayed as a HIP graph).  Every case follows the single-lattice semantics
 * above exactly.
 * --------------------------------------------------------------------- */
typedef struct imexlb_batch imexlb_batch;

/* nxny[2*i..2*i+1] = (nx, ny) of case i; params[5*i..5*i+4] = (pos, radius,
 * ome, rho0, uu) as SetGeometry / DataInput define them.  precision:
 * IMEXLB_F64, IMEXLB_F32 or IMEXLB_F16_F32. */
int imexlb_batch_create(imexlb_batch **b, int ncase, const int32_t *nxny, const double *params, int device,
                        int precision);
/* The same with an elliptic body per case: shapes[2*i..2*i+1] = (aspect,
 * angle_deg) as imexlb_set_geometry_shape; NULL: all circles. */
int imexlb_batch_create_shapes(imexlb_batch **b, int ncase, const int32_t *nxny, const double *params,
                               const double *shapes, int device, int precision);
int imexlb_batch_destroy(imexlb_batch *b);
/* InitUP + InitPDF + the first Collision of every case (same r_vec). */
int imexlb_batch_init(imexlb_batch *b, const double *r_vec);
/* Warm start: InitPDF + the first Collision of every case from given
 * fields, p and u of all cases concatenated in case order, each in the
 * interior layout of imexlb_batch_download_fields ((nx+1)(ny+1) values of
 * p; u[d][y][x]). */
int imexlb_batch_init_fields(imexlb_batch *b, const double *p, const double *u);
/* Warm start of every case from device memory: fields holds ncase FP32
 * stacks [3][H][W], one per case in case order, each applied as
 * imexlb_init_fields_f32 does; then InitPDF + the first Collision. */
int imexlb_batch_init_fields_f32(imexlb_batch *b, const float *fields, int H, int W, double p_scale,
                                 double u_scale, const double *r_vec);
/* Body masks of every case as imexlb_body_mask_f32 writes them, case i at
 * out + i stride (stride >= H W); asynchronous on the batch's stream. */
int imexlb_batch_body_mask_f32(imexlb_batch *b, float *out, int H, int W, int64_t stride);
/* nsteps complete iterations of every case. */
int imexlb_batch_advance(imexlb_batch *b, int64_t nsteps);
/* Shape of the single-step kernel: threads per block (64, 128, 256, 512),
 * nodes per thread (1, 2, 4), persistent blocks taking tiles from a queue (1)
 * or one block per tile (0).  Results do not depend on it, nor do the steps
 * that imexlb_batch_advance makes several per launch. */
int imexlb_batch_set_config(imexlb_batch *b, int block, int cells_per_thread, int persistent);
/* Times every shape over trial_steps single steps (advancing the ensemble)
 * and keeps the fastest; best = (block, cells_per_thread, persistent). */
int imexlb_batch_tune(imexlb_batch *b, int trial_steps, int32_t best[3], double *best_ms_per_step);
/* Waits for every step queued on the batch's stream. */
int imexlb_batch_synchronize(imexlb_batch *b);
/* Momentum-exchange force of every case, F[3*i..3*i+2]. */
int imexlb_batch_forces(imexlb_batch *b, double *F);
/* Monitor of every case (lbm.f90:205-217 per case, as imexlb_monitor):
 * um[i] = max over case i's fluid entries 1..F-1 of sqrt(ux^2+uy^2).  A
 * case with a non-finite velocity gets um[i] = NaN; if any case has one the
 * call returns IMEXLB_E_NAN after filling every um[i] (imexlb_last_error
 * names the number of diverged cases).  Synchronises. */
int imexlb_batch_monitor(imexlb_batch *b, double *um);
/* p and u of case i, interior layout (u[d][y][x]). */
int imexlb_batch_download_fields(imexlb_batch *b, int i, double *p, double *u);
/* [0] nodes of all cases, [1] cases, [2] tiles, [3] device bytes */
int imexlb_batch_info(imexlb_batch *b, int64_t out[4]);
/* [0] to [2] as imexlb_step_form, for every case of the ensemble; [3] windows
 * per launch.  One case that several steps per launch do not suit keeps the
 * whole ensemble on single steps. */
int imexlb_batch_step_form(imexlb_batch *b, int32_t out[4]);

#ifdef __cplusplus
}
#endif
#endif /* IMEXLB_H */
