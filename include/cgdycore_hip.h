/*
 * cgdycore_hip.h -- C ABI of the MI355X (gfx950) spectral-element tendency and
 * Rosenbrock-W step for CGDycore.jl's CompressibleShallow / Dry
 * configuration.
 *
 * Every array argument is a DEVICE pointer with the reference's Julia
 * column-major layout (first index fastest):
 *   U, F, V, Vn, fV        : double (Nz, NumG, 5+NumTr)  AuxG : double (Nz, NumG, 4)
 *   Temp1                  : double (Nz, NumG, >= 5+NumTr)
 *   k                      : double (Nz, NumG, 5+NumTr, 3)
 *   JRhoW, JWRho, JWRhoTh, JRhoThW : double (2, Nz-1, NumG)   tri : double (3, Nz-1, NumG)
 *   Glob  : int64 (N*N, NF), 1-based      DS, DW : double (N, N)
 *   dXdxI : double (3,3,2,N*N,Nz,NF)      J : double (N*N,2,Nz,NF)
 *   X     : double (N*N,2,3,Nz,NF)        M : double (Nz,NumG,2)    dz : double (Nz,NumG)
 * Components 1-5 are rho, u, v, w, rho*theta, then the NumTr tracer
 * densities.  Temp1 may have more components (the reference allocates
 * 8+NumTr); its first 5 hold the hyperviscosity cache of the dynamics and
 * components 6..5+NumTr those of the tracers (FcnGPU.jl:115-126).
 *
 * All calls are ordered on the caller's HIP stream (passed as void*) and
 * return CGD_OK (0) or a negative error code.  The step-path calls
 * (cgd_prepare, cgd_fcn, cgd_jac, cgd_schur, cgd_rw_step, cgd_rw_run,
 * cgd_rw_graph_launch) allocate nothing; only the set-up calls
 * (cgd_ctx_create*, cgd_autotune, cgd_rw_graph_create, cgd_profile_enable)
 * do.  A context is not thread-safe; calls on one context must be issued
 * from one host thread.  Tendencies and steps use arrays of the context:
 * on several streams they run one after the other, in the order of the calls
 * (a call waits for the work that the stream of the last one holds by then).
 * Calls that a caller captures into graphs of its own are not ordered so;
 * their replays must not overlap others of the context.
 */
#ifndef CGDYCORE_HIP_H
#define CGDYCORE_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
  CGD_OK = 0,
  CGD_ERR_ARG = -1,         /* null pointer or bad dimension */
  CGD_ERR_UNSUPPORTED = -2, /* flag combination outside the Dry/CompressibleShallow path */
  CGD_ERR_HIP = -3,         /* a HIP runtime call failed */
  CGD_ERR_STATE = -4        /* context not usable (e.g. creation failed) */
};

/* precision modes (cgd_desc.precision).  CGD_MIXED applies to cgd_rw_step
 * only: the tendency and its DSS are computed and accumulated in FP32; the
 * equation of state, the w-interface balance of pressure gradient and
 * gravity, the horizontal pressure gradient, the theta hyperviscosity (from
 * the FP64 state, with an FP64 cache), the column Jacobian and Schur solve
 * and the Rosenbrock stage arithmetic stay FP64, as does the state V.
 * The fV and k work buffers then hold FP32 data (an FP32 copy of the stage
 * state and, with physics hooks, the FP32 tendency in fV; the stage
 * increments, solved in FP64, stored in FP32 in k).  Tracers
 * (NumTr > 0, with HorLimit, the moist state and microphysics) stay FP64 in
 * this mode: their increments (and tendencies, with microphysics) are
 * components 6.. of the same buffers, beyond the FP32 data.  Columns of more
 * than 64 levels step in FP64, and the other entry points compute in FP64 in
 * either mode. */
enum { CGD_FP64 = 0, CGD_MIXED = 1 };

typedef struct {
  /* dimensions (reference names) */
  int N;      /* OrdPoly + 1, 2..5 */
  int Nz;     /* vertical layers, 2..256 */
  int NF;     /* NumFaces (elements) */
  int NumG;   /* global CG nodes */
  int NumV;   /* must be 5: rho, u, v, w, rho*theta */
  int NumTr;  /* tracers, 0..16 (FP64 in both precision modes) */
  int precision; /* CGD_FP64 or CGD_MIXED */
  /* model switches that select FcnGPU! branches; implemented: Damping
   * (DampingW), Forcing (Held-Suarez), Microphysics (SimpleMicrophysics,
   * Moist state) and HorLimit (the limited horizontal tracer transport,
   * with tracers, FP64); Turbulence, VerticalDiffusion, SurfaceFlux and
   * EDMF must be 0 */
  int HorLimit;
  int Turbulence, VerticalDiffusion, SurfaceFlux, Forcing, Microphysics, Damping, EDMF;
  /* PhysParameters (GlobalVariables.jl:188-230) */
  double Grav, Omega, Rd, Cpd, p0, kappa;
  /* hyperviscosity (Model.HyperDCurl/HyperDGrad/HyperDDiv/HyperDDivW) */
  double HyperDCurl, HyperDGrad, HyperDDiv, HyperDDivW;
  /* static device inputs (reference layouts) */
  const int64_t *Glob;
  const double *DS, *DW, *dXdxI, *J, *X, *M, *dz;
  /* Damping != 0: DampingW (src/GPU/dampingGPU.jl:5-16), a Rayleigh sponge
   * on w above DampH - DampStride: F_w -= DampRelax sin^2(pi/2 (1 - (DampH -
   * zP)/DampStride)) w, with zP (Nz, NumG) the layer-centre heights
   * (GridSizeSphereKernel!, src/DyCore/DiscretizationCG.jl:130-134) */
  double DampH, DampStride, DampRelax;
  const double *zP;
  /* Forcing != 0: HeldSuarezForcing (src/Examples/force.jl:5-27) with the
   * ParamHeldSuarezDrySphere constants (src/Examples/parameters.jl:122-131)
   * and xS (2, NumG) = longitude, latitude of the global nodes */
  double HS_k_a, HS_k_f, HS_k_s, HS_DeltaT_y, HS_DeltaTh_z, HS_T_equator, HS_T_min, HS_sigma_b;
  const double *xS;
  /* State: CGD_DRY or CGD_MOIST (Models.Moist, src/Models/Equation.jl:56-75):
   * the pressure from rho, rho*theta and the vapour and cloud densities at
   * the 1-based components RhoVPos, RhoCPos (tracers, so > 5), with Cpv, Cpl,
   * Rv (PhysParameters); dPresdRhoTh stays the dry one, as in the reference */
  int State, RhoVPos, RhoCPos;
  double Cpv, Cpl, Rv;
  /* HorLimit != 0: the N GLL weights (FE.w), device pointer */
  const double *w;
  /* Kink smoothing of the rho*theta upwind flux, a mode of this library
   * with no counterpart in the reference (0, 0: the reference's exact
   * |wCon| and RecU4 limiter, OperatorKernel.jl:695-696,1044-1059).  With
   * SmoothW > 0, |wCon| -> sqrt(wCon^2 + (SmoothW (dXdxI[3,3] of the layers
   * on both sides of the interface)/2)^2); with SmoothC > 0 the limited
   * face value cL + max(0, min(r, kL r + kR, 1)) (cR - cL), written as
   * cL + minmod(cL - cLL, kL (cL - cLL) + kR (cR - cL), cR - cL), takes the
   * smooth minmod (x + y)/2 - S(M)/2 + S(m)/2, M, m = (x + y +- S(x - y))/2,
   * S(t) = sqrt(t^2 + SmoothC^2) (and likewise the right-biased face).  The
   * tendency is then smooth in the state, as a finite-difference check of
   * the adjoint needs.  Dry FP64 dynamics only (no tracers, HorLimit or
   * mixed precision); the adjoint differentiates the same functions. */
  double SmoothW, SmoothC;
  /* Microphysics != 0 (State = CGD_MOIST): SimpleMicrophysics
   * (src/Models/Microphysics.jl:6-40) through MicrophysicsKernel!
   * (src/GPU/OperatorKernel.jl:1082-1089) after Forcing and before Damping
   * (FcnGPU.jl:953-966): at each point, with T = p / Rm,
   * a = fpvs(T) / (Rv T) - rhoV, b = rhoC (clipped at 0),
   * FPh = RelCloud (a + b - sqrt(a^2 + b^2)) / 2 (evaporation > 0),
   * FR = -Rain FPh; F_rho -= FR, F_rhoV += FPh, F_rhoC -= FPh + FR and
   * F_rho*theta += the latent heating of Microphysics.jl:24-26.  fpvs is
   * Thermodynamics.fpvs (611.2 exp(17.62 (T-T0)/(243.12 + T-T0))), L =
   * L00 - (Cpl - Cpv)(T - T0) (Thermodynamics.jl:27-35,83-85).  The
   * reference's defaults: RelCloud = Rain = 0 (its tests use RelCloud =
   * 0.1), T0 = 273.15, L00 = 2.5e6 (GlobalVariables.jl:199-204,386-387). */
  double RelCloud, Rain, T0, L00;
} cgd_desc;

enum { CGD_DRY = 0, CGD_MOIST = 1 };

typedef struct cgd_ctx cgd_ctx;

/* Validates the descriptor, builds the element colouring and the
 * level-fastest copy of the metric.  Replaces the static part of
 * FcnGPU!'s setup (src/GPU/FcnGPU.jl:552-730) and of CGQuad/MetricStruct
 * consumption; no reference counterpart as a separate call. */
int cgd_ctx_create(const cgd_desc *desc, cgd_ctx **ctx, void *stream);

/* One context over nmem grids ("members", e.g. an ensemble on grids of
 * uneven size) that every entry point below then advances together.  The
 * members must agree on N, Nz, precision and the physical constants; each
 * keeps its own Glob, DS/DW (equal values), metric, M, dz and
 * hyperviscosity.  The batch's arrays concatenate the members along NumG:
 * U, V, F, ... are (Nz, sum_m NumG_m, 5) with member m's nodes at
 * NumG_0 + ... + NumG_{m-1} onward (and likewise k, AuxG, Temp1, the J
 * blocks).  Each member is coloured on its own and a node's contributions are
 * summed in its member's colour order, so a member's results are bit-identical
 * to those of a context built for it alone with the same launch shape, where the
 * members' metrics are of one kind: all on flat uniform layers with the same
 * bits at all levels, or none.  Otherwise the whole batch takes the kernels of
 * the general metric, and a member has the bits of its own context with
 * CGD_METRIC=full, which differ from its default ones by rounding.  No reference
 * counterpart (the reference steps one grid per process; batch variants of
 * the calls above, src/GPU/FcnGPU.jl:552 and src/Integration/RosenbrockSchur.jl:1). */
int cgd_ctx_create_batch(const cgd_desc *members, int nmem, cgd_ctx **ctx, void *stream);
int cgd_ctx_destroy(cgd_ctx *ctx);
const char *cgd_last_error(const cgd_ctx *ctx);

/* FcnPrepareGPU!(U,...) -- src/GPU/DiagnosticKernel.jl:180-241 (PressureKernel!
 * :96-115 with Models.Dry or Models.Moist, src/Models/Equation.jl:25-75).
 * Writes AuxG[:,:,1:3] = (p, T, theta). */
int cgd_prepare(cgd_ctx *ctx, const double *U, double *AuxG, void *stream);

/* FcnGPU!(F,U,...,Models.CompressibleShallow) -- src/GPU/FcnGPU.jl:552-913,
 * with the tracers of DivRhoTrUpwind3New2Kernel! (src/GPU/OperatorKernel.jl:722-759)
 * and HyperViscTracer(Koeff)Kernel! (src/GPU/ViscKernel.jl:169-218,277-327),
 * or with HorLimit LimitKernel! and DivRhoTrUpwind3LimKernel!
 * (src/GPU/HorLimiterKernel.jl:2-196) and no tracer hyperviscosity.
 * Zeroes and overwrites F and Temp1[:,:,1:5+NumTr]; reads p = AuxG[:,:,1]. */
int cgd_fcn(cgd_ctx *ctx, double *F, const double *U, double *Temp1, const double *AuxG, void *stream);

/* Global.TimeStepper.dtauStage, the time step of the limited tracer
 * transport (HorLimit): RosenbrockSchur! sets it to dt
 * (src/Integration/RosenbrockSchur.jl:9), and so do cgd_rw_step and
 * cgd_rw_run; cgd_fcn with HorLimit needs it set. */
int cgd_set_dtau(cgd_ctx *ctx, double dtau);

/* JacSchurGPU!(J,U,...) -- src/DyCore/JacSchur.jl:3-75.  Reads AuxG[:,:,4]
 * (identically zero for State=Dry). */
int cgd_jac(cgd_ctx *ctx, double *JRhoW, double *JWRho, double *JWRhoTh, double *JRhoThW, const double *U,
            const double *AuxG, void *stream);

/* SchurSolveGPU!(k,v,J,fac,...) -- src/Integration/SchurSolve.jl:149-177.
 * k: one stage (Nz,NumG,5+NumTr), tracers k = fac v.  Clobbers v[:,:,1],
 * v[:,:,4], v[:,:,5].
 * comp_tri != 0 rebuilds tri from the J blocks first (J.CompTri). */
int cgd_schur(cgd_ctx *ctx, double *k, double *v, const double *JRhoW, const double *JWRho, const double *JWRhoTh,
              const double *JRhoThW, double *tri, double fac, int comp_tri, void *stream);

/* RosenbrockSchur!(V,dt,...) with SSP-Knoth -- src/Integration/RosenbrockSchur.jl:1-33
 * and src/Integration/RosenbrockMethod.jl:24-48.  The work buffers are the
 * reference's Cache.Vn, Cache.fV, Cache.k, Cache.AuxG, Cache.Temp1 and the
 * JCache blocks; all are caller owned.  V is advanced by one step exactly as
 * the reference's sequence of calls would; the work buffers are scratch.
 * The stage kernel recomputes the frozen Jacobian from Vn
 * instead of storing it, so JRhoW..JRhoThW, tri, Temp1, k[:,:,:,3] and (without
 * physics hooks) fV are left unwritten, AuxG[:,:,1] holds the pressure of the last stage state and
 * AuxG[:,:,2:4] are neither read nor written (AuxG[:,:,4] must be zero, as
 * for State = Dry). */
typedef struct {
  double *Vn, *fV, *k, *AuxG, *Temp1;
  double *JRhoW, *JWRho, *JWRhoTh, *JRhoThW, *tri;
} cgd_rw_work;
int cgd_rw_step(cgd_ctx *ctx, double *V, double dt, const cgd_rw_work *work, void *stream);

/* The Rosenbrock branch of TimeStepper! (src/Integration/TimeStepper.jl:105-109):
 * nsteps calls of cgd_rw_step on one stream.  Each step but the last also
 * writes the pressure (and, in the mixed mode, the FP32 shadow) of its final
 * state, which the next step then uses instead of recomputing them; the
 * result is bit-identical to nsteps separate cgd_rw_step calls. */
int cgd_rw_run(cgd_ctx *ctx, double *V, double dt, const cgd_rw_work *work, int nsteps, void *stream);

/* The schedule and layout cgd_ctx_create chose: the number of element
 * colours (the order in which a node's contributions are summed), the level
 * chunk height of the element kernels before the context's own choice of
 * another one for some of them (which cgd_get_launch_shape reports), and
 * whether the metric is stored in the compact layout (every
 * component except the terrain row dXdxI[3,1:2,:] identical across levels,
 * so stored once per element node; of a batch: that of every member).  The
 * kernels of the layouts agree to rounding.  No reference counterpart. */
int cgd_ctx_info(const cgd_ctx *ctx, int *ncolor, int *chunk_levels, int *compact_metric);

/* Launch shapes (no reference counterpart; the reference fixes its
 * workgroup shapes by NumberThreadGPU, src/DyCore/GlobalVariables.jl:240).
 * In cgd_set_launch_shape a field of 0 keeps the current value.  A context
 * starts with heights chosen by a rule on N, Nz, the metric and the size of
 * the grid.  cgd_get_launch_shape reports the heights that run (chunk_levels:
 * those of cgd_rw_step's tendency), and setting the reported shape, on this
 * context or on another one for the same inputs, changes nothing.  A height
 * that equals the chosen one stands for the whole choice (in the mixed mode
 * the FP64 tendency of cgd_fcn may have another height than the steps', and
 * tracers keep 8 levels); any other is the height of all of a pass's kernels.
 * The workgroup sizes, pass 1's height and pass1_items change no bit; the pass-2
 * chunk height (chunk-interface w sums; in FP64 not on the regular metric of
 * flat uniform layers) and 32-lane columns (the compiler's fused
 * multiply-adds) change rounding only, within the FP64 parity bound.
 * persistent = 1 runs each RW stage of cgd_rw_step as ONE launch (both
 * tendency passes, then the column stage) whose
 * workgroups stay resident and meet at grid-wide barriers where the
 * separate launches have kernel boundaries; the results in FP64 are
 * bit-identical to the separate launches with heights of 8 (on a regular
 * metric with any heights).  It takes the dry dynamics with the compact
 * metric (no tracers, hooks or kink smoothing), N = 4 or 5, Nz <= 64, chunk
 * heights 8, pass1_items 1 and col_block = 64*ceil(8*N*N/64); otherwise
 * CGD_ERR_UNSUPPORTED.  Heights that the context chose give way to 8 while
 * persistent is 1 and stand again afterwards; set heights must be 8.  A barrier wait is bounded (250 ms): should the
 * workgroups not all be resident (another process on the device), the
 * launch ends and cgd_check reports it.
 * Setting a shape drops a captured step graph. */
typedef struct {
  int chunk_levels;       /* levels per workgroup of the fused tendency pass: 8, or 16 for N = 5 */
  int pass1_chunk_levels; /* the same for the first (hyperviscosity) pass; 64: whole columns (compact metric, Nz <= 64) */
  int pass1_items;        /* (element, chunk) items per pass-1 workgroup: 1 or 2 (loads of both in flight) */
  int col_lanes;          /* lanes per column in the stage kernel: 64, or 32 (two columns per wavefront, Nz <= 32) */
  int col_block;          /* threads per stage workgroup: 64, 128, 192 or 256 */
  int persistent;         /* 1: one persistent launch per RW stage; -1: separate launches (the default) */
} cgd_launch_shape;
int cgd_set_launch_shape(cgd_ctx *ctx, const cgd_launch_shape *shape);
int cgd_get_launch_shape(const cgd_ctx *ctx, cgd_launch_shape *shape);

/* Synchronises stream and reports (CGD_ERR_HIP, then clears) a grid
 * barrier of a persistent stage launch that timed out since the last
 * check; CGD_OK otherwise.  No reference counterpart. */
int cgd_check(cgd_ctx *ctx, void *stream);

/* Autotuner: times cgd_rw_step per candidate launch shape on the caller's V
 * and work buffers (per shape the fastest of three timings of reps steps,
 * over two sweeps through the candidates) and keeps the fastest: the
 * element-kernel shapes jointly (both chunk heights, whole columns of pass 1 and
 * pass1_items), then
 * the column shape with the best of them, then separate launches against
 * one persistent launch per stage where the configuration allows it.  The context's shape on entry is
 * kept unless a candidate beats it by more than 1 %.  V, all components,
 * is restored afterwards (the work buffers are scratch).  A set-up call: it allocates a copy of V and
 * synchronises the stream.  chosen (may be null) receives the shape, best_ms
 * the time per step.  No reference counterpart. */
int cgd_autotune(cgd_ctx *ctx, double *V, double dt, const cgd_rw_work *work, int reps, void *stream,
                 cgd_launch_shape *chosen, double *best_ms);

/* Step graph: captures cgd_rw_run(ctx, V, dt, work, nsteps) into a HIP
 * graph held by the context (pointers, dt and launch shapes as at the
 * capture); cgd_rw_graph_launch replays all of them with one launch on
 * stream, advancing V by nsteps steps.  Capture is a set-up call (it
 * synchronises stream and creates a capture stream); a replay allocates
 * nothing.  Profiling must be off while capturing.  No reference
 * counterpart. */
int cgd_rw_graph_create(cgd_ctx *ctx, double *V, double dt, const cgd_rw_work *work, int nsteps, void *stream);
int cgd_rw_graph_launch(cgd_ctx *ctx, void *stream);

/* ---- Set-up on the device (no context; each call synchronises stream and
 * may allocate temporaries).  Errors: a negative code and the message of
 * cgd_setup_error() (per host thread). */
const char *cgd_setup_error(void);

/* JacobiSphere3GPU!(AdaptGrid=Sleve, X, dXdxI, J, FE, F, z, zs, Rad,
 * ::CompressibleShallow) -- src/Grids/JacobiSphere3GPU.jl:24-40, kernel
 * :102-215, with the Sleve height of src/Grids/Adapt.jl:19-31 (etaH, s; the
 * reference's defaults are 0.7 and 0.8).  F: element corners double
 * (4,3,NF); xw: the N GLL nodes; DS: (N,N); z: the Nz+1 layer interfaces
 * (z[Nz+1] = H); zs: surface height (N,N,NF), or NULL for flat terrain.
 * Writes X (N*N,2,3,Nz,NF), dXdxI (3,3,2,N*N,Nz,NF), J (N*N,2,Nz,NF). */
int cgd_jacobi_sphere3(int N, int Nz, int NF, const double *F, const double *xw, const double *DS, const double *z,
                       const double *zs, double Rad, double etaH, double s, double *X, double *dXdxI, double *J,
                       void *stream);

/* MassCGGPU! -- src/DyCore/MassCG.jl:42-75: M (Nz,NumG,2) = sums of J over
 * the element copies of each node, MMass (Nz,NumG) = sums of
 * 0.5 (J1 + J2) w_I w_J (w: the N GLL weights; MMass may be NULL), each in
 * ascending (element, node) order. */
int cgd_mass_cg(int N, int Nz, int NF, int NumG, const int64_t *Glob, const double *J, const double *w, double *M,
                double *MMass, void *stream);

/* cgd_mass_cg without allocating: no counterpart in the reference; for
 * callers that cannot allocate device memory (code under HIP graph capture,
 * tight serving loops, harnesses that forbid hipMalloc).  The same kernels
 * and results as cgd_mass_cg, bit for bit, but the node -> element-copy
 * table lives in a fixed device array of CGD_NOALLOC_MAX_NODES * 17 + 64
 * ints (about 42 MB, held by every GPU the library runs on until the
 * process ends) instead of memory allocated per call; nothing is allocated
 * and nothing is freed.  NumG above CGD_NOALLOC_MAX_NODES (ne = 80 at
 * p = 4) is refused with CGD_ERR_ARG before any device work.  Every call
 * on one GPU uses that GPU's one table, which keeps the last call's
 * contents (the counts are cleared by a fill kernel on every call): calls
 * that overlap on one GPU (other streams or host threads) race.
 * Synchronises stream once (the numbering check). */
#define CGD_NOALLOC_MAX_NODES 614402
int cgd_mass_cg_noalloc(int N, int Nz, int NF, int NumG, const int64_t *Glob, const double *J, const double *w,
                        double *M, double *MMass, void *stream);

/* GridSizeSphereKernel! -- src/DyCore/DiscretizationCG.jl:119-144: dz
 * (Nz,NumG) = |X[:,2,...]| - |X[:,1,...]| and zP (Nz,NumG, may be NULL) =
 * max(|mean of both|-Rad, 0) at each node, taken from its last element copy
 * in (element, node) order. */
int cgd_grid_size_sphere(int N, int Nz, int NF, int NumG, const int64_t *Glob, const double *X, double Rad,
                         double *zP, double *dz, void *stream);

/* The single-rank cubed sphere of ne x ne elements per panel, on the host
 * (no GPU work): CubedGrid -- src/Grids/CubedGrid.jl:1-513 (CubePoint
 * :377-391, InsertFaceEdge :393-441, InsertEdgeEdge :443-462,
 * InsertFaceFace :464-513), Face (src/Grids/Face.jl:48-167),
 * Orientation! (src/Grids/Orientation.jl), RenumberingFace4!
 * (src/Grids/Renumbering.jl) and the one-rank renumbering of
 * src/Grids/SubGridGhost.jl:1-162.  cgd_cubed_sphere_sizes gives the counts
 * (NumNodes = 6(ne-1)^2 + 12(ne-1) + 8, NumEdges = 12 ne^2, NumFaces =
 * 6 ne^2); cgd_cubed_sphere fills host arrays: nodes (NumNodes,3) on the
 * sphere of radius Rad, face_nodes and face_edges (NumFaces,4) and
 * edge_nodes (NumEdges,2), 1-based, in the sub-grid numbering. */
int cgd_cubed_sphere_sizes(int ne, int *NumNodes, int *NumEdges, int *NumFaces);
int cgd_cubed_sphere(int ne, double Rad, double *nodes, int64_t *face_nodes, int64_t *face_edges,
                     int64_t *edge_nodes);

/* NumberingFemCGQuad(Grid, OrdPoly) -- src/DyCore/NumberingFem.jl:21-131,
 * on the device, one thread per face: Glob (NN = (p+1)^2, NF) of 1-based
 * global node numbers (corner nodes, then p-1 numbers per edge in the
 * edge's direction, then (p-1)^2 per face, placed by the reference's Per
 * table) from device copies of cgd_cubed_sphere's face_nodes, face_edges
 * and edge_nodes.  OrdPoly p = 1..4 (the reference's p > 4 branch does not
 * run).  NumG (may be NULL) = NumNodes + NumEdges (p-1) + NF (p-1)^2.
 * Asynchronous on stream. */
int cgd_numbering_cg_quad(int p, int NF, int NumNodes, int NumEdges, const int64_t *face_nodes,
                          const int64_t *face_edges, const int64_t *edge_nodes, int64_t *Glob, int *NumG,
                          void *stream);

/* ---- Output (no context).  InterpolateGPU! / InterpolateRhoGPU! /
 * InterpolateWBGPU! -- src/Outputs/vtkOutputKernel.jl:49-158,215-292: the
 * values at the cell centres of an OrdPrint x OrdPrint sub-grid of every
 * element and layer, cCell (OrdPrint, OrdPrint, Nz, NF), from a global-node
 * field (Nz, NumG) and Inter (OrdPrint, OrdPrint, N, N) = the Lagrange basis
 * at the sub-cell centres (vtkSphere.jl:193-210).  mode 0: c; mode 1: c/rho
 * (rho needed); mode 2: c = w at the layer tops, the cell value
 * 1/2 (w[Iz] + w[Iz-1]) with the free-slip w below the first layer (u, v
 * and dXdxI needed).  Errors: cgd_output_error(). */
const char *cgd_output_error(void);
int cgd_interpolate(int mode, int N, int Nz, int NF, int NumG, int OrdPrint, const int64_t *Glob, const double *Inter,
                    const double *c, const double *rho, const double *u, const double *v, const double *dXdxI,
                    double *cCell, void *stream);

/* Host-only helper (no GPU needed): the element colouring that schedules the
 * DSS.  glob is a HOST int64 (N*N, NF) 1-based array; color receives NF
 * colours (0-based), ncolor their count.  Elements of one colour share no
 * global node; nodes accumulate element contributions in colour order.  No
 * reference counterpart (the reference scatters with atomics,
 * src/GPU/ViscKernel.jl:78-82). */
int cgd_color_elements(const int64_t *glob, int NN, int NF, int NumG, int *color, int *ncolor);

/* Per-kernel timing of the tendency passes with HIP events on the launch
 * stream (used by the benchmark; off by default).  which: 0 = pass 1
 * (hyperviscosity), 1 = pass 2 (fused tendency), 2 = column solve.
 * cgd_profile_enable takes a bit mask of the passes to time (bit which;
 * 0 turns timing off).  Every recorded event is a stream barrier with a
 * cache write-back, so time only what is read. */
int cgd_profile_enable(cgd_ctx *ctx, int on);
int cgd_profile_read(cgd_ctx *ctx, int which, double *total_ms, long long *launches);

/* ---- Adjoint (reverse mode) of the FP64 path.  The reference has no
 * adjoint: these are the transposes of the derivatives of FcnGPU!
 * (src/GPU/FcnGPU.jl:552-968), SchurSolveGPU!
 * (src/Integration/SchurSolve.jl:149-177), JacSchurGPU!
 * (src/DyCore/JacSchur.jl:3-75) and RosenbrockSchur!
 * (src/Integration/RosenbrockSchur.jl:1-33), for the dry configuration
 * without tracers or physics hooks (CGD_ERR_UNSUPPORTED otherwise), in FP64
 * whatever the context's precision.  The RecU4 limiter and the |wCon|
 * upwinding are differentiated on the branch the forward takes, except
 * |wCon| where wCon is zero to rounding (w = 0 on a flat metric): there the
 * mean of its one-sided derivatives (0) is taken.  State
 * cotangents are summed in a fixed order (no atomics), so results are
 * bit-reproducible.  work: device doubles, at least cgd_adjoint_work_size(ctx,
 * nsteps, every) of them (nsteps = 0 for the single-evaluation calls). */
int cgd_adjoint_work_size(cgd_ctx *ctx, int nsteps, int every, size_t *ndoubles);

/* lamU (Nz,NumG,5) = (dF/dU)^T lamF for F = FcnGPU!(U) (with its
 * FcnPrepareGPU! pressure); the forward tendency is recomputed in work. */
int cgd_fcn_adjoint(cgd_ctx *ctx, const double *U, const double *lamF, double *lamU, double *work, void *stream);

/* For k = SchurSolveGPU!(v; J blocks, fac): lamv (Nz,NumG,5) = (dk/dv)^T
 * lamk, and the Jacobian-block cotangents (each (2,Nz-1,NumG)) are ADDED
 * into lJRhoW .. lJRhoThW.  k: the forward result (its w component is the
 * tridiagonal solution); v: the forward right-hand side as it was before
 * the solve (the solve overwrites it). */
int cgd_schur_adjoint(cgd_ctx *ctx, const double *lamk, const double *k, const double *v, const double *JRhoW,
                      const double *JWRho, const double *JWRhoTh, const double *JRhoThW, double fac, double *lamv,
                      double *lJRhoW, double *lJWRho, double *lJWRhoTh, double *lJRhoThW, double *work,
                      void *stream);

/* ADDS (dJ/dU)^T lJ into lamU (rho and rho*theta) for the Jacobian blocks
 * of JacSchurGPU!(U). */
int cgd_jac_adjoint(cgd_ctx *ctx, const double *U, const double *lJRhoW, const double *lJWRho,
                    const double *lJWRhoTh, const double *lJRhoThW, double *lamU, void *stream);

/* One RosenbrockSchur! step from Vn: lamV holds the cotangent of the step's
 * result on entry and that of Vn on return.  The stages are recomputed from
 * Vn with the composed FP64 calls. */
int cgd_rw_step_adjoint(cgd_ctx *ctx, const double *Vn, double dt, double *lamV, double *work, void *stream);

/* nsteps steps from V0 with a checkpoint every `every` steps: lamV holds the
 * cotangent of the final state on entry and that of V0 on return; Vfinal
 * (may be NULL) receives the final state.  The forward run stores
 * ceil(nsteps/every) states, the reverse sweep recomputes each segment's
 * step states from its checkpoint. */
int cgd_rw_adjoint(cgd_ctx *ctx, const double *V0, double dt, int nsteps, int every, double *lamV, double *Vfinal,
                   double *work, void *stream);

/* cgd_rw_adjoint in two halves, for a caller that runs the forward itself
 * and differentiates later (a ChainRulesCore rrule: the forward pass keeps
 * its checkpoints, the pullback uses them).  cgd_rw_forward_ckpt: nsteps
 * steps from V0 into Vfinal, keeping a checkpoint every `every` steps in
 * work.  cgd_rw_adjoint_ckpt: the reverse sweep from those checkpoints;
 * lamV as in cgd_rw_adjoint.  The reverse needs the checkpoints of the last
 * cgd_rw_forward_ckpt (or cgd_rw_adjoint) on this context, with the same
 * dt, nsteps, every and work array, and fails otherwise; work must not be
 * used by other calls in between. */
int cgd_rw_forward_ckpt(cgd_ctx *ctx, const double *V0, double dt, int nsteps, int every, double *Vfinal,
                        double *work, void *stream);
int cgd_rw_adjoint_ckpt(cgd_ctx *ctx, double dt, int nsteps, int every, double *lamV, double *work, void *stream);

#ifdef __cplusplus
}
#endif

#endif
