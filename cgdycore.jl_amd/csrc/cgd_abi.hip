// C ABI (include/cgdycore_hip.h): context set-up, argument validation and
// launch sequencing for the gfx950 kernels in cgd_kernels.hip.
#include "../../include/cgdycore_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "cgd_kernels.hip"

struct cgd_ctx {
  cgd_desc desc{};
  KArgs ka{};
  int N = 0, NN = 0, Nz = 0, NF = 0, NumG = 0;
  // levels per workgroup of pass 2 and of pass 1 (64: whole columns, k_fcn1c)
  // as cgd_get_launch_shape reports them for separate launches, and the ones
  // the context chose: nzt is then 16 levels in FP64 where r16 (k_fcn2r) is set
  int nzt = 0, nzt1 = 0;
  int base_nzt = 8, rule_nzt = 0, rule_nzt1 = 0;
  int r16 = 0;
  int thomas = 0;  // column solve: 0 = cyclic reduction, 1 = serial Thomas (CGD_THOMAS=1)
  int ntr = 0;     // tracers (components 5..4+ntr of the state arrays, 0-based)
  int ncolor = 0;
  std::vector<int> color_off;  // first entry of each colour in the colour list
  int *d_glob = nullptr;       // [NF][NN] 0-based
  int *d_clist = nullptr;      // elements by colour, ascending within one
  int *d_cpy = nullptr, *d_gcpy = nullptr;  // the copies of each element node / global node, colour order
  double *d_e1 = nullptr, *d_e2 = nullptr;  // element copies of the pass-1 cache and of the tendency (5 + NumTr each)
  double *d_met = nullptr, *d_met1 = nullptr, *d_ms = nullptr;
  double *d_metn = nullptr, *d_met1n = nullptr;  // compact metric layout: per element node
  int cm = 0;                                    // 1: compact metric layout
  int reg = 0;                                   // 1: regular compact metric (k_fcn2r)
  double *d_iMn = nullptr;                       // regular metric: 1/(M1+M2) per node
  int mixed = 0;                                 // 1: mixed-precision cgd_rw_step
  int smooth = 0;                                // 1: kink-smoothed upwind flux (SmoothW or SmoothC > 0)
  float *d_ims32 = nullptr;                      // 1/(M1+M2) in FP32 (mixed precision)
  float *d_m32 = nullptr;                        // M in FP32 (mixed precision)
  float *d_metp32 = nullptr;                     // compact per-point metric in FP32 (mixed precision)
  double *d_f4x = nullptr;     // [NF][NN][nchunk] chunk-bottom F4 terms
  int *d_nptr = nullptr, *d_ncopy = nullptr;  // global node -> element copies (colour order)
  double *d_kvis = nullptr;    // [element][3] hyperviscosity coefficients
  // HorLimit: each element's stencil (itself and the elements sharing a node,
  // 13 element numbers), the element bounds of the mixing ratios
  // [tracer][element][Nz], and the stage time step (dtauStage)
  int horlimit = 0;
  double dtau = 0.0;
  // the checkpoints that cgd_rw_forward_ckpt left in a work array, for the
  // reverse sweep of cgd_rw_adjoint_ckpt (nullptr: none)
  const double *ck_work = nullptr;
  double ck_dt = 0.0;
  int ck_nsteps = 0, ck_every = 0;
  int *d_stencil = nullptr;
  double *d_qmin = nullptr, *d_qmax = nullptr;
  // batch of grids (cgd_ctx_create_batch): member m owns elements
  // mem_e0[m]..mem_e0[m+1]-1 and global nodes mem_g0[m]..mem_g0[m+1]-1
  int nmem = 1;
  std::vector<int> mem_e0, mem_g0;
  double *d_M = nullptr, *d_dz = nullptr;  // M and dz in batch numbering (batches only)
  double *d_zP = nullptr, *d_xS = nullptr;  // zP, xS in batch numbering (batches with hooks only)
  Hooks hooks{};                            // Damping / Forcing (pointwise, after the tendency)
  const double *M = nullptr, *dz = nullptr;  // the M and dz the kernels read
  // column launch shape of the fused stage kernel: lanes per column (64,
  // or 32 for two columns per wavefront when Nz <= 32) and workgroup size
  int colw = 64, colblock = 256;
  int items1 = 1;  // pass-1 work items (element, level chunk) per workgroup: 1 or 2
  // one persistent launch per RW stage (k_stage_persist): on/off, its grid
  // (workgroups resident at once), the grid barrier's state and wait bound
  int persistent = 0;
  int pgrid = 0;
  GridBar *d_bar = nullptr;
  long long bar_ticks = 0;
  // the stream of the last call that used the context's own arrays (order_streams)
  hipStream_t last = nullptr;
  bool used = false;
  hipEvent_t ev_last = nullptr;
  // captured step graph (cgd_rw_graph_create)
  hipStream_t gstream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  bool ok = false;
  std::string err;
  // per-pass timing (events on the launch stream)
  int prof = 0;  // bit w: time pass w (0 = pass 1, 1 = pass 2, 2 = column)
  double prof_ms[3] = {0, 0, 0};
  long long prof_n[3] = {0, 0, 0};
  std::vector<hipEvent_t> prof_ev;
  std::vector<int> prof_which, prof_launch;
  int prof_cap = 0, prof_used = 0;
};

// LDS bytes of the element kernels for tendency type R: pass 1 holds D, DW
// and tile sets of 5 and 4; pass 2 an FP64 D and pressure tile, then D, DW,
// two sets of 7 tiles and the per-node horizontal metric
// FP32 element kernels: an FP64 region for the theta hyperviscosity after
// the R-typed LDS (pass 1: D, DW and three tiles; pass 2: DW and three tiles)
template <typename R> static size_t lds_fcn1(const cgd_ctx *c, int nzt1) {
  const size_t r = sizeof(R) * (2 * c->NN + 9 * c->NN * nzt1);
  if (std::is_same<R, double>::value) return r;
  return (r + 7) / 8 * 8 + sizeof(double) * (2 * c->NN + 3 * c->NN * nzt1);
}
template <typename R> static size_t lds_fcn2(const cgd_ctx *c, int nzt) {
  // + the horizontal metric: 12 values per node (compact layout), 10 per point
  // (full layout, FP64)
  const size_t hm = c->cm || !std::is_same<R, double>::value ? 12 * c->NN : 10 * c->NN * nzt;
  const size_t r = sizeof(R) * (2 * c->NN + 14 * c->NN * nzt + hm);
  const size_t base = sizeof(double) * (c->NN + c->NN * nzt);
  if (std::is_same<R, double>::value) return base + r;
  return base + (r + 7) / 8 * 8 + sizeof(double) * (c->NN + 3 * c->NN * nzt);
}

// pass 1 can take whole columns
static bool columns_ok(const cgd_ctx *c) { return c->cm && c->Nz <= 64; }
// k_fcn1c: three tiles of whole columns, one of them FP64
static size_t lds_fcn1c(const cgd_ctx *c, size_t r) { return (size_t)c->NN * 64 * (sizeof(double) + 2 * r); }

// The heights that separate launches run (a persistent one has chunks of 8
// levels, and so has pass 2 of a tendency called beside it).  A height that is
// the context's own choice stands for all of that choice: in pass 2 the FP64
// and the FP32 tendency's, each by its rule, and base_nzt for the tracers'
// kernels; any other is the height of all of them.
static int cache_nzt(const cgd_ctx *c) { return c->nzt1; }
template <typename R> static int tend_nzt(const cgd_ctx *c) {
  if (c->persistent) return 8;
  if (c->nzt != c->rule_nzt) return c->nzt;
  return std::is_same<R, double>::value && c->r16 ? 16 : c->base_nzt;
}
// the levels between the interfaces whose w terms pass 2 leaves in d_f4x
template <typename R> static int f4_nzt(const cgd_ctx *c) {
  return std::is_same<R, double>::value && c->reg && !c->smooth ? 8 : tend_nzt<R>(c);
}
static int tr_cache_nzt(const cgd_ctx *c) { return c->nzt1 == c->rule_nzt1 || c->nzt1 == 64 ? c->base_nzt : c->nzt1; }
static int tr_tend_nzt(const cgd_ctx *c) { return c->nzt == c->rule_nzt ? c->base_nzt : c->nzt; }
static int nchunks(const cgd_ctx *c, int nzt) { return (c->Nz + nzt - 1) / nzt; }
// threads of an element tile of nzt levels
static int tile_block(const cgd_ctx *c, int nzt) { return (c->NN * nzt + 63) / 64 * 64; }

// k_fcn2r: D, DW, 12 tiles, four tiles with the level below, its sums, the
// horizontal metric and 1/(2 M)
static size_t lds_fcn2r(const cgd_ctx *c, int nzt) {
  return sizeof(double) * (2 * c->NN + 12 * c->NN * nzt + 4 * c->NN * (nzt + 1) + 7 * c->NN);
}

static int fail(cgd_ctx *c, int code, const std::string &msg) {
  if (c) c->err = msg;
  return code;
}

#define HIPCHK(ctx, call)                                                                     \
  do {                                                                                        \
    hipError_t e_ = (call);                                                                   \
    if (e_ != hipSuccess)                                                                     \
      return fail(ctx, CGD_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_));      \
  } while (0)

static inline hipStream_t S(void *s) { return reinterpret_cast<hipStream_t>(s); }

static int grid_for(size_t n, int block) {
  size_t g = (n + block - 1) / block;
  return (int)std::min<size_t>(std::max<size_t>(g, 1), 65536);
}

// Element adjacency: elements sharing at least one global node.
static void element_adjacency(const std::vector<int> &g32, int NN, int NF, int NumG, std::vector<int> &aptr,
                              std::vector<int> &adj) {
  std::vector<int> nptr(NumG + 1, 0);
  for (int v : g32) nptr[v + 1]++;
  for (int i = 0; i < NumG; ++i) nptr[i + 1] += nptr[i];
  std::vector<int> nel(nptr[NumG]);
  {
    std::vector<int> fillp(nptr.begin(), nptr.end() - 1);
    for (int e = 0; e < NF; ++e)
      for (int i = 0; i < NN; ++i) nel[fillp[g32[(size_t)e * NN + i]]++] = e;
  }
  aptr.assign(NF + 1, 0);
  adj.clear();
  std::vector<int> mark(NF, -1);
  for (int e = 0; e < NF; ++e) {
    for (int i = 0; i < NN; ++i) {
      const int gn = g32[(size_t)e * NN + i];
      for (int q = nptr[gn]; q < nptr[gn + 1]; ++q) {
        const int o = nel[q];
        if (o != e && mark[o] != e) {
          mark[o] = e;
          adj.push_back(o);
        }
      }
    }
    aptr[e + 1] = (int)adj.size();
  }
}

// Greedy colouring in element order: each element takes the smallest colour
// not used by an adjacent element.  Returns the number of colours, or -1 if
// more than 64 would be needed.
static int color_greedy(int NF, const std::vector<int> &aptr, const std::vector<int> &adj, std::vector<int> &color) {
  color.assign(NF, -1);
  int ncol = 0;
  std::vector<int> mark(64, -1);
  for (int e = 0; e < NF; ++e) {
    for (int q = aptr[e]; q < aptr[e + 1]; ++q)
      if (color[adj[q]] >= 0) mark[color[adj[q]]] = e;
    int col = 0;
    while (col < 64 && mark[col] == e) ++col;
    if (col >= 64) return -1;
    color[e] = col;
    ncol = std::max(ncol, col + 1);
  }
  return ncol;
}

// Four colours by depth-first search with forward checking: the element with
// the fewest admissible colours is coloured next (ties: lowest index), its
// colour is removed from its neighbours' domains, and an emptied domain
// backtracks.  Four colours are the minimum (four elements meet at a vertex
// away from the cube corners); on the cubed sphere such colourings exist and
// are found with almost no backtracking, giving four launches of equal size
// instead of a greedy colouring's long tail of small colours.  Returns false
// when the step budget runs out.
static bool color_four(int NF, const std::vector<int> &aptr, const std::vector<int> &adj, std::vector<int> &color) {
  const long long budget = 64LL * NF + 100000;
  std::vector<unsigned char> dom(NF, 15);
  color.assign(NF, -1);
  struct Frame {
    int e;
    unsigned char rem;
    size_t trail;
  };
  std::vector<Frame> stack;
  std::vector<std::pair<int, unsigned char>> trail;
  // candidates by domain size: a lazy min-structure over (popcount, index)
  std::vector<int> forced;  // elements whose domain shrank to one colour
  int scan = 0;             // all elements below scan are coloured or queued
  auto popc = [](unsigned v) { return __builtin_popcount(v); };
  auto pick = [&]() -> int {
    while (!forced.empty()) {
      const int e = forced.back();
      forced.pop_back();
      if (color[e] < 0) return e;
    }
    int best = -1, bs = 99;
    while (scan < NF && color[scan] >= 0) ++scan;
    for (int e = scan; e < NF; ++e)
      if (color[e] < 0 && popc(dom[e]) < bs) {
        bs = popc(dom[e]);
        best = e;
        if (bs <= 2) break;
      }
    return best;
  };
  long long steps = 0;
  for (;;) {
    const int e0 = pick();
    if (e0 < 0) return true;
    if (++steps > budget) return false;
    stack.push_back({e0, dom[e0], trail.size()});
    bool placed = false;
    while (!stack.empty()) {
      Frame &f = stack.back();
      while (trail.size() > f.trail) {
        dom[trail.back().first] = trail.back().second;
        trail.pop_back();
      }
      color[f.e] = -1;
      if (f.rem == 0) {
        stack.pop_back();
        forced.clear();
        scan = 0;
        continue;
      }
      const int c = __builtin_ctz(f.rem);
      f.rem &= (unsigned char)~(1u << c);
      color[f.e] = c;
      bool fail = false;
      for (int q = aptr[f.e]; q < aptr[f.e + 1] && !fail; ++q) {
        const int b = adj[q];
        if (color[b] < 0 && (dom[b] >> c & 1)) {
          trail.push_back({b, dom[b]});
          dom[b] &= (unsigned char)~(1u << c);
          if (dom[b] == 0) fail = true;
          else if (popc(dom[b]) == 1) forced.push_back(b);
        }
      }
      if (!fail) {
        placed = true;
        break;
      }
      if (++steps > budget) return false;
    }
    if (!placed) return false;
  }
}

// DSS schedule: four balanced colours when the search succeeds, else greedy.
static int color_elements(const std::vector<int> &g32, int NN, int NF, int NumG, std::vector<int> &color) {
  std::vector<int> aptr, adj;
  element_adjacency(g32, NN, NF, NumG, aptr, adj);
  if (color_four(NF, aptr, adj, color)) return 4;
  return color_greedy(NF, aptr, adj, color);
}

extern "C" int cgd_color_elements(const int64_t *glob, int NN, int NF, int NumG, int *color, int *ncolor) {
  if (!glob || !color || !ncolor || NN < 1 || NF < 1 || NumG < 1) return CGD_ERR_ARG;
  std::vector<int> g32((size_t)NN * NF);
  for (size_t i = 0; i < g32.size(); ++i) {
    if (glob[i] < 1 || glob[i] > NumG) return CGD_ERR_ARG;
    g32[i] = (int)(glob[i] - 1);
  }
  std::vector<int> col;
  const int n = color_elements(g32, NN, NF, NumG, col);
  if (n < 0) return CGD_ERR_UNSUPPORTED;
  std::copy(col.begin(), col.end(), color);
  *ncolor = n;
  return CGD_OK;
}

extern "C" const char *cgd_last_error(const cgd_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

extern "C" int cgd_ctx_info(const cgd_ctx *c, int *ncolor, int *chunk_levels, int *compact_metric) {
  if (!c) return CGD_ERR_ARG;
  if (!c->ok) return CGD_ERR_STATE;
  if (ncolor) *ncolor = c->ncolor;
  if (chunk_levels) *chunk_levels = c->persistent ? 8 : tr_tend_nzt(c);
  if (compact_metric) *compact_metric = c->cm;
  return CGD_OK;
}

// Checks one descriptor on its own (dimensions, flags, pointers).
static int validate_desc(cgd_ctx *c, const cgd_desc *d, const std::string &who) {
  if (d->N < 4 || d->N > 5) return fail(c, CGD_ERR_UNSUPPORTED, who + "OrdPoly must be 3 or 4 (N = 4 or 5)");
  if (d->Nz < 3 || d->Nz > 256) return fail(c, CGD_ERR_ARG, who + "Nz must be in [3, 256]");
  if (d->NF < 1 || d->NumG < 1) return fail(c, CGD_ERR_ARG, who + "NF and NumG must be positive");
  if (d->NumV != 5) return fail(c, CGD_ERR_UNSUPPORTED, who + "NumV must be 5 (rho, u, v, w, rho*theta)");
  if (d->NumTr < 0 || d->NumTr > 16) return fail(c, CGD_ERR_UNSUPPORTED, who + "NumTr must be in [0, 16]");
  if (d->precision != CGD_FP64 && d->precision != CGD_MIXED)
    return fail(c, CGD_ERR_UNSUPPORTED, who + "unknown precision mode");
  if (d->Turbulence || d->VerticalDiffusion || d->SurfaceFlux || d->EDMF)
    return fail(c, CGD_ERR_UNSUPPORTED,
                who + "only the CompressibleShallow path is implemented (hooks: Damping, Forcing, Microphysics, "
                      "HorLimit)");
  if (d->Microphysics && d->State != CGD_MOIST)
    return fail(c, CGD_ERR_ARG, who + "Microphysics needs State = Moist (vapour and cloud components)");
  if (d->Microphysics && !(d->RelCloud >= 0.0 && d->Rain >= 0.0 && d->T0 > 0.0 && d->L00 > 0.0))
    return fail(c, CGD_ERR_ARG, who + "Microphysics needs RelCloud >= 0, Rain >= 0, T0 > 0 and L00 > 0");
  if (d->HorLimit && (d->NumTr < 1 || !d->w))
    return fail(c, CGD_ERR_ARG, who + "HorLimit needs tracers (NumTr > 0) and the GLL weights w");
  if (d->Damping && (!d->zP || !(d->DampStride > 0.0) || !(d->DampH > 0.0)))
    return fail(c, CGD_ERR_ARG, who + "Damping needs zP, DampH > 0 and DampStride > 0");
  if (d->Forcing && (!d->xS || !(d->HS_sigma_b > 0.0 && d->HS_sigma_b < 1.0)))
    return fail(c, CGD_ERR_ARG, who + "Forcing needs xS and 0 < HS_sigma_b < 1");
  if (d->State != CGD_DRY && d->State != CGD_MOIST) return fail(c, CGD_ERR_UNSUPPORTED, who + "unknown State");
  if (d->State == CGD_MOIST) {
    const int hi = 5 + d->NumTr;
    if (d->RhoVPos < 6 || d->RhoVPos > hi || d->RhoCPos < 6 || d->RhoCPos > hi || d->RhoVPos == d->RhoCPos)
      return fail(c, CGD_ERR_ARG, who + "Moist needs RhoVPos != RhoCPos among the tracer components 6..5+NumTr");
    if (!(d->Cpv > 0.0 && d->Cpl > 0.0 && d->Rv > 0.0))
      return fail(c, CGD_ERR_ARG, who + "Moist needs Cpv, Cpl, Rv > 0");
  }
  if (!(d->SmoothW >= 0.0) || !(d->SmoothC >= 0.0))
    return fail(c, CGD_ERR_ARG, who + "SmoothW and SmoothC must be >= 0");
  if ((d->SmoothW > 0.0 || d->SmoothC > 0.0) && (d->NumTr > 0 || d->HorLimit || d->precision != CGD_FP64))
    return fail(c, CGD_ERR_UNSUPPORTED,
                who + "kink smoothing is implemented for the dry FP64 dynamics (no tracers, HorLimit or mixed)");
  if (d->HyperDDivW != 0.0)
    return fail(c, CGD_ERR_UNSUPPORTED, who + "HyperDDivW > 0 (w hyperviscosity) is not implemented");
  if (!d->Glob || !d->DS || !d->DW || !d->dXdxI || !d->J || !d->X || !d->M || !d->dz)
    return fail(c, CGD_ERR_ARG, who + "null static input pointer");
  return CGD_OK;
}

// Context over nmem grids ("members") stepped together.  Their meshes are
// concatenated: member m's elements and global nodes follow those of members
// 0..m-1, so the state of the batch is one (Nz, sum NumG, 5) array.  Each
// member is coloured on its own and colour k of the batch is the union of
// the members' colour k, so each node sums its element contributions in the
// order a context of its member alone uses: a member's results are
// bit-identical either way.
static int ctx_build(cgd_ctx *c, const cgd_desc *ds, int nmem, hipStream_t st) {
  int r;
  for (int m = 0; m < nmem; ++m) {
    const std::string who = nmem > 1 ? "member " + std::to_string(m) + ": " : "";
    if ((r = validate_desc(c, &ds[m], who))) return r;
    const cgd_desc &a = ds[0], &b = ds[m];
    if (b.N != a.N || b.Nz != a.Nz || b.precision != a.precision || b.NumTr != a.NumTr)
      return fail(c, CGD_ERR_ARG, who + "N, Nz, NumTr and precision must be the same for every member");
    if (b.Grav != a.Grav || b.Omega != a.Omega || b.Rd != a.Rd || b.Cpd != a.Cpd || b.p0 != a.p0 ||
        b.kappa != a.kappa)
      return fail(c, CGD_ERR_ARG, who + "physical constants must be the same for every member");
    if (b.State != a.State || (a.State == CGD_MOIST && (b.RhoVPos != a.RhoVPos || b.RhoCPos != a.RhoCPos ||
                                                        b.Cpv != a.Cpv || b.Cpl != a.Cpl || b.Rv != a.Rv)))
      return fail(c, CGD_ERR_ARG, who + "State and the moist constants must be the same for every member");
    if (b.Microphysics != a.Microphysics ||
        (a.Microphysics && (b.RelCloud != a.RelCloud || b.Rain != a.Rain || b.T0 != a.T0 || b.L00 != a.L00)))
      return fail(c, CGD_ERR_ARG, who + "Microphysics and its constants must be the same for every member");
    if (b.Damping != a.Damping || b.Forcing != a.Forcing ||
        (a.Damping && (b.DampH != a.DampH || b.DampStride != a.DampStride || b.DampRelax != a.DampRelax)) ||
        (a.Forcing && (b.HS_k_a != a.HS_k_a || b.HS_k_f != a.HS_k_f || b.HS_k_s != a.HS_k_s ||
                       b.HS_DeltaT_y != a.HS_DeltaT_y || b.HS_DeltaTh_z != a.HS_DeltaTh_z ||
                       b.HS_T_equator != a.HS_T_equator || b.HS_T_min != a.HS_T_min ||
                       b.HS_sigma_b != a.HS_sigma_b)))
      return fail(c, CGD_ERR_ARG, who + "physics hooks and their constants must be the same for every member");
    if ((b.HorLimit != 0) != (a.HorLimit != 0))
      return fail(c, CGD_ERR_ARG, who + "HorLimit must be the same for every member");
    if (b.SmoothW != a.SmoothW || b.SmoothC != a.SmoothC)
      return fail(c, CGD_ERR_ARG, who + "SmoothW and SmoothC must be the same for every member");
  }
  const cgd_desc *d = &ds[0];
  c->desc = *d;
  c->mixed = d->precision == CGD_MIXED;
  c->ntr = d->NumTr;
  c->smooth = d->SmoothW > 0.0 || d->SmoothC > 0.0;
  c->ka.smw = d->SmoothW;
  c->ka.smc = d->SmoothC;
  c->nmem = nmem;
  c->N = d->N;
  c->NN = d->N * d->N;
  c->Nz = d->Nz;
  const int NN = c->NN, Nz = c->Nz;
  size_t nf_tot = 0, ng_tot = 0;
  c->mem_e0.assign(nmem + 1, 0);
  c->mem_g0.assign(nmem + 1, 0);
  for (int m = 0; m < nmem; ++m) {
    nf_tot += ds[m].NF;
    ng_tot += ds[m].NumG;
    if (nf_tot >= (size_t)1 << 31 || ng_tot >= (size_t)1 << 31) return fail(c, CGD_ERR_ARG, "grid too large");
    c->mem_e0[m + 1] = (int)nf_tot;
    c->mem_g0[m + 1] = (int)ng_tot;
  }
  if (nf_tot * NN * Nz > (size_t)1 << 40) return fail(c, CGD_ERR_ARG, "grid too large");
  // the element kernels index a field with 32-bit offsets
  if (ng_tot * Nz >= (size_t)1 << 28 || (size_t)NN * Nz >= (size_t)1 << 28)
    return fail(c, CGD_ERR_ARG, "NumG*Nz (summed over members) must be below 2^28");
  c->NF = (int)nf_tot;
  c->NumG = (int)ng_tot;
  const int NF = c->NF, NumG = c->NumG;
  // level chunk height NZT (a template constant): a workgroup is one
  // element x NZT levels, N*N*NZT lanes rounded up to whole wavefronts.
  // 8 levels measured fastest at ne=30, nz=64 (5 and 10 fill the
  // wavefronts better but straddle cache lines); CGD_NZT=16 overrides, and
  // cgd_set_launch_shape / cgd_autotune change it later.
  {
    c->base_nzt = 8;
    if (const char *ev = getenv("CGD_NZT")) {
      const int o = atoi(ev);
      if (o == 16 && c->N == 5) c->base_nzt = o;
    }
    if (const char *ev = getenv("CGD_THOMAS")) c->thomas = atoi(ev) != 0;
  }
  c->colw = 64;
  c->colblock = 256;
  c->items1 = 1;

  // global numbering -> 0-based int32 in batch numbering, range checks, and
  // each member's colouring
  std::vector<int> g32((size_t)NN * NF), color(NF, -1);
  std::vector<double> hds(NN), hdw(NN);
  int ncol = 0;
  for (int m = 0; m < nmem; ++m) {
    const cgd_desc &dm = ds[m];
    std::vector<int64_t> hglob((size_t)NN * dm.NF);
    std::vector<double> mds(NN), mdw(NN);
    HIPCHK(c, hipMemcpyAsync(hglob.data(), dm.Glob, hglob.size() * sizeof(int64_t), hipMemcpyDeviceToHost, st));
    HIPCHK(c, hipMemcpyAsync(mds.data(), dm.DS, NN * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(c, hipMemcpyAsync(mdw.data(), dm.DW, NN * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(c, hipStreamSynchronize(st));
    if (m == 0) {
      hds = mds;
      hdw = mdw;
    } else if (mds != hds || mdw != hdw) {
      return fail(c, CGD_ERR_ARG, "member " + std::to_string(m) + ": DS and DW must be the same for every member");
    }
    std::vector<int> gm(hglob.size());
    for (size_t i = 0; i < gm.size(); ++i) {
      if (hglob[i] < 1 || hglob[i] > dm.NumG) return fail(c, CGD_ERR_ARG, "Glob entry outside 1..NumG");
      gm[i] = (int)(hglob[i] - 1);
      g32[(size_t)c->mem_e0[m] * NN + i] = gm[i] + c->mem_g0[m];
    }
    std::vector<int> cm;
    const int nc = color_elements(gm, NN, dm.NF, dm.NumG, cm);
    if (nc < 0) return fail(c, CGD_ERR_ARG, "element colouring needs more than 64 colours");
    ncol = std::max(ncol, nc);
    std::copy(cm.begin(), cm.end(), color.begin() + c->mem_e0[m]);
  }
  c->ncolor = ncol;
  c->color_off.assign(ncol + 1, 0);
  for (int e = 0; e < NF; ++e) c->color_off[color[e] + 1]++;
  for (int k = 0; k < ncol; ++k) c->color_off[k + 1] += c->color_off[k];
  // elements are stored in the caller's order (neighbours lie close, so the
  // nodes they share are read again while cached); elist: colour by colour,
  // then member, then element number within the member
  std::vector<int> elist(NF);
  {
    std::vector<int> fp(c->color_off.begin(), c->color_off.end() - 1);
    for (int e = 0; e < NF; ++e) elist[fp[color[e]]++] = e;
  }
  // global node -> element copies (e*NN + node) in colour order
  std::vector<int> cptr(NumG + 1, 0), ccopy((size_t)NF * NN);
  for (int v : g32) cptr[v + 1]++;
  for (int i = 0; i < NumG; ++i) cptr[i + 1] += cptr[i];
  {
    std::vector<int> fp(cptr.begin(), cptr.end() - 1);
    for (int q = 0; q < NF; ++q) {
      const int e = elist[q];
      for (int i = 0; i < NN; ++i) ccopy[fp[g32[(size_t)e * NN + i]]++] = e * NN + i;
    }
  }
  // width of the fixed-width lists of the same (an even number)
  int mult = 4;
  for (int gn = 0; gn < NumG; ++gn) mult = std::max(mult, cptr[gn + 1] - cptr[gn]);
  const int cpw = (mult + 1) / 2 * 2;
  // numbering, bit 31 marking the first copy of each node
  std::vector<int> gslot = g32;
  for (int gn = 0; gn < NumG; ++gn)
    if (cptr[gn + 1] > cptr[gn]) gslot[ccopy[cptr[gn]]] |= (int)0x80000000u;
  // hyperviscosity per element (the member's coefficients)
  std::vector<double> kvis((size_t)NF * 3);
  for (int m = 0; m < nmem; ++m)
    for (int e = c->mem_e0[m]; e < c->mem_e0[m + 1]; ++e) {
      kvis[(size_t)e * 3] = ds[m].HyperDCurl;
      kvis[(size_t)e * 3 + 1] = ds[m].HyperDGrad;
      kvis[(size_t)e * 3 + 2] = ds[m].HyperDDiv;
    }
  // HorLimit: the stencil of every element (FE.Stencil, NumberingFem.jl:133-157:
  // the element and those sharing a grid node with it, padded with itself)
  c->horlimit = d->HorLimit != 0;
  std::vector<int> stencil;
  if (c->horlimit) {
    std::vector<int> aptr, adj;
    element_adjacency(g32, NN, NF, NumG, aptr, adj);
    stencil.assign((size_t)NF * 13, 0);
    for (int e = 0; e < NF; ++e) {
      const int q = e;
      if (aptr[e + 1] - aptr[e] > 12) return fail(c, CGD_ERR_ARG, "HorLimit: an element has more than 12 neighbours");
      for (int k = 0; k < 13; ++k) stencil[(size_t)q * 13 + k] = q;
      for (int k = aptr[e]; k < aptr[e + 1]; ++k) stencil[(size_t)q * 13 + 1 + (k - aptr[e])] = adj[k];
    }
    std::vector<double> wg(c->N);
    HIPCHK(c, hipMemcpyAsync(wg.data(), d->w, c->N * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(c, hipStreamSynchronize(st));
    for (int i = 0; i < c->N; ++i) c->ka.wg[i] = wg[i];
  }
  // device buffers (set-up only; nothing is allocated on the step path).
  // The chunk-interface side buffer is sized for the shortest chunk height
  // (8 levels), so the launch shape can change later.
  const size_t npt = (size_t)NF * NN * Nz;
  const size_t ng = (size_t)NumG * Nz;
  const int nchunk_max = (Nz + 7) / 8;
  HIPCHK(c, hipMalloc(&c->d_glob, gslot.size() * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_clist, (size_t)NF * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_cpy, (size_t)NF * NN * cpw * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_gcpy, (size_t)NumG * cpw * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_e1, npt * (5 + c->ntr) * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_e2, npt * (5 + c->ntr) * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_met, npt * CGD_NMET * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_met1, npt * CGD_NMET1 * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_ms, ng * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_f4x, (size_t)NF * NN * nchunk_max * sizeof(double)));
  HIPCHK(c, hipMalloc(&c->d_nptr, cptr.size() * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_ncopy, ccopy.size() * sizeof(int)));
  HIPCHK(c, hipMalloc(&c->d_kvis, kvis.size() * sizeof(double)));
  HIPCHK(c, hipMemcpyAsync(c->d_nptr, cptr.data(), cptr.size() * sizeof(int), hipMemcpyHostToDevice, st));
  HIPCHK(c, hipMemcpyAsync(c->d_ncopy, ccopy.data(), ccopy.size() * sizeof(int), hipMemcpyHostToDevice, st));
  HIPCHK(c, hipMemcpyAsync(c->d_glob, gslot.data(), gslot.size() * sizeof(int), hipMemcpyHostToDevice, st));
  HIPCHK(c, hipMemcpyAsync(c->d_clist, elist.data(), elist.size() * sizeof(int), hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_copy_lists, dim3(grid_for((size_t)NumG + (size_t)NF * NN, 256)), dim3(256), 0, st, c->d_nptr,
                     c->d_ncopy, c->d_glob, NumG, NF * NN, cpw, c->d_gcpy, c->d_cpy);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipMemcpyAsync(c->d_kvis, kvis.data(), kvis.size() * sizeof(double), hipMemcpyHostToDevice, st));
  if (c->horlimit) {
    const size_t nb = (size_t)c->ntr * NF * Nz;
    HIPCHK(c, hipMalloc(&c->d_stencil, stencil.size() * sizeof(int)));
    HIPCHK(c, hipMalloc(&c->d_qmin, nb * sizeof(double)));
    HIPCHK(c, hipMalloc(&c->d_qmax, nb * sizeof(double)));
    HIPCHK(c, hipMemcpyAsync(c->d_stencil, stencil.data(), stencil.size() * sizeof(int), hipMemcpyHostToDevice, st));
  }
  // M and dz in batch numbering (a single grid's arrays are used in place)
  c->hooks.forcing = d->Forcing != 0;
  c->hooks.damping = d->Damping != 0;
  c->hooks.k_a = d->HS_k_a;
  c->hooks.k_f = d->HS_k_f;
  c->hooks.k_s = d->HS_k_s;
  c->hooks.DeltaT_y = d->HS_DeltaT_y;
  c->hooks.DeltaTh_z = d->HS_DeltaTh_z;
  c->hooks.T_equator = d->HS_T_equator;
  c->hooks.T_min = d->HS_T_min;
  c->hooks.sigma_b = d->HS_sigma_b;
  c->hooks.H = d->DampH;
  c->hooks.Stride = d->DampStride;
  c->hooks.Relax = d->DampRelax;
  c->hooks.micro = d->Microphysics != 0;
  c->hooks.RelCloud = d->RelCloud;
  c->hooks.Rain = d->Rain;
  c->hooks.T0 = d->T0;
  c->hooks.L00 = d->L00;
  if (nmem == 1) {
    c->M = d->M;
    c->dz = d->dz;
    c->hooks.zP = d->zP;
    c->hooks.xS = d->xS;
  } else {
    if (d->Damping) HIPCHK(c, hipMalloc(&c->d_zP, ng * sizeof(double)));
    if (d->Forcing) HIPCHK(c, hipMalloc(&c->d_xS, 2 * (size_t)NumG * sizeof(double)));
    for (int m = 0; m < nmem; ++m) {
      const size_t gm = (size_t)ds[m].NumG * Nz, o = (size_t)c->mem_g0[m] * Nz;
      if (d->Damping)
        HIPCHK(c, hipMemcpyAsync(c->d_zP + o, ds[m].zP, gm * sizeof(double), hipMemcpyDeviceToDevice, st));
      if (d->Forcing)
        HIPCHK(c, hipMemcpyAsync(c->d_xS + 2 * (size_t)c->mem_g0[m], ds[m].xS, 2 * (size_t)ds[m].NumG * sizeof(double),
                                 hipMemcpyDeviceToDevice, st));
    }
    c->hooks.zP = c->d_zP;
    c->hooks.xS = c->d_xS;
    HIPCHK(c, hipMalloc(&c->d_M, 2 * ng * sizeof(double)));
    HIPCHK(c, hipMalloc(&c->d_dz, ng * sizeof(double)));
    for (int m = 0; m < nmem; ++m) {
      const size_t gm = (size_t)ds[m].NumG * Nz, o = (size_t)c->mem_g0[m] * Nz;
      for (int t = 0; t < 2; ++t)
        HIPCHK(c, hipMemcpyAsync(c->d_M + t * ng + o, ds[m].M + t * gm, gm * sizeof(double),
                                 hipMemcpyDeviceToDevice, st));
      HIPCHK(c, hipMemcpyAsync(c->d_dz + o, ds[m].dz, gm * sizeof(double), hipMemcpyDeviceToDevice, st));
    }
    c->M = c->d_M;
    c->dz = c->d_dz;
  }
  for (int m = 0; m < nmem; ++m) {
    const size_t nptm = (size_t)ds[m].NF * NN * Nz;
    hipLaunchKernelGGL(k_relayout_metric, dim3(grid_for(nptm, 256)), dim3(256), 0, st, ds[m].dXdxI, ds[m].J,
                       ds[m].X, (size_t)c->mem_e0[m], c->d_met, c->d_met1, NN, Nz, ds[m].NF, d->Omega);
    HIPCHK(c, hipGetLastError());
  }
  hipLaunchKernelGGL(k_msum, dim3(grid_for(ng, 256)), dim3(256), 0, st, c->M, c->d_ms, ng);
  HIPCHK(c, hipGetLastError());
  // compact metric layout when every component but the terrain row has the
  // same bits at all levels (CGD_METRIC=full keeps the full layout)
  {
    const char *ev = getenv("CGD_METRIC");
    const bool allow = !(ev && strcmp(ev, "full") == 0);
    unsigned *d_mask = nullptr;
    unsigned hmask[2] = {~0u, ~0u};
    if (allow) {
      HIPCHK(c, hipMalloc(&d_mask, 2 * sizeof(unsigned)));
      HIPCHK(c, hipMemsetAsync(d_mask, 0, 2 * sizeof(unsigned), st));
      hipLaunchKernelGGL(k_met_invariant, dim3(1024), dim3(256), 0, st, c->d_met, CGD_NMET, NF, NN, Nz, d_mask);
      hipLaunchKernelGGL(k_met_invariant, dim3(1024), dim3(256), 0, st, c->d_met1, CGD_NMET1, NF, NN, Nz,
                         d_mask + 1);
      HIPCHK(c, hipGetLastError());
      HIPCHK(c, hipMemcpyAsync(hmask, d_mask, sizeof(hmask), hipMemcpyDeviceToHost, st));
      HIPCHK(c, hipStreamSynchronize(st));
      HIPCHK(c, hipFree(d_mask));
    }
    unsigned per_point = 0;
    for (int q = 0; q < CGD_NMET; ++q)
      if (met_per_point(q)) per_point |= 1u << q;
    if (allow && (hmask[0] & ~per_point) == 0 && hmask[1] == 0) {
      double *metp = nullptr;
      HIPCHK(c, hipMalloc(&metp, npt * CGD_NMETP * sizeof(double)));
      HIPCHK(c, hipMalloc(&c->d_metn, (size_t)NF * NN * CGD_NMETN * sizeof(double)));
      HIPCHK(c, hipMalloc(&c->d_met1n, (size_t)NF * NN * CGD_NMET1 * sizeof(double)));
      hipLaunchKernelGGL(k_met_compact, dim3(grid_for(npt, 256)), dim3(256), 0, st, c->d_met, c->d_met1, metp,
                         c->d_metn, c->d_met1n, NF, NN, Nz);
      HIPCHK(c, hipGetLastError());
      HIPCHK(c, hipStreamSynchronize(st));
      HIPCHK(c, hipFree(c->d_met));
      HIPCHK(c, hipFree(c->d_met1));
      c->d_met = metp;
      c->d_met1 = nullptr;
      c->cm = 1;
      // regular (CGD_METRIC=compact keeps the general kernel)
      int *d_bad = nullptr, bad = 1;
      HIPCHK(c, hipMalloc(&d_bad, sizeof(int)));
      HIPCHK(c, hipMalloc(&c->d_iMn, (size_t)NumG * sizeof(double)));
      HIPCHK(c, hipMemsetAsync(d_bad, 0, sizeof(int), st));
      hipLaunchKernelGGL(k_met_regular, dim3(2048), dim3(256), 0, st, c->d_metn, c->d_met, c->M, c->d_ms, NF, NN, NumG,
                         Nz, c->d_iMn, d_bad);
      HIPCHK(c, hipGetLastError());
      HIPCHK(c, hipMemcpyAsync(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, st));
      HIPCHK(c, hipStreamSynchronize(st));
      HIPCHK(c, hipFree(d_bad));
      c->reg = !bad && !(ev && strcmp(ev, "compact") == 0);
    }
  }
  if (c->mixed) {
    HIPCHK(c, hipMalloc(&c->d_ims32, ng * sizeof(float)));
    hipLaunchKernelGGL(k_to_f32, dim3(grid_for(ng, 256)), dim3(256), 0, st, c->d_ms, c->d_ims32, ng);
    HIPCHK(c, hipMalloc(&c->d_m32, 2 * ng * sizeof(float)));
    hipLaunchKernelGGL(k_to_f32, dim3(grid_for(2 * ng, 256)), dim3(256), 0, st, c->M, c->d_m32, 2 * ng);
    if (c->cm) {
      const size_t nmp = npt * CGD_NMETP;
      HIPCHK(c, hipMalloc(&c->d_metp32, nmp * sizeof(float)));
      hipLaunchKernelGGL(k_to_f32, dim3(grid_for(nmp, 256)), dim3(256), 0, st, c->d_met, c->d_metp32, nmp);
    }
    HIPCHK(c, hipGetLastError());
  }
  HIPCHK(c, hipStreamSynchronize(st));

  KArgs &a = c->ka;
  a.Nz = Nz;
  a.NumG = NumG;
  a.Grav = d->Grav;
  a.Omega = d->Omega;
  a.Rd = d->Rd;
  a.Cpd = d->Cpd;
  a.p0 = d->p0;
  a.kappa = d->kappa;
  a.Rd_p0 = d->Rd / d->p0;
  a.eos_y = 1.0 / (1.0 - d->kappa);
  a.Rd_Cpd = d->Rd / d->Cpd;
  a.dpd_y = d->kappa / (1.0 - d->kappa);
  // DS, DW arrive column-major (Julia): DS[i,k] at i + N*k
  for (int i = 0; i < c->N; ++i)
    for (int k = 0; k < c->N; ++k) {
      a.D[i * c->N + k] = hds[i + c->N * k];
      a.DWm[i * c->N + k] = hdw[i + c->N * k];
      a.Df[i * c->N + k] = (float)a.D[i * c->N + k];
      a.DWf[i * c->N + k] = (float)a.DWm[i * c->N + k];
    }
  a.glob = c->d_glob;
  a.clist = c->d_clist;
  a.cpy = c->d_cpy;
  a.gcpy = c->d_gcpy;
  a.cpw = cpw;
  a.ecs = npt;
  a.met = c->d_met;
  a.metn = c->d_metn;
  a.met1n = c->d_met1n;
  a.met1 = c->d_met1;
  a.iMs = c->d_ms;
  a.iMs32 = c->d_ims32;
  a.M32 = c->d_m32;
  a.metp32 = c->d_metp32;
  a.M = c->M;
  a.iMn = c->reg ? c->d_iMn : nullptr;
  a.kvis = c->d_kvis;
  a.iv = d->State == CGD_MOIST ? d->RhoVPos - 1 : -1;
  a.ic = d->State == CGD_MOIST ? d->RhoCPos - 1 : -1;
  a.Cpv = d->Cpv;
  a.Cpl = d->Cpl;
  a.Rv = d->Rv;
  // persistent stage launches: the grid barrier (zero)
  HIPCHK(c, hipMalloc(&c->d_bar, sizeof(GridBar)));
  HIPCHK(c, hipMemsetAsync(c->d_bar, 0, sizeof(GridBar), st));
  HIPCHK(c, hipStreamSynchronize(st));
  {
    int dev = 0, khz = 0;
    HIPCHK(c, hipGetDevice(&dev));
    HIPCHK(c, hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    c->bar_ticks = (long long)std::max(khz, 1000) * 250;  // 250 ms
  }
  // Pass 1 over whole columns has a lane per level, so that it pays where most
  // lanes have one.  Kernel times at ne = 30, p = 4, columns against 8-level
  // chunks: nz = 64 115 against 178 us, 61 119 and 190, 57 118 and 184, 48 104
  // and 131; nz = 32 94 and 88 (a step 1.1 % slower).  The steps at 48..64 gain
  // 2 to 6 %.  (44 and 40 would gain too, 3.4 and 1.4 %; the line lies where it
  // was drawn before they were timed.)
  const bool col1 = columns_ok(c) && Nz >= 48;
  // 16 levels per workgroup where that pads no more levels than 8 do (nz = 40,
  // padded to 48: pass 1 15 %, pass 2 25 % slower): 128-byte pieces of the
  // columns, and in pass 2 half the halo levels.
  // Pass 1, where it can't take whole columns and the grid leaves the chip a few
  // rounds of workgroups (the height changes no bit there): a step of 32 grids
  // of 32 levels 1.5 % faster, steps at ne = 20..45, nz = 9..32 0 to 2 %.
  // Pass 2 on a regular metric, where the height changes no bit either:
  // steps with 16 against 8 levels, nz = 64: ne = 60 9.78 and 9.88 ms, ne = 30
  // 2.451 and 2.498, ne = 16 0.725 and 0.720; ne = 30, nz = 48 1.959 and 1.999,
  // 57 and 61 equal; ne = 20, nz = 80 1.623 and 1.634; at nz = 32 the kernel is no
  // faster, so from 48 levels on.
  const bool tall = c->N == 5 && !(((Nz + 7) / 8) & 1);
  const bool p16 = tall && c->cm && !col1 && (size_t)NF * ((Nz + 15) / 16) >= 4096;
  c->r16 = tall && Nz >= 48 && c->reg && !c->smooth;
  c->nzt = c->rule_nzt = c->r16 && !(c->mixed && Nz <= 64) ? 16 : c->base_nzt;  // that of the steps' tendency
  c->nzt1 = c->rule_nzt1 = col1 ? 64 : p16 ? 16 : c->base_nzt;
  c->ok = true;
  return CGD_OK;
}

extern "C" int cgd_ctx_create(const cgd_desc *d, cgd_ctx **out, void *stream) {
  if (!out) return CGD_ERR_ARG;
  *out = nullptr;
  cgd_ctx *c = new cgd_ctx();
  *out = c;
  if (!d) return fail(c, CGD_ERR_ARG, "null descriptor");
  return ctx_build(c, d, 1, S(stream));
}

extern "C" int cgd_ctx_create_batch(const cgd_desc *members, int nmem, cgd_ctx **out, void *stream) {
  if (!out) return CGD_ERR_ARG;
  *out = nullptr;
  cgd_ctx *c = new cgd_ctx();
  *out = c;
  if (!members) return fail(c, CGD_ERR_ARG, "null member array");
  if (nmem < 1 || nmem > 65536) return fail(c, CGD_ERR_ARG, "member count must be in [1, 65536]");
  return ctx_build(c, members, nmem, S(stream));
}

static void graph_free(cgd_ctx *c);
static void prof_free(cgd_ctx *c);

extern "C" int cgd_ctx_destroy(cgd_ctx *c) {
  if (!c) return CGD_ERR_ARG;
  // a context that failed validation holds no device memory: tear it down
  // without touching the HIP runtime
  graph_free(c);
  if (c->gstream) (void)hipStreamDestroy(c->gstream);
  if (c->ev_last) (void)hipEventDestroy(c->ev_last);
  for (void *p : {(void *)c->d_stencil, (void *)c->d_qmin, (void *)c->d_qmax})
    if (p) (void)hipFree(p);
  for (void *p : {(void *)c->d_glob, (void *)c->d_clist, (void *)c->d_cpy, (void *)c->d_gcpy,
                  (void *)c->d_e1, (void *)c->d_e2, (void *)c->d_iMn, (void *)c->d_met, (void *)c->d_met1, (void *)c->d_metn,
                  (void *)c->d_met1n, (void *)c->d_ms, (void *)c->d_ims32, (void *)c->d_m32, (void *)c->d_metp32,
                  (void *)c->d_f4x, (void *)c->d_nptr, (void *)c->d_ncopy, (void *)c->d_kvis,
                  (void *)c->d_M, (void *)c->d_dz, (void *)c->d_zP, (void *)c->d_xS, (void *)c->d_bar})
    if (p) (void)hipFree(p);
  prof_free(c);
  delete c;
  return CGD_OK;
}

static int check(cgd_ctx *c) {
  if (!c) return CGD_ERR_ARG;
  if (!c->ok) return fail(c, CGD_ERR_STATE, "context creation failed: " + c->err);
  return CGD_OK;
}

// Timing of one pass (a group of launches): an event pair is recorded on the
// launch stream; nothing synchronises until cgd_profile_read.  The events
// are created by cgd_profile_enable (never on the step path).
static void prof_begin(cgd_ctx *c, hipStream_t st, int which) {
  if (!(c->prof >> which & 1) || c->prof_used >= c->prof_cap) return;
  (void)hipEventRecord(c->prof_ev[2 * c->prof_used], st);
}
static int prof_end(cgd_ctx *c, hipStream_t st, int which, int launches) {
  if (!(c->prof >> which & 1) || c->prof_used >= c->prof_cap) return CGD_OK;
  HIPCHK(c, hipEventRecord(c->prof_ev[2 * c->prof_used + 1], st));
  c->prof_which.push_back(which);
  c->prof_launch.push_back(launches);
  c->prof_used++;
  return CGD_OK;
}

static void prof_free(cgd_ctx *c) {
  for (hipEvent_t e : c->prof_ev) (void)hipEventDestroy(e);
  c->prof_ev.clear();
  c->prof_which.clear();
  c->prof_launch.clear();
  c->prof_cap = c->prof_used = 0;
}

extern "C" int cgd_profile_enable(cgd_ctx *c, int on) {
  int r = check(c);
  if (r) return r;
  prof_free(c);
  for (int i = 0; i < 3; ++i) c->prof_ms[i] = 0, c->prof_n[i] = 0;
  c->prof = on & 7;
  if (c->prof) {
    const int cap = 4096;
    c->prof_ev.resize(2 * cap);
    for (auto &e : c->prof_ev) HIPCHK(c, hipEventCreate(&e));
    c->prof_cap = cap;
  }
  return CGD_OK;
}

extern "C" int cgd_profile_read(cgd_ctx *c, int which, double *total_ms, long long *launches) {
  int r = check(c);
  if (r) return r;
  if (which < 0 || which > 2 || !total_ms || !launches) return fail(c, CGD_ERR_ARG, "bad profile query");
  // fold recorded pairs into the totals
  for (int i = 0; i < c->prof_used; ++i) {
    HIPCHK(c, hipEventSynchronize(c->prof_ev[2 * i + 1]));
    float ms = 0;
    HIPCHK(c, hipEventElapsedTime(&ms, c->prof_ev[2 * i], c->prof_ev[2 * i + 1]));
    c->prof_ms[c->prof_which[i]] += ms;
    c->prof_n[c->prof_which[i]] += c->prof_launch[i];
  }
  c->prof_used = 0;
  c->prof_which.clear();
  c->prof_launch.clear();
  *total_ms = c->prof_ms[which];
  *launches = c->prof_n[which];
  return CGD_OK;
}


// template dispatch on (N, chunk height, metric layout); R is the tendency
// type (double, or float in the mixed-precision mode)
template <int N, int NZT, bool CM, typename R>
static void fcn1_t(cgd_ctx *c, hipStream_t st, const R *UR, R *E, const double *U64, double *Eth) {
  const int nchunk = (c->Nz + NZT - 1) / NZT, nitems = c->NF * nchunk;
  const dim3 b(tile_block(c, NZT));
  const size_t lds = lds_fcn1<R>(c, NZT);
  if (c->items1 == 2)
    hipLaunchKernelGGL((k_fcn1<N, NZT, CM, R, 2>), dim3((nitems + 1) / 2), b, lds, st, c->ka, nchunk, nitems, UR, E,
                       U64, Eth);
  else
    hipLaunchKernelGGL((k_fcn1<N, NZT, CM, R, 1>), dim3(nitems), b, lds, st, c->ka, nchunk, nitems, UR, E, U64, Eth);
}
template <int N, int NZT, bool CM, typename R>
static void fcn2_t(cgd_ctx *c, hipStream_t st, const double *U, const R *UR, const R *E1, const double *P, R *E2,
                   const double *E1th, double *Cout) {
  const int nchunk = nchunks(c, NZT);
  const dim3 g(c->NF * nchunk), b(tile_block(c, NZT));
  if constexpr (std::is_same<R, double>::value && CM) {
    if (c->reg && !c->smooth) {
      hipLaunchKernelGGL((k_fcn2r<N, NZT>), g, b, lds_fcn2r(c, NZT), st, c->ka, nchunk, U, E1, P, E2, c->d_f4x, Cout);
      return;
    }
  }
  const size_t lds = lds_fcn2<R>(c, NZT);
  R *const F4x = reinterpret_cast<R *>(c->d_f4x);
  if constexpr (std::is_same<R, double>::value) {
    if (c->smooth) {  // kink-smoothed upwind flux (FP64 only)
      hipLaunchKernelGGL((k_fcn2<N, NZT, CM, R, true>), g, b, lds, st, c->ka, nchunk, U, UR, E1, P, E2, F4x, E1th, Cout);
      return;
    }
  }
  hipLaunchKernelGGL((k_fcn2<N, NZT, CM, R, false>), g, b, lds, st, c->ka, nchunk, U, UR, E1, P, E2, F4x, E1th, Cout);
}
#define CGD_DISPATCH(FN, R, NZTV, ...)                             \
  do {                                                             \
    if (c->N == 5 && (NZTV) == 16) {                               \
      if (c->cm) FN<5, 16, true, R>(c, __VA_ARGS__);               \
      else FN<5, 16, false, R>(c, __VA_ARGS__);                    \
    } else if (c->N == 5) {                                        \
      if (c->cm) FN<5, 8, true, R>(c, __VA_ARGS__);                \
      else FN<5, 8, false, R>(c, __VA_ARGS__);                     \
    } else {                                                       \
      if (c->cm) FN<4, 8, true, R>(c, __VA_ARGS__);                \
      else FN<4, 8, false, R>(c, __VA_ARGS__);                     \
    }                                                              \
  } while (0)
// the tracers' element copies: components 5.. of d_e1 and d_e2, FP64 in both modes
template <int N, int NZT, bool CM, typename R>
static void tr1_t(cgd_ctx *c, hipStream_t st, const double *U) {
  const size_t lds = sizeof(double) * (2 * c->NN + 3 * c->NN * NZT);
  const int nchunk = nchunks(c, NZT);
  hipLaunchKernelGGL((k_tr1<N, NZT, CM>), dim3(c->NF * nchunk), dim3(tile_block(c, NZT)), lds, st, c->ka, nchunk,
                     c->ntr, U, c->d_e1 + 5 * c->ka.ecs);
}
template <int N, int NZT, bool CM, typename R>
static void tr2_t(cgd_ctx *c, hipStream_t st, const double *U, double *Cout) {
  const size_t lds = sizeof(double) * (2 * c->NN + 10 * c->NN * NZT);
  const int nchunk = nchunks(c, NZT);
  hipLaunchKernelGGL((k_tr2<N, NZT, CM>), dim3(c->NF * nchunk), dim3(tile_block(c, NZT)), lds, st, c->ka, nchunk,
                     c->ntr, U, c->d_e1 + 5 * c->ka.ecs, Cout, c->d_e2 + 5 * c->ka.ecs);
}

template <int N, int NZT, bool CM, typename R>
static void tr2lim_t(cgd_ctx *c, hipStream_t st, const double *U) {
  const size_t lds = sizeof(double) * (c->NN + 7 * c->NN * NZT);
  const int nchunk = nchunks(c, NZT);
  hipLaunchKernelGGL((k_tr2_lim<N, NZT, CM>), dim3(c->NF * nchunk), dim3(tile_block(c, NZT)), lds, st, c->ka, nchunk,
                     c->ntr, U, c->d_stencil, c->NF, c->d_qmin, c->d_qmax, c->dtau, c->d_e2 + 5 * c->ka.ecs);
}

template <typename R>
static void launch_fcn1(cgd_ctx *c, hipStream_t st, const R *UR, R *E, const double *U64, double *Eth) {
  if (cache_nzt(c) == 64) {
    const size_t lds = lds_fcn1c(c, sizeof(R));
    if (c->N == 5) hipLaunchKernelGGL((k_fcn1c<5, R>), dim3(c->NF), dim3(320), lds, st, c->ka, UR, E, U64, Eth);
    else hipLaunchKernelGGL((k_fcn1c<4, R>), dim3(c->NF), dim3(256), lds, st, c->ka, UR, E, U64, Eth);
    return;
  }
  CGD_DISPATCH(fcn1_t, R, cache_nzt(c), st, UR, E, U64, Eth);
}
template <typename R>
static void launch_fcn2(cgd_ctx *c, hipStream_t st, const double *U, const R *UR, const R *E1, const double *P, R *E2,
                        const double *E1th, double *Cout) {
  CGD_DISPATCH(fcn2_t, R, tend_nzt<R>(c), st, U, UR, E1, P, E2, E1th, Cout);
}

extern "C" int cgd_prepare(cgd_ctx *c, const double *U, double *AuxG, void *stream) {
  int r = check(c);
  if (r) return r;
  if (!U || !AuxG) return fail(c, CGD_ERR_ARG, "cgd_prepare: null array");
  const size_t n = (size_t)c->NumG * c->Nz;
  const auto kernel = c->ka.iv >= 0 ? k_prepare<true> : k_prepare<false>;
  hipLaunchKernelGGL(kernel, dim3(grid_for(n, 256)), dim3(256), 0, S(stream), c->ka, U, AuxG, n);
  HIPCHK(c, hipGetLastError());
  return CGD_OK;
}

// Tendencies and steps use arrays of the context (the element copies, the
// chunk-interface terms, the limiter's bounds): a call on another stream than
// the last one waits for what that stream holds by then.  On one stream this
// is a comparison.  Calls that are being captured are ordered by the capture's
// owner; a last stream that no longer takes an event is waited for.
static int order_streams(cgd_ctx *c, hipStream_t st) {
  if (c->used && st == c->last) return CGD_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIPCHK(c, hipStreamIsCapturing(st, &cap));
  if (cap != hipStreamCaptureStatusNone) return CGD_OK;
  if (c->used) {
    if (!c->ev_last) HIPCHK(c, hipEventCreateWithFlags(&c->ev_last, hipEventDisableTiming));
    hipError_t e = hipStreamIsCapturing(c->last, &cap);
    if (e == hipSuccess && cap == hipStreamCaptureStatusNone) e = hipEventRecord(c->ev_last, c->last);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      HIPCHK(c, hipDeviceSynchronize());
    } else if (cap == hipStreamCaptureStatusNone) {
      HIPCHK(c, hipStreamWaitEvent(st, c->ev_last, 0));
    }
  }
  c->last = st;
  c->used = true;
  return CGD_OK;
}

static bool has_hooks(const cgd_ctx *c) { return c->hooks.forcing || c->hooks.damping || c->hooks.micro; }

// The element copies of the pass-1 cache (FP32 mode: four FP32 components,
// then the FP64 theta cache)
template <typename R> static double *e1_theta(cgd_ctx *c) {
  return std::is_same<R, double>::value ? nullptr : c->d_e1 + 4 * c->ka.ecs;
}

// Both tendency passes.  The dynamics' tendency ends as element copies in
// d_e2; with want_f (cgd_fcn; U = UR, R = double) and wherever physics hooks
// add to it, it is summed into F, and with want_f the cache into Temp1.
// The tracers' likewise (into F for the microphysics too; the steps sum them
// in k_rw_tr).
// U is the FP64 state; UR the state the R-typed terms read (U itself, or
// its FP32 shadow).
template <typename R>
static int run_fcn(cgd_ctx *c, R *F, const double *U, const R *UR, R *Temp1, const double *AuxG, hipStream_t st,
                   bool want_f) {
  int r = order_streams(c, st);
  if (r) return r;
  R *const E1 = reinterpret_cast<R *>(c->d_e1), *const E2 = reinterpret_cast<R *>(c->d_e2);
  double *const E1th = e1_theta<R>(c);
  prof_begin(c, st, 0);
  int launches = 1;
  launch_fcn1<R>(c, st, UR, E1, U, E1th);
  HIPCHK(c, hipGetLastError());
  // the tracers run in FP64 in both modes: their tendencies and caches are
  // components 6.. of the FP64 F and Temp1 (the mixed mode's FP32 dynamics
  // occupies only the first five components' worth of those buffers)
  double *const Fd = reinterpret_cast<double *>(F);
  double *const T1d = reinterpret_cast<double *>(Temp1);
  if (c->ntr > 0 && !c->horlimit) {  // HorLimit: no tracer hyperviscosity (FcnGPU.jl:747-751)
    CGD_DISPATCH(tr1_t, double, tr_cache_nzt(c), st, U);
    HIPCHK(c, hipGetLastError());
    ++launches;
  }
  if ((r = prof_end(c, st, 0, launches))) return r;
  prof_begin(c, st, 1);
  launches = 0;
  launch_fcn2<R>(c, st, U, UR, E1, AuxG, E2, E1th, want_f ? T1d : nullptr);
  HIPCHK(c, hipGetLastError());
  ++launches;
  {
    if (c->ntr > 0 && c->horlimit) {
      // LimitKernel! on the state, then DivRhoTrUpwind3LimKernel!
      if (!(c->dtau > 0.0)) return fail(c, CGD_ERR_ARG, "HorLimit: the stage time step is not set (cgd_set_dtau)");
      const size_t nb = (size_t)c->ntr * c->NF * c->Nz;
      hipLaunchKernelGGL(k_lim_bounds, dim3(grid_for(nb, 256)), dim3(256), 0, st, c->ka, c->NF, c->NN, c->ntr, U,
                         c->d_qmin, c->d_qmax);
      HIPCHK(c, hipGetLastError());
      ++launches;
      CGD_DISPATCH(tr2lim_t, double, tr_tend_nzt(c), st, U);
      HIPCHK(c, hipGetLastError());
      ++launches;
    } else if (c->ntr > 0) {
      CGD_DISPATCH(tr2_t, double, tr_tend_nzt(c), st, U, want_f ? T1d : nullptr);
      HIPCHK(c, hipGetLastError());
      ++launches;
    }
    if (c->ntr > 0 && (want_f || c->hooks.micro)) {
      const size_t ng = (size_t)c->NumG * c->Nz;
      hipLaunchKernelGGL(k_tr_dss, dim3(grid_for(ng, 256), c->ntr), dim3(256), 0, st, c->ka, c->d_e2 + 5 * c->ka.ecs,
                         Fd + 5 * ng, (unsigned)ng);
      HIPCHK(c, hipGetLastError());
      ++launches;
    }
  }
  if (want_f || has_hooks(c)) {
    const dim3 g(grid_for((size_t)c->NumG * c->Nz, 256));
    const R *F4x = reinterpret_cast<const R *>(c->d_f4x);
    if (has_hooks(c))
      hipLaunchKernelGGL((k_dss<R, true>), g, dim3(256), 0, st, c->ka, c->hooks, U, AuxG, E2, F4x, F, Fd,
                         nchunks(c, f4_nzt<R>(c)), f4_nzt<R>(c));
    else
      hipLaunchKernelGGL((k_dss<R, false>), g, dim3(256), 0, st, c->ka, c->hooks, U, AuxG, E2, F4x, F, Fd,
                         nchunks(c, f4_nzt<R>(c)), f4_nzt<R>(c));
    HIPCHK(c, hipGetLastError());
    ++launches;
  }
  return prof_end(c, st, 1, launches);
}

extern "C" int cgd_fcn(cgd_ctx *c, double *F, const double *U, double *Temp1, const double *AuxG, void *stream) {
  int r = check(c);
  if (r) return r;
  if (!F || !U || !Temp1 || !AuxG) return fail(c, CGD_ERR_ARG, "cgd_fcn: null array");
  return run_fcn<double>(c, F, U, U, Temp1, AuxG, S(stream), true);
}

extern "C" int cgd_set_dtau(cgd_ctx *c, double dtau) {
  int r = check(c);
  if (r) return r;
  if (!(dtau > 0.0)) return fail(c, CGD_ERR_ARG, "cgd_set_dtau: dtau must be positive");
  c->dtau = dtau;
  return CGD_OK;
}

// whether the J blocks take 16-byte accesses
static bool aligned16(const double *a, const double *b, const double *d, const double *e) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(d) |
           reinterpret_cast<uintptr_t>(e)) & 15) == 0;
}

extern "C" int cgd_jac(cgd_ctx *c, double *JRhoW, double *JWRho, double *JWRhoTh, double *JRhoThW, const double *U,
                       const double *AuxG, void *stream) {
  int r = check(c);
  if (r) return r;
  if (!JRhoW || !JWRho || !JWRhoTh || !JRhoThW || !U || !AuxG) return fail(c, CGD_ERR_ARG, "cgd_jac: null array");
  const size_t n = (size_t)c->NumG * (c->Nz - 1);
  const size_t ng = (size_t)c->NumG * c->Nz;
  const auto kernel = aligned16(JRhoW, JWRho, JWRhoTh, JRhoThW) ? k_jac<true> : k_jac<false>;
  hipLaunchKernelGGL(kernel, dim3(grid_for(n, 256)), dim3(256), 0, S(stream), c->ka, U, AuxG + 3 * ng, c->dz,
                     JRhoW, JWRho, JWRhoTh, JRhoThW);
  HIPCHK(c, hipGetLastError());
  return CGD_OK;
}

// f(W, Thomas) as integral constants, W the workgroup of a tall column
template <typename F> static void launch_tall(const cgd_ctx *c, F f) {
  auto w = [&](auto th) {
    if (c->Nz <= 128) f(std::integral_constant<int, 128>{}, th);
    else f(std::integral_constant<int, 256>{}, th);
  };
  if (c->thomas) w(std::true_type{});
  else w(std::false_type{});
}

extern "C" int cgd_schur(cgd_ctx *c, double *k, double *v, const double *JRhoW, const double *JWRho,
                         const double *JWRhoTh, const double *JRhoThW, double *tri, double fac, int comp_tri,
                         void *stream) {
  int r = check(c);
  if (r) return r;
  if (!k || !v || !JRhoW || !JWRho || !JWRhoTh || !JRhoThW || !tri) return fail(c, CGD_ERR_ARG, "cgd_schur: null array");
  if (!(fac > 0.0)) return fail(c, CGD_ERR_ARG, "cgd_schur: fac must be positive");
  hipStream_t st = S(stream);
  prof_begin(c, st, 2);
  const double invfac = 1.0 / fac, invfac2 = invfac / fac;
  if (c->Nz <= 64) {
    // 24 words a point past the cache from 2 M points on: a call takes 162 us
    // instead of 166 at 2.46 M (ne = 20, nz = 64), 363 instead of 376 at 5.5 M; at
    // 1.57 M (ne = 16) 107 instead of 102.6, at 0.88 M 61 instead of 55
    const bool a16 = aligned16(JRhoW, JWRho, JWRhoTh, JRhoThW), nt = (size_t)c->NumG * c->Nz >= (size_t)1 << 21;
    const auto kernel = a16 ? (nt ? k_schur_col<true, true> : k_schur_col<true, false>)
                            : (nt ? k_schur_col<false, true> : k_schur_col<false, false>);
    hipLaunchKernelGGL(kernel, dim3((c->NumG + 3) / 4), dim3(256), 0, st, c->ka, k, v, JRhoW, JWRho, JWRhoTh, JRhoThW,
                       tri, fac, invfac2, comp_tri, c->thomas);
  } else
    launch_tall(c, [&](auto w, auto th) {
      constexpr int W = decltype(w)::value;
      constexpr bool TH = decltype(th)::value;
      hipLaunchKernelGGL((k_schur_tall<W, TH>), dim3(c->NumG), dim3(W), 0, st, c->ka, k, v, JRhoW, JWRho, JWRhoTh,
                         JRhoThW, tri, fac, invfac2, comp_tri);
    });
  HIPCHK(c, hipGetLastError());
  if (c->ntr > 0) {
    const size_t ng = (size_t)c->NumG * c->Nz, nt = (size_t)c->ntr * ng;
    hipLaunchKernelGGL(k_tr_scale, dim3(grid_for(nt, 256)), dim3(256), 0, st, v + 5 * ng, k + 5 * ng, fac, nt);
    HIPCHK(c, hipGetLastError());
  }
  return prof_end(c, st, 2, 1);
}

// The stage kernel over all NumG columns, colw lanes each, colblock
// threads per workgroup.
template <typename R, int W>
static void launch_stage(cgd_ctx *c, int is, const RWStage<R> &rw, hipStream_t st) {
  const size_t cols_per_block = (size_t)c->colblock / W;
  const dim3 g((unsigned)(((size_t)c->NumG + cols_per_block - 1) / cols_per_block)), b(c->colblock);
  if (is == 0) hipLaunchKernelGGL((k_rw_stage<0, R, W>), g, b, 0, st, c->ka, rw);
  else if (is == 1) hipLaunchKernelGGL((k_rw_stage<1, R, W>), g, b, 0, st, c->ka, rw);
  else hipLaunchKernelGGL((k_rw_stage<2, R, W>), g, b, 0, st, c->ka, rw);
}

// One persistent launch per stage (k_stage_persist).  It covers the dry
// dynamics of the fused step with the compact metric and 8-level chunks:
// no tracers, physics hooks or kink smoothing (those add launches between
// the passes), N = 4 or 5, and stage workgroups of the element tile's size.
static bool persist_supported(const cgd_ctx *c, std::string *why) {
  const char *w = nullptr;
  if (c->Nz > 64) w = "Nz > 64";
  else if (c->N != 4 && c->N != 5) w = "N must be 4 or 5";
  else if (!c->cm) w = "the metric is not in the compact layout";
  else if (c->ntr > 0) w = "tracers";
  else if (c->hooks.forcing || c->hooks.damping || c->hooks.micro) w = "physics hooks";
  else if (c->smooth) w = "kink smoothing";
  if (w && why) *why = w;
  return !w;
}

template <int N, typename R, int W> static const void *persist_fn(const cgd_ctx *c) {
  if constexpr (std::is_same<R, double>::value)
    if (c->reg) return reinterpret_cast<const void *>(&k_stage_persist<N, true, R, W, true>);
  return reinterpret_cast<const void *>(&k_stage_persist<N, true, R, W, false>);
}
template <typename R> static size_t lds_persist(const cgd_ctx *c) {
  return std::max(lds_fcn1<R>(c, 8), std::is_same<R, double>::value && c->reg ? lds_fcn2r(c, 8) : lds_fcn2<R>(c, 8));
}

// The grid: every workgroup resident at once (the kernel's occupancy per CU
// times the CUs), and no more than the largest phase has work for.
template <typename R, int W> static int persist_grid(cgd_ctx *c, int &G) {
  const void *fn = c->N == 5 ? persist_fn<5, R, W>(c) : persist_fn<4, R, W>(c);
  const size_t lds = lds_persist<R>(c);
  int per_cu = 0, dev = 0, ncu = 0;
  HIPCHK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, tile_block(c, 8), lds));
  HIPCHK(c, hipGetDevice(&dev));
  HIPCHK(c, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  if (per_cu < 1) return fail(c, CGD_ERR_UNSUPPORTED, "persistent stage launch: the kernel does not fit a CU");
  int need = (c->NumG + c->colblock / c->colw - 1) / (c->colblock / c->colw);
  need = std::max(need, c->NF * nchunks(c, 8));
  G = std::max(1, std::min(per_cu * ncu, need));
  return CGD_OK;
}

template <typename R, int W>
static int launch_persist(cgd_ctx *c, int is, const RWStage<R> &rw, const double *U, const R *UR, const double *P,
                          hipStream_t st) {
  int r;
  if (!c->pgrid && (r = persist_grid<R, W>(c, c->pgrid))) return r;
  StagePersist<R> p{};
  p.nf = c->NF;
  p.nchunk1 = p.nchunk = nchunks(c, 8);
  p.UR = UR;
  p.T1 = reinterpret_cast<R *>(c->d_e1);
  p.U = U;
  p.T1th = e1_theta<R>(c);
  p.P = P;
  p.F = reinterpret_cast<R *>(c->d_e2);
  p.F4x = reinterpret_cast<R *>(c->d_f4x);
  p.bar = c->d_bar;
  p.deadline = c->bar_ticks;
  p.stage_blocks = (unsigned)((c->NumG + c->colblock / W - 1) / (c->colblock / W));
  const size_t lds = lds_persist<R>(c);
  const void *fn = c->N == 5 ? persist_fn<5, R, W>(c) : persist_fn<4, R, W>(c);
  RWStage<R> rws = rw;
  void *args[] = {&c->ka, &p, &rws, &is};
  HIPCHK(c, hipLaunchKernel(fn, dim3(c->pgrid), dim3(tile_block(c, 8)), args, lds, st));
  HIPCHK(c, hipGetLastError());
  return CGD_OK;
}

// Fused step: the first pressure, then per stage the two
// tendency passes and one column kernel (Jacobian, tri, stage terms, Schur
// solve, next state and its pressure; the first also stores Vn = V).  With
// R = float (mixed precision) the FP32 tendency and its FP32 state shadow
// share the fV work buffer (the tendency only where hooks need its sums).
template <typename R>
static int rw_step_fused(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, hipStream_t st, double *const k[3],
                         const double A[3][3], const double Cc[3][3], const double Mw[3], double gamma, bool begin,
                         bool more) {
  int r;
  const size_t ng = (size_t)c->NumG * c->Nz, n5 = 5 * ng;
  const size_t nv = (size_t)(5 + c->ntr) * ng;  // one state array (Nz, NumG, 5 + NumTr)
  const bool mixed = std::is_same<R, float>::value;
  R *F = reinterpret_cast<R *>(w->fV);
  R *T1 = reinterpret_cast<R *>(w->Temp1);
  float *V32 = mixed ? reinterpret_cast<float *>(w->fV) + n5 : nullptr;
  const R *UR = mixed ? reinterpret_cast<const R *>(V32) : reinterpret_cast<const R *>(V);
  // the first pressure (and FP32 shadow) of V, unless the previous step of
  // a run wrote them with its final state
  if (begin) {
    hipLaunchKernelGGL(k_rw_begin, dim3(grid_for((ng + 3) / 4, 256)), dim3(256), 0, st, c->ka, V, w->AuxG, V32, ng);
    HIPCHK(c, hipGetLastError());
    if (c->ka.iv >= 0) {
      hipLaunchKernelGGL(k_moist_p, dim3(grid_for(ng, 256)), dim3(256), 0, st, c->ka, V, w->AuxG, ng);
      HIPCHK(c, hipGetLastError());
    }
  }
  for (int is = 0; is < 3; ++is) {
    if (!c->persistent && (r = run_fcn<R>(c, F, V, UR, T1, w->AuxG, st, false))) return r;
    RWStage<R> rw{};
    rw.fV = has_hooks(c) ? F : nullptr;
    rw.Fe = reinterpret_cast<const R *>(c->d_e2);
    rw.V32 = (is < 2 || more) ? V32 : nullptr;
    // the stage increments are stored as R (FP32 in the mixed mode: they
    // are ~dt*F, so their rounding is ~1e-7 of an increment)
    // (FP32 ones pack into the first five components' worth of k, below the
    // FP64 tracer increments at components 6.. of each stage)
    R *kR[3] = {reinterpret_cast<R *>(k[0]), reinterpret_cast<R *>(w->k) + (mixed ? n5 : nv),
                reinterpret_cast<R *>(w->k) + 2 * (mixed ? n5 : nv)};
    for (int j = 0; j < is; ++j) {
      rw.kprev[j] = kR[j];
      rw.cf[j] = Cc[is][j] / dt;
    }
    for (int j = 0; j <= is; ++j) rw.av[j] = (is < 2) ? A[is + 1][j] : Mw[j];
    rw.Vn = w->Vn;
    rw.Vnw = w->Vn;
    rw.dz = c->dz;
    rw.V = V;
    rw.k = is < 2 ? kR[is] : nullptr;  // k_3 is consumed in registers
    rw.P = (is < 2 || more) ? w->AuxG : nullptr;
    rw.F4x = reinterpret_cast<const R *>(c->d_f4x);
    rw.nchunk = nchunks(c, f4_nzt<R>(c));
    rw.nzt = f4_nzt<R>(c);
    rw.fac = dt * gamma;
    rw.invfac = 1.0 / rw.fac;
    rw.invfac2 = rw.invfac / rw.fac;
    rw.thomas = c->thomas;
    if (c->persistent) {  // both passes and the column stage in one launch (timed as the column pass)
      prof_begin(c, st, 2);
      r = c->colw == 32 ? launch_persist<R, 32>(c, is, rw, V, UR, w->AuxG, st)
                        : launch_persist<R, 64>(c, is, rw, V, UR, w->AuxG, st);
      if (r) return r;
      if ((r = prof_end(c, st, 2, 1))) return r;
      continue;
    }
    prof_begin(c, st, 2);
    if (c->Nz > 64) {
      if constexpr (std::is_same<R, double>::value)
        launch_tall(c, [&](auto w, auto th) {
          constexpr int W = decltype(w)::value;
          constexpr bool TH = decltype(th)::value;
          const dim3 g(c->NumG), b(W);
          if (is == 0) hipLaunchKernelGGL((k_rw_stage_tall<0, W, TH>), g, b, 0, st, c->ka, rw);
          else if (is == 1) hipLaunchKernelGGL((k_rw_stage_tall<1, W, TH>), g, b, 0, st, c->ka, rw);
          else hipLaunchKernelGGL((k_rw_stage_tall<2, W, TH>), g, b, 0, st, c->ka, rw);
        });
    } else if (c->colw == 32) launch_stage<R, 32>(c, is, rw, st);
    else launch_stage<R, 64>(c, is, rw, st);
    HIPCHK(c, hipGetLastError());
    if (c->ntr > 0) {  // the tracers' stage terms and next state, FP64 in both modes
      const size_t o = 5 * ng;
      const double *fvt = c->hooks.micro ? w->fV + o : nullptr, *k0 = k[0] + o, *k1 = k[1] + o;
      double *kout = is < 2 ? k[is] + o : nullptr;
      const double cf0 = is > 0 ? Cc[is][0] / dt : 0.0, cf1 = is > 1 ? Cc[is][1] / dt : 0.0;
      const auto kernel = is == 0 ? k_rw_tr<0> : is == 1 ? k_rw_tr<1> : k_rw_tr<2>;
      hipLaunchKernelGGL(kernel, dim3(grid_for(ng, 256), c->ntr), dim3(256), 0, st, c->ka, c->d_e2 + 5 * c->ka.ecs, fvt,
                         k0, k1, cf0, cf1, rw.av[0], rw.av[1], rw.av[2], rw.fac, V + o, w->Vn + o, kout, (unsigned)ng);
      HIPCHK(c, hipGetLastError());
    }
    // Models.Moist: the pressure of the new state needs its tracers too
    if (c->ka.iv >= 0 && rw.P) {
      hipLaunchKernelGGL(k_moist_p, dim3(grid_for(ng, 256)), dim3(256), 0, st, c->ka, V, w->AuxG, ng);
      HIPCHK(c, hipGetLastError());
    }
    if ((r = prof_end(c, st, 2, 1))) return r;
  }
  return CGD_OK;
}

// One SSP-Knoth step as the reference's sequence of calls (FP64): prepare,
// tendency, the Jacobian at the first stage, the stage terms by k_axpy and
// the Schur solves.  Used by the adjoint's forward runs.
static int rw_composed_step(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, hipStream_t st) {
  int r;
  const double A[3][3] = {{0, 0, 0}, {1.0, 0, 0}, {0.25, 0.25, 0}};
  const double Cc[3][3] = {{-1.0, 0, 0}, {-0.0, -1.0, 0}, {-0.75, -0.75, -1.0}};
  const double m3 = 2.0 / 3.0, m2 = 1.0 / 6.0 - (-0.75) * m3, m1 = 1.0 / 6.0 - (-0.75) * m3;
  const double Mw[3] = {m1, m2, m3};
  const double gamma = 1.0;
  const size_t ng = (size_t)c->NumG * c->Nz, n5 = (size_t)(5 + c->ntr) * ng;  // (Nz, NumG, 5 + NumTr)
  double *k[3] = {w->k, w->k + n5, w->k + 2 * n5};
  HIPCHK(c, hipMemcpyAsync(w->Vn, V, n5 * sizeof(double), hipMemcpyDeviceToDevice, st));
  for (int is = 0; is < 3; ++is) {
    if ((r = cgd_prepare(c, V, w->AuxG, st))) return r;
    if ((r = cgd_fcn(c, w->fV, V, w->Temp1, w->AuxG, st))) return r;
    if (is == 0 && (r = cgd_jac(c, w->JRhoW, w->JWRho, w->JWRhoTh, w->JRhoThW, V, w->AuxG, st))) return r;
    const int gb = grid_for(n5, 256);
    if (is > 0) {
      hipLaunchKernelGGL(k_axpy, dim3(gb), dim3(256), 0, st, w->fV, w->fV, k[0], Cc[is][0] / dt, k[1],
                         Cc[is][1] / dt, is, n5);
      HIPCHK(c, hipGetLastError());
    }
    if ((r = cgd_schur(c, k[is], w->fV, w->JRhoW, w->JWRho, w->JWRhoTh, w->JRhoThW, w->tri, dt * gamma, is == 0, st)))
      return r;
    if (is < 2)
      hipLaunchKernelGGL(k_axpy, dim3(gb), dim3(256), 0, st, V, w->Vn, k[0], A[is + 1][0], k[1], A[is + 1][1], is + 1,
                         n5);
    else
      hipLaunchKernelGGL(k_axpy3, dim3(gb), dim3(256), 0, st, V, w->Vn, k[0], Mw[0], k[1], Mw[1], k[2], Mw[2], n5);
    HIPCHK(c, hipGetLastError());
  }
  return CGD_OK;
}

// nsteps SSP-Knoth steps; with the fused path, steps after the first take
// the pressure (and FP32 shadow) that the previous step's last stage wrote
static int rw_run(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, int nsteps, void *stream) {
  int r = check(c);
  if (r) return r;
  if (!V || !w || !w->Vn || !w->fV || !w->k || !w->AuxG || !w->Temp1 || !w->JRhoW || !w->JWRho || !w->JWRhoTh ||
      !w->JRhoThW || !w->tri)
    return fail(c, CGD_ERR_ARG, "cgd_rw_step: null array");
  if (!(dt > 0.0)) return fail(c, CGD_ERR_ARG, "cgd_rw_step: dt must be positive");
  if (nsteps < 1) return fail(c, CGD_ERR_ARG, "cgd_rw_run: nsteps must be positive");
  hipStream_t st = S(stream);
  if ((r = order_streams(c, st))) return r;
  c->dtau = dt;  // Global.TimeStepper.dtauStage = dt (RosenbrockSchur.jl:9)
  // SSP-Knoth: a = alpha/Gamma, c = -inv(Gamma), m = Gamma'\b, gamma = 1
  const double A[3][3] = {{0, 0, 0}, {1.0, 0, 0}, {0.25, 0.25, 0}};
  const double Cc[3][3] = {{-1.0, 0, 0}, {-0.0, -1.0, 0}, {-0.75, -0.75, -1.0}};
  const double m3 = 2.0 / 3.0, m2 = 1.0 / 6.0 - (-0.75) * m3, m1 = 1.0 / 6.0 - (-0.75) * m3;
  const double Mw[3] = {m1, m2, m3};
  const double gamma = 1.0;
  const size_t ng = (size_t)c->NumG * c->Nz, n5 = (size_t)(5 + c->ntr) * ng;  // (Nz, NumG, 5 + NumTr)
  double *k[3] = {w->k, w->k + n5, w->k + 2 * n5};
  // tall columns step in FP64 in either precision mode
  for (int s = 0; s < nsteps; ++s) {
    const bool begin = s == 0, more = s + 1 < nsteps;
    r = c->mixed && c->Nz <= 64 ? rw_step_fused<float>(c, V, dt, w, st, k, A, Cc, Mw, gamma, begin, more)
                                : rw_step_fused<double>(c, V, dt, w, st, k, A, Cc, Mw, gamma, begin, more);
    if (r) return r;
  }
  return CGD_OK;
}

extern "C" int cgd_rw_step(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, void *stream) {
  return rw_run(c, V, dt, w, 1, stream);
}

extern "C" int cgd_rw_run(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, int nsteps, void *stream) {
  return rw_run(c, V, dt, w, nsteps, stream);
}

// ------------------------------------------------------------------------
// Launch shapes, step graphs and the autotuner

static void graph_free(cgd_ctx *c) {
  if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
  if (c->graph) (void)hipGraphDestroy(c->graph);
  c->gexec = nullptr;
  c->graph = nullptr;
}

// Admissible shapes: chunk heights 8 (and 16 for N = 5); 64 lanes per
// column, or 32 when Nz <= 32 and the solve is cyclic reduction; stage
// workgroups of 64..256 threads in whole wavefronts.
// A persistent stage launch (persistent = 1) also needs 8-level chunks in
// both passes, one pass-1 item per workgroup and stage workgroups of the
// element tile's size (256 threads for N = 5, 128 for N = 4).
static bool shape_ok(const cgd_ctx *c, const cgd_launch_shape &sh) {
  auto chunk_ok = [&](int z) { return z == 8 || (z == 16 && c->N == 5); };
  if (!chunk_ok(sh.chunk_levels)) return false;
  if (!chunk_ok(sh.pass1_chunk_levels) && !(sh.pass1_chunk_levels == 64 && columns_ok(c))) return false;
  if (!(sh.pass1_items == 1 || sh.pass1_items == 2)) return false;
  if (!(sh.col_lanes == 64 || (sh.col_lanes == 32 && c->Nz <= 32 && !c->thomas))) return false;
  if (!(sh.col_block >= 64 && sh.col_block <= 256 && sh.col_block % 64 == 0)) return false;
  if (sh.persistent != 1 && sh.persistent != -1) return false;
  if (sh.persistent == 1)
    return persist_supported(c, nullptr) && sh.chunk_levels == 8 && sh.pass1_chunk_levels == 8 &&
           sh.pass1_items == 1 && sh.col_block == tile_block(c, 8);
  return true;
}

static cgd_launch_shape current_shape(const cgd_ctx *c) {
  cgd_launch_shape sh;
  sh.chunk_levels = c->persistent ? 8 : c->nzt;
  sh.pass1_chunk_levels = c->persistent ? 8 : c->nzt1;
  sh.pass1_items = c->items1;
  sh.col_lanes = c->colw;
  sh.col_block = c->colblock;
  sh.persistent = c->persistent ? 1 : -1;
  return sh;
}

static void apply_shape(cgd_ctx *c, const cgd_launch_shape &sh) {
  c->nzt = sh.chunk_levels;
  c->nzt1 = sh.pass1_chunk_levels;
  c->items1 = sh.pass1_items;
  c->colw = sh.col_lanes;
  c->colblock = sh.col_block;
  c->persistent = sh.persistent == 1;
  c->pgrid = 0;  // sized again at the next launch
}

extern "C" int cgd_set_launch_shape(cgd_ctx *c, const cgd_launch_shape *shape) {
  int r = check(c);
  if (r) return r;
  if (!shape) return fail(c, CGD_ERR_ARG, "cgd_set_launch_shape: null shape");
  cgd_launch_shape sh = current_shape(c);
  // a persistent launch takes 8 levels in place of the heights the context
  // chose, which stand again when it is turned off, but not of set ones
  const bool pers = shape->persistent ? shape->persistent == 1 : c->persistent;
  sh.chunk_levels = pers && c->nzt == c->rule_nzt ? 8 : c->nzt;
  sh.pass1_chunk_levels = pers && c->nzt1 == c->rule_nzt1 ? 8 : c->nzt1;
  if (shape->chunk_levels) sh.chunk_levels = shape->chunk_levels;
  if (shape->pass1_chunk_levels) sh.pass1_chunk_levels = shape->pass1_chunk_levels;
  if (shape->pass1_items) sh.pass1_items = shape->pass1_items;
  if (shape->col_lanes) sh.col_lanes = shape->col_lanes;
  if (shape->col_block) sh.col_block = shape->col_block;
  if (shape->persistent) sh.persistent = shape->persistent;
  std::string why;
  if (sh.persistent == 1 && !persist_supported(c, &why))
    return fail(c, CGD_ERR_UNSUPPORTED, "persistent stage launch: not for " + why);
  if (!shape_ok(c, sh))
    return fail(c, CGD_ERR_ARG,
                "launch shape: chunk heights must be 8 (or 16 for N = 5; 64 in pass 1, whole columns, for the compact "
                "metric and Nz <= 64), pass1_items 1 or 2, col_lanes 64 (or 32 "
                "when Nz <= 32 without the Thomas solve), col_block a multiple of 64 in [64, 256], persistent 1 or "
                "-1; a persistent launch takes chunk heights 8, pass1_items 1 and col_block = 64 * ceil(N*N*8 / 64)");
  graph_free(c);  // a captured graph keeps the old shapes
  const int nzt = c->nzt, nzt1 = c->nzt1;
  apply_shape(c, sh);
  if (!shape->chunk_levels) c->nzt = nzt;
  if (!shape->pass1_chunk_levels) c->nzt1 = nzt1;
  return CGD_OK;
}

// The grid barrier's error word (set by a wait past its bound); cleared
// after it is read.
static int bar_status(cgd_ctx *c, hipStream_t st) {
  GridBar hb{};
  HIPCHK(c, hipStreamSynchronize(st));
  HIPCHK(c, hipMemcpyAsync(&hb, c->d_bar, sizeof(hb), hipMemcpyDeviceToHost, st));
  HIPCHK(c, hipStreamSynchronize(st));
  if (!hb.err) return CGD_OK;
  HIPCHK(c, hipMemsetAsync(c->d_bar, 0, sizeof(GridBar), st));
  HIPCHK(c, hipStreamSynchronize(st));
  return fail(c, CGD_ERR_HIP,
              "a persistent stage launch timed out in its grid barrier (its workgroups were not all resident at "
              "once): the steps since the last check are invalid");
}

extern "C" int cgd_check(cgd_ctx *c, void *stream) {
  int r = check(c);
  if (r) return r;
  return bar_status(c, S(stream));
}

extern "C" int cgd_get_launch_shape(const cgd_ctx *c, cgd_launch_shape *shape) {
  if (!c || !shape) return CGD_ERR_ARG;
  if (!c->ok) return CGD_ERR_STATE;
  *shape = current_shape(c);
  return CGD_OK;
}

extern "C" int cgd_rw_graph_create(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, int nsteps,
                                   void *stream) {
  int r = check(c);
  if (r) return r;
  if (nsteps < 1 || nsteps > 10000) return fail(c, CGD_ERR_ARG, "cgd_rw_graph_create: nsteps must be in [1, 10000]");
  if (c->prof) return fail(c, CGD_ERR_STATE, "cgd_rw_graph_create: turn profiling off before capturing");
  graph_free(c);
  if (!c->gstream) HIPCHK(c, hipStreamCreateWithFlags(&c->gstream, hipStreamNonBlocking));
  // the capture records launches only; the caller's earlier work on stream
  // is ordered before the replays by hipGraphLaunch on that stream
  HIPCHK(c, hipStreamSynchronize(S(stream)));
  HIPCHK(c, hipStreamBeginCapture(c->gstream, hipStreamCaptureModeThreadLocal));
  r = rw_run(c, V, dt, w, nsteps, c->gstream);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(c->gstream, &g);
  if (r || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    if (r) return r;
    return fail(c, CGD_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  }
  c->graph = g;
  HIPCHK(c, hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0));
  return CGD_OK;
}

extern "C" int cgd_rw_graph_launch(cgd_ctx *c, void *stream) {
  int r = check(c);
  if (r) return r;
  if (!c->gexec) return fail(c, CGD_ERR_STATE, "cgd_rw_graph_launch: no captured step graph");
  if ((r = order_streams(c, S(stream)))) return r;
  HIPCHK(c, hipGraphLaunch(c->gexec, S(stream)));
  return CGD_OK;
}

extern "C" int cgd_autotune(cgd_ctx *c, double *V, double dt, const cgd_rw_work *w, int reps, void *stream,
                            cgd_launch_shape *chosen, double *best_ms) {
  int r = check(c);
  if (r) return r;
  if (!V || !w) return fail(c, CGD_ERR_ARG, "cgd_autotune: null array");
  if (reps < 1 || reps > 100) return fail(c, CGD_ERR_ARG, "cgd_autotune: reps must be in [1, 100]");
  hipStream_t st = S(stream);
  const int prof = c->prof;
  c->prof = 0;
  graph_free(c);
  const size_t n5 = (size_t)(5 + c->ntr) * c->NumG * c->Nz;  // every component, tracers included
  double *Vsave = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  cgd_launch_shape best = current_shape(c);
  const cgd_launch_shape entry = best;
  const int entry_nzt = c->nzt, entry_nzt1 = c->nzt1;
  double bms = 1e300;
  auto same = [](const cgd_launch_shape &x, const cgd_launch_shape &y) {
    return x.chunk_levels == y.chunk_levels && x.pass1_chunk_levels == y.pass1_chunk_levels &&
           x.pass1_items == y.pass1_items && x.col_lanes == y.col_lanes && x.col_block == y.col_block &&
           x.persistent == y.persistent;
  };
  auto run = [&]() -> int {
    HIPCHK(c, hipMalloc(&Vsave, n5 * sizeof(double)));
    HIPCHK(c, hipEventCreate(&e0));
    HIPCHK(c, hipEventCreate(&e1));
    HIPCHK(c, hipMemcpyAsync(Vsave, V, n5 * sizeof(double), hipMemcpyDeviceToDevice, st));
    // per-step time of one shape: the fastest of three timings of reps steps
    // (robust to clock ramps and other work on the device)
    auto time_shape = [&](const cgd_launch_shape &sh, double &per) -> int {
      apply_shape(c, sh);
      int rr;
      HIPCHK(c, hipMemcpyAsync(V, Vsave, n5 * sizeof(double), hipMemcpyDeviceToDevice, st));
      if ((rr = cgd_rw_step(c, V, dt, w, stream))) return rr;  // warm-up
      per = 1e300;
      for (int t = 0; t < 3; ++t) {
        HIPCHK(c, hipEventRecord(e0, st));
        for (int q = 0; q < reps; ++q)
          if ((rr = cgd_rw_step(c, V, dt, w, stream))) return rr;
        HIPCHK(c, hipEventRecord(e1, st));
        HIPCHK(c, hipEventSynchronize(e1));
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, e0, e1));
        per = std::min(per, (double)ms / reps);
      }
      return sh.persistent == 1 ? bar_status(c, st) : CGD_OK;
    };
    // the fastest of a set of shapes: two sweeps over all of them, each
    // shape keeping its better time, so a drift of the device's speed during
    // a sweep does not favour the shapes timed in its fast part
    // The shape the context had keeps its place unless another is faster by
    // more than 1 %: short timings rank shapes within that margin in either
    // order, and a switch on noise has cost more over long runs than it won.
    auto pick = [&](const std::vector<cgd_launch_shape> &cand, const cgd_launch_shape &keep) -> int {
      std::vector<double> tmin(cand.size(), 1e300);
      for (int sweep = 0; sweep < 2; ++sweep)
        for (size_t i = 0; i < cand.size(); ++i) {
          double per;
          int rr;
          if ((rr = time_shape(cand[i], per))) return rr;
          tmin[i] = std::min(tmin[i], per);
        }
      size_t ib = 0;
      for (size_t i = 1; i < cand.size(); ++i)
        if (tmin[i] < tmin[ib]) ib = i;
      for (size_t i = 0; i < cand.size(); ++i)
        if (same(cand[i], keep) && tmin[i] <= 1.01 * tmin[ib]) ib = i;
      if (!cand.empty()) {
        bms = tmin[ib];
        best = cand[ib];
      }
      return CGD_OK;
    };
    // the element kernels' shapes jointly (both passes' chunk heights and
    // the pass-1 items, which whole columns have none of), then the column
    // shape with the best of them
    int rr;
    std::vector<cgd_launch_shape> cand;
    best.persistent = -1;  // the element and column sweeps time separate launches
    const cgd_launch_shape ek = best;
    for (int z2 : {8, 16})
      for (int z1 : {8, 16, 64})
        for (int it : {1, 2}) {
          cgd_launch_shape sh = ek;
          sh.chunk_levels = z2;
          sh.pass1_chunk_levels = z1;
          sh.pass1_items = it;
          if (shape_ok(c, sh) && (same(sh, ek) || z1 != 64 || it == 1)) cand.push_back(sh);
        }
    if ((rr = pick(cand, ek))) return rr;
    const cgd_launch_shape b1 = best;
    cand.clear();
    for (int l : {64, 32})
      for (int b : {256, 128, 64}) {
        cgd_launch_shape sh = b1;
        sh.col_lanes = l;
        sh.col_block = b;
        if (shape_ok(c, sh)) cand.push_back(sh);
      }
    {
      cgd_launch_shape keep = b1;  // the entry shape's columns with the chosen element shape
      keep.col_lanes = entry.col_lanes;
      keep.col_block = entry.col_block;
      if ((rr = pick(cand, keep))) return rr;
    }
    // separate launches or one persistent launch per stage (with the best
    // column lanes), where the configuration allows the latter
    if (persist_supported(c, nullptr)) {
      const cgd_launch_shape b2 = best;
      cand.clear();
      cgd_launch_shape sep = b2, per = b2;
      sep.persistent = -1;
      per.chunk_levels = per.pass1_chunk_levels = 8;
      per.pass1_items = 1;
      per.col_block = (c->NN * 8 + 63) / 64 * 64;
      per.persistent = 1;
      if (shape_ok(c, sep)) cand.push_back(sep);
      if (shape_ok(c, per)) cand.push_back(per);
      if (cand.size() == 2 && (rr = pick(cand, entry.persistent == 1 ? per : sep))) return rr;
    }
    return CGD_OK;
  };
  r = run();
  // V as it was, whatever happened above
  if (Vsave) {
    const hipError_t e = hipMemcpyAsync(V, Vsave, n5 * sizeof(double), hipMemcpyDeviceToDevice, st);
    const hipError_t e2 = hipStreamSynchronize(st);
    if (!r && (e != hipSuccess || e2 != hipSuccess))
      r = fail(c, CGD_ERR_HIP, std::string("cgd_autotune: restoring V: ") +
                                   hipGetErrorString(e != hipSuccess ? e : e2));
  }
  if (Vsave) (void)hipFree(Vsave);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  apply_shape(c, best);
  if (same(best, entry)) {  // (a persistent launch keeps the heights it stands in for)
    c->nzt = entry_nzt;
    c->nzt1 = entry_nzt1;
  }
  c->prof = prof;
  if (r) return r;
  if (chosen) *chosen = best;
  if (best_ms) *best_ms = bms;
  return CGD_OK;
}

// ------------------------------------------------------------------------
// Adjoint of the FP64 path
#pragma clang fp contract(fast)
#include "cgd_adjoint.hip"
