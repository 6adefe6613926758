// HIP kernels (gfx950) for the spectral-element tendency, the column
// Jacobian / Schur solve and the Rosenbrock-W stage arithmetic.
//
// Data layout in HBM (all level-fastest, so a wavefront's lanes read
// consecutive levels of one column):
//   state / caches   X[v][g][iz]                  (reference (Nz,NumG,NumV))
//   metric (pass 2)  met[e][c][ID][iz], c < 17    (built once from dXdxI/J/X)
//   metric (pass 1)  met1[e][c][ID][iz], c < 5    (S11,S12,S21,S22,J1+J2)
//   DSS mass         Ms[g][iz] = M1 + M2, M[K][g][iz]
//
// Element kernels: one thread per (node, level) point of one element and
// one chunk of NZT (8 or 16) levels; thread t -> node = t / NZT,
// level = t % NZT, so a chunk column fills whole 16-lane DPP rows.
// Horizontal derivatives exchange values through LDS tiles
// tile[f][node][level]; vertical neighbours come from the neighbouring
// lanes by DPP row shifts, with one global load at each chunk edge.
//
// DSS: the element passes write each element's contributions to an array of
// its own, X[c][e*NN + node][iz], all elements in one launch, and the consumer
// of a field sums a node's copies in colour order (a fixed order, no atomics).
// The adjoint's kernels accumulate in place, one launch per element colour
// (no two elements of a colour share a node).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

// Multiply-adds are fused within an expression, by the front end, and not
// wherever the code generator finds them: a kernel body that is inlined in
// two kernels (separate and persistent launches) then rounds the same way.
#pragma clang fp contract(on)

#define CGD_NMAX 5
#define CGD_NMET 17  // pass-2 metric components
#define CGD_NMET1 5  // pass-1 metric components
#define CGD_NMETP 5  // compact layout: components stored per point (terrain row dXdxI[3,1:2,K], Coriolis)
#define CGD_NMETN 12 // compact layout: components stored once per element node

struct KArgs {
  int Nz, NumG;
  double Grav, Omega, Rd, Cpd, p0, kappa;
  double Rd_p0, eos_y, dpd_y;      // Rd/p0, 1/(1-kappa), kappa/(1-kappa)
  double Rd_Cpd;                   // Rd/Cpd
  double D[CGD_NMAX * CGD_NMAX];   // D[i*N + k] = DS[i,k]
  double DWm[CGD_NMAX * CGD_NMAX]; // DW[i*N + k]
  float Df[CGD_NMAX * CGD_NMAX], DWf[CGD_NMAX * CGD_NMAX];  // both in FP32 (mixed precision)
  const int *glob;                 // [e][NN]: 0-based node | bit 31 set on the node's first copy (colour order)
  const int *clist;                // elements by colour (the adjoint kernels' launch order)
  const int *cpy;                  // [e][NN][cpw]: the node's copies e'*NN + node' in colour order, then -1
  const int *gcpy;                 // [NumG][cpw]: the same per global node
  int cpw;                         // a multiple of 2, at least 4
  size_t ecs;                      // NF*NN*Nz: values per component of an element-copy array
  const double *met;               // [e][17][NN][Nz], or [e][5][NN][Nz] in the compact layout
  const double *met1;              // [element][5][NN][Nz] (full layout only)
  const double *metn;              // compact layout: [element][13][NN]
  const double *met1n;             // compact layout: [element][5][NN]
  const double *iMs;               // [NumG][Nz]: 1 / (M1 + M2)
  const float *iMs32;              // the same in FP32 (mixed-precision mode)
  const float *M32;                // M in FP32 (mixed-precision mode)
  const float *metp32;             // compact layout's per-point components in FP32 (mixed precision)
  const double *M;                 // [2][NumG][Nz]
  const double *iMn;               // regular metric (cgd_pass2r_body.inc): [NumG], 1 / (M1 + M2); else null
  const double *kvis;              // [element][3]: HyperDCurl, HyperDGrad, HyperDDiv of the element's grid
  // Models.Moist: 0-based components of the vapour and cloud densities (-1: dry)
  int iv, ic;
  double Cpv, Cpl, Rv;
  double wg[CGD_NMAX];  // GLL weights (HorLimit)
  double smw, smc;      // kink smoothing of the upwind flux (SmoothW, SmoothC; 0: exact)
};

// metric component indices of met (dXdxI[a,b,K] -> dabK, 1-based a,b,K)
enum {
  M111 = 0, M112, M121, M122, M211, M212, M221, M222,
  M311, M312, M321, M322, M331, M332, MJ1, MJ2, MCOR
};

// Compact metric layout, chosen at context creation when every component
// except the terrain row dXdxI[3,1:2,K] and the Coriolis parameter (z/|X|
// of level-scaled positions, invariant only up to rounding) has the same
// bits at all levels of each element node (shallow atmosphere, flat
// terrain, uniform layers): those 12 components are stored once per
// element node, the other 5 per point.  Index of a component in either table:
__host__ __device__ constexpr bool met_per_point(int c) { return (c >= M311 && c <= M322) || c == MCOR; }
__host__ __device__ constexpr int met_pidx(int c) { return c == MCOR ? 4 : c - M311; }
__host__ __device__ constexpr int met_nidx(int c) { return c < M311 ? c : c - 4; }

// ------------------------------------------------------------------------
// Equation of state (src/Models/Equation.jl:25-38,79)
// p = p0 (Rd rho*theta / p0)^(1/(1-kappa)) evaluated as exp(y log x) like
// fast_powGPU; dp/d(rho*theta) = Rd (Rd rho*theta / p0)^(kappa/(1-kappa))
// in the same form.  The constants Rd/p0, 1/(1-kappa), kappa/(1-kappa)
// are formed once on the host.
__device__ __forceinline__ double eos_p(const KArgs &a, double rhoth) {
  return a.p0 * exp(a.eos_y * log(a.Rd_p0 * rhoth));
}
__device__ __forceinline__ double eos_dpdrhoth(const KArgs &a, double rhoth) {
  return a.Rd * exp(a.dpd_y * log(a.Rd_p0 * rhoth));
}

// Julia min/max on non-NaN values
template <typename R> __device__ __forceinline__ R jmin(R a, R b) { return (b < a) ? b : a; }
template <typename R> __device__ __forceinline__ R jmax(R a, R b) { return (b > a) ? b : a; }

// 1/x for normal, finite x: the hardware estimate (v_rcp_f64) refined by two
// Newton-Raphson steps r <- r + r (1 - x r), each at least doubling the
// correct bits; the result is within an ulp or two of the rounded quotient
// (the IEEE division sequence costs about twice as many instructions)
__device__ __forceinline__ double rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ double rabs(double x) { return fabs(x); }
__device__ __forceinline__ float rabs(float x) { return fabsf(x); }

// FP32: v_rcp_f32 (1 ulp) and one Newton-Raphson step
__device__ __forceinline__ float rcp(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(r, fmaf(-x, r, 1.0f), r);
}

// Element i of a field at a uniform base: the byte offset is formed in 32
// bits so the access is a single saddr-form global load/store (scalar base
// + 32-bit vector offset).  Callers keep i * sizeof(T) below 2^31.
template <typename T> __device__ __forceinline__ T &at(T *base, unsigned i) {
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + i * (unsigned)sizeof(T));
}
template <typename T> __device__ __forceinline__ const T &at(const T *base, unsigned i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + i * (unsigned)sizeof(T));
}

// A table that nothing writes while the kernel runs, at a uniform address:
// read through the constant address space, so that the loads are scalar ones
// (the compiler cannot tell the kernel's stores from the tables otherwise).
template <typename T> using Const = const __attribute__((address_space(4))) T *;
template <typename T> __device__ __forceinline__ Const<T> as_const(const T *p) {
  return (Const<T>)reinterpret_cast<uintptr_t>(p);
}

// The value of x in lane `lane` (uniform), on every lane.
__device__ __forceinline__ double readlane_d(double x, int lane) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// RecU4 (src/GPU/OperatorKernel.jl:1044-1059): the J-weighted limited
// reconstruction of c at the face between cL and cR.  The weights
//   kR = JL/(JL+JR) * (JLL+JL)/(JLL+JL+JR),  kL = JL/(JLL+JL) * JR/(JLL+JL+JR)
// share one reciprocal of the product of their three denominators (and
// likewise for the right-biased pair).
template <typename R>
__device__ __forceinline__ void recu4(R cLL, R cL, R cR, R cRR, R JLL, R JL, R JR, R JRR, R &cFL, R &cFR) {
  const R A = JL + JR;
  const R tiny = R(1.e-20), zero = R(0), one = R(1);
  {
    const R B = JLL + JL, C = B + JR;
    const R q = rcp(A * B * C);
    const R kR = (JL * B) * B * q;
    const R kL = (JL * JR) * A * q;
    const R r = (cL - cLL) * rcp(cR - cL + tiny);
    cFL = cL + jmax(zero, jmin(r, jmin(kL * r + kR, one))) * (cR - cL);
  }
  {
    const R B = JRR + JR, C = A + JRR;
    const R q = rcp(A * B * C);
    const R kL = (JR * B) * B * q;
    const R kR = (JR * JL) * A * q;
    const R r = (cR - cRR) * rcp(cL - cR + tiny);
    cFR = cR + jmax(zero, jmin(r, jmin(kR * r + kL, one))) * (cL - cR);
  }
}

// Kink smoothing (cgd_desc.SmoothW / SmoothC, FP64): S(t) = sqrt(t^2 + d^2)
// for |t|, and the smooth minmod
//   sminmod(x, y) = (x + y)/2 - S(M)/2 + S(m)/2,  M, m = (x + y +- S(x - y))/2
// (x + y - max(x, y, 0) - min(x, y, 0) with smooth max and min).  RecU4's
// limited face values in product form, cL + minmod(a, kL a + kR c, c) with
// a = cL - cLL, c = cR - cL, then take it in place of minmod.
__device__ __forceinline__ double sabs(double x, double d) { return sqrt(fma(x, x, d * d)); }
__device__ __forceinline__ double sminmod(double x, double y, double d) {
  const double s = sabs(x - y, d);
  const double M = 0.5 * (x + y + s), m = 0.5 * (x + y - s);
  return 0.5 * (x + y) - 0.5 * sabs(M, d) + 0.5 * sabs(m, d);
}
__device__ __forceinline__ void recu4_smooth(double cLL, double cL, double cR, double cRR, double JLL, double JL,
                                             double JR, double JRR, double d, double &cFL, double &cFR) {
  const double A = JL + JR;
  {
    const double B = JLL + JL, C = B + JR;
    const double q = rcp(A * B * C);
    const double kR = (JL * B) * B * q, kL = (JL * JR) * A * q;
    const double a = cL - cLL, c = cR - cL;
    cFL = cL + sminmod(a, sminmod(kL * a + kR * c, c, d), d);
  }
  {
    const double B = JRR + JR, C = A + JRR;
    const double q = rcp(A * B * C);
    const double kL = (JR * B) * B * q, kR = (JR * JL) * A * q;
    const double a = cR - cRR, c = cL - cR;
    cFR = cR + sminmod(a, sminmod(kR * a + kL * c, c, d), d);
  }
}

// RecU4 split in two: the weights of both sides depend on the layer volumes
// only (computed once, e.g. for several tracers), the limited
// reconstruction on c
template <typename R> struct RecW {
  R kRl, kLl, kLr, kRr;  // left-biased kR, kL; right-biased kL, kR
};
template <typename R> __device__ __forceinline__ RecW<R> recu4_weights(R JLL, R JL, R JR, R JRR) {
  RecW<R> w;
  const R A = JL + JR;
  {
    const R B = JLL + JL, C = B + JR;
    const R q = rcp(A * B * C);
    w.kRl = (JL * B) * B * q;
    w.kLl = (JL * JR) * A * q;
  }
  {
    const R B = JRR + JR, C = A + JRR;
    const R q = rcp(A * B * C);
    w.kLr = (JR * B) * B * q;
    w.kRr = (JR * JL) * A * q;
  }
  return w;
}
// ... of equal volumes
template <typename R> __device__ __forceinline__ RecW<R> recu4_equal() {
  return RecW<R>{R(1) / R(3), R(1) / R(6), R(1) / R(3), R(1) / R(6)};
}
// The upwind flux through an interface with the contravariant mass flux wc
// between cL (below) and cR (above): ((|w| + w)/4 cFL + (w - |w|)/4 cFR is
// w/2 times the upwind side's limited value, so only that side is formed.
template <typename R>
__device__ __forceinline__ R recu4_flux(R cLL, R cL, R cR, R cRR, const RecW<R> &w, R wc) {
  const bool up = wc >= R(0);
  const R c = up ? cL : cR, d = (up ? cR : cL) - c, s = c - (up ? cLL : cRR);
  const R r = s * rcp(d + R(1.e-20));
  const R lim = jmin((up ? w.kLl : w.kRr) * r + (up ? w.kRl : w.kLr), R(1));
  return R(0.5) * wc * (c + jmax(R(0), jmin(r, lim)) * d);
}

// ------------------------------------------------------------------------
// LDS tile helpers
// tile[f][node][level] of values of type R; NZ (levels per chunk) is a
// compile-time constant so that every (tile, node) offset is an instruction
// immediate
template <int N, int NZ, typename R = double> struct Tiles {
  R *t;  // tile base
  __device__ __forceinline__ R &at(int f, int node, int l) const { return t[(f * N * N + node) * NZ + l]; }
};

// sum_k D[I,k] f(k,J)
template <int N, int NZ, typename R>
__device__ __forceinline__ R dx(const R *Dm, const Tiles<N, NZ, R> &T, int f, int I, int J, int l) {
  R s = Dm[I * N] * T.at(f, J * N, l);
#pragma unroll
  for (int k = 1; k < N; ++k) s += Dm[I * N + k] * T.at(f, k + J * N, l);
  return s;
}
// sum_k D[J,k] f(I,k)
template <int N, int NZ, typename R>
__device__ __forceinline__ R dy(const R *Dm, const Tiles<N, NZ, R> &T, int f, int I, int J, int l) {
  R s = Dm[J * N] * T.at(f, I, l);
#pragma unroll
  for (int k = 1; k < N; ++k) s += Dm[J * N + k] * T.at(f, I + k * N, l);
  return s;
}
// sum_k (D[I,k] fx(k,J) + D[J,k] fy(I,k)), pairwise as in the reference loops
template <int N, int NZ, typename R>
__device__ __forceinline__ R dxy(const R *Dm, const Tiles<N, NZ, R> &T, int fx, int fy, int I, int J, int l) {
  R s = Dm[I * N] * T.at(fx, J * N, l) + Dm[J * N] * T.at(fy, I, l);
#pragma unroll
  for (int k = 1; k < N; ++k) s += Dm[I * N + k] * T.at(fx, k + J * N, l) + Dm[J * N + k] * T.at(fy, I + k * N, l);
  return s;
}
// acc + sum_k (D[I,k] fx(k,J) + D[J,k] fy(I,k)), accumulated term by term
template <int N, int NZ, typename R>
__device__ __forceinline__ R dxy_acc(R s, const R *Dm, const Tiles<N, NZ, R> &T, int fx, int fy, int I, int J,
                                     int l) {
#pragma unroll
  for (int k = 0; k < N; ++k) s += Dm[I * N + k] * T.at(fx, k + J * N, l) + Dm[J * N + k] * T.at(fy, I + k * N, l);
  return s;
}
// sum_k (D[I,k] fx(k,J) cx(k,J) + D[J,k] fy(I,k) cy(I,k))
template <int N, int NZ, typename R>
__device__ __forceinline__ R dxy_prod(const R *Dm, const Tiles<N, NZ, R> &T, int fx, int fy, int fc, int I, int J,
                                      int l) {
  R s = Dm[I * N] * T.at(fx, J * N, l) * T.at(fc, J * N, l) + Dm[J * N] * T.at(fy, I, l) * T.at(fc, I, l);
#pragma unroll
  for (int k = 1; k < N; ++k)
    s += Dm[I * N + k] * T.at(fx, k + J * N, l) * T.at(fc, k + J * N, l) +
         Dm[J * N + k] * T.at(fy, I + k * N, l) * T.at(fc, I + k * N, l);
  return s;
}

// Value of x held by the lane D positions below / above in the same 16-lane
// DPP row (row_shr:D / row_shl:D).  Lanes whose source falls outside the
// row keep their own x; callers replace those with a halo load.
template <int D> __device__ __forceinline__ double dpp_from_below(double x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const long long b = __double_as_longlong(x);
  const int lo = (int)(b & 0xffffffffLL), hi = (int)(b >> 32);
  const int rlo = __builtin_amdgcn_update_dpp(lo, lo, 0x110 + D, 0xf, 0xf, false);
  const int rhi = __builtin_amdgcn_update_dpp(hi, hi, 0x110 + D, 0xf, 0xf, false);
  return __longlong_as_double(((long long)rhi << 32) | (unsigned int)rlo);
}
template <int D> __device__ __forceinline__ double dpp_from_above(double x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const long long b = __double_as_longlong(x);
  const int lo = (int)(b & 0xffffffffLL), hi = (int)(b >> 32);
  const int rlo = __builtin_amdgcn_update_dpp(lo, lo, 0x100 + D, 0xf, 0xf, false);
  const int rhi = __builtin_amdgcn_update_dpp(hi, hi, 0x100 + D, 0xf, 0xf, false);
  return __longlong_as_double(((long long)rhi << 32) | (unsigned int)rlo);
}
template <int D> __device__ __forceinline__ float dpp_from_below(float x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const int b = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(b, b, 0x110 + D, 0xf, 0xf, false));
}
template <int D> __device__ __forceinline__ float dpp_from_above(float x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const int b = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(b, b, 0x100 + D, 0xf, 0xf, false));
}

// The same row shifts with zero in the lanes whose source falls outside the
// row (bound_ctrl): the result needs no copy of x to start from, so each
// 32-bit half is one v_mov_b32_dpp.  For callers that replace every such
// lane (and every lane whose source belongs to another node) by a halo load.
template <int D> __device__ __forceinline__ double dppz_from_below(double x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const long long b = __double_as_longlong(x);
  const int rlo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), 0x110 + D, 0xf, 0xf, true);
  const int rhi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x110 + D, 0xf, 0xf, true);
  return __longlong_as_double(((long long)rhi << 32) | (unsigned int)rlo);
}
template <int D> __device__ __forceinline__ double dppz_from_above(double x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  const long long b = __double_as_longlong(x);
  const int rlo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), 0x100 + D, 0xf, 0xf, true);
  const int rhi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x100 + D, 0xf, 0xf, true);
  return __longlong_as_double(((long long)rhi << 32) | (unsigned int)rlo);
}
template <int D> __device__ __forceinline__ float dppz_from_below(float x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x110 + D, 0xf, 0xf, true));
}
template <int D> __device__ __forceinline__ float dppz_from_above(float x) {
  static_assert(D >= 1 && D <= 15, "row shift");
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x100 + D, 0xf, 0xf, true));
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on
// XCD b % 8).  Renumber blocks so that consecutive logical ids -- the level
// chunks of one element, then the next element -- land on the same XCD and
// share its L2 (a chunk's 128-byte lines are also touched by the chunks
// above and below it).
__device__ __forceinline__ int xcd_logical(int b, int G) {
  const int per = G >> 3, rem = G & 7;
  const int x = b & 7, slot = b >> 3;
  return x < rem ? x * (per + 1) + slot : rem * (per + 1) + (x - rem) * per + slot;
}

template <int N, typename R> __device__ __forceinline__ void load_dmats(const KArgs &a, R *Ds, R *DWs) {
  const int t = threadIdx.x;
  if (t < N * N) {
    Ds[t] = R(a.D[t]);
    DWs[t] = R(a.DWm[t]);
  }
}

// any_value: an unspecified value, for a variable that only some lanes set
// (no instruction to initialise it).
// pin computes its arguments here: an empty asm that reads and writes them, so
// that the code generator, which orders arithmetic within a block by its
// own measure, does not hold the inputs of a long block's later sums (LDS
// values, neighbour levels) in registers and spill them.
__device__ __forceinline__ double any_value() { return __builtin_nondeterministic_value(0.0); }
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(float &x) { asm volatile("" : "+v"(x)); }
template <typename R, typename... D> __device__ __forceinline__ void pin(R &x, D &...y) {
  pin(x);
  pin(y...);
}

// Between LDS stores of some lanes of a wavefront and their first reads by other
// lanes of the same one: the hardware keeps a wavefront's LDS accesses in
// order, and this keeps the compiler from moving a read above a store that the
// reading lane does not make.  No instruction, LDS only.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// ------------------------------------------------------------------------
// Pass 1: HyperViscKernel! (src/GPU/ViscKernel.jl:1-84).
// Grid: one workgroup per ITEMS consecutive work items, an
// item being one (element, level chunk).  With ITEMS = 2 the loads of both
// items are issued before the first item's derivative phases, so a wave has
// twice the memory requests in flight (the kernel is latency-bound: its
// waves mostly wait on memory).  nitems = elements x nchunk.
// R is the arithmetic and storage type of the state it reads (U: the state,
// or its FP32 shadow), of the cache it writes and of the LDS tiles: double, or float in
// the mixed-precision mode.
template <typename R> struct Pass1In {
  R S11, S12, S21, S22, Js, iMs;
  R rho, u, v, rth;
  double rho_d, rth_d;  // FP32 kernel: the FP64 rho and rho*theta
  unsigned eo;          // offset of the point in its element's copies
  int e;
  bool valid;
};

// The FP32 (mixed-precision) element kernels compute the theta
// hyperviscosity -- Laplacian of theta in pass 1, the divergence of its
// gradient in pass 2 -- in FP64, from the FP64 state, with an FP64 cache:
// the fourth-order operator amplifies FP32 rounding of theta (and of its
// intermediate derivatives) into the w equation.  Its LDS tiles and
// derivative matrices sit in an FP64 region after the R-typed one.
template <int N, int NZ> struct ThetaHV {
  double *Dd, *DWd;        // D, DW (NN each)
  Tiles<N, NZ, double> A;  // phase-A tile(s)
  Tiles<N, NZ, double> B;  // phase-B tiles
};

template <int N, int NZT, bool CM, typename R>
__device__ __forceinline__ Pass1In<R> pass1_load(const KArgs &a, int nchunk, int nitems, int L,
                                                 const R *__restrict__ U, const double *__restrict__ U64) {
  constexpr int NN = N * N;
  const int Nz = a.Nz;
  const int e = L / nchunk;
  const int chunk = L - (L / nchunk) * nchunk;
  const int t = threadIdx.x;
  const int node = t / NZT, l = t - node * NZT;
  const int iz = chunk * NZT + l;
  const size_t vs = (size_t)a.NumG * Nz;
  const size_t NNZ = (size_t)NN * Nz;
  Pass1In<R> in{};
  in.valid = L < nitems && node < NN && iz < Nz;
  in.e = e;
  in.Js = 1;
  in.iMs = 1;
  if (!in.valid) return in;
  // uniform bases + 32-bit lane offsets (the host checks NumG*Nz < 2^28)
  const int gv = a.glob[(size_t)e * NN + node];
  const unsigned ui = (unsigned)(gv & 0x7fffffff) * (unsigned)Nz + iz;
  __builtin_assume(ui < (1u << 28));
  in.eo = (unsigned)(node * Nz + iz);
  if constexpr (CM) {
    const double *mN = a.met1n + (size_t)e * CGD_NMET1 * NN;
    const unsigned nd = (unsigned)node;
    in.S11 = R(at(mN, nd));
    in.S12 = R(at(mN + NN, nd));
    in.S21 = R(at(mN + 2 * NN, nd));
    in.S22 = R(at(mN + 3 * NN, nd));
    in.Js = R(at(mN + 4 * NN, nd));
  } else {
    const double *metE = a.met1 + (size_t)e * CGD_NMET1 * NNZ;
    const unsigned mo = (unsigned)(node * Nz + iz);
    __builtin_assume(mo < (1u << 28));
    in.S11 = R(at(metE, mo));
    in.S12 = R(at(metE + NNZ, mo));
    in.S21 = R(at(metE + 2 * NNZ, mo));
    in.S22 = R(at(metE + 3 * NNZ, mo));
    in.Js = R(at(metE + 4 * NNZ, mo));
  }
  const R *iMsR = std::is_same<R, double>::value ? reinterpret_cast<const R *>(a.iMs)
                                                  : reinterpret_cast<const R *>(a.iMs32);
  in.iMs = at(iMsR, ui);
  in.rho = at(U, ui);
  in.u = at(U + vs, ui);
  in.v = at(U + 2 * vs, ui);
  if constexpr (std::is_same<R, double>::value) {
    in.rth = at(U + 4 * vs, ui);
  } else {
    in.rho_d = at(U64, ui);
    in.rth_d = at(U64 + 4 * vs, ui);
  }
  return in;
}

// the derivative phases of one item and the write of its element copies
// (E; the FP64 theta cache Eth of the FP32 kernel); every lane of the
// workgroup calls it (two barriers)
template <int N, int NZT, typename R>
__device__ __forceinline__ void pass1_compute(const KArgs &a, const Pass1In<R> &in, const R *Ds, const R *DWs,
                                              const Tiles<N, NZT, R> &T, const Tiles<N, NZT, R> &TB,
                                              R *__restrict__ E, const ThetaHV<N, NZT> &H,
                                              double *__restrict__ Eth) {
  constexpr bool F32 = !std::is_same<R, double>::value;
  constexpr int NN = N * N;
  const int t = threadIdx.x;
  const int node = t / NZT, l = t - node * NZT;
  const bool in_tile = node < NN;
  const int I = node % N, J = node / N;
  const size_t eb = (size_t)in.e * NN * a.Nz;
  R uC = 0, vC = 0, uD = 0, vD = 0, Th = 0;
  if (in.valid) {
    uC = in.S11 * in.v - in.S12 * in.u;  // Curl12
    vC = in.S21 * in.v - in.S22 * in.u;
    uD = in.S11 * in.u + in.S12 * in.v;  // Contra12
    vD = in.S21 * in.u + in.S22 * in.v;
    if constexpr (!F32) Th = in.rth * rcp(in.rho);
  }
  double Thd = 0;
  if constexpr (F32) {
    if (in.valid) Thd = in.rth_d * rcp(in.rho_d);
  }
  if (in_tile) {
    T.at(0, node, l) = uC;
    T.at(1, node, l) = vC;
    T.at(2, node, l) = uD;
    T.at(3, node, l) = vD;
    if constexpr (F32) H.A.at(0, node, l) = Thd;
    else T.at(4, node, l) = Th;
  }
  __syncthreads();
  R Curl = 0, Div = 0, ThCx = 0, ThCy = 0;
  double ThCxd = 0, ThCyd = 0;
  if (in.valid) {
    const R iJs = rcp(in.Js);
    Curl = dxy<N, NZT, R>(Ds, T, 0, 1, I, J, l) * iJs;
    Div = dxy<N, NZT, R>(Ds, T, 2, 3, I, J, l) * iJs;
    if constexpr (F32) {
      const double Dxc = dx<N, NZT, double>(H.Dd, H.A, 0, I, J, l);
      const double Dyc = dy<N, NZT, double>(H.Dd, H.A, 0, I, J, l);
      const double S11 = in.S11, S12 = in.S12, S21 = in.S21, S22 = in.S22;
      const double iJsd = rcp(double(in.Js));
      const double GDx = (S11 * Dxc + S21 * Dyc) * iJsd;
      const double GDy = (S12 * Dxc + S22 * Dyc) * iJsd;
      ThCxd = S11 * GDx + S12 * GDy;
      ThCyd = S21 * GDx + S22 * GDy;
    } else {
      const R Dxc = dx<N, NZT, R>(Ds, T, 4, I, J, l);
      const R Dyc = dy<N, NZT, R>(Ds, T, 4, I, J, l);
      const R GDx = (in.S11 * Dxc + in.S21 * Dyc) * iJs;  // Grad12 with J
      const R GDy = (in.S12 * Dxc + in.S22 * Dyc) * iJs;
      ThCx = in.S11 * GDx + in.S12 * GDy;  // Contra12
      ThCy = in.S21 * GDx + in.S22 * GDy;
    }
  }
  if (in_tile) {
    TB.at(0, node, l) = Curl;
    TB.at(1, node, l) = Div;
    if constexpr (F32) {
      H.B.at(0, node, l) = ThCxd;
      H.B.at(1, node, l) = ThCyd;
    } else {
      TB.at(2, node, l) = ThCx;
      TB.at(3, node, l) = ThCy;
    }
  }
  __syncthreads();
  if (in.valid) {
    const R DxCurl = dx<N, NZT, R>(DWs, TB, 0, I, J, l);
    const R DyCurl = dy<N, NZT, R>(DWs, TB, 0, I, J, l);
    const R DxDiv = dx<N, NZT, R>(DWs, TB, 1, I, J, l);
    const R DyDiv = dy<N, NZT, R>(DWs, TB, 1, I, J, l);
    R DivTh = 0;
    if constexpr (!F32) DivTh = dxy<N, NZT, R>(DWs, TB, 2, 3, I, J, l);
    const R FuC = in.S12 * DxCurl + in.S22 * DyCurl;  // Rot12
    const R FvC = -in.S11 * DxCurl - in.S21 * DyCurl;
    const R FuD = in.S11 * DxDiv + in.S21 * DyDiv;  // Grad12
    const R FvD = in.S12 * DxDiv + in.S22 * DyDiv;
    const R iMs = in.iMs;
    R *Ea = E + eb, *Eb = Ea + a.ecs, *Ec = Eb + a.ecs, *Ed = Ec + a.ecs, *Ee = Ed + a.ecs;
    at(Ea, in.eo) = -FuC * iMs;
    at(Eb, in.eo) = -FvC * iMs;
    at(Ec, in.eo) = FuD * iMs;
    at(Ed, in.eo) = FvD * iMs;
    if constexpr (F32) at(Eth + eb, in.eo) = dxy<N, NZT, double>(H.DWd, H.B, 0, 1, I, J, l) * double(iMs);
    else at(Ee, in.eo) = DivTh * iMs;
  }
}

// U64, Eth: the FP64 state and the FP64 theta cache of the FP32 kernel
// (unused by the FP64 one).  The body is shared by the kernel and by
// fcn1_block, a workgroup's share in a persistent launch (items item*ITEMS
// .. item*ITEMS + ITEMS - 1).
template <int N, int NZT, bool CM, typename R, int ITEMS>
__device__ __forceinline__ void fcn1_block(int item, const KArgs &a, int nchunk, int nitems, const R *__restrict__ U,
                                           R *__restrict__ E, const double *__restrict__ U64,
                                           double *__restrict__ Eth) {
#define CGD_ITEM item
#include "cgd_pass1_body.inc"
#undef CGD_ITEM
}

template <int N, int NZT, bool CM, typename R, int ITEMS>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64) k_fcn1(KArgs a, int nchunk, int nitems,
                                                                       const R *__restrict__ U, R *__restrict__ E,
                                                                       const double *__restrict__ U64,
                                                                       double *__restrict__ Eth) {
#define CGD_ITEM xcd_logical(blockIdx.x, gridDim.x)
#include "cgd_pass1_body.inc"
#undef CGD_ITEM
}

// Pass 1 over whole columns (compact metric, Nz <= 64): one workgroup per
// element, one wavefront per row J of its nodes, lane = level, so a lane
// holds the N nodes of its row.
// - Every load and store is one node's column, a whole run of 8 Nz bytes; the
//   chunked kernel's 64-byte pieces are what bounds it: 711 us at ne = 60,
//   nz = 64 in 8-level chunks, 669 in 16-level ones, 466 in columns.
// - The derivatives along the row need no LDS, and the node's metric, the
//   derivative matrices and the addresses are uniform (scalar registers);
//   only the derivatives across the rows exchange values through LDS.
// The operations are those of k_fcn1, term by term.
template <int N, typename R>
__device__ __forceinline__ void fcn1c_block(int e, const KArgs &a, const R *__restrict__ U, R *__restrict__ E,
                                            const double *__restrict__ U64, double *__restrict__ Eth) {
  constexpr int NN = N * N;
  constexpr bool F32 = !std::is_same<R, double>::value;
  extern __shared__ double smem[];
  double *TD = smem;                                     // theta, then its flux across the rows
  R *T0 = reinterpret_cast<R *>(smem + NN * 64), *T1 = T0 + NN * 64;  // the curl's and the divergence's
  const int Nz = a.Nz;
  const int lane = threadIdx.x & 63, J = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool valid = lane < Nz;
  const unsigned iz = valid ? lane : Nz - 1;
  const size_t vs = (size_t)a.NumG * Nz;
  const Const<int> gE = as_const(a.glob + (size_t)e * NN + J * N);
  const Const<double> mE = as_const(a.met1n + (size_t)e * CGD_NMET1 * NN + J * N);
  const R *iMsR = F32 ? reinterpret_cast<const R *>(a.iMs32) : reinterpret_cast<const R *>(a.iMs);
  const R *Dm = F32 ? reinterpret_cast<const R *>(a.Df) : reinterpret_cast<const R *>(a.D);
  const R *DWm = F32 ? reinterpret_cast<const R *>(a.DWf) : reinterpret_cast<const R *>(a.DWm);
  R u[N], v[N], iMs[N];
  double rho[N], rth[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const size_t c0 = (size_t)(gE[i] & 0x7fffffff) * Nz;
    u[i] = at(U + vs + c0, iz);
    v[i] = at(U + 2 * vs + c0, iz);
    rho[i] = at(U64 + c0, iz);
    rth[i] = at(U64 + 4 * vs + c0, iz);
    iMs[i] = at(iMsR + c0, iz);
  }
  R uC[N], uD[N];
  double Th[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const R S11 = R(mE[i]), S12 = R(mE[NN + i]), S21 = R(mE[2 * NN + i]), S22 = R(mE[3 * NN + i]);
    const int o = (J * N + i) * 64 + lane;
    uC[i] = S11 * v[i] - S12 * u[i];  // Curl12
    T0[o] = S21 * v[i] - S22 * u[i];
    uD[i] = S11 * u[i] + S12 * v[i];  // Contra12
    T1[o] = S21 * u[i] + S22 * v[i];
    Th[i] = rth[i] * rcp(rho[i]);
    TD[o] = Th[i];
  }
  __syncthreads();
  R Curl[N], Div[N];
  double ThCx[N], ThCy[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    R cu = Dm[i * N] * uC[0] + Dm[J * N] * T0[i * 64 + lane];
    R dv = Dm[i * N] * uD[0] + Dm[J * N] * T1[i * 64 + lane];
    double cx = a.D[i * N] * Th[0], cy = a.D[J * N] * TD[i * 64 + lane];
#pragma unroll
    for (int q = 1; q < N; ++q) {
      const int o = (i + q * N) * 64 + lane;
      cu += Dm[i * N + q] * uC[q] + Dm[J * N + q] * T0[o];
      dv += Dm[i * N + q] * uD[q] + Dm[J * N + q] * T1[o];
      cx += a.D[i * N + q] * Th[q];
      cy += a.D[J * N + q] * TD[o];
    }
    const double S11 = R(mE[i]), S12 = R(mE[NN + i]), S21 = R(mE[2 * NN + i]), S22 = R(mE[3 * NN + i]);
    const R Js = R(mE[4 * NN + i]);
    const R iJs = rcp(Js);
    Curl[i] = cu * iJs;
    Div[i] = dv * iJs;
    const double iJd = rcp(double(Js));
    const double gx = (S11 * cx + S21 * cy) * iJd;  // Grad12 with J
    const double gy = (S12 * cx + S22 * cy) * iJd;
    ThCx[i] = S11 * gx + S12 * gy;  // Contra12
    ThCy[i] = S21 * gx + S22 * gy;
    pin(Curl[i], Div[i], ThCx[i], ThCy[i]);
  }
  __syncthreads();  // the tiles have been read
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int o = (J * N + i) * 64 + lane;
    T0[o] = Curl[i];
    T1[o] = Div[i];
    TD[o] = ThCy[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    R xC = DWm[i * N] * Curl[0], yC = DWm[J * N] * T0[i * 64 + lane];
    R xD = DWm[i * N] * Div[0], yD = DWm[J * N] * T1[i * 64 + lane];
    double dt = a.DWm[i * N] * ThCx[0] + a.DWm[J * N] * TD[i * 64 + lane];
#pragma unroll
    for (int q = 1; q < N; ++q) {
      const int o = (i + q * N) * 64 + lane;
      xC += DWm[i * N + q] * Curl[q];
      yC += DWm[J * N + q] * T0[o];
      xD += DWm[i * N + q] * Div[q];
      yD += DWm[J * N + q] * T1[o];
      dt += a.DWm[i * N + q] * ThCx[q] + a.DWm[J * N + q] * TD[o];
    }
    const R S11 = R(mE[i]), S12 = R(mE[NN + i]), S21 = R(mE[2 * NN + i]), S22 = R(mE[3 * NN + i]);
    const R FuC = S12 * xC + S22 * yC;  // Rot12
    const R FvC = -S11 * xC - S21 * yC;
    const R FuD = S11 * xD + S21 * yD;  // Grad12
    const R FvD = S12 * xD + S22 * yD;
    R o1 = -FuC * iMs[i], o2 = -FvC * iMs[i], o3 = FuD * iMs[i], o4 = FvD * iMs[i];
    double o5 = dt * double(iMs[i]);
    pin(o1, o2, o3, o4, o5);
    if (valid) {
      R *Ea = E + ((size_t)e * NN + J * N + i) * Nz;
      at(Ea, iz) = o1;
      at(Ea + a.ecs, iz) = o2;
      at(Ea + 2 * a.ecs, iz) = o3;
      at(Ea + 3 * a.ecs, iz) = o4;
      if constexpr (F32) at(Eth + ((size_t)e * NN + J * N + i) * Nz, iz) = o5;
      else at(Ea + 4 * a.ecs, iz) = o5;
    }
  }
}

template <int N, typename R>
__global__ void __launch_bounds__(N * 64) __attribute__((amdgpu_waves_per_eu(5))) k_fcn1c(KArgs a, const R *__restrict__ U, R *__restrict__ E,
                                                  const double *__restrict__ U64, double *__restrict__ Eth) {
  fcn1c_block<N, R>(xcd_logical(blockIdx.x, gridDim.x), a, U, E, U64, Eth);
}

// ------------------------------------------------------------------------
// Pass 2: HyperViscKoeffKernel! + MomentumVectorInvariantCoriolisKernel! +
// GradFullKernel! + DivRhoTrUpwind3New2Kernel! fused into one element pass
// (src/GPU/ViscKernel.jl:86-167, src/GPU/MomentumKernel.jl:1-178,
// src/GPU/GradKineticKernel.jl:1-129, src/GPU/OperatorKernel.jl:637-720).
// One launch over (element, level chunk) workgroups; the chunks of one
// element are independent.
//
// Phase 0 computes every term that couples levels (vertical momentum
// fluxes, kinetic-energy and pressure differences, the upwind mass and
// theta fluxes through both interfaces of the layer) from the neighbour
// levels, so those values are dead before the LDS phases start.  Each
// thread adds the fluxes of both its interfaces to its own level (the
// reference adds them from the owner of the interface); F4 of interface iz
// combines this layer's upper terms with the layer above's lower terms.
// C holds the pass-1 cache as element copies (each point sums its node's),
// F receives the element copies of the tendency, and Cout (FP64, may be
// null) the summed cache in the layout of Temp1.
// R is the arithmetic and storage type of the tendency (F, the chunk side
// sums F4x), of the hyperviscosity cache C, of the winds and rho*theta
// it reads (UR: the state, or its FP32 shadow) and of the LDS tiles: double,
// or float in the mixed-precision mode.  FP64 in both modes: rho (from the
// FP64 state U), the pressure P, the w-interface balance of pressure
// gradient and gravity (rho, p, J and dXdxI[3,3] in FP64), the horizontal
// pressure gradient (an FP64 tile and derivative) and the theta
// hyperviscosity (its FP64 cache Cth, FP64 tiles and derivatives).
// The body is shared by the kernel and by fcn2_block, one item of a
// persistent launch.
template <int N, int NZT, bool CM, typename R, bool SM>
__device__ __forceinline__ void fcn2_block(int item, const KArgs &a, int nchunk,
                                           const double *__restrict__ U, const R *__restrict__ UR,
                                           const R *__restrict__ C, const double *__restrict__ P,
                                           R *__restrict__ F, R *__restrict__ F4x,
                                           const double *__restrict__ Cth, double *__restrict__ Cout) {
#define CGD_ITEM item
#define CGD_EARLY_HALO false
#include "cgd_pass2_body.inc"
#undef CGD_EARLY_HALO
#undef CGD_ITEM
}

// Waves per SIMD: what fits without spills, 4 in FP64 and 5 in FP32.  The kink-
// smoothed flux (SM) takes 142 registers in the full layout: at 4 waves it
// spilled 14 (2400 elements of 45 levels 376 us, 337 at 3 waves).  In the compact
// layout 3 waves also hold the early halo levels and copies, 154 registers: 5400
// elements of 64 levels 1009 us with 16 spilled at 4 waves, 897 at 3.
template <int N, int NZT, bool CM, typename R, bool SM>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64) __attribute__((amdgpu_waves_per_eu(std::is_same<R, float>::value ? 5 : SM ? 3 : 4))) k_fcn2(KArgs a, int nchunk,
                                               const double *__restrict__ U, const R *__restrict__ UR,
                                               const R *__restrict__ C, const double *__restrict__ P,
                                               R *__restrict__ F, R *__restrict__ F4x,
                                               const double *__restrict__ Cth, double *__restrict__ Cout) {
#define CGD_ITEM xcd_logical(blockIdx.x, gridDim.x)
#define CGD_EARLY_HALO true
#include "cgd_pass2_body.inc"
#undef CGD_EARLY_HALO
#undef CGD_ITEM
}

// Pass 2 for the regular compact metric (FP64): the same terms, reduced by
// what such a metric and mass share between levels and vertical nodes.
template <int N, int NZT>
__device__ __forceinline__ void fcn2r_block(int item, const KArgs &a, int nchunk, const double *__restrict__ U,
                                            const double *__restrict__ C, const double *__restrict__ P,
                                            double *__restrict__ F, double *__restrict__ F4x,
                                            double *__restrict__ Cout) {
#define CGD_ITEM item
#include "cgd_pass2r_body.inc"
#undef CGD_ITEM
}

template <int N, int NZT>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64) __attribute__((amdgpu_waves_per_eu(5)))
    k_fcn2r(KArgs a, int nchunk, const double *__restrict__ U, const double *__restrict__ C,
            const double *__restrict__ P, double *__restrict__ F, double *__restrict__ F4x,
            double *__restrict__ Cout) {
#define CGD_ITEM xcd_logical(blockIdx.x, gridDim.x)
#include "cgd_pass2r_body.inc"
#undef CGD_ITEM
}

// ------------------------------------------------------------------------
// Pointwise physics hooks at the end of FcnGPU! (FcnGPU.jl:953-966), per
// global point: HeldSuarezForcing (src/Examples/force.jl:5-27) on F2, F3, F5
// from rho, u, v, the pressure p and the latitude, then DampingW
// (src/GPU/dampingGPU.jl:5-16) on F4 from w and the layer-centre height.
struct Hooks {
  int forcing, damping, micro;
  double k_a, k_f, k_s, DeltaT_y, DeltaTh_z, T_equator, T_min, sigma_b;
  double H, Stride, Relax;
  double RelCloud, Rain, T0, L00;  // SimpleMicrophysics (Models.Moist state, components a.iv, a.ic)
  const double *xS;  // (2, NumG)
  const double *zP;  // (Nz, NumG)
};
// s: the five components of the dynamics' tendency at point i (R-typed);
// Ftr: the FP64 tendency array, whose components 6.. are the tracers'
template <typename R>
__device__ __forceinline__ void hooks_point(const KArgs &a, const Hooks &hk, const double *__restrict__ U,
                                            const double *__restrict__ P, R (&s)[5], double *__restrict__ Ftr,
                                            size_t i, size_t n) {
  const size_t vs = n;
  if (hk.forcing) {
    const size_t ig = i / a.Nz;
    const double rho = U[i], u = U[vs + i], v = U[2 * vs + i];
    const double lat = hk.xS[2 * ig + 1];
    const double Sigma = P[i] / a.p0;
    const double SigmaPowKappa = exp(a.kappa * log(Sigma));  // fast_powGPU
    const double hf = jmax(0.0, (Sigma - hk.sigma_b) / (1.0 - hk.sigma_b));
    const double coslat = cos(lat), sinlat = sin(lat);
    s[1] = R(double(s[1]) + -(hk.k_f * hf) * u);
    s[2] = R(double(s[2]) + -(hk.k_f * hf) * v);
    const double kT = Sigma < 0.7 ? hk.k_a + (hk.k_s - hk.k_a) * hf * coslat * coslat * coslat * coslat : 0.0;
    double Teq = (hk.T_equator - hk.DeltaT_y * sinlat * sinlat - hk.DeltaTh_z * log(Sigma) * coslat * coslat) *
                 SigmaPowKappa;
    Teq = jmax(hk.T_min, Teq);
    const double DeltaT = kT * (a.p0 * Sigma / (rho * a.Rd) - Teq);
    s[4] = R(double(s[4]) + -rho * DeltaT / SigmaPowKappa);
  }
  if (hk.micro) {
    // SimpleMicrophysics (src/Models/Microphysics.jl:6-40) through
    // MicrophysicsKernel! (OperatorKernel.jl:1082-1089): relaxation of the
    // vapour towards saturation (fpvs, src/Thermodynamics/Thermodynamics.jl:27-35)
    // through cloud, the latent heating in rho*theta (LatHeat, :83-85), and
    // the rain-out fraction Rain of the condensate leaving rho
    const double p = P[i];
    const double Rho = U[i], RhoTh = U[4 * vs + i];
    const double RhoV = jmax(U[(size_t)a.iv * vs + i], 0.0), RhoC = jmax(U[(size_t)a.ic * vs + i], 0.0);
    const double RhoD = Rho - RhoV - RhoC;
    const double Cpml = a.Cpd * RhoD + a.Cpv * RhoV + a.Cpl * RhoC;
    const double Rm = a.Rd * RhoD + a.Rv * RhoV;
    const double T = p / Rm;
    const double T_C = T - hk.T0;
    const double p_vs = 611.2 * exp(17.62 * T_C / (243.12 + T_C));
    const double am = p_vs / (a.Rv * T) - RhoV;
    const double bm = RhoC;
    const double FPh = 0.5 * hk.RelCloud * (am + bm - sqrt(am * am + bm * bm));
    const double L = hk.L00 - (a.Cpl - a.Cpv) * (T - hk.T0);
    const double FR = -FPh * hk.Rain;
    const double lp = log(p / a.p0);
    const double FRhoTh =
        RhoTh * ((-L / (Cpml * T) - lp * (Rm / Cpml) * (a.Rv / Rm + (a.Cpl - a.Cpv) / Cpml) + a.Rv / Rm) * FPh +
                 (1.0 / Rho - lp * (Rm / Cpml) * (a.Cpl / Cpml)) * FR);
    s[0] = R(double(s[0]) + -FR);
    s[4] = R(double(s[4]) + FRhoTh);
    Ftr[(size_t)a.iv * vs + i] += FPh;
    Ftr[(size_t)a.ic * vs + i] += -FPh - FR;
  }
  if (hk.damping) {
    const double z = hk.zP[i];
    if (z >= hk.H - hk.Stride) {
      const double sn = sin(0.5 * M_PI * (1.0 - (hk.H - z) / hk.Stride));
      const double Damp = hk.Relax * (sn * sn);
      s[3] = R(double(s[3]) + -Damp * U[3 * vs + i]);
    }
  }
}

// ------------------------------------------------------------------------
// Tracers (NumTr > 0, FP64): components 5..4+NumTr of U/F (0-based), their
// hyperviscosity caches at the same components of Temp1 (FcnGPU.jl:115-126).
// Each tracer repeats the rho*theta path: HyperViscTracerKernel!
// (ViscKernel.jl:169-218) in pass 1, HyperViscTracerKoeffKernel!
// (:277-327) and the tracer loop of DivRhoTrUpwind3New2Kernel!
// (OperatorKernel.jl:722-759) in pass 2.  The kernels run after the
// corresponding main pass, over (element, level chunk) workgroups, all tracers
// in one launch; like the dynamics' passes they write element copies
// ([tracer][element][node][Nz]) and read the sums of the previous pass's.
// They are bound by the latency of their loads, so pass 2 issues the halo
// levels' with the own level's, and in the compact layout, whose volumes are
// the same at all levels, fits five waves per SIMD.  Per stage, two tracers,
// ne = 24, nz = 40, with one launch per colour and sums in place before:
// pass 1 80 -> 59 us, pass 2 244 -> 187, limited pass 2 352 -> 296.
// Tracers do not feed back on the dynamics.

// metric component c of element e at (node, level), either layout
template <int NN, bool CM>
__device__ __forceinline__ double met_at(const KArgs &a, size_t e, int c, int node, int iz) {
  const size_t Nz = (size_t)a.Nz;
  if (CM) {
    if (met_per_point(c)) return a.met[((e * CGD_NMETP + met_pidx(c)) * NN + node) * Nz + iz];
    return a.metn[(e * CGD_NMETN + met_nidx(c)) * NN + node];
  }
  return a.met[((e * CGD_NMET + c) * NN + node) * Nz + iz];
}

// pass 1: the tracer caches, r = div(grad c) / (M1 + M2) with c = q / rho
template <int N, int NZT, bool CM>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64) k_tr1(KArgs a, int nchunk, int ntr,
                                                                      const double *__restrict__ U,
                                                                      double *__restrict__ E1) {
  constexpr int NN = N * N;
  extern __shared__ double smem[];
  double *Ds = smem, *DWs = Ds + NN;
  Tiles<N, NZT, double> T{Ds + 2 * NN};  // field 0: c; fields 1, 2: the contravariant gradient
  load_dmats<N>(a, Ds, DWs);
  const int Nz = a.Nz;
  const int L = xcd_logical(blockIdx.x, gridDim.x);
  const int e = L / nchunk;
  const int chunk = L - e * nchunk;
  const int t = threadIdx.x;
  const int node = t / NZT, l = t - node * NZT;
  const int iz = chunk * NZT + l;
  const bool in_tile = node < NN;
  const bool valid = in_tile && iz < Nz;
  const int I = node % N, J = node / N;
  const size_t vs = (size_t)a.NumG * Nz;
  double S11 = 0, S12 = 0, S21 = 0, S22 = 0, iJs = 1, iMs = 1, irho = 1;
  size_t ui = 0;
  if (valid) {
    ui = (size_t)(a.glob[e * NN + node] & 0x7fffffff) * Nz + iz;
    if constexpr (CM) {
      const double *mN = a.met1n + (size_t)e * CGD_NMET1 * NN;
      S11 = mN[node];
      S12 = mN[NN + node];
      S21 = mN[2 * NN + node];
      S22 = mN[3 * NN + node];
      iJs = rcp(mN[4 * NN + node]);
    } else {
      const size_t NNZ = (size_t)NN * Nz, mo = (size_t)node * Nz + iz;
      const double *metE = a.met1 + (size_t)e * CGD_NMET1 * NNZ;
      S11 = metE[mo];
      S12 = metE[NNZ + mo];
      S21 = metE[2 * NNZ + mo];
      S22 = metE[3 * NNZ + mo];
      iJs = rcp(metE[4 * NNZ + mo]);
    }
    iMs = a.iMs[ui];
    irho = rcp(U[ui]);
  }
  for (int tr = 0; tr < ntr; ++tr) {
    const size_t off = (size_t)(5 + tr) * vs;
    if (valid) {
      T.at(0, node, l) = U[off + ui] * irho;
    } else if (in_tile) {
      T.at(0, node, l) = 0;
    }
    __syncthreads();
    if (in_tile) {
      double Cx = 0, Cy = 0;
      if (valid) {
        const double Dxc = dx<N, NZT, double>(Ds, T, 0, I, J, l);
        const double Dyc = dy<N, NZT, double>(Ds, T, 0, I, J, l);
        const double GDx = (S11 * Dxc + S21 * Dyc) * iJs;  // Grad12 with J
        const double GDy = (S12 * Dxc + S22 * Dyc) * iJs;
        Cx = S11 * GDx + S12 * GDy;  // Contra12
        Cy = S21 * GDx + S22 * GDy;
      }
      T.at(1, node, l) = Cx;
      T.at(2, node, l) = Cy;
    }
    __syncthreads();
    if (valid)
      E1[tr * a.ecs + ((size_t)e * NN + node) * Nz + iz] = dxy<N, NZT, double>(DWs, T, 1, 2, I, J, l) * iMs;
    __syncthreads();  // the next tracer rewrites the tiles
  }
}

// pass 2: -Kd div(rho grad C) / (M1 + M2) from the cache C, the upwind
// vertical flux of c = q / rho through both interfaces of the layer (the
// same contravariant w and RecU4 weights as rho*theta) and the horizontal
// divergence of (-rho v) c.  As in k_fcn2, the values of the neighbour
// levels come from DPP row shifts (halo loads only at chunk edges), fields
// are addressed by uniform bases plus 32-bit offsets, and the compact
// metric layout is read per node.
template <int N, int NZT, bool CM>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64) __attribute__((amdgpu_waves_per_eu(CM ? 5 : 4)))
    k_tr2(KArgs a, int nchunk, int ntr, const double *__restrict__ U, const double *__restrict__ E1,
          double *__restrict__ Cout, double *__restrict__ E2) {
  constexpr int NN = N * N;
  static_assert(NZT >= 4 && NZT <= 16 && 64 % NZT == 0, "chunk heights 4, 8 or 16 (halo levels share registers)");
  extern __shared__ double smem[];
  double *Ds = smem, *DWs = Ds + NN;
  // fields 0, 1: uc, vc (all tracers); 2..5 and 6..9: C, c, and the
  // rho-weighted contravariant gradient of C, for alternate tracers
  Tiles<N, NZT, double> T{Ds + 2 * NN};
  load_dmats<N>(a, Ds, DWs);
  const int Nz = a.Nz;
  const int L = xcd_logical(blockIdx.x, gridDim.x);
  const int e = L / nchunk;
  const int chunk = L - e * nchunk;
  const int t = threadIdx.x;
  const int node = t / NZT, l = t - node * NZT;
  const int iz = chunk * NZT + l;
  const bool in_tile = node < NN;
  const bool valid = in_tile && iz < Nz;
  const int I = node % N, J = node / N;
  const unsigned vs = (unsigned)a.NumG * (unsigned)Nz;
  const size_t NNZ = (size_t)NN * Nz;
  const bool has_lo = iz > 0, has_hi = iz < Nz - 1;
  const double Kd = a.kvis[3 * e + 2];
  const double *metE = a.met + (size_t)e * (CM ? CGD_NMETP : CGD_NMET) * NNZ;
  const double *metN = CM ? a.metn + (size_t)e * CGD_NMETN * NN : nullptr;
  unsigned ui = 0, mo = 0;
  int cpa = 0, cpb = -1;  // the node's first two element copies
  const int *cpl = a.cpy + ((size_t)e * NN + (in_tile ? node : 0)) * a.cpw;
  bool first = false;
  if (valid) {
    const int gv = a.glob[e * NN + node];
    first = gv < 0;
    cpa = cpl[0];
    cpb = cpl[1];
    ui = (unsigned)(gv & 0x7fffffff) * (unsigned)Nz + iz;
    mo = (unsigned)(node * Nz + iz);
  }
  __builtin_assume(ui < (1u << 28));
  __builtin_assume(mo < (1u << 28));
#define MET(c, off) at(metE + (size_t)(CM ? met_pidx(c) : (c)) * NNZ, mo + (off))
#define METN(c) at(metN + (size_t)met_nidx(c) * NN, (unsigned)node)
#define MET0(c) (CM && !met_per_point(c) ? METN(c) : MET(c, 0))
  const double *Uu = U + vs, *Uv = U + 2 * (size_t)vs, *Uw = U + 3 * (size_t)vs;
  double rho = 1, u = 0, v = 0, w = 0, S11 = 0, S12 = 0, S21 = 0, S22 = 0, Js = 1, iMs = 1;
  double d311 = 0, d312 = 0, d321 = 0, d322 = 0, d331 = 1, d332 = 1;
  if (valid) {
    rho = at(U, ui);
    u = at(Uu, ui);
    v = at(Uv, ui);
    w = at(Uw, ui);
    iMs = at(a.iMs, ui);
    S11 = MET0(M111) + MET0(M112);
    S12 = MET0(M121) + MET0(M122);
    S21 = MET0(M211) + MET0(M212);
    S22 = MET0(M221) + MET0(M222);
    Js = MET0(MJ1) + MET0(MJ2);
    d311 = MET0(M311);
    d312 = MET0(M312);
    d321 = MET0(M321);
    d322 = MET0(M322);
    d331 = MET0(M331);
    d332 = MET0(M332);
  }
  // neighbour levels (a node's chunk is one half of a 16-lane DPP row); the
  // halo loads of the chunk-edge lanes are issued with the own level's
  const int lr = threadIdx.x & 15;
  const bool edge_m1 = l < 1 || lr < 1, edge_m2 = l < 2 || lr < 2;
  const bool edge_p1 = l + 1 >= NZT || lr + 1 > 15, edge_p2 = l + 2 >= NZT || lr + 2 > 15;
  const bool hm1 = valid && has_lo && edge_m1, hm2 = valid && iz >= 2 && edge_m2;
  const bool hp1 = valid && has_hi && edge_p1, hp2 = valid && iz + 2 <= Nz - 1 && edge_p2;
  // (the lanes' lower and upper halo levels share registers: with chunks of at
  // least 4 levels no lane has both: in one of 3 the middle one would)
  double hrho = 1, hu = 0, hv = 0, hw = 0, h31 = 0, h32 = 0, h33 = 0, hJ = 1, hrho2 = 1, hJ2 = 1;
  if (hm1 || hp1) {
    const unsigned uh = hm1 ? ui - 1 : ui + 1;
    hrho = at(U, uh);
    hu = at(Uu, uh);
    hv = at(Uv, uh);
    hw = at(Uw, uh);
    const int off = hm1 ? -1 : 1;
    h31 = at(metE + (size_t)(CM ? met_pidx(M311) : M311) * NNZ + (hm1 ? NNZ : 0), mo + off);
    h32 = at(metE + (size_t)(CM ? met_pidx(M321) : M321) * NNZ + (hm1 ? NNZ : 0), mo + off);
    if constexpr (!CM) {
      h33 = at(metE + (size_t)M331 * NNZ + (hm1 ? NNZ : 0), mo + off);
      hJ = MET(MJ1, off) + MET(MJ2, off);
    }
  }
  if (hm2 || hp2) {
    const int off = hm2 ? -2 : 2;
    hrho2 = at(U, ui + off);
    if constexpr (!CM) hJ2 = MET(MJ1, off) + MET(MJ2, off);
  }
  const double irho = rcp(rho), iJs = rcp(Js);
  double rho_m = dpp_from_below<1>(rho), u_m = dpp_from_below<1>(u), v_m = dpp_from_below<1>(v);
  double w_m = dpp_from_below<1>(w), d312m = dpp_from_below<1>(d312), d322m = dpp_from_below<1>(d322);
  double d332m = CM ? d332 : dpp_from_below<1>(d332);
  double rho_p = dpp_from_above<1>(rho), u_p = dpp_from_above<1>(u), v_p = dpp_from_above<1>(v);
  double d311p = dpp_from_above<1>(d311), d321p = dpp_from_above<1>(d321);
  double d331p = CM ? d331 : dpp_from_above<1>(d331);
  double Jm = CM ? Js : dpp_from_below<1>(Js), Jmm = CM ? Js : dpp_from_below<2>(Js);
  double Jp = CM ? Js : dpp_from_above<1>(Js), Jpp = CM ? Js : dpp_from_above<2>(Js);
  const double irh = rcp(hrho), irh2 = rcp(hrho2);
  if (hm1) {
    rho_m = hrho;
    u_m = hu;
    v_m = hv;
    w_m = hw;
    d312m = h31;
    d322m = h32;
    if constexpr (!CM) {
      d332m = h33;
      Jm = hJ;
    }
  }
  if constexpr (!CM)
    if (hm2) Jmm = hJ2;
  if (hp1) {
    rho_p = hrho;
    u_p = hu;
    v_p = hv;
    d311p = h31;
    d321p = h32;
    if constexpr (!CM) {
      d331p = h33;
      Jp = hJ;
    }
  }
  if constexpr (!CM)
    if (hp2) Jpp = hJ2;
  // clamped levels iz-1, iz-2 >= 0 and iz+2 <= Nz-1 (the reference's max/min);
  // at iz = 0 the shifted values belong to another node's lanes
  if (iz == 0) Jm = Js;
  if (iz == 1) Jmm = Jm;
  if (iz + 2 > Nz - 1) Jpp = Jp;
  // contravariant mass fluxes through the interfaces (Contra3)
  double wlo = 0, wup = 0;
  if (valid && has_lo) wlo = rho_m * (d312m * u_m + d322m * v_m + d332m * w_m) + rho * (d311 * u + d321 * v + d331 * w_m);
  if (valid && has_hi) wup = rho * (d312 * u + d322 * v + d332 * w) + rho_p * (d311p * u_p + d321p * v_p + d331p * w);
  // RecU4 weights of the upper interface (and of the lower one, used by the
  // lanes at a chunk's bottom edge), shared by all tracers
  // (the compact layout's volumes are those of every level)
  const RecW<double> Wup = CM ? recu4_equal<double>() : recu4_weights(Jm, Js, Jp, Jpp);
  const RecW<double> Wlo = CM ? recu4_equal<double>() : recu4_weights(Jmm, Jm, Js, has_hi ? Jp : Js);
  pin(wlo, wup);
  // the tracer-independent tiles: (uc, vc) = Contra12(-rho, u, v)
  if (in_tile) {
    T.at(0, node, l) = -rho * (S11 * u + S12 * v);
    T.at(1, node, l) = -rho * (S21 * u + S22 * v);
  }
  // Contra12 of Grad12 with rho / J: a symmetric matrix
  double Gxx = (S11 * S11 + S12 * S12) * rho * iJs, Gxy = (S11 * S21 + S12 * S22) * rho * iJs;
  double Gyy = (S21 * S21 + S22 * S22) * rho * iJs;
  pin(Gxx, Gxy, Gyy);
  for (int tr = 0; tr < ntr; ++tr) {
    // two sets of per-tracer tiles (C, c, Cx, Cy) used alternately, so a
    // tracer's tiles are never rewritten before every lane has passed the
    // next tracer's first barrier
    const int b = 2 + 4 * (tr & 1);
    const double *Q = U + (size_t)(5 + tr) * vs;
    const double *C = E1 + tr * a.ecs;
    double cown = 0, Cown = 0, Cb = 0, q1 = 0, q2 = 0;
    if (valid) {
      cown = at(Q, ui);
      Cown = C[(size_t)cpa * Nz + iz];
    }
    if (hm1 || hp1) q1 = at(Q, hm1 ? ui - 1 : ui + 1);
    if (hm2 || hp2) q2 = at(Q, hm2 ? ui - 2 : ui + 2);
    if (cpb >= 0) {
      Cb = C[(size_t)cpb * Nz + iz];
      for (int q = 2; q < a.cpw && cpl[q] >= 0; ++q) {
        Cown += Cb;
        Cb = C[(size_t)cpl[q] * Nz + iz];
      }
    }
    cown *= irho;
    double c_m = dpp_from_below<1>(cown), c_mm = dpp_from_below<2>(cown);
    double c_p = dpp_from_above<1>(cown), c_pp = dpp_from_above<2>(cown);
    if (hm1) c_m = q1 * irh;
    if (hm2) c_mm = q2 * irh2;
    if (hp1) c_p = q1 * irh;
    if (hp2) c_pp = q2 * irh2;
    Cown += Cb;
    if (Cout && first) at(Cout + (size_t)(5 + tr) * vs, ui) = Cown;  // Temp1
    if (iz == 0) c_m = cown;
    if (iz == 1) c_mm = c_m;
    if (iz + 2 > Nz - 1) c_pp = c_p;
    if (in_tile) {
      T.at(b, node, l) = Cown;
      T.at(b + 1, node, l) = cown;
    }
    // upper-interface flux; the lower one is the upper flux of the level
    // below, taken from its lane (lanes at a chunk's bottom edge compute it)
    double Fup = 0;
    if (valid && has_hi) Fup = recu4_flux(c_m, cown, c_p, c_pp, Wup, wup);
    double Flo = dpp_from_below<1>(Fup);
    if (valid && has_lo && edge_m1) Flo = recu4_flux(c_mm, c_m, cown, has_hi ? c_p : cown, Wlo, wlo);
    __syncthreads();
    double f = 0;
    if (in_tile) {
      double Cx = 0, Cy = 0;
      if (valid) {
        const double Dxc = dx<N, NZT, double>(Ds, T, b, I, J, l);
        const double Dyc = dy<N, NZT, double>(Ds, T, b, I, J, l);
        Cx = Gxx * Dxc + Gxy * Dyc;
        Cy = Gxy * Dxc + Gyy * Dyc;
        // horizontal transport: sum_k D (uc c) over the element row / column
        f = dxy_prod<N, NZT, double>(Ds, T, 0, 1, b + 1, I, J, l);
        if (has_lo) f += Flo;
        f -= Fup;
      }
      T.at(b + 2, node, l) = Cx;
      T.at(b + 3, node, l) = Cy;
    }
    __syncthreads();
    if (valid) {
      f = (f - Kd * dxy<N, NZT, double>(DWs, T, b + 2, b + 3, I, J, l)) * iMs;
      E2[tr * a.ecs + (size_t)e * NNZ + mo] = f;
    }
  }
#undef MET
#undef METN
#undef MET0
}

// ------------------------------------------------------------------------
// HorLimit (src/GPU/HorLimiterKernel.jl)

// LimitKernel! (HorLimiterKernel.jl:2-22): per tracer, element and
// level, the min and max over the element's nodes of the mixing ratio;
// qmin/qmax[(tr*NF + element)*Nz + iz]
__global__ void k_lim_bounds(KArgs a, int NF, int NN, int ntr, const double *__restrict__ U,
                             double *__restrict__ qmin, double *__restrict__ qmax) {
  const int Nz = a.Nz;
  const size_t vs = (size_t)a.NumG * Nz, n = (size_t)ntr * NF * Nz;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const size_t tq = q / ((size_t)NF * Nz), r = q - tq * NF * Nz;
    const int e = (int)(r / Nz), iz = (int)(r - (size_t)e * Nz);
    const double *Tr = U + (5 + tq) * vs;
    double mn = 1.0 / 0.0, mx = -1.0 / 0.0;
    for (int ID = 0; ID < NN; ++ID) {
      const size_t ui = (size_t)(a.glob[(size_t)e * NN + ID] & 0x7fffffff) * Nz + iz;
      const double v = Tr[ui] / U[ui];
      mn = jmin(mn, v);
      mx = jmax(mx, v);
    }
    qmin[q] = mn;
    qmax[q] = mx;
  }
}

// medianGPU (HorLimiterKernel.jl:389-406)
__device__ __forceinline__ double median3(double a1, double a2, double a3) {
  if (a1 <= a2) {
    if (a2 <= a3) return a2;
    if (a1 <= a3) return a3;
    return a1;
  }
  if (a1 <= a3) return a1;
  if (a2 <= a3) return a3;
  return a2;
}

// The sum of x over the 32 lanes of each half of the wavefront, on every
// lane of the half: each 16-lane row pairwise at strides 8, 4, 2, 1 (lane i
// adds lane i + s, DPP row shifts), then row 0 + row 1 of the half.  This is
// the limiter's level-sum order, which the oracle restates.
__device__ __forceinline__ double half_tree_sum(double x) {
  x = x + dpp_from_above<8>(x);
  x = x + dpp_from_above<4>(x);
  x = x + dpp_from_above<2>(x);
  x = x + dpp_from_above<1>(x);
  const double h0 = readlane_d(x, 0) + readlane_d(x, 16), h1 = readlane_d(x, 32) + readlane_d(x, 48);
  return (threadIdx.x & 32) ? h1 : h0;
}

// DivRhoTrUpwind3LimKernel! (HorLimiterKernel.jl:24-196) for all tracers,
// one thread per (node, level) of an element and
// level chunk: the upwind vertical flux through both interfaces of the
// layer (as k_tr2), then the limited horizontal transport: the predicted
// rho*q and rho after dtau, the mixing ratio clipped to the bounds of the
// element's stencil after a level-wide shift lambda, lambda from the
// reference's secant iteration on the element-level tracer mass.
// Per tracer, three phases and three barriers: (A) the node threads form
// rho*q and rho after dtau and put them in LDS; (B) one wavefront per level
// (lane = node) takes the stencil's bounds and runs the whole iteration,
// every residual a sum over the lanes in node order (readlane), so the sums
// and the iteration's decisions are those of the serial restatement, with
// no barrier inside the iteration; (C) the node threads read the clipped q
// back and write the tendency.  Divisions as in the reference (no
// reciprocals): the iteration's thresholds are absolute.  The DSS mass is
// M1 + M2 (the reference indexes its 3-D M with two indices here).
template <int N, int NZT, bool CM>
__global__ void __launch_bounds__((N * N * NZT + 63) / 64 * 64)
    k_tr2_lim(KArgs a, int nchunk, int ntr, const double *__restrict__ U, const int *__restrict__ stencil,
              int NF, const double *__restrict__ qmin, const double *__restrict__ qmax, double dtau,
              double *__restrict__ E2) {
  constexpr int NN = N * N;
  static_assert(NN <= 32, "a 32-lane half of a wavefront holds the nodes of an element level");
  static_assert(NZT >= 4 && NZT <= 16 && 64 % NZT == 0, "chunk heights 4, 8 or 16 (halo levels share registers)");
  extern __shared__ double smem[];
  double *Ds = smem;
  // tiles 0, 1: uc, vc; 2: c.  Then per (level, node), node fastest: J,
  // and per tracer rho after dtau, rho*q after dtau and the clipped q
  Tiles<N, NZT, double> T{Ds + NN};
  double *wJ = Ds + NN + 3 * NN * NZT, *wS = wJ + NN * NZT, *wT = wS + NN * NZT, *wQ = wT + NN * NZT;
  if (threadIdx.x < NN) Ds[threadIdx.x] = a.D[threadIdx.x];
  const int Nz = a.Nz;
  const int L = xcd_logical(blockIdx.x, gridDim.x);
  const int e = L / nchunk;
  const int chunk = L - e * nchunk;
  const int t = threadIdx.x;
  const int node = t / NZT, l = t - node * NZT;
  const int iz = chunk * NZT + l;
  const bool in_tile = node < NN;
  const bool valid = in_tile && iz < Nz;
  const int I = node % N, J = node / N;
  const size_t vs = (size_t)a.NumG * Nz;
  const bool has_lo = iz > 0, has_hi = iz < Nz - 1;
  auto M = [&](int c, int Lv) { return met_at<NN, CM>(a, (size_t)e, c, node, Lv); };
  size_t ui = 0;
  double rho = 1, u = 0, v = 0, S11 = 0, S12 = 0, S21 = 0, S22 = 0, Js = 1, Ms = 1;
  double wlo = 0, wup = 0, rho_m = 1, rho_mm = 1, rho_p = 1, rho_pp = 1;
  double Jm = 1, Jmm = 1, Jp = 1, Jpp = 1;
  if (valid) {
    ui = (size_t)(a.glob[(size_t)e * NN + node] & 0x7fffffff) * Nz + iz;
    rho = U[ui];
    u = U[vs + ui];
    v = U[2 * vs + ui];
    S11 = M(M111, iz) + M(M112, iz);
    S12 = M(M121, iz) + M(M122, iz);
    S21 = M(M211, iz) + M(M212, iz);
    S22 = M(M221, iz) + M(M222, iz);
    Js = M(MJ1, iz) + M(MJ2, iz);
    Ms = a.M[ui] + a.M[vs + ui];
    const int lm = has_lo ? iz - 1 : iz, lmm = iz >= 2 ? iz - 2 : 0;
    const int lp = has_hi ? iz + 1 : iz, lpp = iz + 2 <= Nz - 1 ? iz + 2 : Nz - 1;
    rho_m = U[ui - iz + lm];
    rho_mm = U[ui - iz + lmm];
    rho_p = U[ui - iz + lp];
    rho_pp = U[ui - iz + lpp];
    Jm = M(MJ1, lm) + M(MJ2, lm);
    Jmm = M(MJ1, lmm) + M(MJ2, lmm);
    Jp = M(MJ1, lp) + M(MJ2, lp);
    Jpp = M(MJ1, lpp) + M(MJ2, lpp);
    // Contra3 at the two interfaces (the reference's operation order); the
    // loads at clamped levels, so that they need no branch and all take one
    // round trip
    const double *um = U + ui - iz + lm, *up = U + ui - iz + lp;
    const double wm = um[3 * vs], w = U[3 * vs + ui];
    const double lo = rho_m * (M(M312, lm) * um[vs] + M(M322, lm) * um[2 * vs] + M(M332, lm) * wm) +
                      rho * (M(M311, iz) * u + M(M321, iz) * v + M(M331, iz) * wm);
    const double hi = rho * (M(M312, iz) * u + M(M322, iz) * v + M(M332, iz) * w) +
                      rho_p * (M(M311, lp) * up[vs] + M(M321, lp) * up[2 * vs] + M(M331, lp) * w);
    if (has_lo) wlo = lo;
    if (has_hi) wup = hi;
  }
  if (in_tile) {
    T.at(0, node, l) = -rho * (S11 * u + S12 * v);  // Contra12(-rho, u, v)
    T.at(1, node, l) = -rho * (S21 * u + S22 * v);
    wJ[l * NN + node] = Js;
  }
  __syncthreads();  // D and the tracer-independent tiles
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int ln = lane & 31, In = ln % N, Jn = ln / N;
  const double eta = 1.e-12, dlFD = 1.e-8, l0 = 0.0;
  // the stencil's bounds of level lw: min / max over the 13 stencil slots
  // (the same addresses on every lane of a half)
  const int *st = stencil + 13 * (size_t)e;
  auto bounds = [&](int tr, int izw, double &qMinS, double &qMaxS) {
    const double *mn = qmin + (size_t)tr * NF * Nz, *mx = qmax + (size_t)tr * NF * Nz;
    qMinS = mn[(size_t)st[0] * Nz + izw];
    qMaxS = mx[(size_t)st[0] * Nz + izw];
    for (int iS = 1; iS < 13; ++iS) {
      qMinS = jmin(mn[(size_t)st[iS] * Nz + izw], qMinS);
      qMaxS = jmax(mx[(size_t)st[iS] * Nz + izw], qMaxS);
    }
  };
  // RecU4 weights of both interfaces, shared by all tracers
  // (the compact layout's volumes are those of every level)
  const RecW<double> Wup = CM ? recu4_equal<double>() : recu4_weights(Jm, Js, Jp, Jpp);
  const RecW<double> Wlo = CM ? recu4_equal<double>() : recu4_weights(Jmm, Jm, Js, has_hi ? Jp : Js);
  // a node's levels sit in one DPP row (or half of one), so the neighbour
  // levels' mixing ratios and the lower interface's flux come from the
  // neighbouring lanes; lanes at a chunk edge load or compute their own
  const int lr = threadIdx.x & 15;
  const bool edge_m1 = l < 1 || lr < 1, edge_m2 = l < 2 || lr < 2;
  const bool edge_p1 = l + 1 >= NZT || lr + 1 > 15, edge_p2 = l + 2 >= NZT || lr + 2 > 15;
  const int lw0 = 2 * wave + (lane >> 5), iz0 = chunk * NZT + lw0;  // this half's first level in phase B
  const bool live0 = 2 * wave < NZT && lw0 < NZT && iz0 < Nz;
  const bool hm1 = valid && has_lo && edge_m1, hm2 = valid && iz >= 2 && edge_m2;
  const bool hp1 = valid && has_hi && edge_p1, hp2 = valid && iz + 2 <= Nz - 1 && edge_p2;
  // (no lane of a chunk of at least 4 levels has a halo level on both sides)
  const double rho1 = hm1 ? rho_m : rho_p, rho2 = hm2 ? rho_mm : rho_pp;
  // this level's tracer density and the halo levels', one tracer ahead
  double Trs_n = 0, q1n = 0, q2n = 0;
  auto load = [&](int tr) {
    const double *Tr = U + (size_t)(5 + tr) * vs;
    if (valid) Trs_n = Tr[ui];
    if (hm1 || hp1) q1n = Tr[hm1 ? ui - 1 : ui + 1];
    if (hm2 || hp2) q2n = Tr[hm2 ? ui - 2 : ui + 2];
  };
  if (ntr > 0) load(0);
  for (int tr = 0; tr < ntr; ++tr) {
    // phase B's bounds of the first level pair, loaded ahead of phase A
    double qMin0 = 0, qMax0 = 0;
    if (live0) bounds(tr, iz0, qMin0, qMax0);
    const double Trs = Trs_n, q1 = q1n, q2 = q2n;
    if (tr + 1 < ntr) load(tr + 1);
    double c = 0, f = 0;
    if (valid) c = Trs / rho;
    double cm = dpp_from_below<1>(c), cmm = dpp_from_below<2>(c);
    double cp = dpp_from_above<1>(c), cpp = dpp_from_above<2>(c);
    const double c1 = q1 / rho1, c2 = q2 / rho2;
    if (hm1) cm = c1;
    if (hm2) cmm = c2;
    if (hp1) cp = c1;
    if (hp2) cpp = c2;
    // clamped levels (the reference's max/min)
    if (!has_lo) cm = c;
    if (iz < 2) cmm = cm;
    if (!has_hi) cp = c;
    if (iz + 2 > Nz - 1) cpp = cp;
    // upwind vertical flux through the upper interface; the lower one is the
    // upper flux of the level below (the unlimited kernel's fluxes)
    double Fup = 0;
    if (valid && has_hi) Fup = recu4_flux(cm, c, cp, cpp, Wup, wup);
    double Flo = dpp_from_below<1>(Fup);
    if (valid && has_lo && edge_m1) Flo = recu4_flux(cmm, cm, c, has_hi ? cp : c, Wlo, wlo);
    if (valid) {
      if (has_lo) f += Flo / Ms;
      if (has_hi) f += -Fup / Ms;
    }
    if (in_tile) T.at(2, node, l) = c;
    __syncthreads();  // (A) c of every node
    double RhoS = 1;
    if (valid) {
      double DivRhoTr = Ds[I * N] * T.at(0, J * N, l) * T.at(2, J * N, l);
      DivRhoTr += Ds[J * N] * T.at(1, I, l) * T.at(2, I, l);
      double DivRho = Ds[I * N] * T.at(0, J * N, l);
      DivRho += Ds[J * N] * T.at(1, I, l);
#pragma unroll
      for (int k = 1; k < N; ++k) {
        DivRhoTr += Ds[I * N + k] * T.at(0, k + J * N, l) * T.at(2, k + J * N, l);
        DivRhoTr += Ds[J * N + k] * T.at(1, I + k * N, l) * T.at(2, I + k * N, l);
        DivRho += Ds[I * N + k] * T.at(0, k + J * N, l);
        DivRho += Ds[J * N + k] * T.at(1, I + k * N, l);
      }
      RhoS = rho + dtau * DivRho / Js;
      wS[l * NN + node] = RhoS;
      wT[l * NN + node] = Trs + dtau * DivRhoTr / Js;
    }
    __syncthreads();  // (B) rho and rho*q after dtau of every node
    // two levels per wavefront, one per 32-lane half (lane = node)
    for (int pr = wave; pr < (NZT + 1) / 2; pr += nwave) {
      const int lw = 2 * pr + (lane >> 5);
      const int izw = chunk * NZT + lw;
      const bool live = lw < NZT && izw < Nz;  // uniform in each half
      const bool node_lane = live && ln < NN;
      double qMinS = qMin0, qMaxS = qMax0, Jl = 0, RhoSl = 1, RhoTrSl = 0;
      if (live && pr != wave) bounds(tr, izw, qMinS, qMaxS);
      if (node_lane) {
        Jl = wJ[lw * NN + ln];
        RhoSl = wS[lw * NN + ln];
        RhoTrSl = wT[lw * NN + ln];
      }
      const double sumJ = half_tree_sum(Jl);
      // the weight J w_I w_J / sum J of the reference's residual terms
      const double wgs = Jl * a.wg[In] * a.wg[Jn] / sumJ, pred = RhoTrSl / RhoSl;
      double q = 0.0;
      // the level's tracer-mass residual of a shift lam (every lane takes
      // part in the reduction); q takes the clipped mixing ratios on `store`
      auto resid = [&](double lam, bool store) {
        const double qq = median3(qMinS, pred + lam, qMaxS);
        if (store) q = qq;
        return half_tree_sum(node_lane ? wgs * (qq * RhoSl - RhoTrSl) : 0.0);
      };
      double resp = resid(l0, true), lp = 0.0, lc = 0.0;
      bool conv = live && !(fabs(resp) <= eta);
      const double resc0 = resid(l0 + dlFD, false);
      if (conv) {
        if (fabs(resc0 - resp) <= 1.e-13) {
          conv = false;
        } else {
          const double alpha = dlFD / (resc0 - resp);
          lp = l0;
          lc = lp - alpha * resp;
          resp = 0.0;  // the reference resets it here
        }
      }
      for (int it = 0; it < 8; ++it) {
        if (__ballot(conv) == 0) break;  // uniform
        const double resc = resid(lc, conv);
        if (conv) {
          if (fabs(resc - resp) <= 1.e-13) {
            conv = false;
          } else {
            const double alpha = (lp - lc) / (resp - resc);
            resp = resc;
            lp = lc;
            lc = lc - alpha * resc;
          }
        }
      }
      if (node_lane) wQ[lw * NN + ln] = q;
    }
    __syncthreads();  // (C) the clipped q of every node
    if (valid) {
      f += (wQ[l * NN + node] * RhoS - Trs) * Js / dtau / Ms;
      E2[tr * a.ecs + ((size_t)e * NN + node) * Nz + iz] = f;
    }
    // the next tracer writes tile 2, wS and wT after barrier (A), and wQ
    // after (B), which every lane reaches only after reading them here
  }
}

// The sum of a global point's element copies E, in colour order.
__device__ __forceinline__ double copies_sum(const KArgs &a, const double *__restrict__ E, unsigned ip) {
  const unsigned g = ip / (unsigned)a.Nz, iz = ip - g * (unsigned)a.Nz;
  const int *cp = a.gcpy + (size_t)g * a.cpw;
  const int c0 = cp[0], c1 = cp[1];
  if (c0 < 0) return 0.0;  // a node of no element
  double v = E[(size_t)c0 * a.Nz + iz];
  if (c1 >= 0) {
    double y = E[(size_t)c1 * a.Nz + iz];
    for (int q = 2; q < a.cpw && cp[q] >= 0; ++q) {
      v += y;
      y = E[(size_t)cp[q] * a.Nz + iz];
    }
    v += y;
  }
  return v;
}

// F of the tracers from their element copies, for callers that want F and
// for the microphysics; tracer blockIdx.y
__global__ void k_tr_dss(KArgs a, const double *__restrict__ E, double *__restrict__ F, unsigned ng) {
  for (unsigned ip = blockIdx.x * blockDim.x + threadIdx.x; ip < ng; ip += gridDim.x * blockDim.x)
    F[(size_t)blockIdx.y * ng + ip] = copies_sum(a, E + blockIdx.y * a.ecs, ip);
}

// SchurSolveBKernel! for the tracers (SchurSolve.jl:106-109): k = fac v
__global__ void k_tr_scale(const double *__restrict__ v, double *__restrict__ k, double fac, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    k[i] = fac * v[i];
}

// Rosenbrock stage arithmetic of the tracers (k = fac v, SchurSolve.jl:106-109):
// v = fV + sum_j cf[j] k_j; k = fac v; V = Vn + sum_j av[j] k_j (+ av[STAGE] k).
// Stage 0 reads V and stores it as Vn.  fV is summed here from the element
// copies E, unless it is given (the microphysics adds to the sums).
// Tracer blockIdx.y; ng points each.
template <int STAGE>
__global__ void k_rw_tr(KArgs a, const double *__restrict__ E, const double *__restrict__ fV,
                        const double *__restrict__ k0, const double *__restrict__ k1, double cf0, double cf1,
                        double av0, double av1, double av2, double fac, double *__restrict__ V,
                        double *__restrict__ Vn, double *__restrict__ kout, unsigned ng) {
  const size_t off = (size_t)blockIdx.y * ng;
  for (unsigned ip = blockIdx.x * blockDim.x + threadIdx.x; ip < ng; ip += gridDim.x * blockDim.x) {
    const size_t i = off + ip;
    double v = fV ? fV[i] : copies_sum(a, E + blockIdx.y * a.ecs, ip);
    double kp0 = 0, kp1 = 0;
    if (STAGE > 0) {
      kp0 = k0[i];
      v = v + cf0 * kp0;
    }
    if (STAGE > 1) {
      kp1 = k1[i];
      v = v + cf1 * kp1;
    }
    const double kc = fac * v;
    double vn;
    if (STAGE == 0) {
      vn = V[i];
      Vn[i] = vn;
    } else {
      vn = Vn[i];
    }
    double r = vn;
    if (STAGE > 0) r = r + av0 * kp0;
    if (STAGE > 1) r = r + av1 * kp1;
    r = r + (STAGE == 0 ? av0 : (STAGE == 1 ? av1 : av2)) * kc;
    V[i] = r;
    if (kout) kout[i] = kc;
  }
}

// The tendency of the dynamics from its element copies E: F = the sum over
// each node's copies in colour order, plus for w the chunk-interface terms
// (the lower-interface terms of the first levels of the chunks above, F4x).
// For callers that want F itself (cgd_fcn) and for the physics hooks (HK),
// which add to the sums before they are stored; without hooks the stage
// kernel sums the copies in registers instead.
template <typename R, bool HK>
__global__ void k_dss(KArgs a, Hooks hk, const double *__restrict__ U, const double *__restrict__ P,
                      const R *__restrict__ E, const R *__restrict__ F4x, R *__restrict__ F, double *__restrict__ Ftr,
                      int nchunk, int nzt) {
  const int Nz = a.Nz;
  const size_t vs = (size_t)a.NumG * Nz;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < vs; i += (size_t)gridDim.x * blockDim.x) {
    const size_t g = i / Nz;
    const int iz = (int)(i - g * Nz);
    const bool edge = nchunk > 1 && (iz + 1) % nzt == 0 && iz + 1 < Nz;
    const int ch = (iz + 1) / nzt;
    R s[5] = {0, 0, 0, 0, 0}, s4 = 0;
    for (int r0 = 0; r0 < a.cpw; r0 += 2) {
      const int2 cq = *reinterpret_cast<const int2 *>(a.gcpy + g * a.cpw + r0);
      if (cq.x < 0) break;
      const int cpq[2] = {cq.x, cq.y};
      R x[2][5], x4[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        x4[j] = 0;
#pragma unroll
        for (int q = 0; q < 5; ++q) x[j][q] = 0;
        if (cpq[j] >= 0) {
          const R *Ec = E + (size_t)cpq[j] * Nz + iz;
#pragma unroll
          for (int q = 0; q < 5; ++q) x[j][q] = Ec[q * a.ecs];
          if (edge) x4[j] = F4x[(size_t)cpq[j] * nchunk + ch];
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int q = 0; q < 5; ++q) s[q] += x[j][q];
        s4 += x4[j];
      }
    }
    if (edge) s[3] += s4;
    if constexpr (HK) hooks_point<R>(a, hk, U, P, s, Ftr, i, vs);
#pragma unroll
    for (int q = 0; q < 5; ++q) F[q * vs + i] = s[q];
  }
}

// Solution of the Schur tridiagonal system of one column, one row per lane
// (rows >= n are the identity).  Row i of the matrix is
// A[i,i-1] x[i-1] + A[i,i] x[i] + A[i,i+1] x[i+1] = rhs with A[i,i-1] =
// tri[3,i-1], A[i,i] = tri[2,i], A[i,i+1] = tri[1,i+1] (the column-oriented
// storage of SchurSolve.jl); lane i holds t0, t1, t2 = tri[1..3, i].
// A column occupies W consecutive lanes (W = 64, or 32 when two columns of
// at most 32 levels share a wavefront); i is the lane within the column.
// The Thomas branch broadcasts with readlane, so it needs W = 64.
template <int W>
__device__ __forceinline__ double col_solve(double t0, double t1, double t2, double rhs, int i, int n, int thomas) {
  static_assert(W == 32 || W == 64, "a column spans half or all of a wavefront");
  const bool row = i < n;
  double sol = 0.0;
  if (W == 64 && thomas) {
    // triSolve!: forward elimination, wave-serial (row j broadcast by readlane)
    double x = t1, b = rhs;
    for (int j = 0; j < n - 1; ++j) {
      const double q = readlane_d(t2, j) / readlane_d(x, j);
      const double bj = readlane_d(b, j);
      if (i == j + 1) {
        x = t1 - q * t0;
        b = b - q * bj;
      }
    }
    // back substitution
    if (i == n - 1) sol = b / x;
    for (int j = n - 2; j >= 0; --j) {
      const double sj1 = readlane_d(sol, j + 1);
      const double t0j1 = readlane_d(t0, j + 1);
      if (i == j) sol = (b - t0j1 * sj1) / x;
    }
  } else {
    // parallel cyclic reduction: log2(W) elimination sweeps, all lanes busy.
    // Rows n..W-1 are identity rows, so for n < 32 the sixth sweep of a
    // 64-lane column is an identity on the (then decoupled) rows and W = 32
    // computes the same solution (up to the compiler's choice of fused
    // multiply-adds in either instantiation).
    double ra = __shfl_up(t2, 1, W), rb = t1, rc = __shfl_down(t0, 1, W), rd = rhs;
    if (i == 0 || !row) ra = 0.0;
    if (i >= n - 1) rc = 0.0;
    if (!row) {
      rb = 1.0;
      rd = 0.0;
    }
#pragma unroll
    for (int st = 1; st < W; st <<= 1) {
      double am = __shfl_up(ra, st, W), bm = __shfl_up(rb, st, W), cm = __shfl_up(rc, st, W),
             dm = __shfl_up(rd, st, W);
      double ap = __shfl_down(ra, st, W), bp = __shfl_down(rb, st, W), cp = __shfl_down(rc, st, W),
             dp = __shfl_down(rd, st, W);
      if (i < st) {
        am = 0.0;
        bm = 1.0;
        cm = 0.0;
        dm = 0.0;
      }
      if (i + st > W - 1) {
        ap = 0.0;
        bp = 1.0;
        cp = 0.0;
        dp = 0.0;
      }
      const double k1 = ra * rcp(bm), k2 = rc * rcp(bp);
      rb = rb - cm * k1 - ap * k2;
      rd = rd - dm * k1 - dp * k2;
      ra = -am * k1;
      rc = -cp * k2;
    }
    sol = rd * rcp(rb);
  }
  return row ? sol : 0.0;
}

// TriDiagKernel! (SchurSolve.jl:45-74) for row i from the J blocks of
// rows i-1, i, i+1 (neighbour rows reached by shuffles)
// (invfac2 = (1/fac)/fac, formed once on the host)
template <int W>
__device__ __forceinline__ void col_tri(double jrw0, double jrw1, double jwr0, double jwr1, double jwt0,
                                        double jwt1, double jtw0, double jtw1, double invfac2, int i, int n,
                                        double &t0, double &t1, double &t2) {
  const double jwr0m = __shfl_up(jwr0, 1, W), jwt0m = __shfl_up(jwt0, 1, W);
  const double jwr1p = __shfl_down(jwr1, 1, W), jwt1p = __shfl_down(jwt1, 1, W);
  t0 = 0;
  t1 = 1;
  t2 = 0;
  if (i < n) {
    t1 = invfac2 - jwr1 * jrw0 - jwr0 * jrw1 - jwt1 * jtw0 - jwt0 * jtw1;
    t0 = (i == 0) ? 0.0 : -jwr0m * jrw0 - jwt0m * jtw0;
    t2 = (i == n - 1) ? 0.0 : -jwr1p * jrw1 - jwt1p * jtw1;
  }
}

// A J block's two entries of one interface: one 16-byte access where the
// caller's arrays are aligned for it (A16), so that a wavefront's access is one
// run instead of two of every other word: k_jac 94 us instead of 97 for 86402
// columns of 64 levels.
typedef double dbl2 __attribute__((ext_vector_type(2)));
template <bool A16> __device__ __forceinline__ void store_pair(double *p, double x, double y) {
  if constexpr (A16) {
    *reinterpret_cast<dbl2 *>(p) = dbl2{x, y};
  } else {
    p[0] = x;
    p[1] = y;
  }
}
// NT: past the cache, for what nothing here reads again.  k_schur_col streams so
// where the call is larger than the last-level cache (256 MB): 24 words a point,
// 86402 columns of 64 levels 184 us instead of 204.  Where its arrays stay in the
// cache from the call before it, a stream loses them: 24578 columns 60 us instead
// of 50, 13826 34 instead of 28.
template <bool NT> __device__ __forceinline__ double load_nt(const double *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT> __device__ __forceinline__ void store_nt(double x, double *p) {
  if constexpr (NT) __builtin_nontemporal_store(x, p);
  else *p = x;
}
template <bool A16, bool NT> __device__ __forceinline__ void load_pair(const double *p, double &x, double &y) {
  if constexpr (A16) {
    const dbl2 *q = reinterpret_cast<const dbl2 *>(p);
    dbl2 v;
    if constexpr (NT) v = __builtin_nontemporal_load(q);
    else v = *q;
    x = v.x;
    y = v.y;
  } else {
    x = p[0];
    y = p[1];
  }
}

// SchurSolveGPU! for Nz <= 64: one wavefront per column, lane = level, so
// every load and store is a coalesced 8*Nz-byte run.  The tri build
// (TriDiagKernel!), the w right-hand side (SchurSolveFKernel!) and the
// back-substitution of rho, rho*theta (SchurSolveBKernel!) are pointwise
// with neighbour lanes reached by shuffles; the tridiagonal system is
// solved by parallel cyclic reduction (default) or, with thomas != 0, by
// the Thomas recurrence of triSolve! run wave-serially in the reference's
// operation order (one useful lane per step, about 2.5x slower).
template <bool A16, bool NT>
__global__ void __launch_bounds__(256) k_schur_col(KArgs a, double *__restrict__ k, double *__restrict__ v,
                                                   const double *__restrict__ JRhoW, const double *__restrict__ JWRho,
                                                   const double *__restrict__ JWRhoTh,
                                                   const double *__restrict__ JRhoThW, double *__restrict__ tri,
                                                   double fac, double invfac2, int comp_tri, int thomas) {
  const int Nz = a.Nz, n = Nz - 1;
  const int i = threadIdx.x & 63;
  const size_t ig = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (ig >= (size_t)a.NumG) return;  // uniform per wavefront
  const size_t vs = (size_t)a.NumG * Nz;
  const size_t c0 = ig * Nz;
  const bool row = i < n, lev = i < Nz;
  const size_t jb = (ig * (size_t)n + i) * 2, tb = (ig * (size_t)n + i) * 3;
  double jrw0 = 0, jrw1 = 0, jwr0 = 0, jwr1 = 0, jwt0 = 0, jwt1 = 0, jtw0 = 0, jtw1 = 0;
  if (row) {
    load_pair<A16, NT>(JRhoW + jb, jrw0, jrw1);
    load_pair<A16, NT>(JWRho + jb, jwr0, jwr1);
    load_pair<A16, NT>(JWRhoTh + jb, jwt0, jwt1);
    load_pair<A16, NT>(JRhoThW + jb, jtw0, jtw1);
  }
  double t0, t1, t2;
  if (comp_tri) {
    col_tri<64>(jrw0, jrw1, jwr0, jwr1, jwt0, jwt1, jtw0, jtw1, invfac2, i, n, t0, t1, t2);
    if (row) {
      tri[tb] = t0;
      tri[tb + 1] = t1;
      tri[tb + 2] = t2;
    }
  } else {
    t0 = 0;
    t1 = 1;
    t2 = 0;
    if (row) {
      t0 = tri[tb];
      t1 = tri[tb + 1];
      t2 = tri[tb + 2];
    }
  }
  double v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
  if (lev) {
    v1 = v[c0 + i];
    v2 = load_nt<NT>(&v[c0 + i + vs]);
    v3 = load_nt<NT>(&v[c0 + i + 2 * vs]);
    v4 = v[c0 + i + 3 * vs];
    v5 = v[c0 + i + 4 * vs];
  }
  const double v1p = __shfl_down(v1, 1), v5p = __shfl_down(v5, 1);
  if (row) {
    v4 = v4 / fac + jwr1 * v1 + jwr0 * v1p + jwt1 * v5 + jwt0 * v5p;
    v[c0 + i + 3 * vs] = v4;
  }
  const double k4 = col_solve<64>(t0, t1, t2, v4, i, n, thomas);
  // SchurSolveBKernel!
  const double k4m = __shfl_up(k4, 1);
  const double jrw1m = __shfl_up(jrw1, 1), jtw1m = __shfl_up(jtw1, 1);
  if (lev) {
    if (i == 0) {
      v1 += jrw0 * k4;
      v5 += jtw0 * k4;
    } else if (i == Nz - 1) {
      v1 += jrw1m * k4m;
      v5 += jtw1m * k4m;
    } else {
      v1 += jrw0 * k4 + jrw1m * k4m;
      v5 += jtw0 * k4 + jtw1m * k4m;
    }
    store_nt<NT>(fac * v1, &k[c0 + i]);
    store_nt<NT>(fac * v2, &k[c0 + i + vs]);
    store_nt<NT>(fac * v3, &k[c0 + i + 2 * vs]);
    store_nt<NT>(k4, &k[c0 + i + 3 * vs]);
    store_nt<NT>(fac * v5, &k[c0 + i + 4 * vs]);
    store_nt<NT>(v1, &v[c0 + i]);
    store_nt<NT>(v5, &v[c0 + i + 4 * vs]);
  }
}

// ------------------------------------------------------------------------
// PressureKernel! with Models.Dry (DiagnosticKernel.jl:96-115)
// Models.Moist (src/Models/Equation.jl:56-75) at one point: kappa_m = R_m / c_pml
// of the dry air, vapour and cloud densities; p = (Rd rho*theta /
// p0^kappa_m)^(1/(1-kappa_m)), T = p / R_m, theta = (p0/p)^kappa_m T
__device__ __forceinline__ void moist_ptth(const KArgs &a, double rho, double rth, double rv, double rc, double &p,
                                           double &T, double &th) {
  const double rd = rho - rv - rc;
  const double Cpml = a.Cpd * rd + a.Cpv * rv + a.Cpl * rc;
  const double Rm = a.Rd * rd + a.Rv * rv;
  const double km = Rm / Cpml;
  p = pow(a.Rd * rth / pow(a.p0, km), 1.0 / (1.0 - km));
  T = p / Rm;
  th = pow(a.p0 / p, km) * T;
}

// theta = (p0/p)^(Rd/Cpd) T: with kappa = Rd/Cpd that is rho*theta / rho, the
// rounded quotient instead of the errors of log, exp and pow after each other.
// The pow was most of the arithmetic: 80 us for 86402 columns of 64 levels,
// whose five arrays take 51 us at the rate of a copy; without it, and with the moist state a
// kernel of its own, 56 us.
template <bool MOIST>
__global__ void k_prepare(KArgs a, const double *__restrict__ U, double *__restrict__ AuxG, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const double rho = U[i], rth = U[i + 4 * n];
    if constexpr (MOIST) {
      double p, T, th;
      moist_ptth(a, rho, rth, U[i + (size_t)a.iv * n], U[i + (size_t)a.ic * n], p, T, th);
      AuxG[i] = p;
      AuxG[i + n] = T;
      AuxG[i + 2 * n] = th;
      continue;
    }
    const double p = eos_p(a, rth);
    const double T = p / (a.Rd * rho);
    AuxG[i] = p;
    AuxG[i + n] = T;
    const bool exact = a.kappa == a.Rd_Cpd && p > 0.0 && p < __builtin_huge_val();
    AuxG[i + 2 * n] = exact ? rth / rho : pow(a.p0 / p, a.Rd_Cpd) * T;
  }
}

// the moist pressure of a state, overwriting the dry one that the fused
// step kernels wrote (only p: FcnGPU! reads AuxG[:,:,1])
__global__ void k_moist_p(KArgs a, const double *__restrict__ V, double *__restrict__ P, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double p, T, th;
    moist_ptth(a, V[i], V[i + 4 * n], V[i + (size_t)a.iv * n], V[i + (size_t)a.ic * n], p, T, th);
    P[i] = p;
  }
}

__global__ void k_fill(double *__restrict__ x, size_t n, double val) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] = val;
}

// JacSchurKernel! (src/DyCore/JacSchur.jl:29-75); p = AuxG[:,:,4]
// JacSchurKernel! (src/DyCore/JacSchur.jl:29-75) for the interface between
// levels L (below) and R (above): the two entries of each block.
struct JacBlocks {
  double rw0, rw1, wr0, wr1, wt0, wt1, tw0, tw1;  // JRhoW, JWRho, JWRhoTh, JRhoThW
};
__device__ __forceinline__ JacBlocks jac_blocks(const KArgs &a, double RhoL, double RhoR, double RhoThL,
                                                double RhoThR, double dPdThL, double dPdThR, double dzL,
                                                double dzR) {
  // the quotients of the reference as products with four reciprocals
  JacBlocks J;
  const double iS = rcp(dzL + dzR), iL = rcp(dzL), iR = rcp(dzR);
  const double RhoF = (RhoL * dzL + RhoR * dzR) * iS;
  const double iRhoF = rcp(RhoF);
  J.rw0 = -RhoF * iL;
  J.rw1 = RhoF * iR;
  J.wt0 = -dPdThR * iRhoF * (2.0 * iS);
  J.wt1 = dPdThL * iRhoF * (2.0 * iS);
  J.wr0 = -a.Grav * dzR * iRhoF * iS;
  J.wr1 = -a.Grav * dzL * iRhoF * iS;
  const double RhoThF = (RhoThL * dzL + RhoThR * dzR) * iS;
  J.tw0 = -RhoThF * iL;
  J.tw1 = RhoThF * iR;
  return J;
}

// JacSchurGPU!: p = AuxG[:,:,4] is added to rho*theta (zero for State = Dry)
template <bool A16>
__global__ void k_jac(KArgs a, const double *__restrict__ U, const double *__restrict__ P4,
                      const double *__restrict__ dz, double *__restrict__ JRhoW, double *__restrict__ JWRho,
                      double *__restrict__ JWRhoTh, double *__restrict__ JRhoThW) {
  const int Nz = a.Nz, n = Nz - 1;
  const size_t total = (size_t)a.NumG * n;
  const size_t vs = (size_t)a.NumG * Nz;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (size_t)gridDim.x * blockDim.x) {
    const size_t ig = q / n;
    const int iz = (int)(q - ig * n);
    const size_t i0 = ig * Nz + iz;
    const double RhoThL = U[i0 + 4 * vs] + P4[i0], RhoThR = U[i0 + 1 + 4 * vs] + P4[i0 + 1];
    const JacBlocks J = jac_blocks(a, U[i0], U[i0 + 1], RhoThL, RhoThR, eos_dpdrhoth(a, RhoThL),
                                   eos_dpdrhoth(a, RhoThR), dz[i0], dz[i0 + 1]);
    const size_t o = 2 * q;
    store_pair<A16>(JRhoW + o, J.rw0, J.rw1);
    store_pair<A16>(JWRhoTh + o, J.wt0, J.wt1);
    store_pair<A16>(JWRho + o, J.wr0, J.wr1);
    store_pair<A16>(JRhoThW + o, J.tw0, J.tw1);
  }
}

// One Rosenbrock-W stage of cgd_rw_step after the tendency
// (RosenbrockSchur.jl:12-32), for Nz <= 64: one wavefront per column,
// lane = level.  Nothing that can be recomputed is stored and re-read:
//  - the frozen Jacobian (JacSchurGPU! of the stage-1 state, which is Vn)
//    and the Schur tri matrix are rebuilt from Vn in every stage, with the
//    same arithmetic as k_jac and the tri build of k_schur_col;
//  - the tendency is summed here from its element copies, in k_dss's
//    order, with the w terms of the interfaces between level chunks;
//  - fV + sum_j (c_ij/dt) k_j, the Schur solve, and the next stage state
//    V = Vn + sum_j a_{i+1,j} k_j (or the final V = Vn + sum_j m_j k_j)
//    follow in registers, and the pressure of the next stage's
//    FcnPrepareGPU! is written with it.
// AuxG[:,:,4] (zero for State = Dry) is not read.  The state, tendency and
// increments are streamed once per stage (several hundred MB against a
// few MB of L2 per XCD), so their loads and stores are non-temporal: at
// ne=60, nz=64 that takes 6 % off the stage kernel's time.
template <typename R> struct RWStage {
  const R *fV;             // this stage's tendency (FP32 in the mixed-precision mode); null: its element copies
  const R *Fe;             // element copies of the tendency
  float *V32;              // FP32 shadow of the next stage state (mixed-precision mode; else null)
  const R *kprev[2];       // k_1, k_2 (earlier stages; FP32 storage in the mixed mode)
  double cf[2];            // c_ij / dt
  double av[3];            // V = Vn + sum_j av[j] k_j, j <= stage
  const double *Vn;        // state at the start of the step (stages 2, 3)
  double *Vnw;             // where stage 1 stores it
  const double *dz;        // (Nz, NumG)
  double *V;               // next stage state, or the final state
  R *k;                    // this stage's increment (null: not stored)
  double *P;               // AuxG[:,:,1] for the next stage (null: not written)
  const R *F4x;            // chunk-interface w terms of k_fcn2
  int nchunk, nzt;
  double fac;              // dt * gamma
  double invfac, invfac2;  // 1/fac and (1/fac)/fac
  int thomas;
};

// A column takes W lanes: W = 64, or W = 32 (Nz <= 32) for two columns per
// wavefront; blockDim.x is any multiple of 64 up to 256.  The body is shared
// by the kernel and by rw_stage_block, workgroup blk's columns in a
// persistent launch.
template <int STAGE, typename R, int W>
__device__ __forceinline__ void rw_stage_block(size_t blk, const KArgs &a, const RWStage<R> &rw) {
#define CGD_ITEM blk
#include "cgd_stage_body.inc"
#undef CGD_ITEM
}

template <int STAGE, typename R, int W>
__global__ void __launch_bounds__(256) k_rw_stage(KArgs a, RWStage<R> rw) {
#define CGD_ITEM blockIdx.x
#include "cgd_stage_body.inc"
#undef CGD_ITEM
}

// ------------------------------------------------------------------------
// Columns taller than a wavefront (64 < Nz <= 256): one workgroup of W = 128
// or 256 threads per column, thread = level.  Values of other levels are
// exchanged through LDS: put() stores four per thread and meets one barrier
// (two buffers in turn, so a buffer is rewritten only after every thread has
// passed the next barrier); the tridiagonal system is solved by cyclic
// reduction as in col_solve.  The loads and stores are whole columns; the
// one-thread-per-column Thomas solve that this replaces took 1132 us for
// 38402 columns of 70 levels, 48 % of a step over terrain at ne = 20.
template <int W> struct TallX {
  double *q;  // LDS: 2 * 4 * W
  int i, ph;
  __device__ __forceinline__ void put(double a, double b, double c, double d) {
    ph ^= 1;
    double *p = q + ph * 4 * W + i;
    p[0] = a;
    p[W] = b;
    p[2 * W] = c;
    p[3 * W] = d;
    __syncthreads();
  }
  __device__ __forceinline__ void put(double a) {
    ph ^= 1;
    q[ph * 4 * W + i] = a;
    __syncthreads();
  }
  // value `f` of the last put at level i + o, or `def` outside the workgroup
  __device__ __forceinline__ double get(int f, int o, double def) const {
    const int j = i + o;
    return j >= 0 && j < W ? q[ph * 4 * W + f * W + j] : def;
  }
};

// (s, lo) - a b, with the rounding errors of the product and of the
// difference (Knuth's two-sum) gathered in lo
__device__ __forceinline__ void sub_product(double &s, double &lo, double a, double b) {
  const double p = a * b, t = s - p, z = t - s;
  lo += ((s - (t - z)) - (p + z)) - fma(a, b, -p);
  s = t;
}

// Solution of the tridiagonal system, one row per thread: cyclic reduction as
// in col_solve, then one step of refinement with the same multipliers (they
// stay in registers, so a sweep exchanges one value) from a residual with its
// rounding errors.  The reduction's rounding grows with the height, as the
// layers get thin against fac: against an extended-precision solve it is ten
// times that of the elimination in order, refined it is smaller than that.
// With TH, triSolve!'s recurrence in its order instead, by one thread in LDS,
// as the Thomas branch of col_solve (kernels of their own: as a branch it made
// the stages 1 % slower).
template <int W, bool TH>
__device__ __forceinline__ double tall_solve(TallX<W> &X, double t0, double t1, double t2, double rhs, int n) {
  constexpr int S = W == 128 ? 7 : 8;
  static_assert(W == 1 << S, "one level per thread");
  if constexpr (TH) {
    X.put(t0, t1, t2, rhs);
    double *p0 = X.q + X.ph * 4 * W, *p1 = p0 + W, *p2 = p1 + W, *pb = p2 + W;
    if (X.i == 0) {
      for (int j = 0; j < n - 1; ++j) {
        const double q = p2[j] / p1[j];
        p1[j + 1] = p1[j + 1] - q * p0[j + 1];
        pb[j + 1] = pb[j + 1] - q * pb[j];
      }
      pb[n - 1] = pb[n - 1] / p1[n - 1];
      for (int j = n - 2; j >= 0; --j) pb[j] = (pb[j] - p0[j + 1] * pb[j + 1]) / p1[j];
    }
    __syncthreads();
    return X.i < n ? pb[X.i] : 0.0;
  }
  const int i = X.i;
  const bool row = i < n;
  X.put(t0, t2, 0.0, 0.0);
  const double a0 = i > 0 && row ? X.get(1, -1, 0.0) : 0.0, c0 = i < n - 1 ? X.get(0, 1, 0.0) : 0.0;
  double ra = a0, rb = row ? t1 : 1.0, rc = c0, rd = row ? rhs : 0.0;
  double k1[S], k2[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int st = 1 << s;
    k1[s] = k2[s] = 0.0;
    if (st < n) {
      X.put(ra, rb, rc, rd);
      const double am = X.get(0, -st, 0.0), bm = X.get(1, -st, 1.0), cm = X.get(2, -st, 0.0), dm = X.get(3, -st, 0.0);
      const double ap = X.get(0, st, 0.0), bp = X.get(1, st, 1.0), cp = X.get(2, st, 0.0), dp = X.get(3, st, 0.0);
      k1[s] = ra * rcp(bm);
      k2[s] = rc * rcp(bp);
      rb = rb - cm * k1[s] - ap * k2[s];
      rd = rd - dm * k1[s] - dp * k2[s];
      ra = -am * k1[s];
      rc = -cp * k2[s];
    }
  }
  const double ib = rcp(rb), x = row ? rd * ib : 0.0;
  X.put(x);
  double r = 0.0;
  if (row) {
    double lo = 0.0;
    r = rhs;
    sub_product(r, lo, t1, x);
    sub_product(r, lo, a0, X.get(0, -1, 0.0));
    sub_product(r, lo, c0, X.get(0, 1, 0.0));
    r += lo;
  }
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int st = 1 << s;
    if (st < n) {
      X.put(r);
      r = r - X.get(0, -st, 0.0) * k1[s] - X.get(0, st, 0.0) * k2[s];
    }
  }
  return row ? x + r * ib : 0.0;
}

// The tri matrix of row i from the J blocks of rows i-1, i, i+1 (as col_tri)
template <int W>
__device__ __forceinline__ void tall_tri(TallX<W> &X, const JacBlocks &J, double invfac2, int n, double &t0,
                                         double &t1, double &t2) {
  const int i = X.i;
  X.put(J.wr0, J.wt0, J.wr1, J.wt1);
  const double wr0m = X.get(0, -1, 0.0), wt0m = X.get(1, -1, 0.0), wr1p = X.get(2, 1, 0.0), wt1p = X.get(3, 1, 0.0);
  t0 = 0.0;
  t1 = 1.0;
  t2 = 0.0;
  if (i < n) {
    t1 = invfac2 - J.wr1 * J.rw0 - J.wr0 * J.rw1 - J.wt1 * J.tw0 - J.wt0 * J.tw1;
    t0 = i == 0 ? 0.0 : -wr0m * J.rw0 - wt0m * J.tw0;
    t2 = i == n - 1 ? 0.0 : -wr1p * J.rw1 - wt1p * J.tw1;
  }
}

// SchurSolveGPU! (as k_schur_col)
template <int W, bool TH>
__global__ void __launch_bounds__(W)
    k_schur_tall(KArgs a, double *__restrict__ k, double *__restrict__ v, const double *__restrict__ JRhoW,
                 const double *__restrict__ JWRho, const double *__restrict__ JWRhoTh,
                 const double *__restrict__ JRhoThW, double *__restrict__ tri, double fac, double invfac2,
                 int comp_tri) {
  __shared__ double lds[8 * W];
  TallX<W> X{lds, (int)threadIdx.x, 0};
  const int Nz = a.Nz, n = Nz - 1, i = X.i;
  const size_t ig = blockIdx.x;
  const size_t vs = (size_t)a.NumG * Nz, c0 = ig * Nz + i;
  const bool row = i < n, lev = i < Nz;
  const size_t jb = (ig * (size_t)n + i) * 2, tb = (ig * (size_t)n + i) * 3;
  JacBlocks J{0, 0, 0, 0, 0, 0, 0, 0};
  if (row)
    J = JacBlocks{JRhoW[jb],   JRhoW[jb + 1],   JWRho[jb],   JWRho[jb + 1],
                  JWRhoTh[jb], JWRhoTh[jb + 1], JRhoThW[jb], JRhoThW[jb + 1]};
  double v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
  if (lev) {
    v1 = v[c0];
    v2 = v[c0 + vs];
    v3 = v[c0 + 2 * vs];
    v4 = v[c0 + 3 * vs];
    v5 = v[c0 + 4 * vs];
  }
  double t0 = 0, t1 = 1, t2 = 0;
  if (comp_tri) {
    tall_tri(X, J, invfac2, n, t0, t1, t2);
    if (row) {
      tri[tb] = t0;
      tri[tb + 1] = t1;
      tri[tb + 2] = t2;
    }
  } else if (row) {
    t0 = tri[tb];
    t1 = tri[tb + 1];
    t2 = tri[tb + 2];
  }
  X.put(v1, v5, 0.0, 0.0);
  const double v1p = X.get(0, 1, 0.0), v5p = X.get(1, 1, 0.0);
  if (row) {
    v4 = v4 / fac + J.wr1 * v1 + J.wr0 * v1p + J.wt1 * v5 + J.wt0 * v5p;
    v[c0 + 3 * vs] = v4;
  }
  const double k4 = tall_solve<W, TH>(X, t0, t1, t2, v4, n);
  X.put(k4, J.rw1, J.tw1, 0.0);
  const double k4m = X.get(0, -1, 0.0), rw1m = X.get(1, -1, 0.0), tw1m = X.get(2, -1, 0.0);
  if (lev) {
    if (row) {
      v1 += J.rw0 * k4;
      v5 += J.tw0 * k4;
    }
    if (i > 0) {
      v1 += rw1m * k4m;
      v5 += tw1m * k4m;
    }
    k[c0] = fac * v1;
    k[c0 + vs] = fac * v2;
    k[c0 + 2 * vs] = fac * v3;
    k[c0 + 3 * vs] = k4;
    k[c0 + 4 * vs] = fac * v5;
    v[c0] = v1;
    v[c0 + 4 * vs] = v5;
  }
}

// The Rosenbrock stage (as k_rw_stage), FP64
template <int STAGE, int W, bool TH>
__global__ void __launch_bounds__(W) k_rw_stage_tall(KArgs a, RWStage<double> rw) {
  __shared__ double lds[8 * W];
  TallX<W> X{lds, (int)threadIdx.x, 0};
  const int Nz = a.Nz, n = Nz - 1, i = X.i;
  const size_t ig = blockIdx.x;
  const size_t vs = (size_t)a.NumG * Nz, c0 = ig * Nz + i;
  const bool row = i < n, lev = i < Nz;
  const double fac = rw.fac;
  double vn[5] = {0, 0, 0, 0, 0}, v[5] = {0, 0, 0, 0, 0}, kp[2][5] = {{0, 0, 0, 0, 0}, {0, 0, 0, 0, 0}};
  double dzi = 1.0;
  if (lev) {
    const double *src = STAGE == 0 ? rw.V : rw.Vn;
#pragma unroll
    for (int q = 0; q < 5; ++q) vn[q] = __builtin_nontemporal_load(&src[c0 + q * vs]);
    if constexpr (STAGE == 0) {
#pragma unroll
      for (int q = 0; q < 5; ++q) __builtin_nontemporal_store(vn[q], &rw.Vnw[c0 + q * vs]);
    }
    dzi = rw.dz[c0];
    if (rw.fV) {
#pragma unroll
      for (int q = 0; q < 5; ++q) v[q] = __builtin_nontemporal_load(&rw.fV[c0 + q * vs]);
    } else {
      const bool edge = rw.nchunk > 1 && (i + 1) % rw.nzt == 0 && i + 1 < Nz;
      const int ch = (i + 1) / rw.nzt;
      const Const<int> cp = as_const(a.gcpy + ig * a.cpw);
      double s4 = 0;
      for (int q = 0; q < a.cpw; ++q) {
        const int c = cp[q];
        if (c < 0) break;
        const double *Ec = rw.Fe + (size_t)c * Nz + i;
#pragma unroll
        for (int f = 0; f < 5; ++f) v[f] += __builtin_nontemporal_load(Ec + f * a.ecs);
        if (edge) s4 += rw.F4x[(size_t)c * rw.nchunk + ch];
      }
      if (edge) v[3] += s4;
    }
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        kp[j][q] = __builtin_nontemporal_load(&rw.kprev[j][c0 + q * vs]);
        v[q] = v[q] + rw.cf[j] * kp[j][q];
      }
    }
  }
  const double dpd = lev ? eos_dpdrhoth(a, vn[4]) : 0.0;
  X.put(vn[0], vn[4], dpd, dzi);
  JacBlocks J{0, 0, 0, 0, 0, 0, 0, 0};
  if (row) J = jac_blocks(a, vn[0], X.get(0, 1, 0.0), vn[4], X.get(1, 1, 0.0), dpd, X.get(2, 1, 0.0), dzi, X.get(3, 1, 1.0));
  double t0, t1, t2;
  tall_tri(X, J, rw.invfac2, n, t0, t1, t2);
  X.put(v[0], v[4], 0.0, 0.0);
  double rhs = 0.0;
  if (row)
    rhs = v[3] * rw.invfac + J.wr1 * v[0] + J.wr0 * X.get(0, 1, 0.0) + J.wt1 * v[4] + J.wt0 * X.get(1, 1, 0.0);
  const double k4 = tall_solve<W, TH>(X, t0, t1, t2, rhs, n);
  X.put(k4, J.rw1, J.tw1, 0.0);
  if (!lev) return;
  if (row) {
    v[0] += J.rw0 * k4;
    v[4] += J.tw0 * k4;
  }
  if (i > 0) {
    const double k4m = X.get(0, -1, 0.0);
    v[0] += X.get(1, -1, 0.0) * k4m;
    v[4] += X.get(2, -1, 0.0) * k4m;
  }
  const double kc[5] = {fac * v[0], fac * v[1], fac * v[2], k4, fac * v[4]};
  if (rw.k) {
#pragma unroll
    for (int q = 0; q < 5; ++q) __builtin_nontemporal_store(kc[q], &rw.k[c0 + q * vs]);
  }
  double rt = 0.0;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    double r = vn[q];
#pragma unroll
    for (int j = 0; j < STAGE; ++j) r = r + rw.av[j] * kp[j][q];
    r = r + rw.av[STAGE] * kc[q];
    __builtin_nontemporal_store(r, &rw.V[c0 + q * vs]);
    if (q == 4) rt = r;
  }
  if (rw.P) rw.P[c0] = eos_p(a, rt);
}

// ------------------------------------------------------------------------
// One persistent launch per Rosenbrock-W stage: pass 1, pass 2, then the
// column stage, in one grid whose
// workgroups are all resident at once (the host sizes the grid from the
// kernel's occupancy).  A grid-wide barrier separates the
// passes, where the ordinary path has kernel boundaries; the arithmetic is
// the same per item, so the results are bit-identical to the ordinary
// launches.
//
// The 8 XCDs each have their own L2, and the L2s are not coherent with each
// other: a workgroup's stores reach the other XCDs after an L2 write-back
// of its XCD (an agent-scope release), and it sees theirs after an L2
// invalidate (an agent-scope acquire).  Both act on the whole L2 of the
// XCD, so the barrier does each once per XCD and barrier, not once per
// workgroup:
// - every wavefront waits for its own stores to reach the L2, then the
//   workgroup arrives on its XCD's counter;
// - the last arrival of an XCD writes the L2 back and arrives on the grid
//   counter; the last of those advances the grid generation;
// - each XCD's last arrival waits for the grid generation, invalidates the
//   L2 and advances its XCD's generation; the XCD's other workgroups wait
//   for that and invalidate only their CU's L1.
// Which workgroups share an XCD is read from the hardware (XCC_ID) and
// counted at the start of each launch, so nothing is assumed about how the
// dispatcher places workgroups (grid_sync).  Waits spin on relaxed loads
// and acquire once when they end.
//
// A wait is bounded: past the deadline (wall-clock ticks) the waiting
// workgroup sets err, and every later wait and launch ends at once, so the
// grid always drains; the host reports err (cgd_check) and clears the
// whole structure.
struct GridBar {
  // the error word, the grid counter and generation, and per XCC_ID value
  // its counter, generation and workgroup count, each in a 128-byte line of
  // its own (the spin loads of one do not queue behind the atomics of
  // another)
  unsigned err, pad0[31], count, pad1[31], gen, pad2[31];
  unsigned arrive[16][32], xgen[16][32], members[16][32];
};

__device__ __forceinline__ unsigned xcc_id() {
  return __builtin_amdgcn_s_getreg((20) | (0 << 6) | ((4 - 1) << 11));  // HW_REG_XCC_ID bits 3:0
}

// Spin until *w differs from v0; false on a timeout or an earlier error.
__device__ __forceinline__ bool bar_wait(const unsigned *w, unsigned v0, GridBar *gb, long long deadline) {
  const long long t0 = wall_clock64();
  while (__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == v0) {
    if (__hip_atomic_load(&gb->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    if (wall_clock64() - t0 > deadline) {
      __hip_atomic_store(&gb->err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(2);
  }
  return true;
}

// Barrier with one L2 write-back and one L2 invalidate per XCD.  nx: the
// workgroups on this XCD; ngroups: the XCDs that hold workgroups (both
// meaningful in thread 0 only).  reset: clear the per-XCD counts of this
// launch (after every workgroup has read its own).
__device__ __forceinline__ void grid_barrier_xcd(GridBar *gb, unsigned xcc, unsigned nx, unsigned ngroups,
                                                 bool reset, long long deadline) {
  __builtin_amdgcn_s_waitcnt(0);  // this wavefront's stores have reached the L2
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned *arrive = &gb->arrive[xcc][0], *xgen = &gb->xgen[xcc][0];
    const unsigned g0 = __hip_atomic_load(&gb->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned x0 = __hip_atomic_load(xgen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // both generations read before arriving
    const unsigned old = __hip_atomic_fetch_add(arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old + 1 == nx) {
      __hip_atomic_store(arrive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // the XCD's L2 write-back
      const unsigned o2 = __hip_atomic_fetch_add(&gb->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (o2 + 1 == ngroups) {
        __hip_atomic_store(&gb->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (reset)
          for (int y = 0; y < 16; ++y) __hip_atomic_store(&gb->members[y][0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&gb->gen, g0 + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        bar_wait(&gb->gen, g0, gb, deadline);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // the XCD's L2 invalidate
      __hip_atomic_store(xgen, x0 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      bar_wait(xgen, x0, gb, deadline);
      asm volatile("buffer_inv sc0" ::: "memory");  // this CU's L1
    }
  }
  __syncthreads();
}

// The n-th grid barrier of a launch (n counts from 0; state in thread 0).
// The first one begins with a round without fences: every workgroup
// arrives on the grid counter, after which the per-XCD counts (added at
// the start of the launch) are complete and each workgroup reads its
// XCD's count and the number of XCDs in use; then it runs as the others.
// The second one clears the counts for the next launch.
__device__ __forceinline__ void grid_sync(GridBar *gb, unsigned &n, unsigned nblk, unsigned xcc, unsigned &nx,
                                          unsigned &ngroups, long long deadline) {
  if (n == 0) {
    __syncthreads();
    if (threadIdx.x == 0) {
      const unsigned g0 = __hip_atomic_load(&gb->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_s_waitcnt(0);  // the generation read (and the count added) before arriving
      const unsigned old = __hip_atomic_fetch_add(&gb->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old + 1 == nblk) {
        __hip_atomic_store(&gb->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&gb->gen, g0 + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        bar_wait(&gb->gen, g0, gb, deadline);
      }
      nx = __hip_atomic_load(&gb->members[xcc][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ngroups = 0;
      for (int y = 0; y < 16; ++y)
        ngroups += __hip_atomic_load(&gb->members[y][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > 0;
    }
  }
  grid_barrier_xcd(gb, xcc, nx, ngroups, n == 1, deadline);
  ++n;
}

template <typename R> struct StagePersist {
  int nf, nchunk1, nchunk;  // elements, level chunks of the passes
  const R *UR;          // pass 1 and pass 2: the state the R-typed terms read
  R *T1;                // hyperviscosity cache (element copies)
  const double *U;      // FP64 state
  double *T1th;         // FP32 mode: the FP64 theta cache (element copies)
  const double *P;      // pressure
  R *F, *F4x;           // tendency, chunk-interface side sums
  GridBar *bar;
  long long deadline;   // barrier wait bound in wall-clock ticks
  unsigned stage_blocks;  // workgroups of the column stage
};

// Pass-1 and pass-2 chunks of 8 levels, blockDim = the element tile
// (N*N*8 lanes rounded up to wavefronts) = the column stage's workgroup.
// stage: 0, 1, 2 (RW stage).  Nothing here is const __restrict__: the
// tendency and caches written by one phase are read by the next.
// Occupancy: 3 waves per SIMD, the most that holds the three phases without
// spilling (4 waves spill 68-136 bytes per lane).
template <int N, bool CM, typename R, int W, bool REG>
__global__ void __launch_bounds__((N * N * 8 + 63) / 64 * 64) __attribute__((amdgpu_waves_per_eu(3)))
    k_stage_persist(KArgs a, StagePersist<R> p, RWStage<R> rw, int stage) {
  if (__hip_atomic_load(&p.bar->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const int G = gridDim.x;
  const int b = xcd_logical(blockIdx.x, G);
  const unsigned xcc = xcc_id() & 15u;
  unsigned nbar = 0, nx = 0, ngroups = 0;
  if (threadIdx.x == 0) __hip_atomic_fetch_add(&p.bar->members[xcc][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int L = b, ni = p.nf * p.nchunk1; L < ni; L += G) {
    fcn1_block<N, 8, CM, R, 1>(L, a, p.nchunk1, ni, p.UR, p.T1, p.U, p.T1th);
    __syncthreads();  // the next item rewrites the LDS tiles
  }
  grid_sync(p.bar, nbar, G, xcc, nx, ngroups, p.deadline);
  for (int L = b, ni = p.nf * p.nchunk; L < ni; L += G) {
    if constexpr (REG && std::is_same<R, double>::value)
      fcn2r_block<N, 8>(L, a, p.nchunk, p.U, p.T1, p.P, p.F, p.F4x, nullptr);
    else
      fcn2_block<N, 8, CM, R, false>(L, a, p.nchunk, p.U, p.UR, p.T1, p.P, p.F, p.F4x, p.T1th, nullptr);
    __syncthreads();
  }
  grid_sync(p.bar, nbar, G, xcc, nx, ngroups, p.deadline);
  for (unsigned s = blockIdx.x; s < p.stage_blocks; s += G) {
    if (stage == 0) rw_stage_block<0, R, W>(s, a, rw);
    else if (stage == 1) rw_stage_block<1, R, W>(s, a, rw);
    else rw_stage_block<2, R, W>(s, a, rw);
  }
}

// Start of cgd_rw_step: the pressure of the first stage's FcnPrepareGPU!
// (the copy Vn = V is made by the first stage kernel), and in the
// mixed-precision mode the FP32 shadow of V.
// Each thread takes four points a grid-stride apart, so their loads and
// EOS chains (exp, log) overlap.
__global__ void k_rw_begin(KArgs a, const double *__restrict__ V, double *__restrict__ P,
                           float *__restrict__ V32, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (; i + 3 * stride < n; i += 4 * stride) {
    double rt[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) rt[u] = V[i + u * stride + 4 * n];
#pragma unroll
    for (int u = 0; u < 4; ++u) P[i + u * stride] = eos_p(a, rt[u]);
    if (V32)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        for (int q = 0; q < 5; ++q) V32[i + u * stride + q * n] = float(V[i + u * stride + q * n]);
  }
  for (; i < n; i += stride) {
    P[i] = eos_p(a, V[i + 4 * n]);
    if (V32)
      for (int q = 0; q < 5; ++q) V32[i + q * n] = float(V[i + q * n]);
  }
}

// FP32 copy of a table (set-up)
__global__ void k_to_f32(const double *__restrict__ x, float *__restrict__ y, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    y[i] = float(x[i]);
}

// y = x0 + a1*x1 (+ a2*x2), evaluated as ((x0 + a1 x1) + a2 x2) like the
// successive broadcasts of RosenbrockSchur!.
__global__ void k_axpy(double *__restrict__ y, const double *__restrict__ x0, const double *__restrict__ x1,
                       double a1, const double *__restrict__ x2, double a2, int nterm, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double r = x0[i];
    if (nterm >= 1) r = r + a1 * x1[i];
    if (nterm >= 2) r = r + a2 * x2[i];
    y[i] = r;
  }
}

// y = x0 + a1 x1 + a2 x2 + a3 x3 (final RW update)
__global__ void k_axpy3(double *__restrict__ y, const double *__restrict__ x0, const double *__restrict__ x1,
                        double a1, const double *__restrict__ x2, double a2, const double *__restrict__ x3, double a3,
                        size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double r = x0[i];
    r = r + a1 * x1[i];
    r = r + a2 * x2[i];
    r = r + a3 * x3[i];
    y[i] = r;
  }
}

// ------------------------------------------------------------------------
// Context set-up: level-fastest metric for the element kernels.
// met[element][c][ID][iz] from dXdxI (3,3,2,NN,Nz,NF), J (NN,2,Nz,NF), X (NN,2,3,Nz,NF)
__global__ void k_relayout_metric(const double *__restrict__ dXdxI, const double *__restrict__ Jm,
                                  const double *__restrict__ X, size_t e0,
                                  double *__restrict__ met, double *__restrict__ met1, int NN, int Nz, int NF,
                                  double Omega) {
  const size_t total = (size_t)NF * NN * Nz;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (size_t)gridDim.x * blockDim.x) {
    const int iz = (int)(q % Nz);
    const size_t r = q / Nz;
    const int ID = (int)(r % NN);
    const size_t e = r / NN;
    const size_t pt = (size_t)ID + (size_t)NN * ((size_t)iz + (size_t)Nz * e);  // (ID, iz, e)
    const double *dp = dXdxI + 18 * pt;  // dXdxI[i,j,K] at dp[i + 3 j + 9 K]
#define DXI(i, j, K) dp[(i - 1) + 3 * (j - 1) + 9 * (K - 1)]
    const double vals[CGD_NMET - 1] = {DXI(1, 1, 1), DXI(1, 1, 2), DXI(1, 2, 1), DXI(1, 2, 2), DXI(2, 1, 1),
                                       DXI(2, 1, 2), DXI(2, 2, 1), DXI(2, 2, 2), DXI(3, 1, 1), DXI(3, 1, 2),
                                       DXI(3, 2, 1), DXI(3, 2, 2), DXI(3, 3, 1), DXI(3, 3, 2),
                                       Jm[(size_t)ID + (size_t)NN * (0 + 2 * ((size_t)iz + (size_t)Nz * e))],
                                       Jm[(size_t)ID + (size_t)NN * (1 + 2 * ((size_t)iz + (size_t)Nz * e))]};
    const size_t NNZ = (size_t)NN * Nz;
    const size_t es = e0 + e;
    const size_t mb = (es * CGD_NMET * NN + ID) * (size_t)Nz + iz;
    for (int c = 0; c < CGD_NMET - 1; ++c) met[mb + c * NNZ] = vals[c];
    // CoriolisShallow at the layer midpoint (Coriolis.jl:16-28, MomentumKernel.jl:156-159)
#define XA(K, c) X[(size_t)ID + (size_t)NN * ((K) + 2 * ((c) + 3 * ((size_t)iz + (size_t)Nz * e)))]
    const double x = 0.5 * (XA(0, 0) + XA(1, 0));
    const double y = 0.5 * (XA(0, 1) + XA(1, 1));
    const double z = 0.5 * (XA(0, 2) + XA(1, 2));
    const double sinlat = z / sqrt(x * x + y * y + z * z);
    met[mb + MCOR * NNZ] = 2.0 * Omega * sinlat;
    const size_t m1 = (es * CGD_NMET1 * NN + ID) * (size_t)Nz + iz;
    met1[m1] = DXI(1, 1, 1) + DXI(1, 1, 2);
    met1[m1 + NNZ] = DXI(1, 2, 1) + DXI(1, 2, 2);
    met1[m1 + 2 * NNZ] = DXI(2, 1, 1) + DXI(2, 1, 2);
    met1[m1 + 3 * NNZ] = DXI(2, 2, 1) + DXI(2, 2, 2);
    met1[m1 + 4 * NNZ] = vals[14] + vals[15];
#undef DXI
#undef XA
  }
}

// The copies of each node, the list of global node g being
// ncopy[nptr[g] .. nptr[g+1]), as fixed-width lists: gcpy[NumG][cpw] per global
// node, cpy[NF*NN][cpw] per element node, -1 past the last copy.
__global__ void k_copy_lists(const int *__restrict__ nptr, const int *__restrict__ ncopy, const int *__restrict__ glob,
                             int NumG, int ne, int cpw, int *__restrict__ gcpy, int *__restrict__ cpy) {
  const size_t n = (size_t)NumG + ne;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
    const bool elem = q >= (size_t)NumG;
    const size_t i = elem ? q - NumG : q;
    const int g = elem ? glob[i] & 0x7fffffff : (int)q;
    int *out = (elem ? cpy : gcpy) + i * cpw;
    const int c0 = nptr[g], c1 = nptr[g + 1];
    for (int r = 0; r < cpw; ++r) out[r] = c0 + r < c1 ? ncopy[c0 + r] : -1;
  }
}

// Whether a compact metric is regular (cgd_pass2r_body.inc): flag[0] is set
// to 1 where it is not.  metn: [NF][12][NN]; met: [NF][5][NN][Nz]; M:
// [2][NumG][Nz].  Where it is, iMn[g] = 1 / (M1 + M2) (ms: that, per point).
__global__ void k_met_regular(const double *__restrict__ metn, const double *__restrict__ met,
                              const double *__restrict__ M, const double *__restrict__ ms, int NF, int NN, int NumG,
                              int Nz, double *__restrict__ iMn, int *__restrict__ flag) {
  bool bad = false;
  const size_t ne = (size_t)NF * NN, np = ne * Nz, ng = (size_t)NumG * Nz;
  const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, st = (size_t)gridDim.x * blockDim.x;
  for (size_t q = t0; q < ne; q += st) {
    const double *m = metn + (q / NN) * CGD_NMETN * NN + q % NN;
    const int pair[6][2] = {{M111, M112}, {M121, M122}, {M211, M212}, {M221, M222}, {M331, M332}, {MJ1, MJ2}};
    for (int k = 0; k < 6; ++k)
      if (!(m[met_nidx(pair[k][0]) * NN] == m[met_nidx(pair[k][1]) * NN])) bad = true;
  }
  for (size_t q = t0; q < np; q += st) {
    const size_t r = q / Nz, e = r / NN, nd = r - e * NN;
    const int iz = (int)(q - r * Nz);
    if (iz + 1 >= Nz) continue;
    const double *m = met + (e * CGD_NMETP * NN + nd) * Nz + iz;
    const size_t cs = (size_t)NN * Nz;
    if (!(m[met_pidx(M312) * cs] == m[met_pidx(M311) * cs + 1] && m[met_pidx(M322) * cs] == m[met_pidx(M321) * cs + 1]))
      bad = true;
  }
  for (size_t q = t0; q < ng; q += st) {
    const size_t g = q / Nz;
    if (!(M[q] == M[ng + q] && M[q] == M[g * Nz])) bad = true;
    if (q == g * Nz) iMn[g] = ms[q];
  }
  if (bad) *flag = 1;
}

// Bit mask of the metric components (met[element][c][node][iz], ncomp
// components) whose value differs between levels of some element node.
__global__ void k_met_invariant(const double *__restrict__ met, int ncomp, int NF, int NN, int Nz,
                                unsigned *__restrict__ mask) {
  unsigned m = 0;
  const size_t total = (size_t)NF * ncomp * NN;  // (element, c, node) columns
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)((q / NN) % ncomp);
    const double *col = met + q * Nz;
    const long long b0 = __double_as_longlong(col[0]);
    for (int iz = 1; iz < Nz; ++iz)
      if (__double_as_longlong(col[iz]) != b0) {
        m |= 1u << c;
        break;
      }
  }
  if (m) atomicOr(mask, m);
}

// Full -> compact metric layout (met_pidx / met_nidx), pass-1 table per node.
__global__ void k_met_compact(const double *__restrict__ met, const double *__restrict__ met1,
                              double *__restrict__ metp, double *__restrict__ metn, double *__restrict__ met1n,
                              int NF, int NN, int Nz) {
  const size_t total = (size_t)NF * NN * Nz;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (size_t)gridDim.x * blockDim.x) {
    const int iz = (int)(q % Nz);
    const size_t r = q / Nz;
    const int node = (int)(r % NN);
    const size_t e = r / NN;
    for (int c = 0; c < CGD_NMET; ++c) {
      const double x = met[((e * CGD_NMET + c) * NN + node) * Nz + iz];
      if (met_per_point(c))
        metp[((e * CGD_NMETP + met_pidx(c)) * NN + node) * Nz + iz] = x;
      else if (iz == 0)
        metn[(e * CGD_NMETN + met_nidx(c)) * NN + node] = x;
    }
    if (iz == 0)
      for (int c = 0; c < CGD_NMET1; ++c)
        met1n[(e * CGD_NMET1 + c) * NN + node] = met1[((e * CGD_NMET1 + c) * NN + node) * Nz];
  }
}

// 1 / (M1 + M2): the DSS weight every element kernel multiplies by
__global__ void k_msum(const double *__restrict__ M, double *__restrict__ iMs, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    iMs[i] = 1.0 / (M[i] + M[i + n]);
}

