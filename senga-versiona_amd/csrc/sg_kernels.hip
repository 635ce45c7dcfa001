// sg_kernels.hip -- CDNA4 kernels of one SENGA+ Runge-Kutta substage (FP64).
//
// Per substage (src/senga2.f:113-159):
//   k_boundt   BOUNDT inflow values at x-left            (src/boundt.f:177-218)
//   k_prim     TEMPER + transport + CHRATE + enthalpies   (src/temper.f, src/chrate.f,
//                                                          src/rhscal.f:515-573,1292-1470,3854-3891)
//   k_pass     every derivative along x and y, then along z (or one direction
//              each) and the RHS terms separable in them  (src/rhscal.f, src/rhsvel.f)
//   k_final    mixed derivatives, cross-direction viscous terms, NSCBC face
//              corrections (src/bounds.f) and the RK register update
//              (src/lincom.f, src/fincom.f)
// Periodic directions use wrapped indices: no halo copies are stored.
#include <math.h>

#include <type_traits>

#include "sg_internal.h"
#include "sg_stencil.h"
#include "sg_mech_h2.h"

namespace sg {

// Point kernels and their helpers: a multiply and an add are fused only
// within one expression, so the fusing does not depend on how the compiler
// lays out the surrounding code (the compiled-mechanism and table-driven
// step loops then give identical results).  The stencil kernels below
// switch back to fusing across statements.
#pragma clang fp contract(on)

#define BLK 256

// Forces x to be materialised here.  Without it the compiler sinks stencil
// sums toward their last use and keeps every neighbour value live across the
// following stages (hundreds of registers in the direction passes).  The empty
// volatile asm is ordered against the LDS barriers, so each derivative is
// formed within its own stage.
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(float &x) { asm volatile("" : "+v"(x)); }

// Scheduling boundary between the phases of a long straight-line kernel, so
// that independent phases are not interleaved (which multiplies live values).
#define SG_PHASE() __builtin_amdgcn_sched_barrier(0)

// Element at byte offset bo of a field.  A 32-bit offset from a uniform field
// base lets loads and stores use the scalar-base addressing form, instead of a
// live 64-bit vector address per field (field byte offsets stay below 2^32,
// which handle creation checks).
template <class T>
__device__ __forceinline__ T &fld(T *base, uint32_t bo) {
  return *(T *)((char *)base + bo);
}

// XCD-aware block order.  Work-groups are dispatched round-robin over the
// chip's 8 XCDs, each with its own L2; consecutive block ids therefore land on
// different L2s and neighbouring tiles (which share stencil halos) miss.  The
// remap gives each XCD one contiguous chunk of logical blocks: hardware block b
// runs on XCD b % 8 as that XCD's (b / 8)-th block, and becomes logical block
// start(XCD) + b / 8.  A bijection on [0, n) for any n.
#define SG_NXCD 8
__device__ __forceinline__ int xcd_block(int b, int n) {
  const int q = n / SG_NXCD, r = n % SG_NXCD;
  const int x = b % SG_NXCD, slot = b / SG_NXCD;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + slot;
}

__device__ __forceinline__ void coords(const Params &P, long idx, int &i, int &j, int &k) {
  int nxy = P.nx * P.ny;
  k = (int)(idx / nxy);
  int r = (int)(idx - (long)k * nxy);
  j = r / P.nx;
  i = r - j * P.nx;
}

// Packed temperature-interval indices: one bit per species (the reference's
// ITNDEX packing, src/com_senga2.h:88-98, with number base NTBASE = 2, which
// holds the two intervals every species has here), species s in bit s.
static_assert(SG_NTINT == 2 && SG_MAX_SPEC <= 32, "one index bit per species in a 32-bit word");
__device__ __forceinline__ int itint_of(uint32_t idx, int s) { return (int)((idx >> s) & 1u); }

// Interval of species s at temperature t: the first interval whose upper
// bound is not below t, the last one otherwise.  With at most two intervals
// (sg_create checks 1 <= ntint <= SG_NTINT) that is one comparison; written
// as a per-lane search loop, the uniform bound was fetched by a vector load
// and waited on inside the loop, once per species.
__device__ __forceinline__ int locate(const sg_config *c, int s, double t) {
  return (c->ntint[s] > 1 && t > c->tinthi[s][0]) ? 1 : 0;
}

__device__ void set_error(int *err, int code, int i, int j, int k) {
  if (atomicCAS(err, 0, code) == 0) {
    err[1] = i + 1;
    err[2] = j + 1;
    err[3] = k + 1;
  }
}

// Member owning flattened block gb of a launch of kind KIND, and the block's
// index lb within that member's own grid.  The map and table are read-only
// for the kernel's lifetime, so these are uniform scalar loads.
// Field pointers read from the member table are generic pointers to the
// compiler; stating that they point to global memory (a no-op conversion on
// this target) lets every access through them use global instead of flat
// instructions, which would otherwise also count against the LDS wait counter
// and stall the LDS-staged stencils.
template <class T>
__device__ __forceinline__ T *as_global(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)(uintptr_t)p;
}
__device__ __forceinline__ Fields global_fields(const Fields &G) {
  Fields F;
  F.tab = as_global(G.tab);
  F.q = as_global(G.q);
  F.run = as_global(G.run);
  F.prim = as_global(G.prim);
  F.rate = as_global(G.rate);
  F.acc = as_global(G.acc);
  F.grad = as_global(G.grad);
  F.itndex = as_global(G.itndex);
  F.face = as_global(G.face);
  F.err = as_global(G.err);
  F.erk = as_global(G.erk);
  F.emax = as_global(G.emax);
  return F;
}

template <int KIND>
__device__ __forceinline__ const Member &member_at(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                                   int gb, int &lb) {
  const Member &M = mem[map[gb]];
  lb = gb - M.blk0[KIND];
  return M;
}

// ---------------------------------------------------------------------------
// BOUNDT for NSBCI3 at x-left (src/boundt.f:177-218; BCDTXL, BCUTXL type 1, BCYTXL)
template <int NS>
__global__ void __launch_bounds__(BLK) k_boundt(const Member *__restrict__ mem, const uint32_t *__restrict__ map) {
  int lb;
  const Member &M = member_at<L_FACE>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  if (!P.inflow_xl) return;
  long t = (long)lb * BLK + threadIdx.x;
  if (t >= (long)P.ny * P.nz) return;
  long p = t * P.nx;  // i = 0
  const long fs = P.fstride;
  double strd = P.drin, stru = P.uin;
  F.q[p] = strd;
  F.q[fs + p] = strd * stru;
  F.q[2 * fs + p] = strd * 0.0;
  F.q[3 * fs + p] = strd * 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) F.q[(5 + s) * fs + p] = strd * P.yrin[s];
}

// BOUNTT for NSBCI3 at x-left (src/bountt.f:195-262)
template <int NS>
__global__ void __launch_bounds__(BLK) k_bountt(const Member *__restrict__ mem, const uint32_t *__restrict__ map) {
  int lb;
  const Member &M = member_at<L_FACE>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  if (!P.inflow_xl) return;
  long t = (long)lb * BLK + threadIdx.x;
  if (t >= (long)P.ny * P.nz) return;
  long p = t * P.nx;
  const long fs = P.fstride;
  double strd = P.drin, stru = P.uin;
  double v[4] = {strd, strd * stru, strd * 0.0, strd * 0.0};
#pragma unroll
  for (int m = 0; m < 4; m++) {
    F.q[m * fs + p] = v[m];
    F.run[m * fs + p] = v[m];
  }
#pragma unroll
  for (int s = 0; s < NS; s++) {
    double y = strd * P.yrin[s];
    F.q[(5 + s) * fs + p] = y;
    F.run[(5 + s) * fs + p] = y;
  }
  // the imposed values carry no RK error (src/bountt.f)
  if (F.erk) {
    for (int m = 0; m < 4; m++) F.erk[m * fs + p] = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) F.erk[(5 + s) * fs + p] = 0.0;
  }
}

// ---------------------------------------------------------------------------
// Point physics: TEMPER (src/temper.f:58-225), conductivity and viscosity
// (src/rhscal.f:515-573, 3854-3891, src/rhsvel.f:926-980), CHRATE
// (src/chrate.f:146-760), primitive variables, diffusivities
// (src/rhscal.f:1292-1346) and species enthalpies (src/rhscal.f:1444-1470).
// Two-interval polynomials are evaluated for both intervals with uniform
// (scalar) coefficients and the result is chosen per point.
// a * b + c for a uniform c, as one VOP3 FMA that reads c from scalar
// registers.  Left to itself the compiler copies c into vector registers and
// uses the two-address FMAC form (two moves and an FMA in FP64, one move and
// an FMA in FP32) at every Horner step.  Same operation, same rounding.
__device__ __forceinline__ double fma_u(double a, double b, double c) {
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
  return r;
}
__device__ __forceinline__ float fma_u(float a, float b, float c) {
  float r;
  asm("v_fma_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
  return r;
}
// A uniform FP64 value into vector registers with one 64-bit move (the
// compiler otherwise copies the two halves with two moves), for the leading
// coefficient that starts each Horner chain.
__device__ __forceinline__ double vmov_u(double c) {
  double r;
  asm("v_mov_b64 %0, %1" : "=v"(r) : "s"(c));
  return r;
}

// the intervals of all species at temperature t, one bit each
template <int NS>
__device__ __forceinline__ uint32_t locate_all(const sg_config *c, const Tables *tb, double t) {
  if (tb->onebound) return t > tb->tbound ? tb->twomask : 0u;
  uint32_t n = 0;
#pragma unroll
  for (int s = 0; s < NS; s++) n += (uint32_t)locate(c, s, t) << s;
  return n;
}

// Horner over the zero-padded SG_NCPMAX-term polynomial of interval it: both
// intervals are evaluated with uniform (scalar) coefficients and the result is
// chosen per point, which is cheaper than choosing every coefficient.
__device__ __forceinline__ double horner(const double (&a)[SG_NTINT][SG_NCPMAX], int it, double x) {
  static_assert(SG_NTINT == 2, "two temperature intervals");
  double f0 = vmov_u(a[0][SG_NCPMAX - 1]), f1 = vmov_u(a[1][SG_NCPMAX - 1]);
#pragma unroll
  for (int m = SG_NCPMAX - 2; m >= 0; m--) {
    f0 = fma_u(f0, x, a[0][m]);
    f1 = fma_u(f1, x, a[1][m]);
  }
  return it ? f1 : f0;
}

// c(it) + x * poly(it)(x) for a two-interval table: formed for both intervals
// with scalar coefficients (a: the two polynomials, c0: the two constants) and
// the result chosen per point (a choice of the coefficients instead costs
// register copies and selects for every one).
__device__ __forceinline__ double horner_c(const double *a, const double *c0, int it, double x) {
  double f0 = vmov_u(a[SG_NCPMAX - 1]), f1 = vmov_u(a[2 * SG_NCPMAX - 1]);
#pragma unroll
  for (int m = SG_NCPMAX - 2; m >= 0; m--) {
    f0 = fma_u(f0, x, a[m]);
    f1 = fma_u(f1, x, a[SG_NCPMAX + m]);
  }
  f0 = fma_u(f0, x, c0[0]);
  f1 = fma_u(f1, x, c0[1]);
  return it ? f1 : f0;
}
// Gibbs function h(it)/T - s(it) ln T - poly(it)(T), both intervals formed, one
// chosen (ovt = 1/T); a: the polynomials, hs: h(0), h(1), s(0), s(1).
__device__ __forceinline__ double gibbs_of(const double *a, const double *hs, int it, double t, double ovt,
                                           double lt) {
  double f0 = vmov_u(a[SG_NCPMAX - 1]), f1 = vmov_u(a[2 * SG_NCPMAX - 1]);
#pragma unroll
  for (int m = SG_NCPMAX - 2; m >= 0; m--) {
    f0 = fma_u(f0, t, a[m]);
    f1 = fma_u(f1, t, a[SG_NCPMAX + m]);
  }
  const double g0 = hs[0] * ovt - hs[2] * lt - f0;
  const double g1 = hs[1] * ovt - hs[3] * lt - f1;
  return it ? g1 : g0;
}

// TEMPER's polynomial sums (src/temper.f:92-128 with the coefficients of
// src/chemin.f:906-916): species s of mass density y in interval it adds its
// terms to tc (E(T) - E) and td (dE/dT).  Where the wave does not agree on the
// intervals, y * c(interval) is formed as y0 * c(0) + y1 * c(1) with exactly
// one of y0, y1 zero: the zero term adds an exact zero, so every sum is the one
// formed with the chosen interval alone, and the coefficients stay uniform.
// Terms above the interval's order add y * 0, which leaves the sums unchanged.
__device__ __forceinline__ void temper_add(const Tables *tb, int s, int it, double y, double (&tc)[6],
                                           double (&td)[6]) {
  const double y0 = it ? 0.0 : y, y1 = it ? y : 0.0;
  tc[0] = tc[0] + y0 * tb->hcp[s][0];
  tc[0] = tc[0] + y1 * tb->hcp[s][1];
  tc[1] = tc[1] + y0 * tb->ct[s][0][0];
  tc[1] = tc[1] + y1 * tb->ct[s][1][0];
  td[1] = tc[1];
#pragma unroll
  for (int m = 2; m <= SG_NCPMAX; m++) {
    tc[m] = tc[m] + y0 * tb->ct[s][0][m - 1];
    tc[m] = tc[m] + y1 * tb->ct[s][1][m - 1];
    td[m] = td[m] + y0 * tb->cp[s][0][m - 1];
    td[m] = td[m] + y1 * tb->cp[s][1][m - 1];
  }
}

// Uniform coefficients, a group ahead.  Left to itself the compiler loads each
// table entry right before its use and waits for it, 366 times in the point
// kernel of 9 species; with 16 species the waves waited for two thirds of
// their time.  pipe() runs use(k, coefficients of group k) for NG groups of up
// to N values: the loads of the next group are issued before the group is
// used, and held there.  With the transport fits in groups (exp_fits) and one
// decision per wave on the temperature intervals, the point kernel between
// substages takes 248 -> 214 us (16 species, 72x60x48), 85 -> 80 us (9
// species, 93x71x57), 29 -> 26 us (24x20x21) and 363 -> 358 us at 128^3, where
// HBM bounds it; mixed 235 -> 228 us, 69 -> 64 us (4-step methane, 96x80x64).
template <int NG, int N, class T, class LOAD, class USE>
__device__ __forceinline__ void pipe(LOAD load, USE use) {
  T c[2][N];
  load(0, c[0]);
#pragma unroll
  for (int g = 0; g < NG; g++) {
    if (g + 1 < NG) {
      load(g + 1, c[(g + 1) & 1]);
      SG_PHASE();
    }
    use(g, c[g & 1]);
    SG_PHASE();
  }
}

// put(s, enthalpy) and put(s, Gibbs function) of every species at t
template <int NS, class IT, class PUT>
__device__ __forceinline__ void enthalpies(const Tables *tb, IT it, double t, PUT put) {
  constexpr int N = 2 * SG_NCPMAX;
  pipe<NS, N + 2, double>(
      [&](int s, double (&c)[N + 2]) {
#pragma unroll
        for (int m = 0; m < N; m++) c[m] = tb->ch[s][m / SG_NCPMAX][m % SG_NCPMAX];
        c[N] = tb->hch[s][0];
        c[N + 1] = tb->hch[s][1];
      },
      [&](int s, const double (&c)[N + 2]) { put(s, horner_c(c, c + N, it(s), t)); });
}
template <int NS, class IT, class PUT>
__device__ __forceinline__ void gibbs_all(const Tables *tb, IT it, double t, double ovt, double lt, PUT put) {
  constexpr int N = 2 * SG_NCPMAX;
  pipe<NS, N + 4, double>(
      [&](int s, double (&c)[N + 4]) {
#pragma unroll
        for (int m = 0; m < N; m++) c[m] = tb->gb[s][m / SG_NCPMAX][m % SG_NCPMAX];
#pragma unroll
        for (int m = 0; m < 2; m++) {
          c[N + m] = tb->gbh[s][m];
          c[N + 2 + m] = tb->gbs[s][m];
        }
      },
      [&](int s, const double (&c)[N + 4]) { put(s, gibbs_of(c, c + N, it(s), t, ovt, lt)); });
}

// The sums over all species; a wave whose points agree on every interval takes
// each species' with that interval's scalar coefficients.
template <int NS>
__device__ __forceinline__ void temper_sums(const Tables *tb, uint32_t idxo, const double (&ry)[NS], double (&tc)[6],
                                            double (&td)[6]) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(idxo);
  if (__ballot(idxo != m0) == 0ull) {
    pipe<NS, 10, double>(
        [&](int s, double (&c)[10]) {
          const int u = itint_of(m0, s);
          c[0] = tb->hcp[s][u];
#pragma unroll
          for (int m = 0; m < 5; m++) c[1 + m] = tb->ct[s][u][m];
#pragma unroll
          for (int m = 1; m < 5; m++) c[5 + m] = tb->cp[s][u][m];
        },
        [&](int s, const double (&c)[10]) {
          const double y = ry[s];
          tc[0] = tc[0] + y * c[0];
          tc[1] = tc[1] + y * c[1];
          td[1] = tc[1];
#pragma unroll
          for (int m = 2; m <= SG_NCPMAX; m++) {
            tc[m] = tc[m] + y * c[m];
            td[m] = td[m] + y * c[4 + m];
          }
        });
  } else {
#pragma unroll
    for (int s = 0; s < NS; s++) temper_add(tb, s, itint_of(idxo, s), ry[s], tc, td);
  }
}
// rho cp = sum over the species of rho Y_k cp_k at the new intervals
template <int NS>
__device__ __forceinline__ double rho_cp(const Tables *tb, uint32_t nidx, const double (&ry)[NS], double t) {
  double cp = 0.0;
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(nidx);
  if (__ballot(nidx != m0) == 0ull) {
    pipe<NS, 5, double>(
        [&](int s, double (&c)[5]) {
          const int u = itint_of(m0, s);
#pragma unroll
          for (int m = 0; m < 5; m++) c[m] = tb->cp[s][u][m];
        },
        [&](int s, const double (&c)[5]) {
          double f = vmov_u(c[4]);
#pragma unroll
          for (int m = 3; m >= 0; m--) f = fma_u(f, t, c[m]);
          cp = cp + ry[s] * f;
        });
  } else {
#pragma unroll
    for (int s = 0; s < NS; s++) cp = cp + ry[s] * horner(tb->cp[s], itint_of(nidx, s), t);
  }
  return cp;
}

// ---------------------------------------------------------------------------
// TEMPIN: bisection from TRIN in 50 K steps, src/tempin.f:55-512
template <int NS, class R>
__global__ void __launch_bounds__(BLK) k_tempin(Params P, const sg_config *__restrict__ c, Fields F) {
  long idx = (long)blockIdx.x * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  const long fs = P.fstride;
  const double *q = F.q;
  double d = q[idx], ru = q[fs + idx], rv = q[2 * fs + idx], rw = q[3 * fs + idx];
  double ry[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) ry[s] = q[(5 + s) * fs + idx];
  double ukuk = (ru * ru + rv * rv + rw * rw) / d;
  double tuk2me = 0.5 * ukuk - q[4 * fs + idx];
  const double toltmp = 1.0e-4, tininc = 5.0e1, tlimlo = 2.0e2, tlimhi = 3.0e3;
  const Tables *tb = F.tab;
  // E(T) - E from the sums over species of the interval t lies in.  Where the
  // species share one interval bound (the usual mechanism) the sums of both
  // intervals are formed once and an evaluation is one polynomial; formed
  // anew for every evaluation, with each lane gathering its interval's
  // coefficients, the bisection took 2.1 ms at 128^3 and 9 species.  The sums
  // are the same either way.
  double ta[6], tc[6];
  if (tb->onebound) {
    ta[0] = tc[0] = tuk2me;
#pragma unroll
    for (int m = 1; m <= 5; m++) ta[m] = tc[m] = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      ta[0] = ta[0] + ry[s] * tb->hcp[s][0];
      tc[0] = tc[0] + ry[s] * tb->hcp[s][1];
#pragma unroll
      for (int m = 1; m <= SG_NCPMAX; m++) {
        ta[m] = ta[m] + ry[s] * tb->ct[s][0][m - 1];
        tc[m] = tc[m] + ry[s] * tb->ct[s][1][m - 1];
      }
    }
  }
  auto resid = [&](double t) {
    if (tb->onebound) {
      const bool hi = t > tb->tbound;
      double r = hi ? tc[5] : ta[5];
#pragma unroll
      for (int m = 4; m >= 0; m--) r = (hi ? tc[m] : ta[m]) + r * t;
      return r;
    }
    double sc[6], sd[6];
    sc[0] = tuk2me;
#pragma unroll
    for (int m = 1; m <= 5; m++) sc[m] = sd[m] = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) temper_add(tb, s, locate(c, s, t), ry[s], sc, sd);
    double r = sc[5];
#pragma unroll
    for (int m = 4; m >= 0; m--) r = sc[m] + r * t;
    return r;
  };
  double tlower = tlimlo, tupper = tlimhi, t = c->trin;
  bool fnconv = true, fail = false;
  double res = resid(t);
  if (fabs(res) < toltmp) {
    fnconv = false;
  } else if (res < 0.0) {
    for (;;) {
      tlower = t;
      t = t + tininc;
      res = resid(t);
      if (fabs(res) < toltmp) { fnconv = false; break; }
      if (res < 0.0) {
        if (t < tlimhi) continue;
        fail = true;
        break;
      }
      tupper = t;
      break;
    }
  } else {
    for (;;) {
      tupper = t;
      t = t - tininc;
      res = resid(t);
      if (fabs(res) < toltmp) { fnconv = false; break; }
      if (res > 0.0) {
        if (t > tlimlo) continue;
        fail = true;
        break;
      }
      tlower = t;
      break;
    }
  }
  if (fail) {
    int i, j, k;
    coords(P, idx, i, j, k);
    set_error(F.err, SG_ETEMPIN, i, j, k);
    return;
  }
  if (fnconv) {
    // bisection: the bracket halves each pass, bounded by 64 passes in double
    for (int it = 0; it < 200; it++) {
      t = 0.5 * (tlower + tupper);
      res = resid(t);
      if (fabs(res) < toltmp) break;
      if (res < 0.0) tlower = t;
      else tupper = t;
    }
  }
  uint32_t nidx = 0;
#pragma unroll
  for (int s = 0; s < NS; s++) nidx += (uint32_t)locate(c, s, t) << s;
  F.itndex[idx] = nidx;
  R *pr = (R *)F.prim;
  pr[P_T * fs + idx] = (R)t;
  double s7 = 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) s7 = s7 + ry[s] * c->rgspec[s];
  pr[P_P * fs + idx] = (R)(t * s7 - P.pofs);
}

// Reciprocals of a[0..N-1] in place with one division (prefix products,
// Montgomery's trick): 3 (N - 1) products instead of N - 1 more divisions.
template <int N>
__device__ __forceinline__ void batch_recip(double (&a)[N]) {
  double pre[N];
  pre[0] = a[0];
#pragma unroll
  for (int k = 1; k < N; k++) pre[k] = pre[k - 1] * a[k];
  double inv = 1.0 / pre[N - 1];
#pragma unroll
  for (int k = N - 1; k > 0; k--) {
    const double ak = a[k];
    a[k] = inv * pre[k - 1];
    inv = inv * ak;
  }
  a[0] = inv;
}

// Transport fits, zero-padded to SG_NTRC terms.
__device__ __forceinline__ double trfit(const double *a, double x) {
  double f = vmov_u(a[SG_NTRC - 1]);
#pragma unroll
  for (int m = SG_NTRC - 2; m >= 0; m--) f = fma_u(f, x, a[m]);
  return f;
}


// exp(x) in FP64 by Tang's table-driven method (P. T. P. Tang, "Table-driven
// implementation of the exponential function in IEEE floating-point
// arithmetic", ACM TOMS 15(2), 1989): x = (64 m + j) ln2/64 + r, |r| <= ln2/128,
// exp(x) = 2^m 2^(j/64) exp(r), with exp(r) - 1 from its degree-5 Taylor
// polynomial (truncation < 4e-17, a third of an ulp).  n ln2/64 is split so
// that n * L1 is exact.
// xt is the 2^(j/64) table (kExp2j) staged in LDS.  Domain: finite x with
// |x| < 2^31 ln2/64 (about 2.3e7), where n fits the 32-bit exponent split.
// There it is within 1 ulp of a correctly rounded exp (measured against glibc
// on 1.2e8 arguments in [-745, 709.7]), gives inf above 709.78 and 0 below
// -745.2; infinite arguments (which would give NaN) are outside the domain,
// and the kernels never pass them: every call's argument is a rate exponent,
// a transport fit or a falloff term of a temperature that TEMPER bounds.
// NaN propagates.  13 VALU instructions and one LDS read, against ~22 for the
// library exp.
static constexpr double kExp2j[64] = {0x1.0000000000000p+0, 0x1.02c9a3e778061p+0, 0x1.059b0d3158574p+0, 0x1.0874518759bc8p+0, 0x1.0b5586cf9890fp+0, 0x1.0e3ec32d3d1a2p+0, 0x1.11301d0125b51p+0, 0x1.1429aaea92de0p+0, 0x1.172b83c7d517bp+0, 0x1.1a35beb6fcb75p+0, 0x1.1d4873168b9aap+0, 0x1.2063b88628cd6p+0, 0x1.2387a6e756238p+0, 0x1.26b4565e27cddp+0, 0x1.29e9df51fdee1p+0, 0x1.2d285a6e4030bp+0, 0x1.306fe0a31b715p+0, 0x1.33c08b26416ffp+0, 0x1.371a7373aa9cbp+0, 0x1.3a7db34e59ff7p+0, 0x1.3dea64c123422p+0, 0x1.4160a21f72e2ap+0, 0x1.44e086061892dp+0, 0x1.486a2b5c13cd0p+0, 0x1.4bfdad5362a27p+0, 0x1.4f9b2769d2ca7p+0, 0x1.5342b569d4f82p+0, 0x1.56f4736b527dap+0, 0x1.5ab07dd485429p+0, 0x1.5e76f15ad2148p+0, 0x1.6247eb03a5585p+0, 0x1.6623882552225p+0, 0x1.6a09e667f3bcdp+0, 0x1.6dfb23c651a2fp+0, 0x1.71f75e8ec5f74p+0, 0x1.75feb564267c9p+0, 0x1.7a11473eb0187p+0, 0x1.7e2f336cf4e62p+0, 0x1.82589994cce13p+0, 0x1.868d99b4492edp+0, 0x1.8ace5422aa0dbp+0, 0x1.8f1ae99157736p+0, 0x1.93737b0cdc5e5p+0, 0x1.97d829fde4e50p+0, 0x1.9c49182a3f090p+0, 0x1.a0c667b5de565p+0, 0x1.a5503b23e255dp+0, 0x1.a9e6b5579fdbfp+0, 0x1.ae89f995ad3adp+0, 0x1.b33a2b84f15fbp+0, 0x1.b7f76f2fb5e47p+0, 0x1.bcc1e904bc1d2p+0, 0x1.c199bdd85529cp+0, 0x1.c67f12e57d14bp+0, 0x1.cb720dcef9069p+0, 0x1.d072d4a07897cp+0, 0x1.d5818dcfba487p+0, 0x1.da9e603db3285p+0, 0x1.dfc97337b9b5fp+0, 0x1.e502ee78b3ff6p+0, 0x1.ea4afa2a490dap+0, 0x1.efa1bee615a27p+0, 0x1.f50765b6e4540p+0, 0x1.fa7c1819e90d8p+0};
struct ExpT {
  double r, tj;
  int ni;
  // the reduction and the table read; value() the rest
  __device__ __forceinline__ void start(double x, const double *xt) {
    const double INV = 0x1.71547652b82fep+6, L1 = 0x1.62e42ff000000p-7, L2 = -0x1.718432a1b0e26p-41;
    // n = nearest integer to x*64/ln2 by the shifter 1.5*2^52: the fused sum
    // rounds to an integer, whose low 32 bits are n (two's complement)
    const double SH = 0x1.8p52;
    const double tsh = __builtin_fma(x, INV, SH);
    const double n = tsh - SH;
    ni = (int)(unsigned)__builtin_bit_cast(unsigned long long, tsh);
    tj = xt[ni & 63];
    r = __builtin_fma(-n, L1, x);
    r = __builtin_fma(-n, L2, r);
  }
  __device__ __forceinline__ double value() const {
    double q = __builtin_fma(r, 1.0 / 120.0, 1.0 / 24.0);
    q = __builtin_fma(q, r, 1.0 / 6.0);
    q = __builtin_fma(q, r, 0.5);
    const double p = __builtin_fma(q, r * r, r);
    return __builtin_ldexp(__builtin_fma(tj, p, tj), ni >> 6);
  }
};
__device__ __forceinline__ double exp_t(double x, const double *xt) {
  ExpT e;
  e.start(x, xt);
  return e.value();
}

// put(i, exp(pre(fit_i(x)))) for the N transport fits at row(i), four at a time:
// their table reads are issued together, and the next four fits' coefficients
// arrive while this group's polynomials are evaluated.
template <int N, class ROW, class PRE, class PUT>
__device__ __forceinline__ void exp_fits(double x, const double *xt, ROW row, PRE pre, PUT put) {
  constexpr int G = 4;
  double c[2][G][SG_NTRC];
  auto load = [&](int g) {
#pragma unroll
    for (int i = 0; i < G; i++)
      if (g * G + i < N) {
        const double *a = row(g * G + i);
#pragma unroll
        for (int m = 0; m < SG_NTRC; m++) c[g & 1][i][m] = a[m];
      }
  };
  load(0);
#pragma unroll
  for (int g = 0; g < (N + G - 1) / G; g++) {
    ExpT e[G];
#pragma unroll
    for (int i = 0; i < G; i++)
      if (g * G + i < N) e[i].start(pre(trfit(c[g & 1][i], x)), xt);
    SG_PHASE();
    if ((g + 1) * G < N) load(g + 1);
    SG_PHASE();
#pragma unroll
    for (int i = 0; i < G; i++)
      if (g * G + i < N) put(g * G + i, e[i].value());
    SG_PHASE();
  }
}
// the same in FP32, where the exponential reads no table: put(i, fit_i(x)),
// eight fits' coefficients ahead
template <int N, class ROW, class PUT>
__device__ __forceinline__ void fits_f(float x, ROW row, PUT put) {
  constexpr int G = 8;
  pipe<(N + G - 1) / G, G * SG_NTRC, float>(
      [&](int g, float (&c)[G * SG_NTRC]) {
#pragma unroll
        for (int i = 0; i < G; i++)
          if (g * G + i < N) {
            const float *a = row(g * G + i);
#pragma unroll
            for (int m = 0; m < SG_NTRC; m++) c[i * SG_NTRC + m] = a[m];
          }
      },
      [&](int g, const float (&c)[G * SG_NTRC]) {
#pragma unroll
        for (int i = 0; i < G; i++)
          if (g * G + i < N) {
            float f = c[i * SG_NTRC + SG_NTRC - 1];
#pragma unroll
            for (int m = SG_NTRC - 2; m >= 0; m--) f = fma_u(f, x, c[i * SG_NTRC + m]);
            put(g * G + i, f);
          }
      });
}
// the species pairs a < b, row by row
template <int NS>
struct Pairs {
  int a[NS * (NS - 1) / 2 + 1] = {}, b[NS * (NS - 1) / 2 + 1] = {};
  constexpr Pairs() {
    int p = 0;
    for (int i = 0; i < NS; i++)
      for (int j = i + 1; j < NS; j++, p++) {
        a[p] = i;
        b[p] = j;
      }
  }
};
template <int NS>
__constant__ constexpr Pairs<NS> kPairs{};

// ---------------------------------------------------------------------------
// CHRATE step loop (src/chrate.f:146-760), shared by the two sources of
// mechanism constants: RtMech reads the runtime configuration and derived
// tables; CtMech<T> reads compile-time tables (a mechanism compiled into the
// library, e.g. MechH2), for which the loop is unrolled over the steps, every
// list length, species index and rate constant becomes an immediate, and the
// per-point concentrations and Gibbs functions stay in registers.  Both run
// the same expressions in the same order on the same values, so they give
// the same results.
//
// The run-time source works from a step's packed record (StepRec), which
// arrives while the step before it is worked on.  Its lists have fixed
// lengths, so that a step's concentrations and Gibbs functions are read from
// LDS together; the fill-up entries multiply by 1 and add 0, which changes
// nothing.  Read list by list from the configuration, with a branch and two
// dependent loads per entry, the point kernel took 216 instead of 198 us (16
// species, 35 steps, 72x60x48) and 65 instead of 56.5 us (8 species, 4 steps
// of fractional orders, mixed, 96x80x64).
//
// A step's lists index a point's concentrations and Gibbs functions in LDS, one
// row of BLK values per species, and these rows decide how many blocks share a
// CU.  The fill-up entries read a row of ones and a row of zeros more, where
// that leaves as many blocks (fill_rows 2); else the species list's, whose
// weights are 0, read species 0 (1), or the reactants' and products' too, a 1
// being chosen in their place (0).  At 64^3, point kernel: 9 species in FP64
// with both rows have three blocks a CU and take 104 us, four blocks and 78 us
// with one; 13 species mixed 101 and 72 us.  Where no block is at stake the
// rows are the cheaper form: 16 species in FP64 220 us with either, 237 with
// none; 12 species 136 with both, 138 with one.
template <class T>
constexpr int list_blocks(int nc, int ng) {   // blocks of a CU, at most four (k_prim also holds exp_t's table)
  const int n = 163840 / (BLK * (nc * (int)sizeof(T) + ng * 8) + (sizeof(T) == 8 ? 512 : 0));
  return n < 4 ? n : 4;
}
template <int NS, class T>
constexpr int fill_rows = list_blocks<T>(NS + 1, NS + 1) == list_blocks<T>(NS, NS) ? 2
                          : list_blocks<T>(NS + 1, NS) == list_blocks<T>(NS, NS) ? 1 : 0;
// rows of the two arrays
template <int NS, class T>
constexpr int rows_c = NS + (fill_rows<NS, T> > 0);
template <int NS, class T>
constexpr int rows_g = NS + (fill_rows<NS, T> > 1);

template <int NS, int ROWS>
struct RtMech {
  const sg_config *c;
  const Tables *tb;
  StepRec r;   // of the step at hand
  static constexpr bool fixed = false;
  static __device__ __forceinline__ int byte(uint32_t w, int b) { return (int)((w >> (8 * b)) & 255u); }
  template <class T, class CY>
  __device__ T conc(T s1, uint32_t list, int len, const int32_t (&all)[SG_MAX_SSL], CY cyv) const {
    T v[SG_NFWD];
#pragma unroll
    for (int q = 0; q < SG_NFWD; q++) {
      const int s = byte(list, q);
      v[q] = cyv(ROWS > 0 || s < NS ? s : 0);
    }
#pragma unroll
    for (int q = 0; q < SG_NFWD; q++)
      if constexpr (ROWS > 0) s1 = s1 * (v[q] > T(0) ? v[q] : T(0));
      else s1 = s1 * (q < len ? (v[q] > T(0) ? v[q] : T(0)) : T(1));
#pragma unroll 1
    for (int q = SG_NFWD; q < len; q++) {
      const T x = cyv(all[q]);
      s1 = s1 * (x > T(0) ? x : T(0));
    }
    return s1;
  }
  template <class T, class CY>
  __device__ T fwd(int st, T s1, CY cyv) const {
    return conc(s1, r.rs, byte(r.len, 2), c->nrspec[st], cyv);
  }
  template <class T, class CY>
  __device__ T rev(int st, T s2, CY cyv) const {
    return conc(s2, r.ps, byte(r.len, 3), c->npspec[st], cyv);
  }
  template <class GB>
  __device__ double gsum(int st, double s2, GB gbv) const {
    double v[SG_NALL];
#pragma unroll
    for (int q = 0; q < SG_NALL; q++) {
      const int s = byte(r.ss[q / 4], q % 4);
      v[q] = gbv(ROWS > 1 || s < NS ? s : 0);
    }
#pragma unroll
    for (int q = 0; q < SG_NALL; q++) s2 = s2 + r.dmu[q] * v[q];
#pragma unroll 1
    for (int q = SG_NALL; q < byte(r.len, 1); q++) s2 = s2 + c->diffmu[st][q] * gbv(c->nsspec[st][q]);
    return s2;
  }
  __device__ double effw(int b, int s) const { return tb->effw[b][s]; }
  __device__ float effwf(int b, int s) const { return tb->effwf[b][s]; }
  __device__ int nst() const { return c->nstep; }
  __device__ int mb(int) const { return byte(r.kind, 0); }
  __device__ int mg(int) const { return byte(r.kind, 1); }
  __device__ int ml(int) const { return byte(r.kind, 2); }
  __device__ int mt(int) const { return byte(r.kind, 3); }
  __device__ int ms(int) const { return byte(r.len, 0); }
  __device__ int nrc(int) const { return byte(r.frac, 0); }
  __device__ int npc(int) const { return byte(r.frac, 1); }
  __device__ double rp(int, int q) const { return r.rp[q]; }
  __device__ double rl(int j, int q) const { return c->rclind[j][q]; }
  __device__ double rt(int j, int q) const { return c->rctroe[j][q]; }
  __device__ double rs(int j, int q) const { return c->rcsrif[j][q]; }
  __device__ int nrcp(int st, int m) const { return c->nrcpec[st][m]; }
  __device__ double crs(int st, int m) const { return c->crspec[st][m]; }
  __device__ float crsf(int st, int m) const { return tb->crspecf[st][m]; }
  __device__ int nss(int st) const { return c->nsslen[st]; }
  __device__ int nssp(int st, int m) const { return c->nsspec[st][m]; }
  __device__ double dmw(int st, int m) const { return c->diffmw[st][m]; }
  __device__ float dmwf(int st, int m) const { return tb->diffmwf[st][m]; }
  __device__ int npcp(int st, int m) const { return c->npcpec[st][m]; }
  __device__ double cps(int st, int m) const { return c->cpspec[st][m]; }
  __device__ float cpsf(int st, int m) const { return tb->cpspecf[st][m]; }
  __device__ double clnten() const { return c->clnten; }
  __device__ bool dense() const { return tb->ratedense != 0; }
  __device__ double nuw(int st, int u) const { return tb->nuw[st][u]; }
  __device__ float nuwf(int st, int u) const { return tb->nuwf[st][u]; }
};

template <class T>
struct CtMech {
  static constexpr bool fixed = true;
  template <class V, class CY>
  __device__ V fwd(int st, V s1, CY cyv) const {
    for (int q = 0; q < T::nrslen[st]; q++) {
      const V x = cyv(T::nrspec[st][q]);
      s1 = s1 * (x > V(0) ? x : V(0));
    }
    return s1;
  }
  template <class V, class CY>
  __device__ V rev(int st, V s2, CY cyv) const {
    for (int q = 0; q < T::npslen[st]; q++) {
      const V x = cyv(T::npspec[st][q]);
      s2 = s2 * (x > V(0) ? x : V(0));
    }
    return s2;
  }
  template <class GB>
  __device__ double gsum(int st, double s2, GB gbv) const {
    for (int q = 0; q < T::nsslen[st]; q++) s2 = s2 + T::diffmu[st][q] * gbv(T::nsspec[st][q]);
    return s2;
  }
  __device__ static constexpr double effw(int b, int s) { return T::ovwmol[s] * T::effy3b[b][s]; }
  __device__ static constexpr float effwf(int b, int s) { return (float)T::ovwmol[s] * (float)T::effy3b[b][s]; }
  __device__ static constexpr int nst() { return T::nstep; }
  __device__ static constexpr int mb(int st) { return T::mblist[st]; }
  __device__ static constexpr int mg(int st) { return T::mglist[st]; }
  __device__ static constexpr int ml(int st) { return T::mllist[st]; }
  __device__ static constexpr int mt(int st) { return T::mtlist[st]; }
  __device__ static constexpr int ms(int st) { return T::mslist[st]; }
  __device__ static constexpr double rp(int st, int q) { return T::rparam[st][q]; }
  __device__ static constexpr double rl(int j, int q) { return T::rclind[j][q]; }
  __device__ static constexpr double rt(int j, int q) { return T::rctroe[j][q]; }
  __device__ static constexpr double rs(int j, int q) { return T::rcsrif[j][q]; }
  __device__ static constexpr int nrc(int st) { return T::nrclen[st]; }
  __device__ static constexpr int nrcp(int st, int m) { return T::nrcpec[st][m]; }
  __device__ static constexpr double crs(int st, int m) { return T::crspec[st][m]; }
  __device__ static constexpr float crsf(int st, int m) { return (float)T::crspec[st][m]; }
  __device__ static constexpr int nss(int st) { return T::nsslen[st]; }
  __device__ static constexpr int nssp(int st, int m) { return T::nsspec[st][m]; }
  __device__ static constexpr double dmw(int st, int m) { return T::diffmw[st][m]; }
  __device__ static constexpr float dmwf(int st, int m) { return (float)T::diffmw[st][m]; }
  __device__ static constexpr int npc(int st) { return T::npclen[st]; }
  __device__ static constexpr int npcp(int st, int m) { return T::npcpec[st][m]; }
  __device__ static constexpr double cps(int st, int m) { return T::cpspec[st][m]; }
  __device__ static constexpr float cpsf(int st, int m) { return (float)T::cpspec[st][m]; }
  __device__ static constexpr double ovw(int s) { return T::ovwmol[s]; }
  __device__ static constexpr float ovwf(int s) { return (float)T::ovwmol[s]; }
  __device__ static constexpr double clnten() { return T::clnten; }
  __device__ static constexpr bool dense() { return T::ratedense != 0; }
  __device__ static constexpr double nuw(int st, int u) { return T::nuw[st][u]; }
  __device__ static constexpr float nuwf(int st, int u) { return (float)T::nuw[st][u]; }
};

// f(st) for every step: unrolled for compile-time tables
template <class M, class Fn>
__device__ __forceinline__ void for_steps(M &m, Fn f) {
  if constexpr (M::fixed) {
#pragma unroll
    for (int st = 0; st < M::nst(); st++) f(st);
  } else {
    // the next step's record arrives while this one is worked on
    StepRec next = m.tb->step[0];
    for (int st = 0; st < m.nst(); st++) {
      m.r = next;
      next = m.tb->step[st + 1];
      f(st);
    }
  }
}

// One step in FP64: rate coefficients with falloff, forward and reverse
// products, added to rate[] (src/chrate.f:177-747).  cyv(s) and gbv(s) give
// the point's molar concentration and Gibbs function of species s, ex(x) the
// exponential.
template <int NS, class M, class CY, class GB, class EX>
__device__ __forceinline__ void chem_step64(const M &m, int st, double t, double lt, double ovt,
                                            const double *ry, CY cyv, GB gbv, double *rate, EX ex) {
  const double ysmall = 1.0e-30, ydenom = 1.0e-15;
  bool flthrd = true;
  double s3 = 0.0;
  const int mb = m.mb(st);
  if (mb != 0) {
#pragma unroll
    for (int s = 0; s < NS; s++) s3 = s3 + ry[s] * m.effw(mb - 1, s);
  }
  double s2 = m.rp(st, 0) + m.rp(st, 1) * lt - m.rp(st, 2) * ovt;
  double s1 = ex(s2);
  const int ml = m.ml(st);
  if (ml != 0) {
    const int j = ml - 1;
    double s4 = m.rl(j, 0) + m.rl(j, 1) * lt - m.rl(j, 2) * ovt;
    s4 = ex(s4);
    double preduc = s3 * s4 / s1;
    double fornow = m.rl(j, 3) * preduc / (1.0 + preduc);  // rl[3] pre-rounded to REAL
    s1 = s1 * fornow;
    s2 = log(s1);
    flthrd = false;
  }
  const int mt = m.mt(st);
  if (mt != 0) {
    const int j = mt - 1;
    double omalph = 1.0 - m.rt(j, 3);
    double s4 = m.rt(j, 0) + m.rt(j, 1) * lt - m.rt(j, 2) * ovt;
    s4 = ex(s4);
    double preduc = s3 * s4 / s1;
    double trats1 = t * m.rt(j, 4), trats2 = -m.rt(j, 5) * ovt, trats3 = t * m.rt(j, 6);
    double ftcent = omalph * ex(trats3) + m.rt(j, 3) * ex(trats1) + ex(trats2);
    ftcent = log10(ftcent);
    double cfactr = m.rt(j, 7) + m.rt(j, 8) * ftcent;
    double enfact = m.rt(j, 9) + m.rt(j, 10) * ftcent;
    double fornow = log10(preduc) + cfactr;
    fornow = fornow / (enfact - m.rt(j, 11) * fornow);
    fornow = 1.0 + fornow * fornow;
    double fbroad = ftcent / fornow;
    fbroad = ex(fbroad * m.clnten());
    fornow = fbroad * preduc / (1.0 + preduc);
    s1 = s1 * fornow;
    s2 = log(s1);
    flthrd = false;
  }
  const int ms = m.ms(st);
  if (ms != 0) {
    const int j = ms - 1;
    double s4 = m.rs(j, 0) + m.rs(j, 1) * lt - m.rs(j, 2) * ovt;
    s4 = ex(s4);
    double preduc = s3 * s4 / s1;
    double fornow = m.rs(j, 4) * ovt;
    double fbroad = m.rs(j, 3) * ex(fornow);
    fornow = t * m.rs(j, 5);
    fbroad = fbroad + ex(fornow);
    fornow = log10(preduc);
    fornow = 1.0 / (1.0 + log10(fornow));
    fbroad = m.rs(j, 6) * ex(fornow * log(fbroad));
    fornow = fbroad * preduc / (1.0 + preduc);
    s1 = s1 * fornow;
    s2 = log(s1);
    flthrd = false;
  }
  s1 = m.fwd(st, s1, cyv);
#pragma unroll 1
  for (int q = 0; q < m.nrc(st); q++) {
    double fornow = cyv(m.nrcp(st, q));
    fornow = fornow > ysmall ? fornow : ysmall;
    fornow = ex(m.crs(st, q) * log(fornow));
    fornow = fornow / (1.0 + ydenom * fornow);
    s1 = s1 * fornow;
  }
  if (m.mg(st) != 0) {
    s2 = m.gsum(st, s2, gbv);
    s2 = ex(s2);
    s2 = m.rev(st, s2, cyv);
#pragma unroll 1
    for (int q = 0; q < m.npc(st); q++) {
      double fornow = cyv(m.npcp(st, q));
      fornow = fornow > ysmall ? fornow : ysmall;
      fornow = ex(m.cps(st, q) * log(fornow));
      fornow = fornow / (1.0 + ydenom * fornow);
      s2 = s2 * fornow;
    }
    s1 = s1 - s2;
  }
  if (mb != 0 && flthrd) s1 = s1 * s3;
  if (m.dense()) {
    // every species once per list: absent species add s1*0, an exact zero;
    // with compile-time tables those terms are not formed at all
#pragma unroll
    for (int u = 0; u < NS; u++)
      if (!M::fixed || m.nuw(st, u) != 0.0) rate[u] = rate[u] + s1 * m.nuw(st, u);
  } else {
    for (int q = 0; q < m.nss(st); q++) {
      int sp = m.nssp(st, q);
      double add = s1 * m.dmw(st, q);
#pragma unroll
      for (int u = 0; u < NS; u++)
        if (u == sp) rate[u] = rate[u] + add;
    }
  }
}

// LINCOM of substage irk (src/lincom.f:53-169) at one point, from the finished
// right-hand sides in the accumulators, then BOUNDT (src/boundt.f:177-218) at
// the inflow plane: the next substage's point kernel starts with it, so that
// between the substages of a step no kernel of its own reads and writes both
// registers (k_final moved 448 of its 608 B per point for them at 9 species).
// v is the stage register's point; of it only density and momentum go to
// memory here (the passes read them), the point kernels store the rest where
// another kernel reads it.
template <int NS, class R>
__device__ __forceinline__ void lincom_point(const Params &P, const Fields &F, const Member &M, int irk, long idx,
                                             double (&v)[5 + NS]) {
  const long fs = P.fstride;
  const uint32_t bo = (uint32_t)idx * 8u, br = (uint32_t)idx * (uint32_t)sizeof(R);
  const R *A = (const R *)F.acc;
  const double lhs = M.rkl[irk - 1], rhsc = M.rkr[irk - 1], erc = M.rke[irk - 1];
  bool in = false;   // a point of the inflow plane, where all but the energy is imposed
  if (P.inflow_xl) in = idx % P.nx == 0;
  if (F.erk) {   // *ERR += RKERR * R, four variables at a time (each load would wait for the store before it)
    for (int q0 = 0; q0 < 5 + NS; q0 += 4) {
      double er[4];
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (q0 + q < 5 + NS) er[q] = fld(F.erk + (q0 + q) * fs, bo) + erc * (double)fld(A + (q0 + q) * fs, br);
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (q0 + q < 5 + NS && (q0 + q == 4 || !in)) fld(F.erk + (q0 + q) * fs, bo) = er[q];
    }
  }
  SG_PHASE();
  R rh[5 + NS];
#pragma unroll
  for (int q = 0; q < 5 + NS; q++) rh[q] = fld(A + q * fs, br);
#pragma unroll
  for (int q = 0; q < 5 + NS; q++) v[q] = fld(F.run + q * fs, bo);
#pragma unroll
  for (int q = 0; q < 5 + NS; q++) {
    const double r = (double)rh[q], old = v[q];
    if (q != 4 && in) {
      v[q] = q == 0 ? P.drin : (q == 1 ? P.drin * P.uin : (q < 4 ? P.drin * 0.0 : P.drin * P.yrin[q < 5 ? 0 : q - 5]));
    } else {
      fld(F.run + q * fs, bo) = old + lhs * r;
      v[q] = old + rhsc * r;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) fld(F.q + q * fs, bo) = v[q];
}
// the rest of the stage register, for the kernels that read it besides the point kernels
template <int NS>
__device__ __forceinline__ void store_stage(const Params &P, const Fields &F, uint32_t bo, double re,
                                            const double (&ry)[NS]) {
  fld(F.q + 4 * P.fstride, bo) = re;
#pragma unroll
  for (int s = 0; s < NS; s++) fld(F.q + (5 + s) * P.fstride, bo) = ry[s];
}

// UPD: the point kernel of a substage after the first, which begins with the
// LINCOM of substage irk.
template <int NS, bool FIX, bool UPD>
__global__ void __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(4))) k_prim(const Member *__restrict__ mem,
    const uint32_t *__restrict__ map, const sg_config *__restrict__ c, const Tables *__restrict__ tb, int irk) {
  int lb;
  const Member &M = member_at<L_POINT>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  // the 2^(j/64) table of exp_t, staged before any thread leaves
  __shared__ double xt[64];
  if (threadIdx.x < 64) xt[threadIdx.x] = kExp2j[threadIdx.x];
  __syncthreads();
  const long idx = (long)lb * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  const uint32_t bo = (uint32_t)idx * 8u;
  const long fs = P.fstride;
  const double *q = F.q;
  double *pr = F.prim;
  // loaded before the update's stores, which they would otherwise wait for
  const uint32_t idxo = fld(F.itndex, bo / 2u);
  double t = fld(pr + P_T * fs, bo);
  double st[5 + NS];
  if constexpr (UPD) {
    lincom_point<NS, double>(P, F, M, irk, idx, st);
  } else {
#pragma unroll
    for (int v = 0; v < 5 + NS; v++) st[v] = fld(q + v * fs, bo);
  }
  const double d = st[0], ru = st[1], rv = st[2], rw = st[3], re = st[4];
  double ry[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) ry[s] = st[5 + s];
  if (UPD && (P.radn || P.ltmask)) store_stage<NS>(P, F, bo, re, ry);
  // --- TEMPER (src/temper.f:58-160) ---
  const double ovd = 1.0 / d;   // one reciprocal for every division by rho
  double ukuk = (ru * ru + rv * rv + rw * rw) * ovd;
  double tc[6], td[6];
  tc[0] = 0.5 * ukuk - re;
#pragma unroll
  for (int m = 1; m <= 5; m++) { tc[m] = 0.0; td[m] = 0.0; }
  temper_sums<NS>(tb, idxo, ry, tc, td);
  double s7 = 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) s7 = s7 + ry[s] * c->rgspec[s];
  const double toltmp = (double)1.0e-10f;  // REAL literal, src/temper.f:33-34
  int iter = 1;
  bool ok = true;
  for (;;) {
    double fp = tc[5], dp = td[5];
#pragma unroll
    for (int m = 4; m >= 1; m--) {
      fp = tc[m] + fp * t;
      dp = td[m] + dp * t;
    }
    fp = tc[0] + fp * t;
    double dt = -fp / dp;
    if (fabs(dt) > toltmp) {
      if (iter < 100) {
        t = t + dt;
        iter++;
        continue;
      }
      ok = false;
    }
    break;
  }
  if (!ok) {
    int i, j, k;
    coords(P, idx, i, j, k);
    set_error(F.err, SG_ETEMPER, i, j, k);
  }
  const uint32_t nidx = locate_all<NS>(c, tb, t);
  const double cp = rho_cp<NS>(tb, nidx, ry, t) * ovd;
  fld(F.itndex, bo / 2u) = nidx;
  SG_PHASE();
  double pres = t * s7;
  fld(pr + P_T * fs, bo) = t;
  fld(pr + P_P * fs, bo) = pres;
  // primitives
  fld(pr + P_U * fs, bo) = ru * ovd;
  fld(pr + P_V * fs, bo) = rv * ovd;
  fld(pr + P_W * fs, bo) = rw * ovd;
  fld(pr + P_E * fs, bo) = re * ovd;
  // --- conductivity (src/rhscal.f:515-573) ---
  double lam, transp, wmomix = 0.0;
  if (!P.mixavg) {
    double fornow = P.alamda * exp_t(P.rlamda * log(t), xt);
    lam = fornow * cp;
    transp = fornow;
  } else {
    transp = log(t / P.tdifgb);
    // the divisions X_k / lambda_k share one (batch_recip; a few ulp from the
    // reference's quotients)
    double c1 = 0.0, c2 = 0.0, c3 = 0.0, ictr[NS];
    exp_fits<NS>(transp, xt, [&](int s) { return c->condco[s]; }, [](double f) { return f; },
                 [&](int s, double ctr) {
                   ictr[s] = ctr;
                   c1 = c1 + (ry[s] * c->ovwmol[s]) * ctr;
                 });
    batch_recip<NS>(ictr);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      double fornow = ry[s] * c->ovwmol[s];
      c2 = c2 + fornow * ictr[s];
      c3 = c3 + fornow;
    }
    c3 = 1.0 / c3;
    c1 = c1 * c3;
    c2 = c2 * c3;
    lam = 0.5 * (c1 + 1.0 / c2);
    wmomix = d * c3;
  }
  fld(pr + P_LAM * fs, bo) = lam;
  if (P.mixw || P.mixp) {
    // ln(mixture molar mass), ln(pressure) and the reciprocal molar mass for
    // the molar-mass and pressure diffusion terms (src/rhscal.f:951-985, 2374)
    fld(pr + P_LNW * fs, bo) = log(wmomix);
    fld(pr + P_LNP * fs, bo) = log(pres);
    fld(pr + P_OVW * fs, bo) = 1.0 / wmomix;
  }
  SG_PHASE();
  // --- chemistry (src/chrate.f:146-760) on rho Y ---
  {
    double rate[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) rate[s] = 0.0;
    const double lt = log(t), ovt = 1.0 / t;
    // Gibbs functions of all species at this temperature, each formed as
    // src/chrate.f:612-632 forms it for every step it enters
    double gibbs[NS];
    if constexpr (FIX) {
      // not a species ahead: the unrolled step loop has room for a Gibbs
      // function only where it is first used (all formed here, the kernel
      // spilled 5 to 7 registers: 797 instead of 744 B per point moved)
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const double hs[4] = {tb->gbh[s][0], tb->gbh[s][1], tb->gbs[s][0], tb->gbs[s][1]};
        gibbs[s] = gibbs_of(tb->gb[s][0], hs, itint_of(nidx, s), t, ovt, lt);
      }
    } else {
      gibbs_all<NS>(tb, [&](int s) { return itint_of(nidx, s); }, t, ovt, lt, [&](int s, double g) { gibbs[s] = g; });
    }
    if constexpr (FIX) {
      using MT = CtMech<MechH2>;
      double cy[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) cy[s] = ry[s] * MT::ovw(s);
      MT m0;
      for_steps(m0, [&](int st) {
        chem_step64<NS>(MT{}, st, t, lt, ovt, ry, [&](int s) { return cy[s]; }, [&](int s) { return gibbs[s]; },
                        rate, [&](double x) { return exp_t(x, xt); });
      });
    } else {
      // Molar concentrations and Gibbs functions of this point in LDS, so
      // that a step's species lists (uniform, known only at run time) index
      // them with one LDS read instead of a select over all species.
      __shared__ double lcy[rows_c<NS, double>][BLK], lgb[rows_g<NS, double>][BLK];
      const int tl = threadIdx.x;
      if constexpr (rows_c<NS, double> > NS) lcy[NS][tl] = 1;
      if constexpr (rows_g<NS, double> > NS) lgb[NS][tl] = 0;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        lcy[s][tl] = ry[s] * c->ovwmol[s];
        lgb[s][tl] = gibbs[s];
      }
      RtMech<NS, fill_rows<NS, double>> mr{c, tb};
      for_steps(mr, [&](int st) {
        chem_step64<NS>(mr, st, t, lt, ovt, ry, [&](int s) { return lcy[s][tl]; }, [&](int s) { return lgb[s][tl]; },
                        rate, [&](double x) { return exp_t(x, xt); });
      });
    }
#pragma unroll
    for (int s = 0; s < NS; s++) fld(F.rate + s * fs, bo) = rate[s];
  }
  // --- mass fractions and enthalpies (src/rhscal.f:1444-1470) ---
  double y[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) y[s] = ry[s] * ovd;
  double hmix = 0.0;
  enthalpies<NS>(tb, [&](int s) { return itint_of(nidx, s); }, t, [&](int s, double h) {
    fld(pr + prim_y(P, s), bo) = y[s];
    fld(pr + prim_h(P, s), bo) = h;
    hmix = hmix + h * y[s];
  });
  fld(pr + P_HMIX * fs, bo) = hmix;
  SG_PHASE();
  if (!P.mixavg) {
#pragma unroll
    for (int s = 0; s < NS; s++) fld(pr + prim_rd(P, s), bo) = transp * c->olewis[s];
    fld(pr + P_MU * fs, bo) = transp * P.prantl;
  } else {
    // binary diffusion (src/rhscal.f:1311-1346), with Y_j + tol formed again
    // where it is used rather than held through the pair loop
    double c1t = 0.0;
#pragma unroll
    for (int js = 0; js < NS; js++) c1t = c1t + (y[js] + 1.0e-12);
    // The reference's term (Y_j + tol) W_j^-1 / CTRANS, CTRANS = exp(f) p_g / p,
    // is formed as ((Y_j + tol) W_j^-1 (p / p_g)) * exp(-f): no division or
    // pressure product per pair (a few ulp from the reference's operation
    // order), and the species' final divisions share one (batch_recip).
    const double ppd = pres / P.pdifgb;
    if (tb->diffsym) {
      double yw2p[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) yw2p[s] = ((y[s] + 1.0e-12) * c->ovwmol[s]) * ppd;
      // D_ij = D_ji: one fit per unordered pair a < b, its term added to both
      // sums.  Visiting the pairs row by row delivers the terms of every sum
      // in increasing species order, the reference's order.  The reference
      // sums over every j and subtracts the j = k term; the sums here skip
      // it (no fit and exp for the 9 self pairs; the same sum up to the
      // rounding of that addition and subtraction).
      double cs[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) cs[s] = 0.0;
      exp_fits<NS * (NS - 1) / 2>(transp, xt, [&](int p) { return c->diffco[kPairs<NS>.a[p]][kPairs<NS>.b[p]]; },
                                  [](double f) { return -f; },
                                  [&](int p, double ictd) {
                                    const int a = kPairs<NS>.a[p], b = kPairs<NS>.b[p];
                                    cs[a] = cs[a] + yw2p[b] * ictd;
                                    cs[b] = cs[b] + yw2p[a] * ictd;
                                  });
      double c2[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) c2[s] = cs[s] * wmomix;
      batch_recip<NS>(c2);
#pragma unroll
      for (int s = 0; s < NS; s++) fld(pr + prim_rd(P, s), bo) = d * (c1t - (y[s] + 1.0e-12)) * c2[s];
    } else {
      double yt[NS], yw2[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        yt[s] = y[s] + 1.0e-12;
        yw2[s] = yt[s] * c->ovwmol[s];
      }
#pragma unroll
      for (int s = 0; s < NS; s++) {
        double c2 = 0.0, self = 0.0;
#pragma unroll
        for (int js = 0; js < NS; js++) {
          const double term = yw2[js] * (exp_t(-trfit(c->diffco[s][js], transp), xt) * ppd);
          c2 = c2 + term;
          if (js == s) self = term;
        }
        double c1 = c1t - yt[s];
        c2 = c2 - self;
        c2 = c2 * wmomix;
        fld(pr + prim_rd(P, s), bo) = d * c1 / c2;
      }
    }
    SG_PHASE();
    // Wilke viscosity (src/rhscal.f:3854-3891).  sqrt(mu_s / mu_j) is formed
    // as sqrt(mu_s) / sqrt(mu_j), with sqrt(mu_s) = exp(fit_s / 2) (one exp
    // instead of exp and square root) and mu_s = sqrt(mu_s)^2; the
    // reciprocals 1/sqrt(mu_j) share one division, and so do the divisions
    // mu_s / sum_s (batch_recip).
    double mus[NS], sq[NS], rsq[NS], yw[NS];
    exp_fits<NS>(transp, xt, [&](int s) { return c->viscco[s]; }, [](double f) { return 0.5 * f; },
                 [&](int s, double v) {
                   sq[s] = v;
                   rsq[s] = v;
                   mus[s] = v * v;
                 });
#pragma unroll
    for (int s = 0; s < NS; s++) yw[s] = y[s] * c->ovwmol[s];
    batch_recip<NS>(rsq);
    double c1 = 0.0, wc2[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) wc2[s] = 0.0;
    pipe<(NS * NS + 7) / 8, 16, double>(
        [&](int g, double (&w)[16]) {
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const int k = g * 8 + i;
            if (k < NS * NS) {
              w[i] = c->wilko2[k / NS][k % NS];
              w[8 + i] = c->wilko1[k / NS][k % NS];
            }
          }
        },
        [&](int g, const double (&w)[16]) {
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const int k = g * 8 + i, s = k / NS, js = k % NS;
            if (k < NS * NS) {
              double fornow = js == s ? 1.0 : sq[s] * rsq[js];
              fornow = 1.0 + fornow * w[i];
              fornow = w[8 + i] * fornow * fornow;
              wc2[s] = wc2[s] + yw[js] * fornow;
            }
          }
        });
    batch_recip<NS>(wc2);
#pragma unroll
    for (int s = 0; s < NS; s++) c1 = c1 + yw[s] * (mus[s] * wc2[s]);
    fld(pr + P_MU * fs, bo) = c1;
  }
  // face data for NSCBC: cp and mixture gas constant (src/rhscal.f:72-131)
  if (P.inflow_xl || P.outflow_xr) {
    int i, j, k;
    coords(P, idx, i, j, k);
    if (i == 0 || i == P.nx - 1) {
      long nf = (long)P.ny * P.nz;
      double *fc = F.face + (i == 0 ? 0 : (long)nface(P.ns) * nf);
      long fq = (long)k * P.ny + j;
      fc[F_CP * nf + fq] = cp;
      fc[F_RR * nf + fq] = s7 * ovd;
    }
  }
}

// Mixed form, after the point kernel: FP32 holds exp(x) only for x in about
// (-87, 88), and outside the mechanism's range [P.chlo, P.chhi] (worked out
// on the host) a rate coefficient could underflow to zero before a falloff
// division, or overflow before its product with small concentrations, and
// give NaN (or lose a reverse rate) where FP64 gives finite values.  The
// points whose temperature lies outside that range get their rates formed
// again here in FP64 (chem_step64 with the library exp, from the FP64 rho Y_k
// and the stored FP32 temperature) and stored in FP32; a block with no such
// point returns after reading its temperatures.
template <int NS, bool FIX>
__global__ void __launch_bounds__(BLK) k_rate64(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                                const sg_config *__restrict__ c, const Tables *__restrict__ tb) {
  int lb;
  const Member &M = member_at<L_POINT>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  const long idx = (long)lb * BLK + threadIdx.x;
  const long fs = P.fstride;
  const double t = idx < P.npts ? (double)((const float *)F.prim)[P_T * fs + idx] : 1000.0;
  const bool out = idx < P.npts && !(t >= P.chlo && t <= P.chhi);
  if (!__syncthreads_or(out)) return;
  if (!out) return;   // no barrier below
  double ry[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) ry[s] = F.q[(5 + s) * fs + idx];
  const double lt = log(t), ovt = 1.0 / t;
  double gibbs[NS], rate[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) rate[s] = 0.0;
  gibbs_all<NS>(tb, [&](int s) { return locate(c, s, t); }, t, ovt, lt, [&](int s, double g) { gibbs[s] = g; });
  auto ex = [](double x) { return exp(x); };
  if constexpr (FIX) {
    using MT = CtMech<MechH2>;
    MT m0;
    for_steps(m0, [&](int st) {
      chem_step64<NS>(MT{}, st, t, lt, ovt, ry, [&](int s) { return ry[s] * MT::ovw(s); },
                      [&](int s) { return gibbs[s]; }, rate, ex);
    });
  } else {
    // species lists index the point's values at run time: from LDS, one
    // slot per thread (as in k_prim)
    __shared__ double lcy[rows_c<NS, double>][BLK], lgb[rows_g<NS, double>][BLK];
    const int tl = threadIdx.x;
    if constexpr (rows_c<NS, double> > NS) lcy[NS][tl] = 1.0;
    if constexpr (rows_g<NS, double> > NS) lgb[NS][tl] = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      lcy[s][tl] = ry[s] * c->ovwmol[s];
      lgb[s][tl] = gibbs[s];
    }
    RtMech<NS, fill_rows<NS, double>> mr{c, tb};
    for_steps(mr, [&](int st) {
      chem_step64<NS>(mr, st, t, lt, ovt, ry, [&](int s) { return lcy[s][tl]; }, [&](int s) { return lgb[s][tl]; },
                      rate, ex);
    });
  }
  float *rt = (float *)F.rate;
#pragma unroll
  for (int s = 0; s < NS; s++) rt[s * fs + idx] = (float)rate[s];
}

// Soret / Dufour, after the point kernel: ln(T/TDIFGB), the thermal
// diffusion ratio TDRMIX of each light species relative to the other light
// species (src/rhscal.f:1353-1410) and T * TDRMIX, from the stage register
// and the stored temperature (rounded to FP32 in the mixed form).  A kernel
// of its own, so that the point kernels keep their registers.
template <int NS, class R>
__global__ void __launch_bounds__(BLK) k_tdr(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                             const sg_config *__restrict__ c) {
  int lb;
  const Member &M = member_at<L_POINT>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  if (!P.ltmask) return;
  const Fields F = global_fields(M.F);
  const long idx = (long)lb * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  const long fs = P.fstride;
  R *pr = (R *)F.prim;
  const double d = F.q[idx], ovd = 1.0 / d;
  double ry[NS];
  double c3 = 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    ry[s] = F.q[(5 + s) * fs + idx];
    c3 = c3 + ry[s] * c->ovwmol[s];
  }
  const double wmomix = d * (1.0 / c3);
  const double t = (double)pr[P_T * fs + idx];
  pr[P_LNT * fs + idx] = (R)log(t / P.tdifgb);
  const double combo2 = t / P.tdifgb;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    if (!((P.ltmask >> k) & 1u)) continue;
    double tdr = 0.0;
#pragma unroll
    for (int j = 0; j < NS; j++) {
      if (j == k || !((P.ltmask >> j) & 1u)) continue;
      tdr = tdr + (ry[j] * ovd) * c->ovwmol[j] * wmomix * trfit(c->tdrcco[k][j], combo2);
    }
    tdr = tdr * (ry[k] * ovd) * wmomix * c->ovwmol[k];
    pr[prim_tdr(P, k) + idx] = (R)tdr;
    pr[prim_tt(P, k) + idx] = (R)(t * tdr);
  }
}

// Optically thin radiation (src/radcal.f:36-111, called at src/rhscal.f:810):
// the energy equation loses 4 sigma K_P (T^4 - T_ref^4), with the Planck mean
// absorption coefficient K_P = sum over the radiating species r of a_r(T) p_r,
// p_r = rho Y_r R_r T (the conserved rho Y_r, as RHSCAL holds it there).  Added
// in FP64 to the energy accumulator the x pass has just written.
template <int NS, class R>
__global__ void __launch_bounds__(BLK) k_radn(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                              const sg_config *__restrict__ c) {
  int lb;
  const Member &M = member_at<L_POINT>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  if (!P.radn) return;
  const Fields F = global_fields(M.F);
  const long idx = (long)lb * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  const long fs = P.fstride;
  const double t = (double)((const R *)F.prim)[P_T * fs + idx];
  double kp = 0.0;
  for (int r = 0; r < c->nsprad; r++) {
    const int nk = c->nkprad[r];
    double pl = c->akprad[r][nk - 1];
    for (int q = nk - 2; q >= 0; q--) pl = pl * t + c->akprad[r][q];
    const int k = c->nsprid[r];
    kp = kp + pl * (F.q[(5 + k) * fs + idx] * c->rgspec[k] * t);
  }
  const double t4 = t * t * t * t, tr = c->trefrn;
  const double trfrth = tr * tr * tr * tr;
  const double foursb = 4.0 * 5.67037321e-08;   // FOUR * STEFBO (src/com_senga2.h:221-222)
  R *A = (R *)F.acc;
  A[4 * fs + idx] += (R)(-(foursb * kp * (t4 - trfrth)));
}

// FP32 quotient and reciprocal from the hardware reciprocal (v_rcp_f32, about
// 1 ulp; the quotient within 2 ulp) instead of the IEEE-exact FP32 division
// sequence (~10 instructions each), for the FP32 transport and chemistry of
// the mixed-precision point kernel.  Operands there are normal numbers.
__device__ __forceinline__ float rf(float y) { return __builtin_amdgcn_rcpf(y); }
__device__ __forceinline__ float qf(float x, float y) { return x * __builtin_amdgcn_rcpf(y); }

// One step of the mixed-precision form: the rate exponents and Gibbs sums
// assembled in FP64, everything else in FP32 (as chem_step64 otherwise).
template <int NS, class M, class CY, class GB>
__device__ __forceinline__ void chem_stepmx(const M &m, int st, float tf, double lt, double ovt, const float *ryf,
                                            CY cyv, GB gbv, float *rate) {
  const float ysmall = 1.0e-30f, ydenom = 1.0e-15f;
  bool flthrd = true;
  float s3 = 0.0f;
  const int mb = m.mb(st);
  if (mb != 0) {
#pragma unroll
    for (int s = 0; s < NS; s++) s3 = s3 + ryf[s] * m.effwf(mb - 1, s);
  }
  double s2d = m.rp(st, 0) + m.rp(st, 1) * lt - m.rp(st, 2) * ovt;
  float s1 = __expf((float)s2d);
  const int ml = m.ml(st);
  if (ml != 0) {
    const int j = ml - 1;
    float s4 = __expf((float)(m.rl(j, 0) + m.rl(j, 1) * lt - m.rl(j, 2) * ovt));
    float preduc = qf(s3 * s4, s1);
    float fornow = qf((float)m.rl(j, 3) * preduc, 1.0f + preduc);
    s1 = s1 * fornow;
    s2d = (double)__logf(s1);
    flthrd = false;
  }
  const int mt = m.mt(st);
  if (mt != 0) {
    const int j = mt - 1;
    float omalph = 1.0f - (float)m.rt(j, 3);
    float s4 = __expf((float)(m.rt(j, 0) + m.rt(j, 1) * lt - m.rt(j, 2) * ovt));
    float preduc = qf(s3 * s4, s1);
    float trats1 = tf * (float)m.rt(j, 4), trats2 = (float)(-m.rt(j, 5) * ovt), trats3 = tf * (float)m.rt(j, 6);
    float ftcent = omalph * __expf(trats3) + (float)m.rt(j, 3) * __expf(trats1) + __expf(trats2);
    ftcent = __log10f(ftcent);
    float cfactr = (float)m.rt(j, 7) + (float)m.rt(j, 8) * ftcent;
    float enfact = (float)m.rt(j, 9) + (float)m.rt(j, 10) * ftcent;
    float fornow = __log10f(preduc) + cfactr;
    fornow = qf(fornow, enfact - (float)m.rt(j, 11) * fornow);
    fornow = 1.0f + fornow * fornow;
    float fbroad = qf(ftcent, fornow);
    fbroad = __expf(fbroad * (float)m.clnten());
    fornow = qf(fbroad * preduc, 1.0f + preduc);
    s1 = s1 * fornow;
    s2d = (double)__logf(s1);
    flthrd = false;
  }
  const int ms = m.ms(st);
  if (ms != 0) {
    const int j = ms - 1;
    float s4 = __expf((float)(m.rs(j, 0) + m.rs(j, 1) * lt - m.rs(j, 2) * ovt));
    float preduc = qf(s3 * s4, s1);
    float fornow = (float)(m.rs(j, 4) * ovt);
    float fbroad = (float)m.rs(j, 3) * __expf(fornow);
    fornow = tf * (float)m.rs(j, 5);
    fbroad = fbroad + __expf(fornow);
    fornow = __log10f(preduc);
    fornow = rf(1.0f + __log10f(fornow));
    fbroad = (float)m.rs(j, 6) * __expf(fornow * __logf(fbroad));
    fornow = qf(fbroad * preduc, 1.0f + preduc);
    s1 = s1 * fornow;
    s2d = (double)__logf(s1);
    flthrd = false;
  }
  s1 = m.fwd(st, s1, cyv);
#pragma unroll 1
  for (int q = 0; q < m.nrc(st); q++) {
    float fornow = cyv(m.nrcp(st, q));
    fornow = fornow > ysmall ? fornow : ysmall;
    fornow = __expf(m.crsf(st, q) * __logf(fornow));
    fornow = qf(fornow, 1.0f + ydenom * fornow);
    s1 = s1 * fornow;
  }
  if (m.mg(st) != 0) {
    s2d = m.gsum(st, s2d, gbv);
    float s2 = __expf((float)s2d);
    s2 = m.rev(st, s2, cyv);
#pragma unroll 1
    for (int q = 0; q < m.npc(st); q++) {
      float fornow = cyv(m.npcp(st, q));
      fornow = fornow > ysmall ? fornow : ysmall;
      fornow = __expf(m.cpsf(st, q) * __logf(fornow));
      fornow = qf(fornow, 1.0f + ydenom * fornow);
      s2 = s2 * fornow;
    }
    s1 = s1 - s2;
  }
  if (mb != 0 && flthrd) s1 = s1 * s3;
  if (m.dense()) {
#pragma unroll
    for (int u = 0; u < NS; u++)
      if (!M::fixed || m.nuwf(st, u) != 0.0f) rate[u] = rate[u] + s1 * m.nuwf(st, u);
  } else {
    for (int q = 0; q < m.nss(st); q++) {
      int sp = m.nssp(st, q);
      float add = s1 * m.dmwf(st, q);
#pragma unroll
      for (int u = 0; u < NS; u++)
        if (u == sp) rate[u] = rate[u] + add;
    }
  }
}

// Mixed-precision point physics: the temperature Newton iteration, the
// primitive variables and the enthalpies are formed in FP64 as in k_prim and
// stored in FP32; transport and chemistry run in FP32 with the hardware
// exp2/log2 based intrinsics, except that the rate exponents (ln k = ln A +
// n ln T - E/RT, Gibbs sums) are assembled in FP64 before the FP32
// exponential, since they are differences of O(10..100) terms.
template <int NS, bool FIX, bool UPD>
__global__ void __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(4))) k_prim_mx(const Member *__restrict__ mem,
    const uint32_t *__restrict__ map, const sg_config *__restrict__ c, const Tables *__restrict__ tb, int irk) {
  int lb;
  const Member &M = member_at<L_POINT>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  const long idx = (long)lb * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  const uint32_t bo = (uint32_t)idx * 8u, b4 = (uint32_t)idx * 4u;
  const long fs = P.fstride;
  const double *q = F.q;
  float *pr = (float *)F.prim;
  // loaded before the update's stores, which they would otherwise wait for
  const uint32_t idxo = fld(F.itndex, bo / 2u);
  double t = (double)fld(pr + P_T * fs, b4);
  double st[5 + NS];
  if constexpr (UPD) {
    lincom_point<NS, float>(P, F, M, irk, idx, st);
  } else {
#pragma unroll
    for (int v = 0; v < 5 + NS; v++) st[v] = fld(q + v * fs, bo);
  }
  const double d = st[0], ru = st[1], rv = st[2], rw = st[3], re = st[4];
  double ry[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) ry[s] = st[5 + s];
  // --- TEMPER (src/temper.f:58-160) ---
  const double ovd = 1.0 / d;   // one reciprocal for every division by rho
  double ukuk = (ru * ru + rv * rv + rw * rw) * ovd;
  double tc[6], td[6];
  tc[0] = 0.5 * ukuk - re;
#pragma unroll
  for (int m = 1; m <= 5; m++) { tc[m] = 0.0; td[m] = 0.0; }
  temper_sums<NS>(tb, idxo, ry, tc, td);
  double s7 = 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) s7 = s7 + ry[s] * c->rgspec[s];
  const double toltmp = (double)1.0e-10f;  // REAL literal, src/temper.f:33-34
  int iter = 1;
  bool ok = true;
  for (;;) {
    double fp = tc[5], dp = td[5];
#pragma unroll
    for (int m = 4; m >= 1; m--) {
      fp = tc[m] + fp * t;
      dp = td[m] + dp * t;
    }
    fp = tc[0] + fp * t;
    double dt = -fp / dp;
    if (fabs(dt) > toltmp) {
      if (iter < 100) {
        t = t + dt;
        iter++;
        continue;
      }
      ok = false;
    }
    break;
  }
  if (!ok) {
    int i, j, k;
    coords(P, idx, i, j, k);
    set_error(F.err, SG_ETEMPER, i, j, k);
  }
  const uint32_t nidx = locate_all<NS>(c, tb, t);
  const double cp = rho_cp<NS>(tb, nidx, ry, t) * ovd;
  fld(F.itndex, bo / 2u) = nidx;
  SG_PHASE();
  double pres = t * s7;
  if (UPD) {   // also where k_rate64 takes the stored temperature's rates
    const double ts = (double)(float)t;
    if (P.radn || P.ltmask || !(ts >= P.chlo && ts <= P.chhi)) store_stage<NS>(P, F, bo, re, ry);
  }
  fld(pr + P_T * fs, b4) = (float)(t);
  fld(pr + P_P * fs, b4) = (float)(pres - P.pofs);
  // primitives
  fld(pr + P_U * fs, b4) = (float)(ru * ovd);
  fld(pr + P_V * fs, b4) = (float)(rv * ovd);
  fld(pr + P_W * fs, b4) = (float)(rw * ovd);
  fld(pr + P_E * fs, b4) = (float)(re * ovd);
  // --- conductivity (src/rhscal.f:515-573), FP32 ---
  const float tf = (float)t;
  float lam = 0.0f, transp = 0.0f, wmomix = 0.0f;
  if (!P.mixavg) {
    float fornow = (float)P.alamda * __expf((float)P.rlamda * __logf(tf));
    lam = fornow * (float)cp;
    transp = fornow;
  }
  float ryf[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) ryf[s] = (float)ry[s];
  const float df = (float)d;
  if (P.mixavg) {
    transp = __logf(tf * (float)(1.0 / P.tdifgb));
    float c1 = 0.0f, c2 = 0.0f, c3 = 0.0f;
    fits_f<NS>(transp, [&](int s) { return tb->condf[s]; }, [&](int s, float f) {
      float ctr = __expf(f);
      float fornow = ryf[s] * tb->ovwf[s];
      c1 = c1 + fornow * ctr;
      c2 = c2 + qf(fornow, ctr);
      c3 = c3 + fornow;
    });
    c3 = rf(c3);
    c1 = c1 * c3;
    c2 = c2 * c3;
    lam = 0.5f * (c1 + rf(c2));
    wmomix = df * c3;
  }
  fld(pr + P_LAM * fs, b4) = lam;
  if (P.mixw || P.mixp) {
    // ln(mixture molar mass), ln(pressure) and the reciprocal molar mass for
    // the molar-mass and pressure diffusion terms (src/rhscal.f:951-985, 2374),
    // formed in FP64
    double sw = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) sw = sw + ry[s] * c->ovwmol[s];
    const double wm = d * (1.0 / sw);
    fld(pr + P_LNW * fs, b4) = (float)log(wm);
    fld(pr + P_LNP * fs, b4) = (float)log(pres);
    fld(pr + P_OVW * fs, b4) = (float)(1.0 / wm);
  }
  SG_PHASE();
  // --- chemistry (src/chrate.f:146-760) on rho Y ---
  {
    float rate[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) rate[s] = 0.0f;
    const double lt = log(t), ovt = 1.0 / t;
    double gibbs[NS];
    gibbs_all<NS>(tb, [&](int s) { return itint_of(nidx, s); }, t, ovt, lt, [&](int s, double g) { gibbs[s] = g; });
    if constexpr (FIX) {
      using MT = CtMech<MechH2>;
      float cy[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) cy[s] = ryf[s] * MT::ovwf(s);
      MT m0;
      for_steps(m0, [&](int st) {
        chem_stepmx<NS>(MT{}, st, tf, lt, ovt, ryf, [&](int s) { return cy[s]; }, [&](int s) { return gibbs[s]; },
                        rate);
      });
    } else {
      __shared__ float lcy[rows_c<NS, float>][BLK];
      __shared__ double lgb[rows_g<NS, float>][BLK];
      const int tl = threadIdx.x;
      if constexpr (rows_c<NS, float> > NS) lcy[NS][tl] = 1;
      if constexpr (rows_g<NS, float> > NS) lgb[NS][tl] = 0;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        lcy[s][tl] = ryf[s] * tb->ovwf[s];
        lgb[s][tl] = gibbs[s];
      }
      RtMech<NS, fill_rows<NS, float>> mr{c, tb};
      for_steps(mr, [&](int st) {
        chem_stepmx<NS>(mr, st, tf, lt, ovt, ryf, [&](int s) { return lcy[s][tl]; }, [&](int s) { return lgb[s][tl]; },
                        rate);
      });
    }
#pragma unroll
    for (int s = 0; s < NS; s++) fld((float *)F.rate + s * fs, b4) = rate[s];
  }
  // --- mass fractions and enthalpies (src/rhscal.f:1444-1470), FP64, stored FP32 ---
  float y[NS];
  double hmix = 0.0;
  enthalpies<NS>(tb, [&](int s) { return itint_of(nidx, s); }, t, [&](int s, double h) {
    const double yd = ry[s] * ovd;
    y[s] = (float)yd;
    fld(pr + prim_y(P, s), b4) = y[s];
    fld(pr + prim_h(P, s), b4) = (float)h;
    hmix = hmix + h * yd;
  });
  fld(pr + P_HMIX * fs, b4) = (float)hmix;
  SG_PHASE();
  if (!P.mixavg) {
#pragma unroll
    for (int s = 0; s < NS; s++) fld(pr + prim_rd(P, s), b4) = transp * tb->olewf[s];
    fld(pr + P_MU * fs, b4) = transp * (float)P.prantl;
  } else {
    // binary diffusion (src/rhscal.f:1311-1346), FP32
    float yt[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) yt[s] = y[s] + 1.0e-12f;
    float c1t = 0.0f;
#pragma unroll
    for (int js = 0; js < NS; js++) c1t = c1t + yt[js];
    const float ppd = (float)(pres / P.pdifgb);
    float yw2[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) yw2[s] = yt[s] * tb->ovwf[s];
    auto fit = [&](const float *a) {
      float f = a[SG_NTRC - 1];
#pragma unroll
      for (int m = SG_NTRC - 2; m >= 0; m--) f = fma_u(f, transp, a[m]);
      return f;
    };
    if (tb->diffsym) {
      // as in the FP64 kernel: one fit per unordered pair a < b, the pressure
      // ratio folded into the pair weights, no self pairs
      float cs[NS], yw2p[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        cs[s] = 0.0f;
        yw2p[s] = yw2[s] * ppd;
      }
      fits_f<NS * (NS - 1) / 2>(transp, [&](int p) { return tb->difff[kPairs<NS>.a[p]][kPairs<NS>.b[p]]; },
                                [&](int p, float f) {
                                  const int a = kPairs<NS>.a[p], b = kPairs<NS>.b[p];
                                  const float ictd = __expf(-f);
                                  cs[a] = cs[a] + yw2p[b] * ictd;
                                  cs[b] = cs[b] + yw2p[a] * ictd;
                                });
#pragma unroll
      for (int s = 0; s < NS; s++) {
        float c1 = c1t - yt[s];
        float c2 = cs[s] * wmomix;
        fld(pr + prim_rd(P, s), b4) = qf(df * c1, c2);
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; s++) {
        float c2 = 0.0f, self = 0.0f;
#pragma unroll
        for (int js = 0; js < NS; js++) {
          const float term = yw2[js] * (__expf(-fit(tb->difff[s][js])) * ppd);
          c2 = c2 + term;
          if (js == s) self = term;
        }
        float c1 = c1t - yt[s];
        c2 = (c2 - self) * wmomix;
        fld(pr + prim_rd(P, s), b4) = qf(df * c1, c2);
      }
    }
    SG_PHASE();
    // Wilke viscosity (src/rhscal.f:3854-3891), FP32
    float mus[NS], sq[NS], rsq[NS], yw[NS];
    fits_f<NS>(transp, [&](int s) { return tb->viscf[s]; }, [&](int s, float f) {
      mus[s] = __expf(f);
      sq[s] = __builtin_amdgcn_sqrtf(mus[s]);
      rsq[s] = rf(sq[s]);
      yw[s] = y[s] * tb->ovwf[s];
    });
    float c1 = 0.0f, c2 = 0.0f;
    pipe<(NS * NS + 15) / 16, 32, float>(
        [&](int g, float (&w)[32]) {
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const int k = g * 16 + i;
            if (k < NS * NS) {
              w[i] = tb->wilk2f[k / NS][k % NS];
              w[16 + i] = tb->wilk1f[k / NS][k % NS];
            }
          }
        },
        [&](int g, const float (&w)[32]) {
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const int k = g * 16 + i, s = k / NS, js = k % NS;
            if (k < NS * NS) {
              float fornow = js == s ? 1.0f : sq[s] * rsq[js];
              fornow = 1.0f + fornow * w[i];
              fornow = w[16 + i] * fornow * fornow;
              c2 = js ? c2 + yw[js] * fornow : yw[js] * fornow;
              if (js == NS - 1) c1 = c1 + yw[s] * qf(mus[s], c2);
            }
          }
        });
    fld(pr + P_MU * fs, b4) = c1;
  }
  // face data for NSCBC: cp and mixture gas constant (src/rhscal.f:72-131)
  if (P.inflow_xl || P.outflow_xr) {
    int i, j, k;
    coords(P, idx, i, j, k);
    if (i == 0 || i == P.nx - 1) {
      long nf = (long)P.ny * P.nz;
      double *fc = F.face + (i == 0 ? 0 : (long)nface(P.ns) * nf);
      long fq = (long)k * P.ny + j;
      fc[F_CP * nf + fq] = cp;
      fc[F_RR * nf + fq] = s7 * ovd;
    }
  }
}

#pragma clang fp contract(fast)

// ---------------------------------------------------------------------------
// Derivative passes: all derivatives along one direction, or along x and y,
// and the RHS terms separable in them.  x with y, then z (with the
// molecular-transport options: x, y and z each, whose terms take the
// registers).
//
// A block owns a tile of 16 x 16 points; one of its waves takes the
// hydrodynamic fields and every other one up to SPMAX species, each lane four
// points in a row.  A wave stages its own fields one after the other into an
// LDS tile of its own with a 5-deep halo and evaluates their stencils from
// there, so the waves of a block run without barriers but for the resident
// rho u_d tiles at the start and the sums over species at the end.  What
// bounds this: one point per lane read 667 LDS values per point and direction
// (59% of the LDS cycles of the y pass, 16 waves a CU), and a joint x-y pass
// of that form held every species' sums of both directions in each lane and
// spilled.  Four points per lane share a 14-value window along the rows (14
// LDS reads instead of 40), and three species a wave leave the registers for
// both directions.  At 128^3 (9 species) the passes took 0.335 (x) + 0.285
// (y) + 0.295 (z) ms in FP64 and 0.217 + 0.157 + 0.166 ms in FP32; x with y
// now takes 0.408 (0.272 interior, 0.136 edge tiles) and z 0.268 ms in FP64,
// 0.250 and 0.148 in FP32, the x-y pass reading the primitives once (1305 ->
// 790 B per point of HBM traffic).
// Products with rho u_d (e rho u_d, Y rho u_d and the momentum fluxes rho u_d
// u_b) are formed inside the stencils from two tiles.
//
// Bounded x direction (pass_xtiles): rows of large grids are split in two
// launches.  Edge tiles at each end of a row hold every closure row (i < 5,
// i > nx - 6) and evaluate their x stencils with per-column weights; interior
// tiles between them take the interior stencil everywhere and reach no further
// than 5 points into the edge tiles.  Grids whose tiles fit the chip at once
// take edge tiles all along the row, in one launch.  xp: 0 every x tile of a
// row (periodic x, and the y and z passes); 1 the interior tiles of a bounded
// row; 2 its edge tiles.

// The block of a pass: a tile of 16 x-points times 16 rows along y (or along
// z, DV = 2), worked by one wave for the hydrodynamic fields and one wave per
// SPW species.  DX: the x derivatives; DV: the y (1) or z (2) derivatives.  A
// pass takes x with y, or one direction.
template <int DX, int DV, int NS, class R, bool EXT>
struct PassTile {
  static constexpr int ND = DX + (DV != 0);
  static constexpr int T = 16, NP = T * T;                 // points of the tile
  static constexpr int HX = DX ? 5 : 0, HV = DV ? 5 : 0;   // halo
  // species a wave: what its registers hold (a direction more, or the transport
  // options, cost more values per species and point).  Three instead of four
  // with the transport options: 16 species, 48^3, FP64 z 81 -> 69 us, y 81 ->
  // 67, x 75 -> 64 and edge tiles 73 -> 58 us (7 waves instead of 5 a block, 6
  // to 10 spilled registers instead of 16 to 35).
  static constexpr int SPMAX = ND == 2 || EXT ? 3 : 4;
  static constexpr int NG = (NS + SPMAX - 1) / SPMAX;      // species waves
  static constexpr int SPW = (NS + NG - 1) / NG;
  static constexpr int NW = 1 + NG, NT = 64 * NW;
  static_assert(!DX || NW == pass_waves(NS), "the wave count pass_split assumes");
  // LDS tile: rows padded so that the four rows a wave reads at once (4 apart)
  // start on different banks
  static constexpr int LXU = T + 2 * HX, LV = T + 2 * HV;
  static constexpr int LX = DX ? (sizeof(R) == 8 ? 28 : 36) : 20;
  static constexpr int LR = LX * LV;
  static constexpr int LN = LXU * T + 2 * HV * T;          // staged values: no corners
  static constexpr int NIT = (LN + 63) / 64;               // per lane of the staging wave
  static constexpr int LS = LR + NIT * 64 - LN;            // the pad takes the surplus lanes' stores
  static constexpr int NRED = 2 + ND;                      // sums over the waves: energy, vt, ucor per direction
  // tile coordinates of staged value l: the rows with their x halo, then the
  // rows of the halo along the other direction
  static __device__ __forceinline__ void coords(int l, int &tx, int &tv) {
    if (l < LXU * T) {
      tx = l % LXU;
      tv = HV + l / LXU;
    } else {
      const int m = l - LXU * T, r = m / T;
      tx = HX + m % T;
      tv = r < 5 ? r : r + T;
    }
  }
  static __device__ __forceinline__ int slot(int l) {
    if (l >= LN) return LR + l - LN;
    int tx, tv;
    coords(l, tx, tv);
    return tv * LX + tx;
  }
};

// Registers: an FP64 wave holds its species' right-hand sides and gradients
// of four points per lane (36 values with two directions) beside a 14-value
// stencil window, which takes the 256 registers of two waves per SIMD: 224 in z
// at 9 species, all and 6 to 9 spilled in the x-y pass (18 to 26 where 5, 7 or
// 8 species make uneven waves, up to 46 at 10 to 12 and 93 at 16 to 18, where
// it is still faster than x and y apart: 153 against 105 + 72 us at 64^3 and 16
// species); FP32 fits three (x with y) and four waves.
// With one spill per lane and field the z pass was 40% slower, hence the sums
// kept in LDS and the branches that end in a barrier of their own.
template <int DX, int DV, bool BND, int NS, class R, int XP = 0, bool EXT = false>
__global__ void __launch_bounds__((PassTile<DX, DV, NS, R, EXT>::NT))
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 8 ? 2 : (DX + (DV != 0) == 2 ? 3 : 4)))) k_pass(
    const Member *__restrict__ mem, const uint32_t *__restrict__ map) {
  static_assert(XP == 0 || (DX && (XP == 1) != BND), "interior x tiles take the periodic form, edge tiles the bounded one");
  static_assert(!EXT || DX + (DV != 0) == 1, "the passes with the transport options take one direction each");
  using T_ = PassTile<DX, DV, NS, R, EXT>;
  constexpr int ND = T_::ND, T = T_::T, HX = T_::HX, HV = T_::HV, LX = T_::LX, LN = T_::LN, NIT = T_::NIT,
                NP = T_::NP, NW = T_::NW, NT = T_::NT, SPW = T_::SPW;
  constexpr int KIND = XP == 2 ? L_PASSXE : (DX ? L_PASSX : (DV == 1 ? L_PASSY : L_PASSZ));
  constexpr bool RMW = !DX;   // the x part writes the accumulators, the others add to them
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  int lb;
  const Member &M = member_at<KIND>(mem, map, xcd_block(blockIdx.x, gridDim.x), lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  // tile origin: x0, and row v0 along y (z for DV = 2) in plane w0
  const int nv = DV == 2 ? P.nz : P.ny, nw = DV == 2 ? P.ny : P.nz;
  const int nbx = pass_xtiles(P, XP), nbv = (nv + T - 1) / T;
  int bv, w0;
  if (DV == 2) {   // planes before rows of tiles, so that x rows of one z follow each other
    w0 = (lb / nbx) % nw;
    bv = lb / (nbx * nw);
  } else {
    bv = (lb / nbx) % nbv;
    w0 = lb / (nbx * nbv);
  }
  const int x0 = pass_x0(P, XP, lb % nbx), v0 = bv * T;
  // this lane's points: column x, rows 4 q .. 4 q + 3 of the tile
  const int lx = lane & 15, q4 = (lane >> 4) * 4;
  const int i = x0 + lx;
  const bool inx = i < (XP == 1 ? P.nx - PASS_EW : P.nx);
  auto elem = [&](int x, int v) {
    return (uint32_t)(((DV == 2 ? v : w0) * P.ny + (DV == 2 ? w0 : v)) * P.nx + x);
  };
  auto active = [&](int r) { return inx && v0 + q4 + r < nv; };
  // byte offset of point r in a field (past the end of a partial tile, of the
  // last point inside: loads need no test, only stores do)
  const int vend = nv - 1 - (v0 + q4);
  const uint32_t pbs = (uint32_t)(DV == 2 ? P.ny * P.nx : P.nx) * (uint32_t)sizeof(R);
  const uint32_t pb0 = elem(i < P.nx ? i : P.nx - 1, v0 + q4) * (uint32_t)sizeof(R);
  auto pb = [&](int r) { return pb0 + (uint32_t)(r < vend ? r : vend) * pbs; };
  // source element of staged value l (wrapped when periodic, clamped when
  // bounded; a second clamp keeps what partial tiles do not use inside)
  auto gsrc = [&](int l) {
    int tx, tv;
    T_::coords(l, tx, tv);
    int gx = x0 + tx - HX, gv = v0 + tv - HV;
    auto wrap = [](int g, int n) { return g < 0 ? g + n : (g >= n ? g - n : g); };
    if (DX) gx = BND ? (gx < 0 ? 0 : gx) : wrap(gx, P.nx);
    if (DV) gv = wrap(gv, nv);
    return elem(gx < P.nx ? gx : P.nx - 1, gv < nv ? gv : nv - 1);
  };
  // rho u_d of the pass directions, 1/(mixture molar mass) (EXT), and what
  // every wave needs per point: the divergence of rho u over the directions,
  // and (EXT) the derivatives of ln W, ln p and ln T
  __shared__ R tmd[ND][T_::LR];
  __shared__ R tow[EXT ? T_::LR : 1];
  __shared__ R tdiv[NP];
  __shared__ R text[EXT ? 6 : 1][NP];
  // one field per wave at a time
  __shared__ R tbuf[NW][T_::LS];
  R *const tb = tbuf[wv];
  // the waves' sums at every point: energy, divergence of the correction
  // velocity and its components.  Each lane keeps its own points' sums here
  // (24 to 32 registers fewer), and the waves' are added at the end.
  __shared__ R tsum[NW][T_::NRED][NP];
  const long fs = P.fstride;
  const R *pr = (const R *)F.prim;
  // a wave's own staging: fetch() issues the loads of a field into registers,
  // put() stores them to the wave's tile.  No barrier: LDS accesses of a wave
  // take effect in order, and no other wave touches the tile.  The next
  // field's loads are in flight while this one's stencils are evaluated.
  uint32_t go[NIT];
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    const int l = lane + 64 * it;
    go[it] = gsrc(l < LN ? l : LN - 1) * (uint32_t)sizeof(R);
  }
  uint32_t slots[(NIT + 1) / 2];   // LDS positions, two to a register
#pragma unroll
  for (int it = 0; it < NIT; it += 2)
    slots[it / 2] = (uint32_t)T_::slot(lane + 64 * it) | (it + 1 < NIT ? (uint32_t)T_::slot(lane + 64 * (it + 1)) << 16 : 0u);
  // fields in flight: two where the registers allow it (FP64 z pass 277 ->
  // 267 us at 128^3; FP32 spilled, 154 -> 164 us)
  constexpr int DEPTH = !EXT && !DX && sizeof(R) == 8 ? 2 : 1;
  R pf[DEPTH][NIT];
  auto fetch = [&](int k, const R *src) {
#pragma unroll
    for (int it = 0; it < NIT; it++) pf[k % DEPTH][it] = fld(src, go[it]);
  };
  auto put_v = [&](const R (&val)[NIT]) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < NIT; it++) tb[(slots[it / 2] >> (16 * (it & 1))) & 0xffff] = val[it];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto put = [&](int k) { put_v(pf[k % DEPTH]); };
  // the k-th field of a wave: of the hydrodynamic wave, and (without the
  // transport options, whose stages depend on the species) of a species wave
  const int s0 = (wv - 1) * SPW;   // first species of a species wave
  auto has = [&](int q) { return NS % SPW == 0 || s0 + q < NS; };
  auto fetch_h = [&](int k) {
    constexpr int order[9] = {P_MU, P_P, P_LAM, P_T, P_E, P_U, P_V, P_W, P_HMIX};
    if (k < 9) fetch(k, pr + order[k] * fs);
  };
  auto fetch_s = [&](int k) {
    const int sp = s0 + k / 3;
    if (k < 3 * SPW && has(k / 3))
      fetch(k, pr + (k % 3 == 0 ? prim_rd(P, sp) : (k % 3 == 1 ? prim_y(P, sp) : prim_h(P, sp))));
  };
  // bounded x: the tile columns' closure rows, as weights of f(q) - f(0),
  // q = -5..-1, 1..5 (first and second derivative)
  __shared__ R wrow[BND ? 20 : 1][T];
  if (BND) {
    for (int e = t; e < 20 * T; e += NT) {
      const int x = x0 + e % T;
      const int row = x < 5 ? 1 + x : (x > P.nx - 6 && x < P.nx ? 6 + (P.nx - 1 - x) : 0);
      wrow[e / T][e % T] = (R)F.tab->rowd[row][e / T];
    }
  }
  // rho u_d (and 1/W) to LDS by all waves together; their loads go out first,
  // then those of each wave's first fields
  constexpr int NMD = (LN + NT - 1) / NT;
  R mreg[ND + EXT][NMD];
#pragma unroll
  for (int it = 0; it < NMD; it++) {
    const int l = t + it * NT;
    const uint32_t g = gsrc(l < LN ? l : LN - 1);
#pragma unroll
    for (int dd = 0; dd < ND; dd++)
      mreg[dd][it] = (R)fld(F.q + (long)(1 + (DX && dd == 0 ? 0 : DV)) * fs, g * 8u);
    if constexpr (EXT) mreg[ND][it] = fld(pr + (long)P_OVW * fs, g * (uint32_t)sizeof(R));
  }
#pragma unroll
  for (int k = 0; k < DEPTH; k++) {
    if (wv == 0) fetch_h(k);
    else fetch_s(k);
  }
#pragma unroll
  for (int it = 0; it < NMD; it++) {
    const int l = t + it * NT;
    if (l < LN) {
      const int s = T_::slot(l);
#pragma unroll
      for (int dd = 0; dd < ND; dd++) tmd[dd][s] = mreg[dd][it];
      if constexpr (EXT) tow[s] = mreg[ND][it];
    }
  }
  const Interior<R> &C = interior(P, R(0));
  // LDS position of the first row of this lane's window (5 rows before its
  // first point when the pass has a row direction), and of its point r
  const int lw = q4 * LX + lx + HX;
  auto lp = [&](int r) { return lw + (r + HV) * LX; };
  constexpr int VD = ND - 1;   // index of the row direction
  // First and second derivative, and first derivative of the product with
  // rho u_d, of a staged field at the lane's four points: along the rows from
  // one window of 14 values, along x from a window of 11 per point.
  // WANT: bit 0 first, bit 1 second derivative, bit 2 derivative of the
  // product; each (direction, point) is handed to use(dd, r, g1, g2, gp) as it
  // is formed, so that no set of results is held
  auto ders = [&](auto want, const R *tile, R (&c)[4], auto use) {
    constexpr int W = decltype(want)::value;
    if constexpr (DV != 0) {
      R wn[14];
#pragma unroll
      for (int k = 0; k < 14; k++) wn[k] = tile[lw + k * LX];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        c[r] = wn[r + 5];
        pin(c[r]);
      }
      R a1[4], a2[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        auto at = [&](int kk) { return wn[r + kk - 3]; };
        a1[r] = W & 1 ? d1_in<R>(C, DV, at) : R(0);
        a2[r] = W & 2 ? d2_in<R>(C, DV, at) : R(0);
        if (W & 4) {
          if (W & 1) pin(a1[r]);
          if (W & 2) pin(a2[r]);
        } else {
          use(VD, r, a1[r], a2[r], R(0));
        }
      }
      if (W & 4) {
#pragma unroll
        for (int k = 0; k < 14; k++) wn[k] = wn[k] * tmd[VD][lw + k * LX];
#pragma unroll
        for (int r = 0; r < 4; r++)
          use(VD, r, a1[r], a2[r], d1_in<R>(C, DV, [&](int kk) { return wn[r + kk - 3]; }));
      }
      SG_PHASE();
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) c[r] = tile[lp(r)];
    }
    if constexpr (DX != 0 && BND) {
      // closure rows: the column's weights one after the other, over the four
      // points; the next neighbour's values are read while this one's are used
      R s1[4], s2[4], sp[4], cm[4], v[2][4];
      auto read = [&](int q) {
        const int e = q & 1, o = q < 5 ? q - 5 : q - 4;
#pragma unroll
        for (int r = 0; r < 4; r++) v[e][r] = tile[lp(r) + o];
      };
      read(0);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s1[r] = s2[r] = sp[r] = R(0);
        cm[r] = W & 4 ? c[r] * tmd[0][lp(r)] : R(0);
      }
#pragma unroll
      for (int q = 0; q < 10; q++) {
        const int e = q & 1, o = q < 5 ? q - 5 : q - 4;
        R m[4];
        if (W & 4) {
#pragma unroll
          for (int r = 0; r < 4; r++) m[r] = tmd[0][lp(r) + o];
        }
        const R wa = wrow[q][lx], wb = W & 2 ? wrow[10 + q][lx] : R(0);
        if (q < 9) read(q + 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const R f = v[e][r] - c[r];
          if (W & 1) s1[r] = s1[r] + wa * f;
          if (W & 2) s2[r] = s2[r] + wb * f;
          if (W & 4) sp[r] = sp[r] + wa * (v[e][r] * m[r] - cm[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if (W & 1) pin(s1[r]);
          if (W & 2) pin(s2[r]);
          if (W & 4) pin(sp[r]);
        }
        SG_PHASE();
      }
#pragma unroll
      for (int r = 0; r < 4; r++) use(0, r, s1[r] * C.ovdel[0], s2[r] * C.ovdl2[0], sp[r] * C.ovdel[0]);
    } else if constexpr (DX != 0) {
      // interior rows: the five pairs of neighbours one after the other, over
      // the four points (a window per point would hold more values); the next
      // pair's values are read while this one's are used
      R s1[4], s2[4], sp[4], fp[2][4], fm[2][4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        fp[0][r] = tile[lp(r) + 1];
        fm[0][r] = tile[lp(r) - 1];
      }
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const int e = q & 1;
        R gp[4], gm[4];
        if (W & 4) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            gp[r] = tmd[0][lp(r) + q + 1];
            gm[r] = tmd[0][lp(r) - q - 1];
          }
        }
        if (q < 4) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            fp[e ^ 1][r] = tile[lp(r) + q + 2];
            fm[e ^ 1][r] = tile[lp(r) - q - 2];
          }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const R p = fp[e][r], m = fm[e][r];
          if (W & 1) s1[r] = q ? s1[r] + C.ac[q] * (p - m) : C.ac[q] * (p - m);
          if (W & 2) {
            const R f = (p - c[r]) - (c[r] - m);
            s2[r] = q ? s2[r] + C.sc[q] * f : C.sc[q] * f;
          }
          if (W & 4) {
            const R f = p * gp[r] - m * gm[r];
            sp[r] = q ? sp[r] + C.ac[q] * f : C.ac[q] * f;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if (W & 1) pin(s1[r]);
          if (W & 2) pin(s2[r]);
          if (W & 4) pin(sp[r]);
        }
        SG_PHASE();
      }
#pragma unroll
      for (int r = 0; r < 4; r++)
        use(0, r, W & 1 ? s1[r] * C.ovdel[0] : R(0), W & 2 ? s2[r] * C.ovdl2[0] : R(0),
            W & 4 ? sp[r] * C.ovdel[0] : R(0));
    }
  };
  using W1 = std::integral_constant<int, 1>;
  using W12 = std::integral_constant<int, 3>;
  using W14 = std::integral_constant<int, 5>;
  using W124 = std::integral_constant<int, 7>;
  auto dir = [](int dd) { return DX && dd == 0 ? 0 : DV; };
  // boundary-plane flags of the x direction (src/bcinit.f; y and z are
  // periodic), false in every other direction
  const bool atL = BND && i == 0, atR = BND && i == P.nx - 1;
  auto zf = [&](const int *flag, int dd) { return BND && dd == 0 && ((atL && flag[0]) || (atR && flag[1])); };
  // ADB zeroing of the correction-velocity divergence acts on the face planes
  const bool zadb_any = (i == 0 && P.fadb[0]) || (i == P.nx - 1 && P.fadb[1]);
  // x-face points of an NSCBC case: copies of what the NSCBC kernel reads go
  // to the face arrays (of the tiles of a bounded x direction only the edge
  // tiles hold such points), a field's four points under one test.  (One test
  // per value, and the chemical rates and pressure loaded where they were
  // copied, cost 40 of the edge tiles' 164 us at 128^3; now 136 us.)  The test and the address are formed where they are used, so that they
  // hold no registers through the pass.
  auto face = [&]() {
    return (!DX || XP == 2) && inx && (P.inflow_xl || P.outflow_xr) && (i == 0 || i == P.nx - 1);
  };
  const long fnf = (long)P.ny * P.nz;
  auto face_at = [&](int slot, int r) -> double & {
    const int v = v0 + q4 + r, j = DV == 2 ? w0 : v, k = DV == 2 ? v : w0;
    return F.face[(i == 0 ? 0 : (long)nface(P.ns) * fnf) + (long)slot * fnf + (long)k * P.ny + j];
  };
  auto face_put = [&](int slot, const R (&val)[4]) {
    if (face()) {
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (active(r)) face_at(slot, r) = (double)val[r];
    }
  };
  __syncthreads();
  // the divergence of rho u, each row of the lanes' points by one wave
  for (int r = wv; r < 4; r += NW) {
    R dm = R(0);
    if constexpr (DX != 0) {
      const R *m = tmd[0] + lp(r);
      if constexpr (BND) {
        for (int q = 0; q < 10; q++) dm = dm + wrow[q][lx] * (m[q < 5 ? q - 5 : q - 4] - m[0]);
        dm = dm * C.ovdel[0];
      } else {
        dm = d1_in<R>(C, 0, [&](int kk) { return m[kk - 8]; });
      }
    }
    if constexpr (DV != 0) {
      const R d = d1_in<R>(C, DV, [&](int kk) { return tmd[VD][lp(r) + (kk - 8) * LX]; });
      dm = DX ? dm + d : d;
    }
    tdiv[(q4 + r) * T + lx] = dm;
  }
  // EXT: first and second derivatives of ln W, ln p and ln(T/TDIFGB)
  // (src/rhscal.f:945-1004), the three fields spread over the species waves
  if constexpr (EXT) {
    if (wv > 0) {
      R hold[NIT];
#pragma unroll
      for (int it = 0; it < NIT; it++) hold[it] = pf[0][it];
      for (int f = wv - 1; f < 3; f += NW - 1) {
        fetch(0, pr + (f == 0 ? P_LNW : (f == 1 ? P_LNP : P_LNT)) * fs);
        put(0);
        R c[4];
        ders(W12{}, tb, c, [&](int, int r, R g1, R g2, R) {
          text[2 * f][(q4 + r) * T + lx] = g1;
          text[2 * f + 1][(q4 + r) * T + lx] = g2;
        });
      }
#pragma unroll
      for (int it = 0; it < NIT; it++) pf[0][it] = hold[it];
    }
  }
  __syncthreads();
  auto divm = [&](int r) { return tdiv[(q4 + r) * T + lx]; };
  auto md0 = [&](int dd, int r) { return tmd[dd][lp(r)]; };
  R *A = (R *)F.acc;
  R *const ts = &tsum[wv][0][q4 * T + lx];
  auto sum_at = [&](int v, int r) -> R & { return ts[v * NP + r * T]; };
  R aE[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    aE[r] = R(0);
    if (wv > 0) {
#pragma unroll
      for (int v = 1; v < T_::NRED; v++) sum_at(v, r) = R(0);
    }
  }
  // The waves' sums, added over the species waves: divergence of the
  // correction velocity and its components.  Every wave passes exactly one
  // barrier here, each on its own side of the branch below, so that neither
  // side's values hold registers on the other.
  R vt[4], uc[ND][4];
  auto add_waves = [&]() {
#pragma unroll
    for (int r = 0; r < 4; r++) sum_at(0, r) = aE[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int p = (q4 + r) * T + lx;
      vt[r] = R(0);
#pragma unroll
      for (int dd = 0; dd < ND; dd++) uc[dd][r] = R(0);
#pragma unroll
      for (int w = 1; w < NW; w++) {
        vt[r] = vt[r] + tsum[w][1][p];
#pragma unroll
        for (int dd = 0; dd < ND; dd++) uc[dd][r] = uc[dd][r] + tsum[w][2 + dd][p];
      }
    }
  };
  if (wv == 0) {
    R hm0[4], ghm[ND][4];
    // accumulator v of point r; what a pass adds to is loaded a stage before,
    // ahead of that stage's prefetch (loads return in order)
    R o[4];
    auto load_old = [&](int v) {
#pragma unroll
      for (int r = 0; r < 4; r++) o[r] = RMW ? fld(A + (long)v * fs, pb(r)) : R(0);
    };
    auto add = [&](int v, int r, R x) { fld(A + (long)v * fs, pb(r)) = RMW ? o[r] + x : x; };
    // ---------------- hydrodynamic fields: mu, p, lambda, T, e, u, v, w, h_mix
    // Results leave for memory after the next put(), before the next loads go
    // out: the wait for those loads would otherwise wait for the stores too.
    R c[4], mu0[4], p0[4], dp[ND][4], dmu[ND][4];
    put(0);
    fetch_h(DEPTH);
    ders(W1{}, tb, mu0, [&](int dd, int r, R g1, R, R) {
      dmu[dd][r] = g1;
      pin(dmu[dd][r]);
    });
    // pressure, less PRUN(IPREF,JPREF,KPREF) (src/rhsvel.f:741)
    const R pref = pr[(long)P_P * fs];
#pragma unroll
    for (int it = 0; it < NIT; it++) pf[1 % DEPTH][it] = pf[1 % DEPTH][it] - pref;
    put(1);
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (active(r)) {
#pragma unroll
        for (int dd = 0; dd < ND; dd++) fld((R *)F.grad + (long)dir(dd) * fs, pb(r)) = dmu[dd][r];   // for the final kernel
      }
    fetch_h(1 + DEPTH);
    ders(W1{}, tb, p0, [&](int dd, int r, R g1, R, R) {
      dp[dd][r] = g1;
      pin(dp[dd][r]);
    });
#pragma unroll
    for (int r = 0; r < 4; r++) p0[r] = p0[r] + pref + (R)P.pofs;   // stored pressure is p - pofs
    // heat conduction (src/rhscal.f:427-797)
    put(2);
#pragma unroll
    for (int dd = 0; dd < ND; dd++) face_put(dir(dd) == 0 ? F_DPDX : (dir(dd) == 1 ? F_DPDY : F_DPDZ), dp[dd]);
    fetch_h(2 + DEPTH);
    {
      R lam[4], dl[ND][4];
      ders(W1{}, tb, lam, [&](int dd, int r, R g1, R, R) {
        dl[dd][r] = zf(P.fcon, dd) ? R(0) : g1;
        pin(dl[dd][r]);
      });
      put(3);
      fetch_h(3 + DEPTH);
      ders(W12{}, tb, c, [&](int dd, int r, R g1, R g2, R) {
        aE[r] = aE[r] + dl[dd][r] * g1 + lam[r] * (zf(P.fcon, dd) ? R(0) : g2);
        pin(aE[r]);
      });
    }
    // continuity and energy convection (src/rhscal.f:141-415)
    put(4);
    if (DX) face_put(F_T, c);
    load_old(0);
    fetch_h(4 + DEPTH);
    ders(W14{}, tb, c, [&](int dd, int r, R g1, R, R gp) {
      aE[r] = aE[r] - R(0.5) * (gp + md0(dd, r) * g1);
      pin(aE[r]);
    });
#pragma unroll
    for (int r = 0; r < 4; r++) {
      aE[r] = aE[r] - R(0.5) * c[r] * divm(r);
      pin(aE[r]);
    }
    // momentum: split convection from the resident rho u_d tiles and the
    // staged u_b (src/rhsvel.f:348-729, 1312-2110; the reference forms the
    // fluxes rho u*v in y, rho u*w and rho v*w in z as rho u_b * u_d: the
    // same quantity, rounded differently in its last bit), pressure gradient
    // and work (src/rhsvel.f:741-917), separable viscous terms
    // (src/rhsvel.f:1462-2305)
    R res[4], gx[ND][4];   // the component's right-hand side; its gradients (face copies)
    auto face_of = [&](int a) {   // face copies of the stage before component a
      if (a == 0) {
        if (DX) face_put(F_E, c);
        return;
      }
      if (DX) {
        face_put(F_U + a - 1, c);
        face_put(F_DUX + a - 1, gx[0]);
      }
      if (DV == 1 && a < 3) face_put(F_DUY + a - 1, gx[VD]);
      if (DV == 2 && a != 2) face_put(a == 1 ? F_DUZ : F_DWZ, gx[VD]);
    };
#pragma unroll
    for (int a = 0; a < 3; a++) {
      R s[4], tv[4];
#pragma unroll
      for (int r = 0; r < 4; r++) s[r] = tv[r] = R(0);
      put(5 + a);
      // of the stage before: continuity, or the previous component's momentum
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (active(r)) add(a, r, a ? res[r] : -divm(r));
      face_of(a);
      load_old(1 + a);
      fetch_h(5 + a + DEPTH);
      ders(W124{}, tb, c, [&](int dd, int r, R g1, R g2, R gp) {
        const int d = dir(dd);
        s[r] = s[r] - R(0.5) * (gp + md0(dd, r) * g1);
        const R f = a == d ? mu0[r] * (R)P.fthd : mu0[r];
        tv[r] = tv[r] + (zf(a == d ? P.fvsn : P.fvst, dd) ? R(0) : f * g2);
        if (a == d) {
          s[r] = s[r] - dp[dd][r];
          aE[r] = aE[r] - c[r] * dp[dd][r] - p0[r] * g1;
          pin(aE[r]);
        }
        pin(s[r]); pin(tv[r]);
        if (!DX || XP == 2) {
          gx[dd][r] = g1;
          pin(gx[dd][r]);
        }
      });
#pragma unroll
      for (int r = 0; r < 4; r++) {
        aE[r] = aE[r] + tv[r] * c[r];
        pin(aE[r]);
        res[r] = s[r] + tv[r] - R(0.5) * c[r] * divm(r);
        pin(res[r]);
      }
    }
    put(8);
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (active(r)) add(3, r, res[r]);
    face_of(3);
    load_old(4);
    ders(W1{}, tb, hm0, [&](int dd, int r, R g1, R, R) {
      ghm[dd][r] = zf(P.fdif, dd) || zf(P.fadb, dd) ? R(0) : g1;
      pin(ghm[dd][r]);
    });
    add_waves();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int p = (q4 + r) * T + lx;
#pragma unroll
      for (int w = 1; w < NW; w++) aE[r] = aE[r] + tsum[w][0][p];
      aE[r] = aE[r] - hm0[r] * (zadb_any ? R(0) : vt[r]);
#pragma unroll
      for (int dd = 0; dd < ND; dd++) aE[r] = aE[r] - ghm[dd][r] * uc[dd][r];
      if (active(r)) add(4, r, aE[r]);
    }
  } else {
    R aY[SPW][4], dYz[ND][SPW][4], hp[4];   // hp: the last species' enthalpy
    constexpr bool LATE = sizeof(R) == 4;
    // ---------------- species (src/rhscal.f:1030-3944)
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      const int sp = s0 + q;
      if (!has(q)) break;
      R c[4], rd[4], drD[ND][4];
      R er[EXT ? NIT : 1];
      if constexpr (EXT) {
#pragma unroll
        for (int it = 0; it < NIT; it++) er[it] = pf[0][it];
      }
      put(3 * q);
      if (DX && !EXT && LATE && q > 0) face_put(face_h(P.ns, sp - 1), hp);
      if (EXT) fetch(0, pr + prim_y(P, sp));
      else fetch_s(3 * q + DEPTH);
      ders(W1{}, tb, rd, [&](int dd, int r, R g1, R, R) {
        drD[dd][r] = g1;
        pin(drD[dd][r]);
      });
      if constexpr (EXT) {
#pragma unroll
        for (int it = 0; it < NIT; it++) er[it] = er[it] * pf[0][it];   // rho D_k Y_k, staged below
      }
      put(3 * q + 1);
      if (EXT) fetch(0, pr + prim_h(P, sp));
      else fetch_s(3 * q + 1 + DEPTH);
      // dif: the diffusive flux divergence without the correction velocity;
      // dife: as it enters the energy
      R dif[4], dife[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        aY[q][r] = dif[r] = dife[r] = R(0);
      }
      ders(W124{}, tb, c, [&](int dd, int r, R g1, R g2, R gp) {
        aY[q][r] = aY[q][r] - R(0.5) * (gp + md0(dd, r) * g1);
        const R g = drD[dd][r] * g1 + rd[r] * g2;
        dif[r] = dif[r] + (zf(P.fdif, dd) ? R(0) : g);
        if (BND) dife[r] = dife[r] + (zf(P.fdif, dd) || zf(P.fadb, dd) ? R(0) : g);
        sum_at(2 + dd, r) += rd[r] * g1;
        dYz[dd][q][r] = g1;
        pin(aY[q][r]); pin(dif[r]); pin(dYz[dd][q][r]);
        if (BND) pin(dife[r]);
      });
#pragma unroll
      for (int r = 0; r < 4; r++) {
        aY[q][r] = aY[q][r] + dif[r] - R(0.5) * c[r] * divm(r);
        sum_at(1, r) += dif[r];
        if (!BND) dife[r] = dif[r];
        pin(aY[q][r]);
      }
      // (FP64 has no registers to hold these until after the next put())
      auto face_y0 = [&]() {
        if (DX) {
          face_put(F_NSCAL + sp, dYz[0][q]);
          face_put(face_y(P.ns, sp), c);
        }
      };
      if (!LATE) face_y0();
      put(3 * q + 2);
      if (LATE) face_y0();
      const bool more = q + 1 < SPW && has(q + 1);
      const bool ltsp = EXT && ((P.ltmask >> sp) & 1u);
      if (EXT) {
        if (ltsp) fetch(0, pr + prim_tdr(P, sp));
        else if (more) fetch(0, pr + prim_rd(P, sp + 1));
      } else {
        fetch_s(3 * q + 2 + DEPTH);
      }
      R (&h)[4] = hp;
      if constexpr (!EXT) {
        ders(W1{}, tb, h, [&](int dd, int r, R g1, R, R) {
          const bool z = zf(P.fdif, dd) || zf(P.fadb, dd);
          aE[r] = aE[r] + ((z ? R(0) : g1) * dYz[dd][q][r]) * rd[r];
          pin(aE[r]);
        });
        if (DX && !LATE) face_put(face_h(P.ns, sp), h);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          aE[r] = aE[r] + h[r] * dife[r];
          pin(aE[r]);
#pragma unroll
          for (int dd = 0; dd < ND; dd++) dYz[dd][q][r] = zf(P.fdif, dd) ? R(0) : dYz[dd][q][r];
        }
      } else {
        R dh[4], dhu[4], hu[4], rdY[4], tdr[4], gt[4];
        ders(W1{}, tb, h, [&](int, int r, R g1, R, R) {
          dh[r] = g1;
          pin(dh[r]);
        });
        if (DX) face_put(face_h(P.ns, sp), h);
        const bool zdif = zf(P.fdif, 0), zdifadb = zdif || zf(P.fadb, 0);
        // one transport option: flux s7 * grad(l), its derivative ds, with
        // the enthalpy ut and its derivative dut
        auto term = [&](int r, R s7, R ds, R d1l, R d2l, R ut, R dut) {
          sum_at(2, r) += s7 * d1l;
          const R f = ds * d1l + d2l * s7;
          const R m = zdif ? R(0) : f, me = zdifadb ? R(0) : f;
          aY[q][r] = aY[q][r] + m;
          sum_at(1, r) += m;
          aE[r] = aE[r] + me * ut + (zdifadb ? R(0) : dut) * d1l * s7;
          pin(aY[q][r]); pin(aE[r]);
        };
#pragma unroll
        for (int r = 0; r < 4; r++) {
          hu[r] = h[r];
          dhu[r] = dh[r];
          rdY[r] = rd[r] * c[r];
        }
        if (ltsp) {
          // TDRMIX and T * TDRMIX of this species.  Dufour: the species
          // enthalpy carries R_k T TDRMIX through the heat-flux terms up to
          // the Soret terms (src/rhscal.f:1549-1566, 2832-2845).  Soret:
          // rho D_k Y_k TDRMIX with ln(T/TDIFGB) (src/rhscal.f:2757-3758),
          // differentiated as the reference forms STORE7 (src/rhscal.f:2768);
          // its heat-flux terms take the species enthalpy without the Dufour
          // part
          R e7[NIT];
#pragma unroll
          for (int it = 0; it < NIT; it++) e7[it] = er[it] * pf[0][it];
          put(0);
          fetch(0, pr + prim_tt(P, sp));
#pragma unroll
          for (int r = 0; r < 4; r++) {
            tdr[r] = tb[lp(r)];
            pin(tdr[r]);
          }
          R dum[4];
          if (P.soret) {
            put_v(e7);
            ders(W1{}, tb, dum, [&](int, int r, R g1, R, R) {
              gt[r] = g1;
              pin(gt[r]);
            });
          }
          put(0);
          if (more) fetch(0, pr + prim_rd(P, sp + 1));
          if (P.dufour) {
            const R rgk = (R)F.tab->rgs[sp];
            ders(W1{}, tb, dum, [&](int, int r, R g1, R, R) {
              dhu[r] = dh[r] + rgk * g1;
              pin(dhu[r]);
            });
#pragma unroll
            for (int r = 0; r < 4; r++) hu[r] = h[r] + rgk * dum[r];
          }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          aE[r] = aE[r] + hu[r] * dife[r] + (zdifadb ? R(0) : dhu[r]) * dYz[0][q][r] * rd[r];
          dYz[0][q][r] = zdif ? R(0) : dYz[0][q][r];
          pin(aE[r]); pin(dYz[0][q][r]);
        }
        auto ex = [&](int f, int r) { return text[f][(q4 + r) * T + lx]; };
        // molar-mass (src/rhscal.f:1970-2364) and pressure (2365-2759)
        // diffusion.  The heat-flux term with the species enthalpy gradient
        // takes rho D_k in its x component, where the reference's STORE4
        // holds it at that point instead of dh/dx (src/rhscal.f:1887,
        // 2071-2103, 2467-2499).
        R dum[4];
        if (P.mixw) {
          put_v(er);
          ders(W1{}, tb, dum, [&](int, int r, R g1, R, R) {
            term(r, rdY[r], g1, ex(0, r), ex(1, r), hu[r], DX ? rd[r] : dhu[r]);
          });
        }
        if (P.mixp) {
          const R wk = (R)F.tab->wmol[sp];
#pragma unroll
          for (int it = 0; it < NIT; it++) {
            const int l = lane + 64 * it;
            er[it] = er[it] * (R(1) - wk * tow[l < LN ? T_::slot(l) : 0]);
          }
          put_v(er);
          ders(W1{}, tb, dum, [&](int, int r, R g1, R, R) {
            term(r, rdY[r] * (R(1) - wk * tow[lp(r)]), g1, ex(2, r), ex(3, r), hu[r], DX ? rd[r] : dhu[r]);
          });
        }
        if (ltsp && P.soret) {
#pragma unroll
          for (int r = 0; r < 4; r++) term(r, rdY[r] * tdr[r], gt[r], ex(4, r), ex(5, r), h[r], dh[r]);
        }
      }
    }
    // what the stores add to, and the points' own Y_k (read again instead of
    // held through the pass), loaded before the barrier and the first store
    R old[SPW][4], y0[SPW][4];
#pragma unroll
    for (int q = 0; q < SPW; q++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (has(q)) {
          old[q][r] = fld((DX ? (const R *)F.rate : A + 5 * fs) + (long)(s0 + q) * fs, pb(r));
          y0[q][r] = fld(pr + prim_y(P, s0 + q), pb(r));
        }
    add_waves();
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      if (!has(q)) break;
      if (DX) face_put(face_rate(P.ns, s0 + q), old[q]);
      if (DX && !EXT && LATE && (q + 1 == SPW || !has(q + 1))) face_put(face_h(P.ns, s0 + q), hp);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        R s = aY[q][r] - y0[q][r] * vt[r];
#pragma unroll
        for (int dd = 0; dd < ND; dd++) s = s - dYz[dd][q][r] * uc[dd][r];
        if (active(r)) fld(A + (long)(5 + s0 + q) * fs, pb(r)) = old[q][r] + s;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// NSCBC face corrections (src/bounds.f:115-206 preparation, NSBCI3 at x-left
// 610-682, NSBCO1 at x-right 1296-1458), one thread per face point.  They are
// additive in the right-hand sides and depend only on fields the passes have
// written, so they are formed here for the 2 ny nz face points and the final
// kernel adds them.  Inside the final kernel they made every wave (each
// holds a face lane when a row is one or two waves long) run the FP64 face
// code, and raised its register count.
#define NSCBC_BLK 64   // one wave per block: the face points spread over every CU
template <int NS, class R>
__global__ void __launch_bounds__(NSCBC_BLK) k_nscbc(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                                     const sg_config *__restrict__ c) {
  int lb;
  const Member &M = member_at<L_FACE2>(mem, map, blockIdx.x, lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  const long nf = (long)P.ny * P.nz;
  const long t = (long)lb * NSCBC_BLK + threadIdx.x;
  if (t >= 2 * nf) return;
  const int side = t >= nf ? 1 : 0;
  const long fq = t - side * nf;
  if (side == 0 ? !P.inflow_xl : !P.outflow_xr) return;
  const int k = (int)(fq / P.ny), j = (int)(fq - (long)k * P.ny);
  const int i = side ? P.nx - 1 : 0;
  const long idx = ((long)k * P.ny + j) * P.nx + i;
  // the face point's values, from the copies the passes wrote into the face
  // arrays (contiguous over the face); each held in the working precision
  // exactly as the passes read it
  const double *fc = F.face + (i == 0 ? 0 : (long)nface(P.ns) * nf) + fq;
  auto fv = [&](int slot) { return (R)fc[slot * nf]; };
  const R u = fv(F_U), v = fv(F_V), w = fv(F_W);
  const R dux = fv(F_DUX), dvy = fv(F_DVY), dwz = fv(F_DWZ);
  R rD = R(0), rU = R(0), rV = R(0), rW = R(0), rE = R(0);
  R rY[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) rY[s] = R(0);
  constexpr bool BND = true;
  {
    const double strg = fc[F_CP * nf], strr = fc[F_RR * nf];
    const double strt = fv(F_T);
    const double strd = F.q[idx];
    double gam1 = strg - strr;
    const double stre = fv(F_E) - gam1 * strt;
    gam1 = strr / gam1;
    const double ovgm = 1.0 / gam1;
    double fornow = strg * gam1 * strt;
    const double acou = sqrt(fornow), ova2 = 1.0 / fornow;
    double strh[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) strh[s] = fv(face_h(P.ns, s)) - strg * strt * c->rgspec[s] / strr;
    if (i == 0 && P.inflow_xl) {
      // NSBCI3, src/bounds.f:610-682 (imposed values have zero time derivative)
      // drho/dx at the face (src/rhscal.f:3966-3990), one-sided closure row
      const Sten Sx = make_sten<BND>(i, P.nx, 1);
      const double drdx = d1<BND>(P, Sx, 0, [&](int kk) { return F.q[idx + Sx.o[kk]]; });
      double bcl1 = dux, bcl2 = drdx, bcl3 = fv(F_DVX), bcl4 = fv(F_DWX), bcl5 = fc[F_DPDX * nf];
      fornow = strd * acou * bcl1;
      bcl1 = 0.5 * (u - acou) * (bcl5 - fornow);
      bcl2 = u * (bcl2 - bcl5 * ova2);
      bcl3 = u * bcl3;
      bcl4 = u * bcl4;
      bcl5 = 0.5 * (u + acou) * (bcl5 + fornow);
      fornow = bcl1 - strd * acou * 0.0;
      bcl2 = -0.0 - ova2 * (bcl1 + fornow) - bcl2;
      bcl3 = -0.0 - bcl3;
      bcl4 = -0.0 - bcl4;
      bcl5 = fornow - bcl5;
      rE = rE - bcl2 * stre - bcl3 * strd * v - bcl4 * strd * w - bcl5 * (ova2 * stre + u / acou + ovgm);
#pragma unroll
      for (int s = 0; s < NS; s++) {
        double bcly = fv(face_rate(P.ns, s)) / strd - 0.0 - u * fc[(F_NSCAL + s) * nf];
        rE = rE - bcly * strd * strh[s];
      }
    }
    if (i == P.nx - 1 && P.outflow_xr) {
      // NSBCO1, src/bounds.f:1296-1458 (pointwise in/outflow switch and local-Mach beta off)
      const double bet = 0.050;
      const double strp = (double)((const R *)F.prim)[(long)P_P * P.fstride + idx] + P.pofs;
      const double t51 = -v * fc[F_DPDY * nf] - w * fc[F_DPDZ * nf];
      const double t52 = -strp * (dvy + dwz);
      const double t2b = -v * fv(F_DUY) - w * fv(F_DUZ);
      const double tt1 = t51 + t52 * (gam1 + 1.0) - strd * acou * t2b;
      double sorp = 0.0;
#pragma unroll
      for (int s = 0; s < NS; s++) sorp = sorp + strh[s] * fv(face_rate(P.ns, s));
      sorp = -sorp * gam1;
      double bcl1 = 0.5 * (u - acou) * (fc[F_DPDX * nf] - strd * acou * dux);
      bcl1 = 0.5 * sorp + P.cobcxr * acou * (strp - P.pinfxr) + 0.5 * (1.0 - bet) * tt1 - bcl1;
      rD = rD - bcl1 * ova2;
      rU = rU - bcl1 * ova2 * (u - acou);
      rV = rV - bcl1 * ova2 * v;
      rW = rW - bcl1 * ova2 * w;
      rE = rE - bcl1 * (ova2 * stre - u / acou + ovgm);
#pragma unroll
      for (int s = 0; s < NS; s++) rY[s] = rY[s] - bcl1 * ova2 * fv(face_y(P.ns, s));
    }
  }
  double *cr = F.face + (long)side * nface(P.ns) * nf + (long)face_corr(P.ns) * nf + fq;
  cr[0] = rD;
  cr[nf] = rU;
  cr[2 * nf] = rV;
  cr[3 * nf] = rW;
  cr[4 * nf] = rE;
#pragma unroll
  for (int s = 0; s < NS; s++) cr[(5 + s) * nf] = rY[s];
}

// ---------------------------------------------------------------------------
// Final kernel: cross-direction viscous terms (src/rhsvel.f:992-2185), NSCBC
// face corrections (added; formed by k_nscbc) and the RK register update
// (src/lincom.f:53-169, src/fincom.f:54-168).
//
// Between the substages of a step only the cross terms are formed here (CROSS)
// and go back to the accumulators; the register update moves to the next
// point kernel (lincom_point).  At 128^3 and 9 species that is 154 us in FP64
// and 97 us mixed (bounded x; periodic about a fifth less) against 294 and 231
// us with the update, while the point kernel grows by 50 and 60 us; an RK step takes
// 6.74 -> 6.42 ms and 4.41 -> 4.18 ms.
//
// A tile twice as deep (16 x 8 x 8, 512 threads) stages 19 values a point instead
// of 27 and gains nothing by it: the mean launch of a step at 9 species, with
// tiles of depth 8 and 4, takes 1160 and 1200 us (256^3, bounded, FP64), 183
// and 184 (128^3), 63 and 61 (80x80x96), 78 and 70 (81x83x90); mixed 863 and
// 825, 134 and 124, 51 and 44, 63 and 54.
//
// A block owns an FX x FY x FZ tile of points, NPT per thread along z.  The
// six mixed derivatives (d2u/dxdy, d2u/dxdz, d2v/dxdy, d2v/dydz, d2w/dxdz,
// d2w/dydz) read their diagonal neighbours from u, v and w staged one at a
// time into an LDS tile with a 5-deep halo in every direction (wrapped where
// periodic, clamped where bounded), instead of 120 neighbour loads per point.
struct FinalTile {
  static constexpr int FX = 16, FY = 8, FZ = 4;
  static constexpr int NPT = FX * FY * FZ / BLK;   // points per thread
  static constexpr int ZS = BLK / (FX * FY);       // z stride between a thread's points
  static constexpr int GX = FX + 10, GY = FY + 10, GZ = FZ + 10, GN = GX * GY * GZ;
};

// The per-point part of the final kernel at (i, j, k), given its six mixed
// derivatives.
// CROSS: the terms go back to the accumulators (the next substage's point
// kernel does the register update); only momentum and energy have any, and
// the x-face points their NSCBC corrections.
template <bool BND, int NS, class R, bool CROSS>
__device__ __forceinline__ void final_point(const Params &P, const Fields &F, const sg_config *__restrict__ c,
                                            int i, int j, int k, int mode, double lhs, double rhsc, double erc,
                                            double *__restrict__ out, R uxy, R vxy, R uxz, R wxz, R vyz, R wyz,
                                            R u, R v, R w, R dux, R dvy, R dwz, R sxy, R sxz, R syz) {
  const long idx = ((long)k * P.ny + j) * P.nx + i;
  const long fs = P.fstride;
  constexpr int ES = (int)sizeof(R);      // bytes per element of the FP32/FP64 fields
  const uint32_t bo = (uint32_t)idx * (uint32_t)ES, bo8 = (uint32_t)idx * 8u;
  const R *pr = (const R *)F.prim;
  const R mu = fld(pr + P_MU * fs, bo);   // u, v, w come from the staged tile
  const R *G = (const R *)F.grad;
  auto gr = [&](int q) { return fld(G + q * fs, bo); };
  R *A = (R *)F.acc;
  R rD = CROSS ? R(0) : fld(A, bo), rU = fld(A + fs, bo), rV = fld(A + 2 * fs, bo), rW = fld(A + 3 * fs, bo),
    rE = fld(A + 4 * fs, bo);
  auto fz = [&](const int *fl, int dir) {
    int m = dir == 0 ? i : (dir == 1 ? j : k);
    int n = dir == 0 ? P.nx : (dir == 1 ? P.ny : P.nz);
    return (m == 0 && fl[2 * dir]) || (m == n - 1 && fl[2 * dir + 1]);
  };
  const R fthd = (R)P.fthd, tthd = (R)P.tthd;
  const R dmux = gr(0), dmuy = gr(1), dmuz = gr(2);
  // normal stresses with viscosity gradients
  {
    R sxx = fthd * dux - tthd * (dvy + dwz);
    rE = rE + mu * sxx * dux;
    R t = fz(P.fvsn, 0) ? R(0) : sxx * dmux;
    rU = rU + t;
    rE = rE + u * t;
    R syy = fthd * dvy - tthd * (dux + dwz);
    rE = rE + mu * syy * dvy;
    t = fz(P.fvsn, 1) ? R(0) : syy * dmuy;
    rV = rV + t;
    rE = rE + v * t;
    R szz = fthd * dwz - tthd * (dux + dvy);
    rE = rE + mu * szz * dwz;
    t = fz(P.fvsn, 2) ? R(0) : szz * dmuz;
    rW = rW + t;
    rE = rE + w * t;
  }
  {  // xy pair
    const R S7 = sxy;   // du/dy + dv/dx
    const R ma = uxy, mb = vxy;
    R t = fz(P.fvsn, 0) ? R(0) : tthd * mu * mb;
    rU = rU - t; rE = rE - u * t;
    t = fz(P.fvsn, 1) ? R(0) : tthd * mu * ma;
    rV = rV - t; rE = rE - v * t;
    t = fz(P.fvst, 1) ? R(0) : mu * mb + S7 * dmuy;
    rU = rU + t; rE = rE + u * t;
    t = fz(P.fvst, 0) ? R(0) : mu * ma + S7 * dmux;
    rV = rV + t; rE = rE + v * t;
    rE = rE + mu * S7 * S7;
  }
  {  // xz pair
    const R S7 = sxz;   // du/dz + dw/dx
    const R ma = uxz, mb = wxz;
    R t = fz(P.fvsn, 0) ? R(0) : tthd * mu * mb;
    rU = rU - t; rE = rE - u * t;
    t = fz(P.fvsn, 2) ? R(0) : tthd * mu * ma;
    rW = rW - t; rE = rE - w * t;
    t = fz(P.fvst, 2) ? R(0) : mu * mb + S7 * dmuz;
    rU = rU + t; rE = rE + u * t;
    t = fz(P.fvst, 0) ? R(0) : mu * ma + S7 * dmux;
    rW = rW + t; rE = rE + w * t;
    rE = rE + mu * S7 * S7;
  }
  {  // yz pair
    const R S7 = syz;   // dv/dz + dw/dy
    const R ma = vyz, mb = wyz;
    R t = fz(P.fvsn, 1) ? R(0) : tthd * mu * mb;
    rV = rV - t; rE = rE - v * t;
    t = fz(P.fvsn, 2) ? R(0) : tthd * mu * ma;
    rW = rW - t; rE = rE - w * t;
    t = fz(P.fvst, 2) ? R(0) : mu * mb + S7 * dmuz;
    rV = rV + t; rE = rE + v * t;
    t = fz(P.fvst, 1) ? R(0) : mu * ma + S7 * dmuy;
    rW = rW + t; rE = rE + w * t;
    rE = rE + mu * S7 * S7;
  }
  if constexpr (CROSS) {
    if (BND && (i == 0 || i == P.nx - 1)) {   // NSCBC faces, as below
      const long nf = (long)P.ny * P.nz, fq = (long)k * P.ny + j;
      const double *cr = F.face + (i == 0 ? 0 : (long)nface(P.ns) * nf) + (long)face_corr(P.ns) * nf + fq;
      rU = rU + (R)cr[nf];
      rV = rV + (R)cr[2 * nf];
      rW = rW + (R)cr[3 * nf];
      rE = rE + (R)cr[4 * nf];
      R a[1 + NS];   // every load before the first store
      a[0] = fld(A, bo) + (R)cr[0];
#pragma unroll
      for (int s = 0; s < NS; s++) a[1 + s] = fld(A + (5 + s) * fs, bo) + (R)cr[(5 + s) * nf];
      fld(A, bo) = a[0];
#pragma unroll
      for (int s = 0; s < NS; s++) fld(A + (5 + s) * fs, bo) = a[1 + s];
    }
    fld(A + fs, bo) = rU;
    fld(A + 2 * fs, bo) = rV;
    fld(A + 3 * fs, bo) = rW;
    fld(A + 4 * fs, bo) = rE;
    return;
  }
  R rY[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) rY[s] = fld(A + (5 + s) * fs, bo);
  // ---------------- NSCBC faces: corrections formed by k_nscbc
  if (BND && (i == 0 || i == P.nx - 1)) {
    const long nf = (long)P.ny * P.nz, fq = (long)k * P.ny + j;
    const double *cr = F.face + (i == 0 ? 0 : (long)nface(P.ns) * nf) + (long)face_corr(P.ns) * nf + fq;
    rD = rD + (R)cr[0];
    rU = rU + (R)cr[nf];
    rV = rV + (R)cr[2 * nf];
    rW = rW + (R)cr[3 * nf];
    rE = rE + (R)cr[4 * nf];
#pragma unroll
    for (int s = 0; s < NS; s++) rY[s] = rY[s] + (R)cr[(5 + s) * nf];
  }
  // ---------------- register update
  R Rv[5 + NS];
  Rv[0] = rD; Rv[1] = rU; Rv[2] = rV; Rv[3] = rW; Rv[4] = rE;
#pragma unroll
  for (int s = 0; s < NS; s++) Rv[5 + s] = rY[s];
  if (mode == 2) {
#pragma unroll
    for (int vv2 = 0; vv2 < 5 + NS; vv2++) out[vv2 * fs + idx] = Rv[vv2];
    return;   // no register update
  }
  // The solution register of every variable is loaded before the first
  // store: the stores could alias the loads as far as the compiler knows, so
  // a load after a store would cost a memory round trip per variable.
  double old[5 + NS];
#pragma unroll
  for (int vv2 = 0; vv2 < 5 + NS; vv2++) old[vv2] = fld(F.run + vv2 * fs, bo8);
  if (sizeof(R) == 4 && mode == 1 && P.renorm) {
    // mixed form with renormalisation: FINCOM, then the species of the new
    // solution rescaled in FP64 so that they sum to the new density
    double nw[5 + NS];
#pragma unroll
    for (int vv2 = 0; vv2 < 5 + NS; vv2++) {
      const int slot = vv2 < 5 ? vv2 : 5;
      if (i >= P.rklo[slot]) {
        if (F.erk) fld(F.erk + vv2 * fs, bo8) += erc * (double)Rv[vv2];
        nw[vv2] = old[vv2] + lhs * (double)Rv[vv2];
      } else {
        nw[vv2] = old[vv2];
      }
    }
    if (i >= P.rklo[5]) {
      double sy = 0.0;
#pragma unroll
      for (int s = 0; s < NS; s++) sy = sy + nw[5 + s];
      const double f = nw[0] / sy;
#pragma unroll
      for (int s = 0; s < NS; s++) nw[5 + s] = nw[5 + s] * f;
    }
#pragma unroll
    for (int vv2 = 0; vv2 < 5 + NS; vv2++) {
      const int slot = vv2 < 5 ? vv2 : 5;
      if (i >= P.rklo[slot]) fld(F.run + vv2 * fs, bo8) = nw[vv2];
      fld(F.q + vv2 * fs, bo8) = i >= P.rklo[slot] ? nw[vv2] : (double)Rv[vv2];
    }
    return;
  }
#pragma unroll
  for (int vv2 = 0; vv2 < 5 + NS; vv2++) {
    const int slot = vv2 < 5 ? vv2 : 5;
    double *runv = F.run + vv2 * fs, *qv = F.q + vv2 * fs;
    if (i >= P.rklo[slot]) {
      if (F.erk) fld(F.erk + vv2 * fs, bo8) += erc * (double)Rv[vv2];   // *ERR += RKERR * R
      if (mode == 0) {
        fld(runv, bo8) = old[vv2] + lhs * (double)Rv[vv2];
        fld(qv, bo8) = old[vv2] + rhsc * (double)Rv[vv2];
      } else {
        double nw = old[vv2] + lhs * (double)Rv[vv2];
        fld(runv, bo8) = nw;
        fld(qv, bo8) = nw;
      }
    } else {
      fld(qv, bo8) = (double)Rv[vv2];
    }
  }
}

template <bool BND, int NS, class R, bool CROSS>
__global__ void __launch_bounds__(BLK) k_final(const Member *__restrict__ mem, const uint32_t *__restrict__ map,
                                               const sg_config *__restrict__ c, int irk, double *__restrict__ out) {
  using FT = FinalTile;
  constexpr int FX = FT::FX, FY = FT::FY, FZ = FT::FZ, NPT = FT::NPT, GX = FT::GX, GY = FT::GY, GZ = FT::GZ;
  int lb;
  const Member &M = member_at<L_FINAL>(mem, map, xcd_block(blockIdx.x, gridDim.x), lb);
  const Params P = M.P;
  const Fields F = global_fields(M.F);
  // substage irk: LINCOM (mode 0) or FINCOM at the last substage (mode 1);
  // irk = 0 writes the right-hand side to out (mode 2)
  const int mode = irk == 0 ? 2 : (irk < 5 ? 0 : 1);
  const double lhs = irk ? M.rkl[irk - 1] : 0.0, rhsc = irk ? M.rkr[irk - 1] : 0.0,
               erc = irk ? M.rke[irk - 1] : 0.0;
  // bounded x: mixed-derivative row weights (uniform row form); the field tile
  __shared__ R mtab[BND ? SG_NROW * 7 : 1];   // in the working precision
  __shared__ R tile[FT::GN];
  const int t = threadIdx.x;
  if (BND && t < SG_NROW * 7) mtab[t] = (R)(&F.tab->mixw[0][0])[t];   // ordered by the first staging barrier
  // first-derivative row weights W1 of the x closure rows (the passes' table)
  __shared__ R wtab1[BND ? SG_NROW * 5 : 1];
  if (BND && t < SG_NROW * 5) wtab1[t] = (R)F.tab->roww[t / 5][t % 5];
  const int nx = P.nx, ny = P.ny, nz = P.nz;
  const int nbx = (nx + FX - 1) / FX, nby = (ny + FY - 1) / FY;
  const int x0 = (lb % nbx) * FX, y0 = ((lb / nbx) % nby) * FY, z0 = (lb / (nbx * nby)) * FZ;
  const int lx = t % FX, ly = (t / FX) % FY, lz0 = t / (FX * FY);
  const int i = x0 + lx, j = y0 + ly;
  // x closure row of this thread's points; waves holding any closure row use
  // the uniform row form, others the interior diagonal stencil
  int row = 0;
  if (BND && i < nx) {
    if (i < 5) row = 1 + i;
    else if (i > nx - 6) row = 6 + (nx - 1 - i);
  }
  const bool xedge = BND && __ballot(row != 0) != 0;
  int pk[5] = {0, 0, 0, 0, 0};
  if (xedge) {
#pragma unroll
    for (int q = 0; q < 5; q++) pk[q] = c_mix_row_offsets.w[row][q];
  }
  Sten S0;
  S0.mode = 0;
  const long fs = P.fstride;
  const R *pr = (const R *)F.prim;
  // halo index along one direction: wrapped when periodic, clamped when
  // bounded; a second clamp keeps the halo of points past the end of a
  // partial tile (whose results are not used) inside the field
  auto hidx = [&](int g, int n, bool bounded) {
    if (bounded) return g < 0 ? 0 : (g >= n ? n - 1 : g);
    g = g < 0 ? g + n : (g >= n ? g - n : g);
    return g < n ? g : n - 1;
  };
  // staging: the tile is GX*GY columns of GZ values; thread t fetches
  // columns t, t + BLK, all loads in flight at once, into registers and then
  // stores them to LDS.  The next field's fetch is issued before the current
  // field's derivatives are evaluated.  Column offsets are per thread, plane
  // offsets are uniform.  Only what the field's stencils read is fetched: u
  // the (x, y) and (x, z) planes of its points, v (x, y) and (y, z), w (x, z)
  // and (y, z).
  constexpr int NCOL = GX * GY, NC = (NCOL + BLK - 1) / BLK;
  uint32_t co[NC];
  bool inx[NC], iny[NC];
#pragma unroll
  for (int q = 0; q < NC; q++) {
    const int cc = t + q * BLK, tx = cc % GX, ty = cc / GX;
    const bool ok = cc < NCOL;
    inx[q] = ok && tx >= 5 && tx < 5 + FX;
    iny[q] = ok && ty >= 5 && ty < 5 + FY;
    co[q] = ok ? (uint32_t)(hidx(y0 - 5 + ty, ny, false) * nx + hidx(x0 - 5 + tx, nx, BND)) : 0u;
  }
  R stg[NC][GZ];
  auto columns = [&](auto field, auto f) {   // f(q, z) for the column values field 0, 1, 2 (u, v, w) needs
    constexpr int FLD = decltype(field)::value;
#pragma unroll
    for (int q = 0; q < NC; q++) {
      const bool halo = FLD == 0 ? iny[q] : (FLD == 1 ? inx[q] : inx[q] || iny[q]);   // z halo
      const bool in = FLD == 2 ? halo : t + q * BLK < NCOL;
      if (in) {
#pragma unroll
        for (int z = 5; z < 5 + FZ; z++) f(q, z);
      }
      if (halo) {
#pragma unroll
        for (int z = 0; z < 5; z++) {
          f(q, z);
          f(q, z + 5 + FZ);
        }
      }
    }
  };
  auto fetch = [&](auto field) {
    const R *f = pr + (P_U + decltype(field)::value) * fs;
    columns(field, [&](int q, int z) {
      const uint32_t zo = (uint32_t)hidx(z0 - 5 + z, nz, false) * (uint32_t)(nx * ny);
      stg[q][z] = fld(f, (zo + co[q]) * (uint32_t)sizeof(R));
    });
  };
  auto store = [&](auto field) {
    columns(field, [&](int q, int z) { tile[z * NCOL + t + q * BLK] = stg[q][z]; });
  };
  using FU = std::integral_constant<int, 0>;
  using FV = std::integral_constant<int, 1>;
  using FW = std::integral_constant<int, 2>;
  auto base = [&](int p) { return (lz0 + p * FT::ZS + 5) * GX * GY + (ly + 5) * GX + (lx + 5); };
  auto mix_x = [&](int B, int d2) {   // d2 = 1: (x, y); d2 = 2: (x, z)
    const int s2 = d2 == 1 ? GX : GX * GY;
    auto g = [&](int a, int b) { return tile[B + a + b * s2]; };
    if (xedge) {
      // fresh copies of the row offsets for every call, so that the
      // neighbour addresses are formed per call instead of being kept live
      // for the whole kernel (they would set its occupancy)
      int pq[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        pq[q] = pk[q];
        asm volatile("" : "+v"(pq[q]));
      }
      return dmix_rows<R>(P, pq, 0, d2, [&](int q) { return mtab[BND ? row * 7 + q : 0]; }, g);
    }
    return dmix<false, R>(P, S0, 0, d2, [&](int k1, int k2) { return g(k1 - 8, k2 - 8); });
  };
  auto mix_yz = [&](int B) {
    return dmix<false, R>(P, S0, 1, 2, [&](int k1, int k2) { return tile[B + (k1 - 8) * GX + (k2 - 8) * GX * GY]; });
  };
  // first derivatives of the staged field: x with the closure rows where the
  // wave holds them (the passes' rows and weights), y and z interior (the
  // supported cases are periodic there)
  auto d1x = [&](int B) {
    if (xedge) {
      // a first derivative reads entries 0..9 (P1, M1) of the packed row,
      // words 0..2; all three loads are issued before the fences, which
      // would otherwise wait for each load in turn
      int pq[5] = {0, 0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 3; q++) pq[q] = c_row_offsets.w[row][q];
#pragma unroll
      for (int q = 0; q < 3; q++) asm volatile("" : "+v"(pq[q]));
      return d1_rows<R>(P, pq, 0, [&](int q) { return wtab1[BND ? row * 5 + q : 0]; },
                        [&](int q) { return tile[B + q]; });
    }
    return d1<false, R>(P, S0, 0, [&](int kk) { return tile[B + kk - 8]; });
  };
  auto d1y = [&](int B) { return d1<false, R>(P, S0, 1, [&](int kk) { return tile[B + (kk - 8) * GX]; }); };
  auto d1z = [&](int B) { return d1<false, R>(P, S0, 2, [&](int kk) { return tile[B + (kk - 8) * GX * GY]; }); };
  // the derivatives, and each point's own u, v, w read back from the tile
  // (the values a global load would give) for the per-point part.  The
  // velocity gradients the viscous terms use are formed here from the tile
  // too, instead of being written by the passes and read back: du/dx, dv/dy,
  // dw/dz and the sums du/dy + dv/dx, du/dz + dw/dx, dv/dz + dw/dy, each
  // added in that order
  R uxy[NPT], uxz[NPT], vxy[NPT], vyz[NPT], wxz[NPT], wyz[NPT], uc[NPT], vc[NPT], wc[NPT];
  R dux[NPT], dvy[NPT], dwz[NPT], sxy[NPT], sxz[NPT], syz[NPT];
  fetch(FU{});
  store(FU{});
  __syncthreads();
  fetch(FV{});
#pragma unroll
  for (int p = 0; p < NPT; p++) {
    uc[p] = tile[base(p)];
    uxy[p] = mix_x(base(p), 1);
    uxz[p] = mix_x(base(p), 2);
    pin(uxy[p]); pin(uxz[p]);
    dux[p] = d1x(base(p));
    sxy[p] = d1y(base(p));
    sxz[p] = d1z(base(p));
    pin(dux[p]); pin(sxy[p]); pin(sxz[p]);
  }
  __syncthreads();
  store(FV{});
  __syncthreads();
  fetch(FW{});
#pragma unroll
  for (int p = 0; p < NPT; p++) {
    vc[p] = tile[base(p)];
    vxy[p] = mix_x(base(p), 1);
    vyz[p] = mix_yz(base(p));
    pin(vxy[p]); pin(vyz[p]);
    sxy[p] = sxy[p] + d1x(base(p));
    dvy[p] = d1y(base(p));
    syz[p] = d1z(base(p));
    pin(sxy[p]); pin(dvy[p]); pin(syz[p]);
  }
  __syncthreads();
  store(FW{});
  __syncthreads();
#pragma unroll
  for (int p = 0; p < NPT; p++) {
    wc[p] = tile[base(p)];
    wxz[p] = mix_x(base(p), 2);
    wyz[p] = mix_yz(base(p));
    pin(wxz[p]); pin(wyz[p]);
    sxz[p] = sxz[p] + d1x(base(p));
    syz[p] = syz[p] + d1y(base(p));
    dwz[p] = d1z(base(p));
    pin(sxz[p]); pin(syz[p]); pin(dwz[p]);
  }
#pragma unroll
  for (int p = 0; p < NPT; p++) {
    const int k = z0 + lz0 + p * FT::ZS;
    if (i < nx && j < ny && k < nz)
      final_point<BND, NS, R, CROSS>(P, F, c, i, j, k, mode, lhs, rhsc, erc, out, uxy[p], vxy[p], uxz[p], wxz[p],
                              vyz[p], wyz[p], uc[p], vc[p], wc[p], dux[p], dvy[p], dwz[p], sxy[p], sxz[p], syz[p]);
  }
}

// ---------------------------------------------------------------------------
// The nine operators on one field (parity of the stencil device functions).
template <bool BX, bool BY, bool BZ>
__global__ void __launch_bounds__(BLK) k_derivs(Params P, const double *__restrict__ f, double *__restrict__ out) {
  long idx = (long)blockIdx.x * BLK + threadIdx.x;
  if (idx >= P.npts) return;
  int i, j, k;
  coords(P, idx, i, j, k);
  const Sten Sx = make_sten<BX>(i, P.nx, 1);
  const Sten Sy = make_sten<BY>(j, P.ny, (int)P.sy);
  const Sten Sz = make_sten<BZ>(k, P.nz, (int)P.sz);
  const long n = P.npts;
  out[idx] = d1<BX>(P, Sx, 0, [&](int q) { return f[idx + Sx.o[q]]; });
  out[n + idx] = d1<BY>(P, Sy, 1, [&](int q) { return f[idx + Sy.o[q]]; });
  out[2 * n + idx] = d1<BZ>(P, Sz, 2, [&](int q) { return f[idx + Sz.o[q]]; });
  out[3 * n + idx] = d2<BX>(P, Sx, 0, [&](int q) { return f[idx + Sx.o[q]]; });
  out[4 * n + idx] = d2<BY>(P, Sy, 1, [&](int q) { return f[idx + Sy.o[q]]; });
  out[5 * n + idx] = d2<BZ>(P, Sz, 2, [&](int q) { return f[idx + Sz.o[q]]; });
  out[6 * n + idx] = dmix<BX>(P, Sx, 0, 1, [&](int a, int b) { return f[idx + Sx.o[a] + Sy.o[b]]; });
  out[7 * n + idx] = dmix<BX>(P, Sx, 0, 2, [&](int a, int b) { return f[idx + Sx.o[a] + Sz.o[b]]; });
  out[8 * n + idx] = dmix<BY>(P, Sy, 1, 2, [&](int a, int b) { return f[idx + Sy.o[a] + Sz.o[b]]; });
}

// ---------------------------------------------------------------------------
// Launchers, instantiated for the species count SG_NS of this translation
// unit (the build compiles one object per supported count, in parallel).

static inline unsigned grid_for(long n) { return (unsigned)((n + BLK - 1) / BLK); }

template <int NS>
void launch_tempin_t(const Params &P, const sg_config *dcfg, const Fields &F, hipStream_t st) {
  if (P.precision) hipLaunchKernelGGL((k_tempin<NS, float>), dim3(grid_for(P.npts)), dim3(BLK), 0, st, P, dcfg, F);
  else hipLaunchKernelGGL((k_tempin<NS, double>), dim3(grid_for(P.npts)), dim3(BLK), 0, st, P, dcfg, F);
}
template <int NS>
void launch_boundt_t(const Launch &L, hipStream_t st) {
  hipLaunchKernelGGL(k_boundt<NS>, dim3(L.nblk[L_FACE]), dim3(BLK), 0, st, L.mem, L.map[L_FACE]);
}
template <int NS>
void launch_bountt_t(const Launch &L, hipStream_t st) {
  hipLaunchKernelGGL(k_bountt<NS>, dim3(L.nblk[L_FACE]), dim3(BLK), 0, st, L.mem, L.map[L_FACE]);
}
template <int NS, bool FIX, bool UPD>
static void launch_prim_u(const Launch &L, int irk, hipStream_t st) {
  const dim3 g(L.nblk[L_POINT]), b(BLK);
  const uint32_t *map = L.map[L_POINT];
  if (L.precision) hipLaunchKernelGGL((k_prim_mx<NS, FIX, UPD>), g, b, 0, st, L.mem, map, L.c, L.tab, irk);
  else hipLaunchKernelGGL((k_prim<NS, FIX, UPD>), g, b, 0, st, L.mem, map, L.c, L.tab, irk);
}
template <int NS, bool FIX>
static void launch_prim_k(const Launch &L, int irk, hipStream_t st) {
  if (irk) launch_prim_u<NS, FIX, true>(L, irk, st);
  else launch_prim_u<NS, FIX, false>(L, 0, st);
}
template <int NS>
void launch_prim_t(const Launch &L, int irk, hipStream_t st) {
  bool fixed = false;
  if constexpr (NS == MechH2::nspec) {
    fixed = L.mechfix != 0;
    if (fixed) launch_prim_k<NS, true>(L, irk, st);
  }
  if (!fixed) launch_prim_k<NS, false>(L, irk, st);
  if (L.precision) {   // mixed form: FP64 rates where FP32 cannot hold them
    const dim3 g(L.nblk[L_POINT]), b(BLK);
    bool fix = false;
    if constexpr (NS == MechH2::nspec) fix = L.mechfix != 0;
    if (fix) hipLaunchKernelGGL((k_rate64<NS, NS == MechH2::nspec>), g, b, 0, st, L.mem, L.map[L_POINT], L.c, L.tab);
    else hipLaunchKernelGGL((k_rate64<NS, false>), g, b, 0, st, L.mem, L.map[L_POINT], L.c, L.tab);
  }
  if (L.ext) {   // Soret / Dufour quantities of the members that need them
    const dim3 g(L.nblk[L_POINT]), b(BLK);
    if (L.precision) hipLaunchKernelGGL((k_tdr<NS, float>), g, b, 0, st, L.mem, L.map[L_POINT], L.c);
    else hipLaunchKernelGGL((k_tdr<NS, double>), g, b, 0, st, L.mem, L.map[L_POINT], L.c);
  }
}
template <int NS, class R, int DX, int DV, bool EXT>
static void launch_pass_w(const Launch &L, hipStream_t st) {
  const int k = DX ? L_PASSX : (DV == 1 ? L_PASSY : L_PASSZ);
  const dim3 b(PassTile<DX, DV, NS, R, EXT>::NT);
  if constexpr (DX != 0) {
    if (L.bndx) {
      // interior tiles of the bounded rows, then their edge tiles
      if (L.nblk[k] > 0)
        hipLaunchKernelGGL((k_pass<DX, DV, false, NS, R, 1, EXT>), dim3(L.nblk[k]), b, 0, st, L.mem, L.map[k]);
      hipLaunchKernelGGL((k_pass<DX, DV, true, NS, R, 2, EXT>), dim3(L.nblk[L_PASSXE]), b, 0, st, L.mem,
                         L.map[L_PASSXE]);
      return;
    }
  }
  hipLaunchKernelGGL((k_pass<DX, DV, false, NS, R, 0, EXT>), dim3(L.nblk[k]), b, 0, st, L.mem, L.map[k]);
}
// x with y and z, or (EXT, the passes with the molecular-transport options) x, y and z
template <int NS, class R>
static void launch_pass_r(int dir, const Launch &L, hipStream_t st) {
  if (L.ext) {
    if (dir == 0) launch_pass_w<NS, R, 1, 0, true>(L, st);
    else if (dir == 1) launch_pass_w<NS, R, 0, 1, true>(L, st);
    else launch_pass_w<NS, R, 0, 2, true>(L, st);
  } else {
    if (dir == 0) launch_pass_w<NS, R, 1, 1, false>(L, st);
    else if (dir == 2) launch_pass_w<NS, R, 0, 2, false>(L, st);
  }
}
template <int NS>
void launch_pass_t(int dir, const Launch &L, hipStream_t st) {
  if (L.precision) launch_pass_r<NS, float>(dir, L, st);
  else launch_pass_r<NS, double>(dir, L, st);
}
template <int NS>
void launch_nscbc_t(const Launch &L, hipStream_t st) {
  const dim3 g(L.nblk[L_FACE2]), b(NSCBC_BLK);
  if (L.precision) hipLaunchKernelGGL((k_nscbc<NS, float>), g, b, 0, st, L.mem, L.map[L_FACE2], L.c);
  else hipLaunchKernelGGL((k_nscbc<NS, double>), g, b, 0, st, L.mem, L.map[L_FACE2], L.c);
}
template <int NS>
void launch_radn_t(const Launch &L, hipStream_t st) {
  const dim3 g(L.nblk[L_POINT]), b(BLK);
  if (L.precision) hipLaunchKernelGGL((k_radn<NS, float>), g, b, 0, st, L.mem, L.map[L_POINT], L.c);
  else hipLaunchKernelGGL((k_radn<NS, double>), g, b, 0, st, L.mem, L.map[L_POINT], L.c);
}
template <int NS, bool CROSS>
static void launch_final_c(const Launch &L, int irk, double *out, hipStream_t st) {
  const dim3 g(L.nblk[L_FINAL]), b(BLK);
  const uint32_t *map = L.map[L_FINAL];
  if (L.precision) {
    if (L.bndx) hipLaunchKernelGGL((k_final<true, NS, float, CROSS>), g, b, 0, st, L.mem, map, L.c, irk, out);
    else hipLaunchKernelGGL((k_final<false, NS, float, CROSS>), g, b, 0, st, L.mem, map, L.c, irk, out);
  } else {
    if (L.bndx) hipLaunchKernelGGL((k_final<true, NS, double, CROSS>), g, b, 0, st, L.mem, map, L.c, irk, out);
    else hipLaunchKernelGGL((k_final<false, NS, double, CROSS>), g, b, 0, st, L.mem, map, L.c, irk, out);
  }
}
template <int NS>
void launch_final_t(const Launch &L, int irk, double *out, hipStream_t st) {
  launch_final_c<NS, false>(L, irk, out, st);
}
template <int NS>
void launch_cross_t(const Launch &L, hipStream_t st) {
  launch_final_c<NS, true>(L, 0, nullptr, st);
}

#ifdef SG_NS
template void launch_tempin_t<SG_NS>(const Params &, const sg_config *, const Fields &, hipStream_t);
template void launch_boundt_t<SG_NS>(const Launch &, hipStream_t);
template void launch_bountt_t<SG_NS>(const Launch &, hipStream_t);
template void launch_prim_t<SG_NS>(const Launch &, int, hipStream_t);
template void launch_cross_t<SG_NS>(const Launch &, hipStream_t);
template void launch_pass_t<SG_NS>(int, const Launch &, hipStream_t);
template void launch_nscbc_t<SG_NS>(const Launch &, hipStream_t);
template void launch_radn_t<SG_NS>(const Launch &, hipStream_t);
template void launch_final_t<SG_NS>(const Launch &, int, double *, hipStream_t);
#endif

#ifdef SG_DERIVS
// ADAPTT error norm (src/adaptt.f:60-160): max over variables and points of
// |ERR| / (|RUN| + norm_v) with the norms of src/dtinit.f:138-145.  A NaN
// never exceeds the running maximum, as in the reference's comparisons.
__global__ void __launch_bounds__(BLK) k_errmax(Params P, Fields F) {
  __shared__ double red[BLK / 64];
  const long idx = (long)blockIdx.x * BLK + threadIdx.x;
  double tot = 0.0;
  if (idx < P.npts) {
    const long fs = P.fstride;
    for (int v = 0; v < 5 + P.ns; v++) {
      const double nrm = v == 0 ? 0.0 : (v < 4 ? 1.0e-6 : (v == 4 ? 1.0e-2 : 1.0e-10));
      const double f = fabs(F.erk[v * fs + idx]) / (fabs(F.run[v * fs + idx]) + nrm);
      if (f > tot) tot = f;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const double u = __shfl_down(tot, o, 64);
    if (u > tot) tot = u;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = tot;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLK / 64; w++)
      if (red[w] > tot) tot = red[w];
    // non-negative doubles order like their bit patterns
    atomicMax(F.emax, (unsigned long long)__double_as_longlong(tot));
  }
}

__global__ void __launch_bounds__(BLK) k_zero(double *p, long n) {
  const long idx = (long)blockIdx.x * BLK + threadIdx.x;
  if (idx < n) p[idx] = 0.0;
}

void member_blocks(const Params &P, int nblk[L_NKIND]) {
  nblk[L_FACE] = (int)grid_for((long)P.ny * P.nz);
  nblk[L_FACE2] = (int)((2L * P.ny * P.nz + NSCBC_BLK - 1) / NSCBC_BLK);
  nblk[L_POINT] = (int)grid_for(P.npts);
  auto tiles = [&](int tx, int ty, int tz) {
    return ((P.nx + tx - 1) / tx) * ((P.ny + ty - 1) / ty) * ((P.nz + tz - 1) / tz);
  };
  nblk[L_FINAL] = tiles(FinalTile::FX, FinalTile::FY, FinalTile::FZ);
  // passes: every tile of a row (periodic x), or of bounded rows the interior
  // tiles (L_PASSX) and the edge tiles (L_PASSXE); y goes with x where the
  // launch has no transport options
  const long rows = (long)((P.ny + 15) / 16) * P.nz;
  nblk[L_PASSX] = (int)(pass_xtiles(P, P.bnd[0] ? 1 : 0) * rows);
  nblk[L_PASSXE] = P.bnd[0] ? (int)(pass_xtiles(P, 2) * rows) : 0;
  nblk[L_PASSY] = pass_xy(P) ? 0 : tiles(16, 16, 1);
  nblk[L_PASSZ] = tiles(16, 1, 16);
}

void launch_errmax(const Params &P, const Fields &F, hipStream_t st) {
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(BLK), 0, st, (double *)F.emax, 1L);
  hipLaunchKernelGGL(k_errmax, dim3(grid_for(P.npts)), dim3(BLK), 0, st, P, F);
}

void launch_zero(double *p, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_zero, dim3(grid_for(n)), dim3(BLK), 0, st, p, n);
}

void launch_derivs(const Params &P, const double *f, double *out, hipStream_t st) {
  dim3 g(grid_for(P.npts)), b(BLK);
  if (P.bnd[0]) hipLaunchKernelGGL((k_derivs<true, false, false>), g, b, 0, st, P, f, out);
  else hipLaunchKernelGGL((k_derivs<false, false, false>), g, b, 0, st, P, f, out);
}
#endif

}  // namespace sg
