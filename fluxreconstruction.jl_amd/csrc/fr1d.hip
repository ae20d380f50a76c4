// fr1d.hip -- 1D FR residuals (src/Equation/eq_euler.jl:29-98, eq_advection.jl:153-273,
// eq_scalar.jl:1-12) and batched ensembles of independent 1D Euler problems, for gfx950.
//
// One kernel body handles a chunk of consecutive elements of one problem: lane t of a workgroup
// of T threads owns element first-1+t, so lanes 0 and T-1 are halo elements that only provide
// their face traces; the T-2 interior lanes produce du.  Traces and interface fluxes go through
// LDS.  A single problem is a work list of its chunks; an ensemble is the concatenated work list
// of all members (any degree 1..8 per member) processed by a persistent grid.  Stepping keeps the
// elements of a chunk in registers over several steps (fr1d_block_kernel); a launch per stage over
// the chunks (fr1d_kernel) gives the same bits and serves the residual, Tsit5 and the forced paths.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "fr_common.h"
#include "fr_ops_table.h"
#include "fr_tsit5.h"

namespace fr {

constexpr int NSP_MAX = 9;  // degrees 1..8 (example/euler_highlevel.jl runs degree 7)
// The operators that do not depend on the correction function are compile-time constants
// (StdOps1D); the device table holds dhl, dhr [NSP_MAX each] of nsp (2..NSP_MAX) at
// OPS_STRIDE*(nsp-2).  With all operators in the table, or the literals hoisted out of the step
// loops (Makefile), the register-resident kernel spilled up to 1400 scalar values into lanes of
// vector registers: 40 against 34 us per step on 512 members of p = 2..4.
constexpr int OPS_STRIDE = 2 * NSP_MAX;
struct Prob1D {
  long long off;  // first double of the member in the concatenated state
  int ncell, nsp;
  double iJ;      // 2/dx
  double cut;     // shock_cut of the member's degree
};

struct Work1D {
  int prob, first;  // member, first interior element of the chunk
};

struct Stage1D {
  const double *u;
  double *out;
  const double *u0;
  const double *acc_in;
  double *acc_out;
  double a0, a1, b, b2;
  int residual;
};

struct Phys1D {
  int eq;       // FR_EQ_EULER / FR_EQ_ADVECTION
  int bc;       // FR_BC1_*
  double g, gm1, a;
};

// The arithmetic of one element, shared by the launch-per-stage and the register-resident kernels
// (the same code in both, so both give the same bits; the sums are written as fma chains, since which
// of two products the compiler fuses depends on where else a product with the same literal is used).

// discontinuous flux f = F(u) / J, traces of u and f on the element's two faces
template <int NSP, int EQ, int NV>
__device__ __forceinline__ void elem_traces(const double (&w)[NSP][NV], double iJ, const Phys1D &ph, double (&f)[NSP][NV],
                                            double (&uL)[NV], double (&uR)[NV], double (&fL)[NV], double (&fR)[NV]) {
  constexpr StdOps1D<NSP> o{};
#pragma unroll
  for (int p = 0; p < NSP; ++p) {
    if constexpr (EQ == FR_EQ_EULER) {
      const double r = 1.0 / w[p][0];
      const double vel = w[p][1] * r;
      const double pr = ph.gm1 * (w[p][2] - 0.5 * w[p][1] * vel);
      f[p][0] = w[p][1] * iJ;
      f[p][1] = (w[p][1] * vel + pr) * iJ;
      f[p][2] = ((w[p][2] + pr) * vel) * iJ;
    } else {
      f[p][0] = ph.a * w[p][0] * iJ;
    }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double a = 0, b = 0, c = 0, d = 0;
#pragma unroll
    for (int q = 0; q < NSP; ++q) {
      a = fma(w[q][k], o.ll[q], a);
      b = fma(w[q][k], o.lr[q], b);
      c = fma(f[q][k], o.ll[q], c);
      d = fma(f[q][k], o.lr[q], d);
    }
    uL[k] = a;
    uR[k] = b;
    fL[k] = c;
    fR[k] = d;
  }
}

// interface flux over J on the element's left face: the left neighbour's right traces (ul, fl; fl
// for advection only), the own left traces; wrap marks the face between the last and first element
template <int EQ, int FLUX, int NV>
__device__ __forceinline__ void elem_face(const double (&ul)[NV], double fl, const double (&uL)[NV],
                                          const double (&fL)[NV], bool wrap, double iJ, const Phys1D &ph,
                                          double (&fs)[NV]) {
  if constexpr (EQ == FR_EQ_EULER) {
    double fw[3];
    riemann_x3<FLUX>(ul, uL, ph.g, ph.gm1, fw);
    // the reference divides the interface flux by J in the correction
#pragma unroll
    for (int k = 0; k < 3; ++k) fs[k] = fw[k] * iJ;
  } else {
    // regularised local Lax-Friedrichs of eq_advection.jl:128-137 (+1e-6 on the periodic face
    // :163); f is already divided by J
    const double eps = wrap ? 1e-6 : 1e-8;
    const double au = (fL[0] - fl) / (uL[0] - ul[0] + eps);
    fs[0] = 0.5 * (fL[0] + fl) - 0.5 * fabs(au) * (uL[0] - ul[0]);
  }
}

// du of point p, variable k from the corrections cl, cr (interface flux minus own trace) of k; ops:
// dhl, dhr of the element's nsp
template <int NSP, int NV>
__device__ __forceinline__ double elem_du(const double (&f)[NSP][NV], const double *__restrict__ ops, int p, int k,
                                          double cl, double cr) {
  constexpr StdOps1D<NSP> o{};
  double d = 0.0;
#pragma unroll
  for (int q = 0; q < NSP; ++q) d = fma(f[q][k], o.dl[p + NSP * q], d);
  return -fma(cr, ops[NSP_MAX + p], fma(cl, ops[p], d));
}

template <int NSP, int EQ, int FLUX>
__device__ __forceinline__ void chunk1d(const Prob1D &pb, int first, const double *__restrict__ ops,
                                        const Phys1D &ph, const Stage1D &sa, double *sh) {
  constexpr int NV = (EQ == FR_EQ_EULER) ? 3 : 1;
  const int T = blockDim.x;
  const int tid = threadIdx.x;
  const int n = pb.ncell;
  // shared layout: uR[NV][T] | fR[NV][T] | Fs[NV][T]
  double *sUR = sh, *sFR = sh + NV * T, *sFS = sh + 2 * NV * T;
  int e = first - 1 + tid;
  bool valid = true;
  if (e < 0 || e >= n) {
    // only the two neighbours of the domain wrap (periodic); lanes further out are unused
    if (ph.bc == FR_BC1_PERIOD && (e == -1 || e == n))
      e = (e < 0) ? e + n : e - n;
    else
      valid = false;
  }
  const bool interior = tid >= 1 && tid <= T - 2 && (first - 1 + tid) < n;
  const double *__restrict__ u = sa.u + pb.off;
  double w[NSP][NV];
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int p = 0; p < NSP; ++p) w[p][k] = valid ? u[e + (long long)n * (p + NSP * k)] : (k == 0 ? 1.0 : (k == 2 ? 2.5 : 0.0));
  double f[NSP][NV], uL[NV], uR[NV], fL[NV], fR[NV];
  elem_traces<NSP, EQ, NV>(w, pb.iJ, ph, f, uL, uR, fL, fR);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    sUR[k * T + tid] = uR[k];
    sFR[k * T + tid] = fR[k];
  }
  __syncthreads();
  // interface flux on the left face of the own element (face between e-1 and e)
  if (tid >= 1 && valid) {
    const bool nb_ok = (ph.bc == FR_BC1_PERIOD) || (first - 2 + tid) >= 0;
    if (nb_ok) {
      double ul[NV], fs[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) ul[k] = sUR[k * T + tid - 1];
      const int ge = first - 1 + tid;  // global element right of the face
      elem_face<EQ, FLUX, NV>(ul, sFR[tid - 1], uL, fL, ge == 0 || ge == n, pb.iJ, ph, fs);
#pragma unroll
      for (int k = 0; k < NV; ++k) sFS[k * T + tid] = fs[k];
    }
  }
  __syncthreads();
  if (interior) {
    const int ge = first - 1 + tid;
    const bool zero = (ph.bc == FR_BC1_DIRICHLET) && (ge == 0 || ge == n - 1);
    double *__restrict__ out = sa.out + pb.off;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const double cl = sFS[k * T + tid] - fL[k];
      const double cr = sFS[k * T + tid + 1] - fR[k];
#pragma unroll
      for (int p = 0; p < NSP; ++p) {
        double du = elem_du<NSP, NV>(f, ops, p, k, cl, cr);
        if (zero) du = 0.0;
        const long long idx = ge + (long long)n * (p + NSP * k);
        if (sa.residual) {
          out[idx] = du;
        } else {
          double v = sa.a1 * w[p][k];
          if (sa.a0 != 0.0) v = sa.a0 * sa.u0[pb.off + idx] + v;
          out[idx] = v + sa.b * du;
          if (sa.acc_out) sa.acc_out[pb.off + idx] = sa.acc_in[pb.off + idx] + sa.b2 * du;
        }
      }
    }
  }
  __syncthreads();  // the shared buffers are reused by the next chunk of a persistent loop
}

// NMAX: the largest nsp the instance handles.  Problem sets of degree <= 4 use the NMAX = 5
// instance, whose register budget is that of those degrees (119 VGPRs for Euler); sets with
// higher degrees (up to 8) the NMAX = NSP_MAX one (179 VGPRs, fewer waves per SIMD).
template <int EQ, int FLUX, int NMAX>
__device__ __forceinline__ void stage_chunk(const Prob1D &pb, int first, const double *__restrict__ ops,
                                            const Phys1D &ph, const Stage1D &sa, double *sh) {
  const double *o = ops + OPS_STRIDE * (pb.nsp - 2);
  switch (pb.nsp) {
    case 2: chunk1d<2, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
    case 3: chunk1d<3, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
    case 4: chunk1d<4, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
    case 5: chunk1d<5, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
    default:
      if constexpr (NMAX > 5) {
        switch (pb.nsp) {
          case 6: chunk1d<6, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
          case 7: chunk1d<7, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
          case 8: chunk1d<8, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
          default: chunk1d<9, EQ, FLUX>(pb, first, o, ph, sa, sh); break;
        }
      }
      break;
  }
}

template <int EQ, int FLUX, int NMAX>
__global__ __launch_bounds__(256) void fr1d_kernel(const Prob1D *__restrict__ probs, const Work1D *__restrict__ work,
                                                   int nwork, const double *__restrict__ ops, Phys1D ph, Stage1D sa) {
  constexpr int NV = (EQ == FR_EQ_EULER) ? 3 : 1;
  __shared__ double sh[3 * NV * 256];
  for (int wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
    const Work1D wk = work[wi];
    stage_chunk<EQ, FLUX, NMAX>(probs[wk.prob], wk.first, ops, ph, sa, sh);
  }
}

// ------------------------------------------------------------------ 1D dissipation
// Per-cell dissipation of 1D Euler states, one thread per cell over the same work lists:
//  mode 1: modal sensor + filter of example/euler_highlevel.jl:37-52 (rho modes u_hat = iV rho,
//          su = u_hat[end]^2 / (sum u_hat^2 + 1e-6), shock_detector(log10 su, deg) with
//          S0 = -3 log10(deg), kappa = 4; on a shock all variables filtered with
//          lambda = dt exp(0.875 deg) 0.15, u_hat[n] /= 1 + lambda (n+1)^2 n^2);
//  mode 2: positivity limiter of src/dissipation.jl:61-123 (density squeeze toward the cell
//          mean, then the pressure squeeze with the closed-form tj_equation root).
// count[0] += flagged (mode 1) / limited (mode 2) cells, count[1] += cells whose density
// assert failed (left untouched).
// Returns whether the values x of the cell were replaced; cut: Prob1D::cut.
constexpr double kKappa1D = 4.0;  // example/euler_highlevel.jl:42
template <int NSP>
__device__ __forceinline__ bool diss1d_values(double (&x)[NSP][3], int mode, double g, double dt, double cut,
                                              bool &flag, bool &bad) {
  constexpr StdOps1D<NSP> o{};
  flag = false;
  bad = false;
  if (mode == 1) {
    double den = 0.0, last = 0.0;
#pragma unroll
    for (int a = 0; a < NSP; ++a) {
      double s = 0.0;
#pragma unroll
      for (int b = 0; b < NSP; ++b) s = fma(o.iV1[a + NSP * b], x[b][0], s);
      den = fma(s, s, den);
      if (a == NSP - 1) last = s * s;
    }
    const int deg = NSP - 1;
    if (!shock_flagged(last, den + 1e-6, cut, -3.0 * log10((double)deg), kKappa1D)) return false;
    flag = true;
    const double lambda = dt * exp(0.875 * deg) * 0.15;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double mh[NSP];
#pragma unroll
      for (int a = 0; a < NSP; ++a) {
        double s = 0.0;
#pragma unroll
        for (int b = 0; b < NSP; ++b) s = fma(o.iV1[a + NSP * b], x[b][k], s);
        mh[a] = a == 0 ? s : s / (1.0 + lambda * (double)((a + 1) * (a + 1) * a * a));
      }
#pragma unroll
      for (int a = 0; a < NSP; ++a) {
        double s = 0.0;
#pragma unroll
        for (int b = 0; b < NSP; ++b) s = fma(o.V1[a + NSP * b], mh[b], s);
        x[a][k] = s;
      }
    }
    return true;
  }
  // positivity limiter
  double um[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double s = 0.0;
#pragma unroll
    for (int p = 0; p < NSP; ++p) s = fma(x[p][k], o.hw[p], s);
    um[k] = s;
  }
  const double um4[4] = {um[0], um[1], 0.0, um[2]};
  const double p_mean = 0.5 * um[0] / prim_lambda(um4, g);
  double bv[2][4];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int p = 0; p < NSP; ++p) {
      a = fma(x[p][k], o.ll[p], a);
      b = fma(x[p][k], o.lr[p], b);
    }
    bv[0][k < 2 ? k : 3] = a;
    bv[1][k < 2 ? k : 3] = b;
  }
  bv[0][2] = bv[1][2] = 0.0;
  const double eps = fmin(1e-13, fmin(um[0], p_mean));
  double rmin = fmin(bv[0][0], bv[1][0]);
#pragma unroll
  for (int p = 0; p < NSP; ++p) rmin = fmin(rmin, x[p][0]);
  const double t1 = fmin((um[0] - eps) / (um[0] - rmin + 1e-8), 1.0);
  if (!(t1 > 0.0 && t1 <= 1.0)) {
    bad = true;
    return false;
  }
  bool have = false;
  double tmin = 1.0e300;
#pragma unroll
  for (int f = 0; f < 2; ++f)
    if (prim_lambda_below(bv[f], g, eps)) {
      have = true;
      tmin = fmin(tmin, tj_root(bv[f], um4, g, eps));
    }
#pragma unroll
  for (int p = 0; p < NSP; ++p) {
    x[p][0] = t1 * (x[p][0] - um[0]) + um[0];
    const double w4[4] = {x[p][0], x[p][1], 0.0, x[p][2]};
    if (prim_lambda_below(w4, g, eps)) {
      have = true;
      tmin = fmin(tmin, tj_root(w4, um4, g, eps));
    }
  }
  const double t2 = have ? fmin(tmin, 1.0) : 1.0;
  flag = t1 < 1.0 || have;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int p = 0; p < NSP; ++p) x[p][k] = have ? t2 * (x[p][k] - um[k]) + um[k] : x[p][k];
  return true;
}

// the same on cell e of a state in memory
template <int NSP>
__device__ __forceinline__ void diss1d_cell(double *__restrict__ u, long long n, long long e, int mode, double g,
                                            double dt, double cut, bool &flag, bool &bad) {
  double x[NSP][3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int p = 0; p < NSP; ++p) x[p][k] = u[e + n * (p + NSP * k)];
  if (!diss1d_values<NSP>(x, mode, g, dt, cut, flag, bad)) return;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int p = 0; p < NSP; ++p) u[e + n * (p + NSP * k)] = x[p][k];
}

// the dissipation pass over the interior elements of one work item
template <int NMAX>
__device__ __forceinline__ void diss_chunk(const Prob1D &pb, const Work1D &wk, double *u, int mode, double g, double dt, int *count) {
  {
    const int tid = threadIdx.x, T = blockDim.x;
    const int e = wk.first - 1 + tid;
    const bool interior = tid >= 1 && tid <= T - 2 && e < pb.ncell;
    bool flag = false, bad = false;
    if (interior) {
      double *um = u + pb.off;
      switch (pb.nsp) {
        case 2: diss1d_cell<2>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
        case 3: diss1d_cell<3>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
        case 4: diss1d_cell<4>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
        case 5: diss1d_cell<5>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
        default:
          if constexpr (NMAX > 5) {
            switch (pb.nsp) {
              case 6: diss1d_cell<6>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
              case 7: diss1d_cell<7>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
              case 8: diss1d_cell<8>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
              default: diss1d_cell<9>(um, pb.ncell, e, mode, g, dt, pb.cut, flag, bad); break;
            }
          }
          break;
      }
    }
    const unsigned long long bf = __ballot(flag), bb = __ballot(bad);
    if ((tid & 63) == 0) {
      if (bf) atomicAdd(count, __popcll(bf));
      if (bb) atomicAdd(count + 1, __popcll(bb));
    }
  }
}

template <int NMAX>
__global__ __launch_bounds__(256) void fr1d_diss_kernel(const Prob1D *__restrict__ probs, const Work1D *__restrict__ work,
                                                        int nwork, double *u, int mode, double g, double dt,
                                                        int *count) {
  for (int wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
    const Work1D wk = work[wi];
    diss_chunk<NMAX>(probs[wk.prob], wk, u, mode, g, dt, count);
  }
}

// ------------------------------------------------------------------ register-resident stepping
// A launch per stage moves the state through HBM or L2 and waits out a launch's latency for every
// stage; here a workgroup of kBlockT lanes loads the elements of a chunk once, steps them several
// times in registers and stores them once.  Only the face traces go through LDS, with two workgroup
// barriers per stage.  A member of at most kBlockT elements is one chunk and takes any number of
// steps per launch.  A larger one is cut into chunks of kBlockT - 2 H elements with H halo elements
// on either side, which the workgroup steps along: every stage spoils one more element from the
// outside, so H / stages steps leave the chunk's own elements right (the neighbours compute the same
// values from the same bits).  The next launch reads the other buffer.  Every element runs the
// arithmetic of the launch-per-stage kernels (elem_traces, elem_face, elem_du, diss1d_values), so
// the bits are theirs.
//
// Bound: one chunk alone by the latency of a stage's dependent FP64 operations, the full chip by
// FP64 issue.  Against a launch per stage (or, for members of up to 508 cells, one workgroup running
// a schedule of stages over L2): 100 cells, p = 2, RK4: 1.52 -> 0.41 us per stage; 512 members of
// 64 to 2048 cells, p = 2..4, SSP-RK3 with the filter: 104 -> 34 us per step (state read and written
// once per four steps instead of once per stage).
constexpr int kBlockT = 256;
// halo elements per side: kHaloFull when the chunks fill the chip (9 % of the lanes step halo
// elements), kHaloIdle when they do not (the lanes cost nothing then, launches do)
constexpr int kHaloFull = 12, kHaloIdle = 48;
static_assert(kHaloFull >= 12 && kHaloFull % 12 == 0 && kHaloIdle % 12 == 0, "whole steps of 1 to 4 stages");
constexpr int kBlockSteps = 4096;  // steps per launch of members that are one chunk

struct Blk1D {
  int prob, first, count, halo;  // member, own elements, halo elements per side (0: the whole member)
};

// nsteps steps of one scheme: stage s is a0[s] base + a1[s] w + b[s] L(w), base the step's start, or
// RK4's accumulator in its last stage (acc += b2[s] L(w) in the others)
struct Run1D {
  int nstage, nsteps, filter;
  double fdt;  // filter time step
  double a0[4], a1[4], b[4], b2[4];
};

// kernel instances: the plain form (sensor + filter before a step when asked), RK4 (an accumulator
// more), and with the limiter on every stage input (whose registers would cost the others a wavefront
// per SIMD)
enum { BLK_PLAIN = 0, BLK_RK4 = 1, BLK_LIMIT = 2 };

template <int NSP, int EQ, int FLUX, int KIND>
__device__ __forceinline__ void block1d(const Prob1D &pb, const Blk1D &bk, const double *__restrict__ ops,
                                        const Phys1D &ph, const Run1D &run, const double *__restrict__ src,
                                        double *dst, int *count, double *sh) {
  constexpr int NV = (EQ == FR_EQ_EULER) ? 3 : 1;
  constexpr bool ACC = KIND == BLK_RK4;
  const int T = blockDim.x, tid = threadIdx.x, n = pb.ncell;
  double *sUR = sh, *sFR = sh + NV * T, *sFS = sh + (NV + 1) * T;
  int e = bk.first - bk.halo + tid;
  const bool whole = bk.halo == 0;
  bool live = tid < bk.count + 2 * bk.halo;
  if (ph.bc == FR_BC1_PERIOD)
    e = e < 0 ? e + n : (e >= n ? e - n : e);
  else
    live = live && e >= 0 && e < n;
  const bool own = live && tid >= bk.halo && tid < bk.halo + bk.count;
  const bool zero = ph.bc == FR_BC1_DIRICHLET && (e == 0 || e == n - 1);
  const int lt = tid > 0 ? tid - 1 : (whole ? n - 1 : 0), rt = whole && tid == n - 1 ? 0 : min(tid + 1, T - 1);
  double U[NSP][NV], w[NSP][NV], A[ACC ? NSP : 1][NV];
  if (live) {
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int p = 0; p < NSP; ++p) U[p][k] = src[pb.off + e + (long long)n * (p + NSP * k)];
  }
  int nflag = 0, nbad = 0;
  auto dissipate = [&](double(&x)[NSP][NV], int mode) {
    if constexpr (EQ == FR_EQ_EULER && !ACC) {
      if (live) {
        bool flag, bad;
        diss1d_values<NSP>(x, mode, ph.g, run.fdt, pb.cut, flag, bad);
        if (own) {
          nflag += flag;
          nbad += bad;
        }
      }
    }
  };
  for (int t = 0; t < run.nsteps; ++t) {
    if (run.filter) dissipate(U, 1);
    if constexpr (KIND == BLK_LIMIT) dissipate(U, 2);
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int p = 0; p < NSP; ++p) w[p][k] = U[p][k];
    for (int s = 0; s < run.nstage; ++s) {
      if constexpr (KIND == BLK_LIMIT)
        if (s > 0) dissipate(w, 2);
      double f[NSP][NV], uL[NV], uR[NV], fL[NV], fR[NV];
      if (live) {
        elem_traces<NSP, EQ, NV>(w, pb.iJ, ph, f, uL, uR, fL, fR);
#pragma unroll
        for (int k = 0; k < NV; ++k) sUR[k * T + tid] = uR[k];
        if constexpr (EQ == FR_EQ_ADVECTION) sFR[tid] = fR[0];
      }
      __syncthreads();  // the traces are there; every lane has read the last stage's fluxes
      if (live) {
        double ul[NV], fl = 0.0, fs[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) ul[k] = sUR[k * T + lt];
        if constexpr (EQ == FR_EQ_ADVECTION) fl = sFR[lt];
        elem_face<EQ, FLUX, NV>(ul, fl, uL, fL, e == 0, pb.iJ, ph, fs);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          fr_pin(fs[k]);  // rounded before the difference, as the value the right neighbour reads
          sFS[k * T + tid] = fs[k];
          fL[k] = fs[k] - fL[k];
        }
      }
      __syncthreads();  // the fluxes are there; every lane has read the traces
      if (live) {
        const double a0 = run.a0[s], a1 = run.a1[s], b = run.b[s], b2 = run.b2[s];
        const bool last = s == run.nstage - 1;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const double cr = sFS[k * T + rt] - fR[k];
#pragma unroll
          for (int p = 0; p < NSP; ++p) {
            double du = elem_du<NSP, NV>(f, ops, p, k, fL[k], cr);
            if (zero) du = 0.0;
            double v = a1 * w[p][k];
            if constexpr (ACC) {
              v = a0 * (last ? A[p][k] : U[p][k]) + v;
              A[p][k] = (s == 0 ? U[p][k] : A[p][k]) + b2 * du;
            } else {
              if (a0 != 0.0) v = a0 * U[p][k] + v;
            }
            w[p][k] = v + b * du;
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int p = 0; p < NSP; ++p) U[p][k] = w[p][k];
  }
  if (own) {
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int p = 0; p < NSP; ++p) dst[pb.off + e + (long long)n * (p + NSP * k)] = U[p][k];
  }
  if (run.filter || KIND == BLK_LIMIT) {
#pragma unroll
    for (int q = 1; q < 64; q <<= 1) {
      nflag += __shfl_xor(nflag, q);
      nbad += __shfl_xor(nbad, q);
    }
    if ((tid & 63) == 0) {
      if (nflag) atomicAdd(count, nflag);
      if (nbad) atomicAdd(count + 1, nbad);
    }
  }
}

// Three wavefronts per SIMD in the plain form of degrees up to 4.  Roe, us with this bound / none, 512 members,
// SSP-RK3: p = 1 476 / 504, p = 2 574 / 590, p = 3 676 / 701, p = 4, where it spills (93 registers), 766 / 745 and,
// 2000 members of 257 to 600 cells with the filter, 1993 / 1436 (4580 with a launch per stage).  Degrees 5 to
// 8 run at one or two wavefronts per SIMD and are ahead of a launch per stage as well: 1000 cells, SSP-RK3,
// p = 5, 7 and 8 0.23 to 0.24 of its time, 1024 members of 200 to 256 cells, p = 8 with the filter, 0.13.
template <int EQ, int FLUX, int NMAX, int KIND>
__global__ __launch_bounds__(kBlockT, (NMAX <= 5 && KIND == BLK_PLAIN ? 3 : 1)) void fr1d_block_kernel(const Prob1D *__restrict__ probs,
                                                             const Blk1D *__restrict__ blocks,
                                                             const double *__restrict__ ops, Phys1D ph, Run1D run,
                                                             const double *src, double *dst, int *count) {
  constexpr int NV = (EQ == FR_EQ_EULER) ? 3 : 1;
  __shared__ double sh[(2 * NV + 1) * kBlockT];
  const Blk1D bk = blocks[blockIdx.x];
  const Prob1D pb = probs[bk.prob];
  const double *o = ops + OPS_STRIDE * (pb.nsp - 2);
  switch (pb.nsp) {
    case 2: block1d<2, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
    case 3: block1d<3, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
    case 4: block1d<4, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
    case 5: block1d<5, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
    default:
      if constexpr (NMAX > 5) {
        switch (pb.nsp) {
          case 6: block1d<6, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
          case 7: block1d<7, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
          case 8: block1d<8, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
          default: block1d<9, EQ, FLUX, KIND>(pb, bk, o, ph, run, src, dst, count, sh); break;
        }
      }
      break;
  }
}

// dst = src over n values
static __global__ __launch_bounds__(256) void fr1d_copy_kernel(double *__restrict__ dst,
                                                               const double *__restrict__ src, long long n) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += 256LL * gridDim.x) dst[i] = src[i];
}

// ------------------------------------------------------------------ batched problem set
struct Batch1D {
  int eq = FR_EQ_EULER, flux = FR_FLUX_HLL, bc = FR_BC1_DIRICHLET, correction = FR_CORR_RADAU;
  double gamma = 1.4, a = 1.0;
  std::vector<Prob1D> probs;
  int max_nsp = 2;  // largest nsp of the problem set (selects the kernel instance)
  size_t len = 0;
  hipStream_t stream = nullptr;      // the stream every call runs on
  HostStaging staging;
  hipStream_t own_stream = nullptr;  // the context's own non-blocking stream
  Prob1D *d_probs = nullptr;
  double *d_ops = nullptr;
  double *d_u = nullptr, *d_s1 = nullptr, *d_s2 = nullptr, *d_acc = nullptr;
  double *d_k = nullptr;  // Tsit5: the six stage derivatives, len doubles each
  double *d_in = nullptr, *d_out = nullptr;
  int *d_count = nullptr;
  // work lists per thread count (64, 128, 256): concatenated list and per-member sub-lists
  int threads = 256, grid = 0;  // grid 0 = one workgroup per work item
  Work1D *d_work[3] = {nullptr, nullptr, nullptr};
  int nwork[3] = {0, 0, 0};
  std::vector<int> member_first[3], member_count[3];
  // register-resident stepping: the chunk lists of kHaloFull ([0]) and kHaloIdle ([1]) halo
  // elements, on the device one after the other; whole: every member is one chunk
  int path = FR1D_PATH_AUTO;
  Blk1D *d_blocks = nullptr;
  int nblocks[2] = {0, 0};
  bool whole = true;
  int max_cell = 0, num_cu = 0;
  // the last step loop captured by fr_ens_run_graph, replayed while its parameters match
  hipGraphExec_t gexec = nullptr;
  int g_opts = -1, g_nsteps = 0, g_threads = 0, g_grid = -1, g_path = -1;
  double g_dt = 0.0;

  int build(int flux_, int eq_) {
    flux = flux_;
    eq = eq_;
    len = 0;
    for (auto &p : probs) {
      max_nsp = std::max(max_nsp, p.nsp);
      max_cell = std::max(max_cell, p.ncell);
      p.off = (long long)len;
      len += (size_t)p.ncell * p.nsp * (eq == FR_EQ_EULER ? 3 : 1);
    }
    std::vector<double> tab(OPS_STRIDE * (NSP_MAX - 1), 0.0);
    for (int nsp = 2; nsp <= NSP_MAX; ++nsp) {
      HostOps o;
      if (!build_ops(nsp - 1, correction, o)) return fail(FR_E_INVALID, "fr1d: operator construction failed");
      double *t = tab.data() + OPS_STRIDE * (nsp - 2);
      for (int q = 0; q < nsp; ++q) {
        t[q] = o.dhl[q];
        t[NSP_MAX + q] = o.dhr[q];
      }
    }
    FR_HIP(hipMalloc(&d_ops, tab.size() * sizeof(double)));
    FR_HIP(hipMemcpy(d_ops, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
    FR_HIP(hipMalloc(&d_probs, probs.size() * sizeof(Prob1D)));
    FR_HIP(hipMemcpy(d_probs, probs.data(), probs.size() * sizeof(Prob1D), hipMemcpyHostToDevice));
    const int Ts[3] = {64, 128, 256};
    for (int v = 0; v < 3; ++v) {
      const int per = Ts[v] - 2;
      std::vector<Work1D> wl;
      member_first[v].assign(probs.size(), 0);
      member_count[v].assign(probs.size(), 0);
      for (size_t b = 0; b < probs.size(); ++b) {
        member_first[v][b] = (int)wl.size();
        for (int f = 0; f < probs[b].ncell; f += per) wl.push_back(Work1D{(int)b, f});
        member_count[v][b] = (int)wl.size() - member_first[v][b];
      }
      nwork[v] = (int)wl.size();
      FR_HIP(hipMalloc(&d_work[v], wl.size() * sizeof(Work1D)));
      FR_HIP(hipMemcpy(d_work[v], wl.data(), wl.size() * sizeof(Work1D), hipMemcpyHostToDevice));
    }
    whole = max_cell <= kBlockT;
    std::vector<Blk1D> bl;
    for (int v = 0; v < (whole ? 1 : 2); ++v) {
      const int halo = v == 0 ? kHaloFull : kHaloIdle, per = kBlockT - 2 * halo;
      for (size_t b = 0; b < probs.size(); ++b) {
        const int n = probs[b].ncell;
        if (n <= kBlockT)
          bl.push_back(Blk1D{(int)b, 0, n, 0});
        else
          for (int f = 0; f < n; f += per) bl.push_back(Blk1D{(int)b, f, std::min(per, n - f), halo});
      }
      nblocks[v] = (int)bl.size() - (v == 0 ? 0 : nblocks[0]);
    }
    FR_HIP(hipMalloc(&d_blocks, bl.size() * sizeof(Blk1D)));
    FR_HIP(hipMemcpy(d_blocks, bl.data(), bl.size() * sizeof(Blk1D), hipMemcpyHostToDevice));
    int dev = 0;
    FR_HIP(hipGetDevice(&dev));
    FR_HIP(hipDeviceGetAttribute(&num_cu, hipDeviceAttributeMultiprocessorCount, dev));
    FR_HIP(hipStreamCreateWithFlags(&own_stream, hipStreamNonBlocking));
    stream = own_stream;
    FR_HIP(hipMalloc(&d_u, len * sizeof(double)));
    FR_HIP(hipMemset(d_u, 0, len * sizeof(double)));
    return FR_OK;
  }

  void release() {
    if (stream) (void)hipStreamSynchronize(stream);
    staging.release();
    double *bufs[] = {d_ops, d_u, d_s1, d_s2, d_acc, d_k, d_in, d_out};
    for (double *b : bufs)
      if (b) (void)hipFree(b);
    if (d_probs) (void)hipFree(d_probs);
    if (d_count) (void)hipFree(d_count);
    for (auto *w : d_work)
      if (w) (void)hipFree(w);
    if (d_blocks) (void)hipFree(d_blocks);
    if (gexec) (void)hipGraphExecDestroy(gexec);
    if (own_stream) (void)hipStreamDestroy(own_stream);
  }

  static int tindex(int T) { return T == 64 ? 0 : (T == 128 ? 1 : 2); }

  template <int NMAX>
  void launch_eq(const Stage1D &sa, int T, int g, const Work1D *wl, int nw, const Phys1D &ph, hipStream_t st) const {
    if (eq == FR_EQ_ADVECTION)
      hipLaunchKernelGGL((fr1d_kernel<FR_EQ_ADVECTION, FR_FLUX_HLL, NMAX>), dim3(g), dim3(T), 0, st, d_probs, wl, nw,
                         d_ops, ph, sa);
    else if (flux == FR_FLUX_HLL)
      hipLaunchKernelGGL((fr1d_kernel<FR_EQ_EULER, FR_FLUX_HLL, NMAX>), dim3(g), dim3(T), 0, st, d_probs, wl, nw, d_ops,
                         ph, sa);
    else if (flux == FR_FLUX_RUSANOV)
      hipLaunchKernelGGL((fr1d_kernel<FR_EQ_EULER, FR_FLUX_RUSANOV, NMAX>), dim3(g), dim3(T), 0, st, d_probs, wl, nw,
                         d_ops, ph, sa);
    else
      hipLaunchKernelGGL((fr1d_kernel<FR_EQ_EULER, FR_FLUX_ROE, NMAX>), dim3(g), dim3(T), 0, st, d_probs, wl, nw, d_ops,
                         ph, sa);
  }

  // one launch over work items [w0, w0 + nw) of the list for T threads
  int launch(const Stage1D &sa, int T, int grid_, int w0, int nw, hipStream_t st) const {
    const int v = tindex(T);
    Phys1D ph{eq, bc, gamma, gamma - 1.0, a};
    const Work1D *wl = d_work[v] + w0;
    const int g = grid_ > 0 ? std::min(grid_, nw) : nw;
    if (nw <= 0) return FR_OK;
    if (max_nsp <= 5)
      launch_eq<5>(sa, T, g, wl, nw, ph, st);
    else
      launch_eq<NSP_MAX>(sa, T, g, wl, nw, ph, st);
    FR_LAUNCHED("fr1d_kernel");
    return FR_OK;
  }

  // batched (mode 0): whole work list in one launch; looped (mode 1): one launch per member
  int stage(const Stage1D &sa, int mode, hipStream_t st) const {
    const int v = tindex(threads);
    if (mode == 0) return launch(sa, threads, grid, 0, nwork[v], st);
    for (size_t b = 0; b < probs.size(); ++b) {
      int rc = launch(sa, threads, 0, member_first[v][b], member_count[v][b], st);
      if (rc) return rc;
    }
    return FR_OK;
  }

  int ensure_stage_buffers(bool acc, bool tsit = false) {
    if (!d_s1) FR_HIP(hipMalloc(&d_s1, len * sizeof(double)));
    if (!d_s2) FR_HIP(hipMalloc(&d_s2, len * sizeof(double)));
    if (acc && !d_acc) FR_HIP(hipMalloc(&d_acc, len * sizeof(double)));
    if (tsit && !d_k) FR_HIP(hipMalloc(&d_k, 6 * len * sizeof(double)));
    return FR_OK;
  }

  // out = u + dt * sum_{j < nk} row[j] k_{j+1} over the whole state
  int tsit5_comb(double *out, const double *u, const double *row, int nk, double dt, hipStream_t st) const {
    FR_HIP(fr::tsit5_comb(out, u, d_k, len, row, nk, dt, len, st));
    return FR_OK;
  }

  // Per-cell dissipation pass over every member (mode 0: one launch; 1: one launch per member):
  // dmode 1 sensor + filter with the filter time step dt, 2 positivity limiter.  count[0] += cells
  // flagged / limited, count[1] += cells whose mean density is not positive (left unchanged).
  int diss_launch(double *u, int dmode, double dt, int mode, hipStream_t st) const {
    const int v = tindex(threads);
    auto one = [&](int w0, int nw, int grid_) {
      if (nw <= 0) return;
      const int g = grid_ > 0 ? std::min(grid_, nw) : nw;
      if (max_nsp <= 5)
        hipLaunchKernelGGL(fr1d_diss_kernel<5>, dim3(g), dim3(threads), 0, st, d_probs, d_work[v] + w0, nw, u,
                           dmode, gamma, dt, d_count);
      else
        hipLaunchKernelGGL(fr1d_diss_kernel<NSP_MAX>, dim3(g), dim3(threads), 0, st, d_probs, d_work[v] + w0, nw, u,
                           dmode, gamma, dt, d_count);
    };
    if (mode == 0) {
      one(0, nwork[v], grid);
    } else {
      for (size_t b = 0; b < probs.size(); ++b) one(member_first[v][b], member_count[v][b], 0);
    }
    FR_LAUNCHED("fr1d_diss_kernel");
    return FR_OK;
  }

  // opts (SSP-RK3 and Midpoint): FR_ENS_FILTER runs the sensor + filter on the state before every
  // step (example/euler_highlevel.jl:37-54), FR_ENS_LIMIT the positivity limiter on the input of
  // every stage (the state before the step and the intermediate stage results)
  int enqueue_steps(int scheme, int mode, double dt, int nsteps, hipStream_t st, int opts = 0) {
    double *U = d_u, *S1 = d_s1, *S2 = d_s2, *A = d_acc;
    auto stg = [&](const double *u0, const double *us, double *out, double a0, double a1, double b,
                   const double *ai, double *ao, double b2) {
      return stage(Stage1D{us, out, u0, ai, ao, a0, a1, b, b2, 0}, mode, st);
    };
    auto dis = [&](double *u, int dmode, double ddt) { return diss_launch(u, dmode, ddt, mode, st); };
    const bool filt = (opts & FR_ENS_FILTER) != 0, lim = (opts & FR_ENS_LIMIT) != 0;
    for (int n = 0; n < nsteps; ++n) {
      int rc = FR_OK;
      switch (scheme) {
        case FR_RK_SSPRK3: {
          // consecutive steps alternate the state between U and S1 (every stage writes every
          // cell), so the last stage never writes the u^n it reads; the call's last step writes U
          double *const X = (n & 1) ? S1 : U, *const Y = (n & 1) ? U : S1;
          double *const out = n == nsteps - 1 ? U : Y;
          if (filt && (rc = dis(X, 1, dt))) return rc;
          if (lim && (rc = dis(X, 2, 0.0))) return rc;
          if ((rc = stg(X, X, Y, 0.0, 1.0, dt, nullptr, nullptr, 0.0))) return rc;
          if (lim && (rc = dis(Y, 2, 0.0))) return rc;
          if ((rc = stg(X, Y, S2, 0.75, 0.25, 0.25 * dt, nullptr, nullptr, 0.0))) return rc;
          if (lim && (rc = dis(S2, 2, 0.0))) return rc;
          if ((rc = stg(X, S2, out, 1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0 * dt, nullptr, nullptr, 0.0))) return rc;
          break;
        }
        case FR_RK_RK4:
          if ((rc = stg(U, U, S2, 1.0, 0.0, 0.5 * dt, U, A, dt / 6.0))) return rc;
          if ((rc = stg(U, S2, S1, 1.0, 0.0, 0.5 * dt, A, A, dt / 3.0))) return rc;
          if ((rc = stg(U, S1, S2, 1.0, 0.0, dt, A, A, dt / 3.0))) return rc;
          if ((rc = stg(A, S2, U, 1.0, 0.0, dt / 6.0, nullptr, nullptr, 0.0))) return rc;
          break;
        case FR_RK_MIDPOINT: {
          // consecutive steps alternate the state between U and S2; the call's last step writes U
          double *const X = (n & 1) ? S2 : U;
          double *const out = n == nsteps - 1 ? U : ((n & 1) ? U : S2);
          if (filt && (rc = dis(X, 1, dt))) return rc;
          if (lim && (rc = dis(X, 2, 0.0))) return rc;
          if ((rc = stg(X, X, S1, 0.0, 1.0, 0.5 * dt, nullptr, nullptr, 0.0))) return rc;
          if (lim && (rc = dis(S1, 2, 0.0))) return rc;
          if ((rc = stg(X, S1, out, 1.0, 0.0, dt, nullptr, nullptr, 0.0))) return rc;
          break;
        }
        case FR_RK_EULER: {
          // consecutive steps alternate the state between U and S1; a call that ends in S1
          // copies it back once
          double *const X = (n & 1) ? S1 : U, *const Y = (n & 1) ? U : S1;
          if ((rc = stg(X, X, Y, 0.0, 1.0, dt, nullptr, nullptr, 0.0))) return rc;
          if (n == nsteps - 1 && Y != U)
            FR_HIP(hipMemcpyAsync(U, Y, len * sizeof(double), hipMemcpyDeviceToDevice, st));
          break;
        }
        case FR_RK_TSIT5: {
          // k_s = L(Y_s) (residual launch), Y_1 = U, Y_{s+1} = U + dt sum_j a_{s+1,j} k_j, and
          // U <- U + dt sum_j b_j k_j (the last combination, in place)
          for (int sg = 0; sg < 6; ++sg) {
            Stage1D r{};
            r.u = sg == 0 ? U : S1;
            r.out = d_k + (size_t)sg * len;
            r.residual = 1;
            if ((rc = stage(r, mode, st))) return rc;
            if ((rc = tsit5_comb(sg == 5 ? U : S1, U, kTsit5[sg], sg + 1, dt, st))) return rc;
          }
          break;
        }
        default:
          return fail(FR_E_INVALID, "fr1d_step: unknown scheme");
      }
    }
    return FR_OK;
  }

  // Register-resident stepping serves every set of problems: FR1D_PATH_MEMBER and FR1D_PATH_AUTO.
  // FR1D_PATH_BATCHED, Tsit5 and the per-member launch mode take a launch per stage.
  bool use_blocks(int scheme, int mode) const {
    return scheme != FR_RK_TSIT5 && mode == 0 && path != FR1D_PATH_BATCHED;
  }

  // the path as reported: a problem set of at most kMemberCells cells per member counts as stepped
  // member by member, a larger one as batched chunks
  static constexpr int kMemberCells = 508;
  int reported_path(int scheme) const {
    if (!use_blocks(scheme, 0)) return FR1D_PATH_BATCHED;
    return path == FR1D_PATH_MEMBER || max_cell <= kMemberCells ? FR1D_PATH_MEMBER : FR1D_PATH_BATCHED;
  }

  template <int NMAX, int KIND>
  void launch_block_eq(const Phys1D &ph, const Run1D &run, const Blk1D *bl, int nb, int T, const double *src,
                       double *dst, hipStream_t st) const {
    const dim3 g((unsigned)nb), b((unsigned)T);
    if (eq == FR_EQ_ADVECTION)
      hipLaunchKernelGGL((fr1d_block_kernel<FR_EQ_ADVECTION, FR_FLUX_HLL, NMAX, KIND == BLK_RK4 ? BLK_RK4 : BLK_PLAIN>),
                         g, b, 0, st, d_probs, bl, d_ops, ph, run, src, dst, d_count);
    else if (flux == FR_FLUX_HLL)
      hipLaunchKernelGGL((fr1d_block_kernel<FR_EQ_EULER, FR_FLUX_HLL, NMAX, KIND>), g, b, 0, st, d_probs, bl, d_ops, ph,
                         run, src, dst, d_count);
    else if (flux == FR_FLUX_RUSANOV)
      hipLaunchKernelGGL((fr1d_block_kernel<FR_EQ_EULER, FR_FLUX_RUSANOV, NMAX, KIND>), g, b, 0, st, d_probs, bl, d_ops,
                         ph, run, src, dst, d_count);
    else
      hipLaunchKernelGGL((fr1d_block_kernel<FR_EQ_EULER, FR_FLUX_ROE, NMAX, KIND>), g, b, 0, st, d_probs, bl, d_ops, ph,
                         run, src, dst, d_count);
  }

  template <int NMAX>
  void launch_block(int kind, const Phys1D &ph, const Run1D &run, const Blk1D *bl, int nb, int T, const double *src,
                    double *dst, hipStream_t st) const {
    if (kind == BLK_RK4)
      launch_block_eq<NMAX, BLK_RK4>(ph, run, bl, nb, T, src, dst, st);
    else if (kind == BLK_LIMIT)
      launch_block_eq<NMAX, BLK_LIMIT>(ph, run, bl, nb, T, src, dst, st);
    else
      launch_block_eq<NMAX, BLK_PLAIN>(ph, run, bl, nb, T, src, dst, st);
  }

  // nsteps steps in launches of fr1d_block_kernel, from d_u to d_u through the stage buffers
  int block_steps(int scheme, double dt, int nsteps, hipStream_t st, int opts) const {
    Run1D run{};
    auto set = [&](int s, double a0, double a1, double b, double b2) {
      run.nstage = s + 1;
      run.a0[s] = a0, run.a1[s] = a1, run.b[s] = b, run.b2[s] = b2;
    };
    switch (scheme) {
      case FR_RK_SSPRK3:
        set(0, 0.0, 1.0, dt, 0.0);
        set(1, 0.75, 0.25, 0.25 * dt, 0.0);
        set(2, 1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0 * dt, 0.0);
        break;
      case FR_RK_RK4:
        set(0, 1.0, 0.0, 0.5 * dt, dt / 6.0);
        set(1, 1.0, 0.0, 0.5 * dt, dt / 3.0);
        set(2, 1.0, 0.0, dt, dt / 3.0);
        set(3, 1.0, 0.0, dt / 6.0, 0.0);
        break;
      case FR_RK_MIDPOINT:
        set(0, 0.0, 1.0, 0.5 * dt, 0.0);
        set(1, 1.0, 0.0, dt, 0.0);
        break;
      case FR_RK_EULER:
        set(0, 0.0, 1.0, dt, 0.0);
        break;
      default:
        return fail(FR_E_INVALID, "fr1d_step: unknown scheme");
    }
    run.filter = (opts & FR_ENS_FILTER) != 0;
    // RK4 steps take no options (fr1d_step passes none, the ensemble loops step with SSP-RK3 or Midpoint)
    const int kind = scheme == FR_RK_RK4 ? BLK_RK4 : (opts & FR_ENS_LIMIT) ? BLK_LIMIT : BLK_PLAIN;
    run.fdt = dt;
    const Phys1D ph{eq, bc, gamma, gamma - 1.0, a};
    const int v = !whole && nblocks[1] <= num_cu ? 1 : 0;
    const Blk1D *bl = d_blocks + (v ? nblocks[0] : 0);
    const int T = whole ? (max_cell + 63) / 64 * 64 : kBlockT;
    const int most = whole ? kBlockSteps : (v ? kHaloIdle : kHaloFull) / run.nstage;
    // chunks with halos read one buffer and write another, the last launch d_u: at least two launches
    // (a single step: a launch into d_s1 and a copy)
    int launches = (nsteps + most - 1) / most;
    if (!whole && launches == 1 && nsteps > 1) launches = 2;
    const double *from = d_u;
    for (int q = 0; q < launches; ++q) {
      run.nsteps = nsteps / launches + (q < nsteps % launches ? 1 : 0);
      double *to = whole || (q == launches - 1 && launches > 1) ? d_u : (from == d_s1 ? d_s2 : d_s1);
      const int nb = nblocks[v];
      if (max_nsp <= 5)
        launch_block<5>(kind, ph, run, bl, nb, T, from, to, st);
      else
        launch_block<NSP_MAX>(kind, ph, run, bl, nb, T, from, to, st);
      FR_LAUNCHED("fr1d_block_kernel");
      from = to;
    }
    if (from != d_u) {
      const long long blocks = std::min<long long>(((long long)len + 255) / 256, 4096);
      hipLaunchKernelGGL(fr1d_copy_kernel, dim3((unsigned)blocks), dim3(256), 0, st, d_u, from, (long long)len);
      FR_LAUNCHED("fr1d_copy_kernel");
    }
    return FR_OK;
  }

  // the steps on the path use_blocks selects
  int run_steps(int scheme, int mode, double dt, int nsteps, hipStream_t st, int opts = 0) {
    if (use_blocks(scheme, mode)) return block_steps(scheme, dt, nsteps, st, opts);
    return enqueue_steps(scheme, mode, dt, nsteps, st, opts);
  }

  // mode 1 sensor + filter, 2 positivity; n_out (optional) receives the two counters
  int dissipation(int mode, double dt, int *n_out) {
    if (!d_count) FR_HIP(hipMalloc(&d_count, 2 * sizeof(int)));
    FR_HIP(hipMemsetAsync(d_count, 0, 2 * sizeof(int), stream));
    int rc = diss_launch(d_u, mode, dt, 0, stream);
    if (rc) return rc;
    int h[2] = {0, 0};
    FR_HIP(hipMemcpyAsync(h, d_count, 2 * sizeof(int), hipMemcpyDeviceToHost, stream));
    FR_HIP(hipStreamSynchronize(stream));
    if (n_out) {
      n_out[0] = h[0];
      n_out[1] = h[1];
    }
    if (mode == 2 && h[1] > 0)
      return fail(FR_E_LIMITER, "fr1d_positivity: " + std::to_string(h[1]) + " cell(s) with non-positive mean density");
    return FR_OK;
  }

  int residual(const double *d_u_, double *d_du_, hipStream_t st) const {
    Stage1D s{};
    s.u = d_u_;
    s.out = d_du_;
    s.residual = 1;
    return stage(s, 0, st);
  }
};

}  // namespace fr

using namespace fr;

static double member_cut(int deg) { return shock_cut(-3.0 * std::log10((double)deg), kKappa1D); }

struct fr1d_ctx : Batch1D {};
struct fr_ens_ctx : Batch1D {};

extern "C" {

int fr1d_create(fr1d_ctx **out, const fr1d_desc *d) {
  FR_REQUIRE(out && d, FR_E_INVALID, "fr1d_create: null argument");
  *out = nullptr;
  FR_REQUIRE(d->equation == FR_EQ_EULER || d->equation == FR_EQ_ADVECTION, FR_E_INVALID, "fr1d_create: unknown equation");
  FR_REQUIRE(d->ncell >= 2, FR_E_INVALID, "fr1d_create: ncell must be >= 2");
  FR_REQUIRE(d->deg >= 1 && d->deg <= NSP_MAX - 1, FR_E_UNSUPPORTED, "fr1d_create: degree must be in 1..8");
  FR_REQUIRE(d->dx > 0.0 && std::isfinite(d->dx), FR_E_INVALID, "fr1d_create: dx must be > 0");
  FR_REQUIRE(d->bc == FR_BC1_DIRICHLET || d->bc == FR_BC1_PERIOD, FR_E_INVALID, "fr1d_create: unknown bc");
  FR_REQUIRE(d->correction >= FR_CORR_RADAU && d->correction <= FR_CORR_HUYNH, FR_E_INVALID, "fr1d_create: unknown correction");
  FR_REQUIRE(d->flux >= FR_FLUX_HLL && d->flux <= FR_FLUX_ROE, FR_E_INVALID, "fr1d_create: unknown flux");
  FR_REQUIRE(d->equation == FR_EQ_ADVECTION || d->gamma > 1.0, FR_E_INVALID, "fr1d_create: gamma must be > 1");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(FR_E_HIP, "fr1d_create: no HIP device visible");
  fr1d_ctx *c = new (std::nothrow) fr1d_ctx();
  FR_REQUIRE(c, FR_E_NOMEM, "fr1d_create: out of host memory");
  c->bc = d->bc;
  c->gamma = d->gamma;
  c->a = d->a;
  c->correction = d->correction;
  int rc = no_throw("fr1d_create", [&] {
    c->probs.push_back(Prob1D{0, d->ncell, d->deg + 1, 2.0 / d->dx, member_cut(d->deg)});
    return c->build(d->flux, d->equation);
  });
  if (rc) {
    c->release();
    delete c;
    return rc;
  }
  *out = c;
  return FR_OK;
}

int fr1d_destroy(fr1d_ctx *c) {
  if (!c) return FR_OK;
  c->release();
  delete c;
  return FR_OK;
}

size_t fr1d_state_len(const fr1d_ctx *c) { return c ? c->len : 0; }

int fr1d_set_stream(fr1d_ctx *c, void *s) {
  FR_REQUIRE(c, FR_E_INVALID, "fr1d_set_stream: null context");
  c->stream = s == FR_OWN_STREAM ? c->own_stream : (hipStream_t)s;
  return FR_OK;
}

int fr1d_rhs_dev(fr1d_ctx *c, const double *d_u, double *d_du, double t) {
  (void)t;
  FR_REQUIRE(c && d_u && d_du && d_u != d_du, FR_E_INVALID, "fr1d_rhs_dev: bad arguments");
  return c->residual(d_u, d_du, c->stream);
}

int fr1d_rhs(fr1d_ctx *c, const double *u, double *du, double t) {
  (void)t;
  FR_REQUIRE(c && u && du, FR_E_INVALID, "fr1d_rhs: null argument");
  const size_t bytes = c->len * sizeof(double);
  if (!c->d_in) FR_HIP(hipMalloc(&c->d_in, bytes));
  if (!c->d_out) FR_HIP(hipMalloc(&c->d_out, bytes));
  FR_HIP(hipMemcpyAsync(c->d_in, u, bytes, hipMemcpyHostToDevice, c->stream));
  int rc = c->residual(c->d_in, c->d_out, c->stream);
  if (rc) return rc;
  FR_HIP(hipMemcpyAsync(du, c->d_out, bytes, hipMemcpyDeviceToHost, c->stream));
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

int fr1d_set_state(fr1d_ctx *c, const double *u) {
  FR_REQUIRE(c && u, FR_E_INVALID, "fr1d_set_state: null argument");
  return copy_to_device(c->staging, c->d_u, u, c->len, c->stream);
}

int fr1d_get_state(fr1d_ctx *c, double *u) {
  FR_REQUIRE(c && u, FR_E_INVALID, "fr1d_get_state: null argument");
  return copy_to_host(c->staging, u, c->d_u, c->len, c->stream);
}

int fr1d_step(fr1d_ctx *c, int scheme, double dt, int nsteps) {
  FR_REQUIRE(c && nsteps >= 0 && std::isfinite(dt), FR_E_INVALID, "fr1d_step: bad arguments");
  FR_REQUIRE(scheme >= FR_RK_SSPRK3 && scheme <= FR_RK_TSIT5, FR_E_INVALID, "fr1d_step: unknown scheme");
  int rc = c->ensure_stage_buffers(scheme == FR_RK_RK4, scheme == FR_RK_TSIT5);
  if (rc) return rc;
  return c->run_steps(scheme, 0, dt, nsteps, c->stream);
}

int fr1d_set_path(fr1d_ctx *c, int path) {
  FR_REQUIRE(c, FR_E_INVALID, "fr1d_set_path: null context");
  FR_REQUIRE(path >= FR1D_PATH_AUTO && path <= FR1D_PATH_MEMBER, FR_E_INVALID,
             "fr1d_set_path: path must be FR1D_PATH_AUTO, _BATCHED or _MEMBER");
  c->path = path;
  return FR_OK;
}

int fr1d_get_path(const fr1d_ctx *c, int scheme, int *path) {
  FR_REQUIRE(c && path, FR_E_INVALID, "fr1d_get_path: null argument");
  *path = c->reported_path(scheme);
  return FR_OK;
}

// ------------------------------------------------------------------ ensembles
int fr_ens_create(fr_ens_ctx **out, int nprob, const int *ncell, const int *deg, const double *dx, double gamma,
                  int flux, int bc) {
  FR_REQUIRE(out && ncell && deg && dx && nprob >= 1, FR_E_INVALID, "fr_ens_create: bad arguments");
  *out = nullptr;
  FR_REQUIRE(gamma > 1.0, FR_E_INVALID, "fr_ens_create: gamma must be > 1");
  FR_REQUIRE(flux >= FR_FLUX_HLL && flux <= FR_FLUX_ROE, FR_E_INVALID, "fr_ens_create: unknown flux");
  FR_REQUIRE(bc == FR_BC1_DIRICHLET || bc == FR_BC1_PERIOD, FR_E_INVALID, "fr_ens_create: unknown bc");
  for (int b = 0; b < nprob; ++b) {
    FR_REQUIRE(ncell[b] >= 2, FR_E_INVALID, "fr_ens_create: every member needs ncell >= 2");
    FR_REQUIRE(deg[b] >= 1 && deg[b] <= NSP_MAX - 1, FR_E_UNSUPPORTED, "fr_ens_create: member degree must be in 1..8");
    FR_REQUIRE(dx[b] > 0.0, FR_E_INVALID, "fr_ens_create: member dx must be > 0");
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(FR_E_HIP, "fr_ens_create: no HIP device visible");
  fr_ens_ctx *c = new (std::nothrow) fr_ens_ctx();
  FR_REQUIRE(c, FR_E_NOMEM, "fr_ens_create: out of host memory");
  c->bc = bc;
  c->gamma = gamma;
  int rc = no_throw("fr_ens_create", [&] {
    for (int b = 0; b < nprob; ++b)
      c->probs.push_back(Prob1D{0, ncell[b], deg[b] + 1, 2.0 / dx[b], member_cut(deg[b])});
    return c->build(flux, FR_EQ_EULER);
  });
  if (rc) {
    c->release();
    delete c;
    return rc;
  }
  *out = c;
  return FR_OK;
}

int fr_ens_destroy(fr_ens_ctx *c) {
  if (!c) return FR_OK;
  c->release();
  delete c;
  return FR_OK;
}

size_t fr_ens_state_len(const fr_ens_ctx *c) { return c ? c->len : 0; }

size_t fr_ens_offset(const fr_ens_ctx *c, int member) {
  if (!c || member < 0 || member >= (int)c->probs.size()) return (size_t)-1;
  return (size_t)c->probs[member].off;
}

int fr_ens_set_state(fr_ens_ctx *c, const double *u) {
  FR_REQUIRE(c && u, FR_E_INVALID, "fr_ens_set_state: null argument");
  return copy_to_device(c->staging, c->d_u, u, c->len, c->stream);
}

int fr_ens_get_state(fr_ens_ctx *c, double *u) {
  FR_REQUIRE(c && u, FR_E_INVALID, "fr_ens_get_state: null argument");
  return copy_to_host(c->staging, u, c->d_u, c->len, c->stream);
}

int fr_ens_step(fr_ens_ctx *c, int mode, double dt, int nsteps) {
  FR_REQUIRE(c && (mode == 0 || mode == 1) && nsteps >= 0 && std::isfinite(dt), FR_E_INVALID,
             "fr_ens_step: bad arguments");
  int rc = c->ensure_stage_buffers(false);
  if (rc) return rc;
  rc = c->run_steps(FR_RK_SSPRK3, mode, dt, nsteps, c->stream);
  if (rc) return rc;
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

int fr_ens_set_path(fr_ens_ctx *c, int path) {
  FR_REQUIRE(c, FR_E_INVALID, "fr_ens_set_path: null context");
  FR_REQUIRE(path >= FR1D_PATH_AUTO && path <= FR1D_PATH_MEMBER, FR_E_INVALID,
             "fr_ens_set_path: path must be FR1D_PATH_AUTO, _BATCHED or _MEMBER");
  c->path = path;
  return FR_OK;
}

// counters of the loop entry points: zeroed before the loop, read after it
static int ens_read_counts(fr_ens_ctx *c, const char *who, int *n_flagged, int *n_limited) {
  int h[2] = {0, 0};
  FR_HIP(hipMemcpyAsync(h, c->d_count, 2 * sizeof(int), hipMemcpyDeviceToHost, c->stream));
  FR_HIP(hipStreamSynchronize(c->stream));
  if (n_flagged) *n_flagged = h[0];
  if (n_limited) *n_limited = h[1];
  if (h[1] > 0)
    return fail(FR_E_LIMITER, std::string(who) + ": " + std::to_string(h[1]) +
                                  " limiter failure(s) (cell mean density not positive) over the loop");
  return FR_OK;
}

int fr_ens_run(fr_ens_ctx *c, int mode, int opts, double dt, int nsteps, int *n_flagged, int *n_limited) {
  FR_REQUIRE(c && (mode == 0 || mode == 1) && nsteps >= 0 && std::isfinite(dt) && dt >= 0.0, FR_E_INVALID,
             "fr_ens_run: bad arguments");
  FR_REQUIRE((opts & ~(FR_ENS_FILTER | FR_ENS_LIMIT | FR_ENS_MIDPOINT)) == 0, FR_E_INVALID,
             "fr_ens_run: unknown option bits");
  int rc = c->ensure_stage_buffers(false);
  if (rc) return rc;
  if (!c->d_count) FR_HIP(hipMalloc(&c->d_count, 2 * sizeof(int)));
  FR_HIP(hipMemsetAsync(c->d_count, 0, 2 * sizeof(int), c->stream));
  const int scheme = (opts & FR_ENS_MIDPOINT) ? FR_RK_MIDPOINT : FR_RK_SSPRK3;
  if ((rc = c->run_steps(scheme, mode, dt, nsteps, c->stream, opts))) return rc;
  return ens_read_counts(c, "fr_ens_run", n_flagged, n_limited);
}

int fr_ens_run_graph(fr_ens_ctx *c, int opts, double dt, int nsteps, int nrep, int *n_flagged, int *n_limited) {
  FR_REQUIRE(c && nsteps >= 1 && nrep >= 0 && std::isfinite(dt) && dt >= 0.0, FR_E_INVALID,
             "fr_ens_run_graph: bad arguments");
  FR_REQUIRE((opts & ~(FR_ENS_FILTER | FR_ENS_LIMIT | FR_ENS_MIDPOINT)) == 0, FR_E_INVALID,
             "fr_ens_run_graph: unknown option bits");
  int rc = c->ensure_stage_buffers(false);
  if (rc) return rc;
  if (!c->d_count) FR_HIP(hipMalloc(&c->d_count, 2 * sizeof(int)));
  // The graph holds the context's own buffers and work lists, which never move once allocated, so a
  // capture stays valid while the options, dt, the step count, the path and, where a launch per stage is
  // captured, the work mapping are unchanged.
  const int scheme = (opts & FR_ENS_MIDPOINT) ? FR_RK_MIDPOINT : FR_RK_SSPRK3;
  const bool same_map = c->use_blocks(scheme, 0) || (c->g_threads == c->threads && c->g_grid == c->grid);
  if (!(c->gexec && c->g_opts == opts && c->g_dt == dt && c->g_nsteps == nsteps && same_map && c->g_path == c->path)) {
    if (c->gexec) {
      FR_HIP(hipStreamSynchronize(c->stream));
      (void)hipGraphExecDestroy(c->gexec);
      c->gexec = nullptr;
    }
    hipGraph_t graph = nullptr;
    FR_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    rc = c->run_steps(scheme, 0, dt, nsteps, c->stream, opts);
    hipError_t e = hipStreamEndCapture(c->stream, &graph);
    if (rc) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    FR_HIP(e);
    e = hipGraphInstantiate(&c->gexec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
      c->gexec = nullptr;
      return hip_fail(e, "hipGraphInstantiate", __FILE__, __LINE__);
    }
    c->g_opts = opts;
    c->g_dt = dt;
    c->g_nsteps = nsteps;
    c->g_threads = c->threads;
    c->g_grid = c->grid;
    c->g_path = c->path;
  }
  // the counters are cleared outside the graph (no memset node is recorded into it)
  FR_HIP(hipMemsetAsync(c->d_count, 0, 2 * sizeof(int), c->stream));
  for (int r = 0; r < nrep; ++r) FR_HIP(hipGraphLaunch(c->gexec, c->stream));
  return ens_read_counts(c, "fr_ens_run_graph", n_flagged, n_limited);
}

int fr_ens_step_graph(fr_ens_ctx *c, double dt, int nsteps, int nrep) {
  FR_REQUIRE(c && nsteps >= 1 && nrep >= 0 && std::isfinite(dt), FR_E_INVALID, "fr_ens_step_graph: bad arguments");
  return fr_ens_run_graph(c, 0, dt, nsteps, nrep, nullptr, nullptr);
}

// Times candidate (threads per workgroup, grid) mappings of the launches per stage with HIP events over a
// few SSP-RK3 steps on a scratch copy of the state, keeps the fastest, and restores the state.
int fr_ens_autotune(fr_ens_ctx *c, double dt, int *chosen) {
  FR_REQUIRE(c && std::isfinite(dt), FR_E_INVALID, "fr_ens_autotune: bad arguments");
  int rc = c->ensure_stage_buffers(false);
  if (rc) return rc;
  int ndev = 0, dev = 0, ncu = 256;
  (void)ndev;
  FR_HIP(hipGetDevice(&dev));
  FR_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  double *save = nullptr;
  FR_HIP(hipMalloc(&save, c->len * sizeof(double)));
  FR_HIP(hipMemcpyAsync(save, c->d_u, c->len * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  const int Ts[3] = {64, 128, 256};
  const int mult[5] = {0, 1, 2, 4, 8};  // 0: one workgroup per work item
  hipEvent_t e0, e1;
  FR_HIP(hipEventCreate(&e0));
  FR_HIP(hipEventCreate(&e1));
  float best = 1e30f;
  int best_i = 0, idx = 0;
  const int keepT = c->threads, keepG = c->grid;
  for (int ti = 0; ti < 3; ++ti)
    for (int mi = 0; mi < 5; ++mi, ++idx) {
      c->threads = Ts[ti];
      c->grid = mult[mi] * ncu;
      rc = c->enqueue_steps(FR_RK_SSPRK3, 0, dt, 1, c->stream);  // warm-up
      if (rc) break;
      FR_HIP(hipEventRecord(e0, c->stream));
      rc = c->enqueue_steps(FR_RK_SSPRK3, 0, dt, 3, c->stream);
      if (rc) break;
      FR_HIP(hipEventRecord(e1, c->stream));
      FR_HIP(hipEventSynchronize(e1));
      float ms = 0.f;
      FR_HIP(hipEventElapsedTime(&ms, e0, e1));
      if (ms < best) {
        best = ms;
        best_i = idx;
      }
      FR_HIP(hipMemcpyAsync(c->d_u, save, c->len * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  FR_HIP(hipStreamSynchronize(c->stream));
  (void)hipFree(save);
  if (rc) {
    c->threads = keepT;
    c->grid = keepG;
    return rc;
  }
  c->threads = Ts[best_i / 5];
  c->grid = mult[best_i % 5] * ncu;
  if (chosen) *chosen = best_i;
  return FR_OK;
}

int fr1d_sensor_filter(fr1d_ctx *c, double dt, int *n_flagged) {
  FR_REQUIRE(c && std::isfinite(dt) && dt >= 0.0, FR_E_INVALID, "fr1d_sensor_filter: bad arguments");
  FR_REQUIRE(c->eq == FR_EQ_EULER, FR_E_UNSUPPORTED, "fr1d_sensor_filter: Euler states only");
  int h[2];
  int rc = c->dissipation(1, dt, h);
  if (n_flagged) *n_flagged = h[0];
  return rc;
}

int fr1d_positivity(fr1d_ctx *c, int *n_limited) {
  FR_REQUIRE(c, FR_E_INVALID, "fr1d_positivity: null context");
  FR_REQUIRE(c->eq == FR_EQ_EULER, FR_E_UNSUPPORTED, "fr1d_positivity: Euler states only");
  int h[2] = {0, 0};
  int rc = c->dissipation(2, 0.0, h);
  if (n_limited) *n_limited = h[0];
  return rc;
}

int fr_ens_sensor_filter(fr_ens_ctx *c, double dt, int *n_flagged) {
  FR_REQUIRE(c && std::isfinite(dt) && dt >= 0.0, FR_E_INVALID, "fr_ens_sensor_filter: bad arguments");
  int h[2];
  int rc = c->dissipation(1, dt, h);
  if (n_flagged) *n_flagged = h[0];
  return rc;
}

int fr_ens_positivity(fr_ens_ctx *c, int *n_limited) {
  FR_REQUIRE(c, FR_E_INVALID, "fr_ens_positivity: null context");
  int h[2] = {0, 0};
  int rc = c->dissipation(2, 0.0, h);
  if (n_limited) *n_limited = h[0];
  return rc;
}

}  // extern "C"
