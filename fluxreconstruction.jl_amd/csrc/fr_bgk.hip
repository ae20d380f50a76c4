// fr_bgk.hip -- 2D discrete-velocity BGK flux reconstruction on periodic uniform quads, and
// batched ensembles of such problems that differ in the relaxation time, for gfx950.
//
// Tensorises example/bgk_wave.jl:69-129: per solution point the conserved moments over the
// velocity grid give the Maxwellian (KitBase moments_conserve / conserve_prim / maxwellian in 2D);
// every discrete velocity is advected by FR with the upwind (Heaviside-blended) interface flux and
// relaxes to the Maxwellian, du = -(div f + corrections) + (M - f) / tau.
//
// State f(i, j, k, l, a, b, member), column-major: the cell index is fastest, so a wavefront of
// consecutive cells reads contiguous memory for a fixed (point, velocity).  Two paths:
// - states that the caches serve, members of few cells, and points beyond what the other path's offsets and
//   launches reach (BgkCtx::large): moments (one thread per solution point, loop over the velocities, FP64 sums; it
//   also writes the separable Maxwellian factors of the point), then transport + relaxation + RK stage (one workgroup per (member, velocity, 16 x 16 cell tile), one thread per cell; the upwind
//   traces of the neighbours come from LDS or from the halo threads);
// - larger states: a stage kernel that walks a tile through a range of velocities and leaves partial
//   velocity sums of its result, and a closure that adds them per point and writes the factors, so no
//   stage reads the state a second time for its moments.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <type_traits>
#include <utility>
#include <vector>

#include "fr_common.h"

namespace fr {

constexpr int BT = 16;  // tile edge in cells (BT x BT threads)

template <int NSP>
struct BgkTileOps {
  double ll[NSP], lr[NSP], dl[NSP * NSP], dhl[NSP], dhr[NSP];
};

struct BgkGeo {
  int nx, ny, nu, nv, nmem;
  int per, ngrp;      // velocities per group, groups
  int tsh;            // log2 of the tile's width
  long long cells;    // nx * ny
  long long npts;     // nx * ny * nsp^2 (one velocity plane)
  long long mstride;  // doubles per member
  double iJx, iJy, gamma;
};

struct BgkStage {
  const double *u, *u0;
  double *out;
  double a0, a1, b;
  int residual;
};

// moments cons[member][c][pt] (rho, rho U, rho V, E) of every solution point, and the separable
// Maxwellian M(a, b) = Ea[a] * Eb[b] of every point: Ea[member][a][pt] = exp(-lambda (u_a - U)^2),
// Eb[member][b][pt] = rho lambda / pi exp(-lambda (v_b - V)^2), so that the transport kernel spends
// one multiplication per value on it.  A wavefront takes 64 consecutive points (the lanes); nq
// wavefronts of the workgroup share a point group and split its velocity rows b between them (nq
// > 1 when the points alone give the chip too few wavefronts).  The partial sums are combined in
// LDS in a fixed order, and each wavefront then writes its share of the factors.
constexpr int MQ = 4;  // wavefronts per workgroup of the moments kernel
__global__ __launch_bounds__(64 * MQ) void bgk_moments_kernel(BgkGeo g, const double *__restrict__ f,
                                                              const double *__restrict__ uv,
                                                              const double *__restrict__ vv,
                                                              const double *__restrict__ wu,
                                                              const double *__restrict__ wv, double *cons,
                                                              double *__restrict__ tab, int nq) {
  __shared__ double sm[MQ][4][64];
  __shared__ double sp[MQ][4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = w % nq, grp = w / nq;
  const long long t = (blockIdx.x * (long long)(MQ / nq) + grp) * 64 + lane;
  const bool act = t < g.npts * g.nmem;
  const long long mem = act ? t / g.npts : 0, p = act ? t % g.npts : 0;
  double m[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    const double *fm = f + mem * g.mstride + p;
    double r4[4][4] = {};  // four independent chains per moment
    const int b0 = q * g.nv / nq, b1 = (q + 1) * g.nv / nq;
    for (int b = b0; b < b1; ++b) {
      const double vb = vv[b], wb = wv[b];
      const double *fb = fm + g.npts * (long long)g.nu * b;
      int a = 0;
      for (; a + 4 <= g.nu; a += 4) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double fv = fb[g.npts * (long long)(a + r)];
          const double ua = uv[a + r], wt = wu[a + r] * wb;
          r4[r][0] += wt * fv;
          r4[r][1] += wt * ua * fv;
          r4[r][2] += wt * vb * fv;
          r4[r][3] += wt * 0.5 * (ua * ua + vb * vb) * fv;
        }
      }
      for (; a < g.nu; ++a) {
        const double fv = fb[g.npts * (long long)a];
        const double ua = uv[a], wt = wu[a] * wb;
        r4[0][0] += wt * fv;
        r4[0][1] += wt * ua * fv;
        r4[0][2] += wt * vb * fv;
        r4[0][3] += wt * 0.5 * (ua * ua + vb * vb) * fv;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) m[c] = (r4[0][c] + r4[1][c]) + (r4[2][c] + r4[3][c]);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) sm[w][c][lane] = m[c];
  __syncthreads();
  if (q == 0) {
    double mm[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      double v = sm[w][c][lane];
      for (int r = 1; r < nq; ++r) v += sm[w + r][c][lane];
      mm[c] = v;
    }
    const double rho = mm[0], U = mm[1] / mm[0], V = mm[2] / mm[0];
    const double lam = 0.5 * mm[0] / (g.gamma - 1.0) / (mm[3] - 0.5 * (mm[1] * mm[1] + mm[2] * mm[2]) / mm[0]);
    sp[grp][0][lane] = rho;
    sp[grp][1][lane] = U;
    sp[grp][2][lane] = V;
    sp[grp][3][lane] = lam;
    if (act) {
      double *o = cons + mem * 4 * g.npts + p;
      o[0] = mm[0];
      o[g.npts] = mm[1];
      o[2 * g.npts] = mm[2];
      o[3 * g.npts] = mm[3];
    }
  }
  __syncthreads();
  if (!act) return;
  const double rho = sp[grp][0][lane], U = sp[grp][1][lane], V = sp[grp][2][lane], lam = sp[grp][3][lane];
  double *ta = tab + mem * (long long)(g.nu + g.nv) * g.npts + p;
  for (int a = q * g.nu / nq; a < (q + 1) * g.nu / nq; ++a) {
    const double du = uv[a] - U;
    ta[g.npts * (long long)a] = exp(-lam * (du * du));
  }
  const double c0 = rho * (lam / M_PI);
  for (int b = q * g.nv / nq; b < (q + 1) * g.nv / nq; ++b) {
    const double dv = vv[b] - V;
    ta[g.npts * (long long)(g.nu + b)] = c0 * exp(-lam * (dv * dv));
  }
}

template <int NSP>
__global__ __launch_bounds__(BT *BT) void bgk_rhs_kernel(BgkGeo g, BgkTileOps<NSP> ops, const double *__restrict__ uv,
                                                         const double *__restrict__ vv,
                                                         const double *__restrict__ tau,
                                                         const double *__restrict__ tab, BgkStage sa) {
  __shared__ double sx[BT + 1][BT][NSP];  // x-face upwind trace, face fx between cells fx-1 and fx
  __shared__ double sy[BT + 1][BT][NSP];  // y-face upwind trace, face fy between rows fy-1 and fy
  const int tiles_x = (g.nx + BT - 1) / BT, tiles_y = (g.ny + BT - 1) / BT;
  long long bid = blockIdx.x;
  const int tile = (int)(bid % (tiles_x * tiles_y));
  bid /= (tiles_x * tiles_y);
  const int vel = (int)(bid % ((long long)g.nu * g.nv));
  const int mem = (int)(bid / ((long long)g.nu * g.nv));
  const int a = vel % g.nu, b = vel / g.nu;
  const double ua = uv[a], vb = vv[b];
  const bool posx = ua > 0.0, posy = vb > 0.0;  // heaviside of the velocity components
  const int tx = threadIdx.x % BT, ty = threadIdx.x / BT;
  const int i0 = (tile % tiles_x) * BT, j0 = (tile / tiles_x) * BT;
  const int ncx = min(BT, g.nx - i0), ncy = min(BT, g.ny - j0);
  const int i = i0 + tx, j = j0 + ty;
  const bool act = tx < ncx && ty < ncy;
  const long long cells = (long long)g.nx * g.ny;
  const long long vbase = mem * g.mstride + g.npts * (long long)vel;
  const double *__restrict__ fv = sa.u + vbase;
  auto idx = [&](int ci, int cj, int k, int l) -> long long {
    return (long long)ci + (long long)g.nx * cj + cells * (k + NSP * l);
  };
  double w[NSP][NSP];  // w[k][l]
  if (act) {
#pragma unroll
    for (int l = 0; l < NSP; ++l)
#pragma unroll
      for (int k = 0; k < NSP; ++k) w[k][l] = fv[idx(i, j, k, l)];
  }
  // own flux traces (f_flux = velocity * f / J)
  double fL[NSP], fR[NSP], gB[NSP], gT[NSP];
  if (act) {
#pragma unroll
    for (int l = 0; l < NSP; ++l) {
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        const double fl = ua * w[q][l] * g.iJx;
        s0 += fl * ops.ll[q];
        s1 += fl * ops.lr[q];
      }
      fL[l] = s0;
      fR[l] = s1;
      // downwind face of the cell carries its trace to the neighbour
      if (posx)
        sx[tx + 1][ty][l] = s1;
      else
        sx[tx][ty][l] = s0;
    }
#pragma unroll
    for (int k = 0; k < NSP; ++k) {
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        const double gl = vb * w[k][q] * g.iJy;
        s0 += gl * ops.ll[q];
        s1 += gl * ops.lr[q];
      }
      gB[k] = s0;
      gT[k] = s1;
      if (posy)
        sy[ty + 1][tx][k] = s1;
      else
        sy[ty][tx][k] = s0;
    }
  }
  // halo: the upwind neighbour cells of the tile edges (periodic wrap)
  const int t = threadIdx.x;
  if (t < 2 * BT) {
    const bool xside = t < BT;
    const int pos = t % BT;
    if (xside && pos < ncy) {
      const int hi = posx ? (i0 - 1 + g.nx) % g.nx : (i0 + ncx) % g.nx;
      const int hj = j0 + pos;
      const int fx = posx ? 0 : ncx;
#pragma unroll
      for (int l = 0; l < NSP; ++l) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NSP; ++q) s += ua * fv[idx(hi, hj, q, l)] * g.iJx * (posx ? ops.lr[q] : ops.ll[q]);
        sx[fx][pos][l] = s;
      }
    } else if (!xside && pos < ncx) {
      const int hj = posy ? (j0 - 1 + g.ny) % g.ny : (j0 + ncy) % g.ny;
      const int hi = i0 + pos;
      const int fy = posy ? 0 : ncy;
#pragma unroll
      for (int k = 0; k < NSP; ++k) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NSP; ++q) s += vb * fv[idx(hi, hj, k, q)] * g.iJy * (posy ? ops.lr[q] : ops.ll[q]);
        sy[fy][pos][k] = s;
      }
    }
  }
  __syncthreads();
  if (!act) return;
  const double itau = 1.0 / tau[mem];
  const double *__restrict__ Ea = tab + (long long)mem * (g.nu + g.nv) * g.npts + g.npts * (long long)a;
  const double *__restrict__ Eb = tab + (long long)mem * (g.nu + g.nv) * g.npts + g.npts * (long long)(g.nu + b);
  double *__restrict__ out = sa.out + vbase;
#pragma unroll
  for (int l = 0; l < NSP; ++l)
#pragma unroll
    for (int k = 0; k < NSP; ++k) {
      // x: upwind interface fluxes on the left / right faces of row l
      const double FsL = posx ? sx[tx][ty][l] : fL[l];
      const double FsR = posx ? fR[l] : sx[tx + 1][ty][l];
      const double GsB = posy ? sy[ty][tx][k] : gB[k];
      const double GsT = posy ? gT[k] : sy[ty + 1][tx][k];
      double dfx = 0.0, dfy = 0.0;
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        dfx += ua * w[q][l] * g.iJx * ops.dl[k + NSP * q];
        dfy += vb * w[k][q] * g.iJy * ops.dl[l + NSP * q];
      }
      const long long pt = (long long)i + (long long)g.nx * j + cells * (k + NSP * l);
      const double M = Eb[pt] * Ea[pt];
      const double fc = w[k][l];
      const double r = -(dfx + (FsL - fL[l]) * ops.dhl[k] + (FsR - fR[l]) * ops.dhr[k] + dfy +
                         (GsB - gB[k]) * ops.dhl[l] + (GsT - gT[k]) * ops.dhr[l]) +
                       (M - fc) * itau;
      const long long o = idx(i, j, k, l);
      if (sa.residual) {
        out[o] = r;
      } else {
        double v = sa.a1 * fc;
        if (sa.a0 != 0.0) v = sa.a0 * sa.u0[vbase + o] + v;
        out[o] = v + sa.b * r;
      }
    }
}

// ------------------------------------------------------------------ states above kBgkStream
// Cells of a workgroup's tile, 64 x BC/64, 32 x BC/32 or 16 x BC/16 (bgk_tile): 256 where nsp wavefronts
// per 64 cells leave the registers that a line needs, fewer above.
template <int NSP>
constexpr int kBgkCells = NSP <= 3 ? 256 : NSP == 4 ? 128 : 64;
// whether the stage kernel also sums its result (at nsp = 5 the sums' registers would be spilled)
template <int NSP>
constexpr bool kBgkSums = NSP < 5;
// Bytes of a state up to which the cached path is the faster one.  Three steps, cached path / this one:
// 8 MB (20 x 33, p = 2, 16 x 11 velocities) 225 / 271 us, 32 MB 328 / 342, 68 MB 620 / 517, 97 MB
// (57 x 43, p = 2, 24 x 24) 1207 / 727.
constexpr size_t kBgkStream = 64u << 20;
// Grids inside one 16 x 16 tile with up to kBgkFewVel velocities are then many members, and a workgroup per
// member and velocity range leaves most lanes without a cell: the line rises as the share of lanes with
// one falls, bgk_fill of bytes per share.  One step, cached path / this one, 70 and 300 MB, 12 x 12
// velocities: 1 x 1 cells, p = 2, 1.78 and 1.63 times as long here, 4 x 4 1.65 and 1.29, 6 x 6 1.36 and 1.02, 8 x 8
// 1.20 and 0.89, 12 x 12 0.99 and 0.80; p = 3: 4 x 4 1.06 and 1.00, 6 x 6 0.85 and 0.65, 10 x 10 (two of its tiles)
// 1.16 and 0.98; p = 4 0.2 to 0.7 everywhere.  With more velocities (few points, whose sums the cached path forms
// one after another) 0.1 to 0.7: 1 x 1 cells, p = 2, 1079 x 1079 velocities 0.24, 8 x 8, p = 1, 202 x 202 0.24.
constexpr int kBgkFewVel = 48 * 48;
constexpr size_t bgk_fill(int nsp, long long tiles) {
  return nsp >= 5 ? 0 : nsp == 4 && tiles == 1 ? 32u << 20 : 48u << 20;
}

// Operators by the sign of the velocity component (0: positive, 1: otherwise).  Upwind, only the face
// towards the neighbour has a correction: D carries its own-trace part, D = dl - dhl ll' (positive) or
// dl - dhr lr' (D[k][q], rounded once from long double), nb forms the neighbour's trace there, dh
// weighs it.
template <int NSP>
struct BgkOps {
  double D[2][NSP * NSP], nb[2][NSP], dh[2][NSP];
};

// per velocity: u iJx, v iJy, the weights w, w u, w v, w (u^2 + v^2) / 2 of the moments, the signs
// (BgkOps) and the velocity indices
struct BgkVel {
  double cx, cy, w[4];
  int sx, sy, a, b;
};

// Velocity sums.  The velocities (a fastest) are cut into ngrp groups of `per`; the sums of a group
// run in velocity order and are kept as part[member][group][moment][point], so the stage kernel
// (which sums its results as it forms them) and bgk_partial_kernel (which reads a state) give the
// same bits.
__device__ __forceinline__ void bgk_add(double *m, const BgkVel &e, double f) {
#pragma unroll
  for (int c = 0; c < 4; ++c) m[c] += e.w[c] * f;
}

__global__ __launch_bounds__(256) void bgk_partial_kernel(BgkGeo g, const double *__restrict__ f,
                                                          const BgkVel *__restrict__ vt, double *__restrict__ part) {
  const unsigned nb = (unsigned)((g.npts + 255) / 256);
  const long long p = (blockIdx.x % nb) * 256LL + threadIdx.x;
  if (p >= g.npts) return;
  const int grp = blockIdx.x / nb % g.ngrp, mem = blockIdx.x / nb / g.ngrp;
  const int v0 = grp * g.per, v1 = min(v0 + g.per, g.nu * g.nv);
  const double *fb = f + mem * g.mstride + p;
  double m[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int v = v0; v < v1; ++v) bgk_add(m, vt[v], fb[g.npts * v]);
  double *o = part + ((long long)mem * g.ngrp + grp) * 4 * g.npts + p;
#pragma unroll
  for (int c = 0; c < 4; ++c) o[g.npts * c] = m[c];
}

// Closure: the sums of all groups, the primitive variables (KitBase conserve_prim at gamma) and the
// separable Maxwellian M(a, b) = Ea[a] * Eb[b] of every point: Ea[member][a][pt] =
// exp(-lambda (u_a - U)^2), Eb[member][b][pt] = rho lambda / pi exp(-lambda (v_b - V)^2), so that the
// stage kernel spends one multiplication per value on it.  A wavefront takes 64 consecutive points;
// the four wavefronts of a workgroup share them and split the groups (group = wavefront mod 4, added
// in wavefront order) and then the factors.
__global__ __launch_bounds__(64 * MQ) void bgk_close_kernel(BgkGeo g, const double *__restrict__ part,
                                                            const double *__restrict__ uv,
                                                            const double *__restrict__ vv, double *__restrict__ tab) {
  __shared__ double sm[MQ][4][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const long long t = blockIdx.x * 64LL + lane;
  const bool act = t < g.npts * g.nmem;
  const long long mem = act ? t / g.npts : 0, p = act ? t % g.npts : 0;
  double m[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    const double *pb = part + mem * g.ngrp * 4 * g.npts + p;
#pragma unroll 4
    for (int r = q; r < g.ngrp; r += MQ)
#pragma unroll
      for (int c = 0; c < 4; ++c) m[c] += pb[g.npts * (4LL * r + c)];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) sm[q][c][lane] = m[c];
  __syncthreads();
  if (!act) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) m[c] = (sm[0][c][lane] + sm[1][c][lane]) + (sm[2][c][lane] + sm[3][c][lane]);
  const double rho = m[0], U = m[1] / m[0], V = m[2] / m[0];
  const double lam = 0.5 * m[0] / (g.gamma - 1.0) / (m[3] - 0.5 * (m[1] * m[1] + m[2] * m[2]) / m[0]);
  double *ta = tab + mem * (long long)(g.nu + g.nv) * g.npts + p;
  for (int a = q; a < g.nu; a += MQ) {
    const double du = uv[a] - U;
    ta[g.npts * (long long)a] = exp(-lam * (du * du));
  }
  const double c0 = rho * (lam / M_PI);
  for (int b = q; b < g.nv; b += MQ) {
    const double dv = vv[b] - V;
    ta[g.npts * (long long)(g.nu + b)] = c0 * exp(-lam * (dv * dv));
  }
}

// Transport + relaxation + RK stage of a tile over one group of velocities.  A thread
// holds the points (k, line) of one cell, so the line is uniform over a wavefront and the moments of
// the result stay in 4 nsp registers over the whole group.  Per velocity: the tile and the one upwind
// column and row go to LDS (two buffers in turn: one barrier), the loads of the next velocity are put
// in flight, and each thread forms its x sums from its registers and its y sums from LDS.
// No branch lies around a load or a store, so the waits count them exactly and a wavefront never
// waits for its own stores: places outside the grid repeat the last cell of their row and column
// (and store its values again).  COMBINE: with the a0 u0 term.  Buffer access with 32-bit offsets inside one
// velocity's plane of points (below 4 GiB, large()) spends no vector instruction on addresses.
// 128 x 128, p = 2, 24 x 24 velocities (679 MB a state): 317 us for the first stage, 423 us with u0 (4.6
// and 5.0 TB/s; a plain copy of 1 GB reaches 5.0), against 135 us of moments and 360 / 578 us of the
// cached path's transport.  64-cell tiles 357 / 491 us; waits for every load and store 570 us; stores
// without the streaming hint 4-5 % slower; 128 registers (34 spilled) 1085 us.
template <int NSP, bool COMBINE>
__global__ __launch_bounds__(kBgkCells<NSP> *NSP) void bgk_stage_kernel(BgkGeo g, BgkOps<NSP> ops,
                                                            const BgkVel *__restrict__ vt,
                                                            const double *__restrict__ tau,
                                                            const double *__restrict__ tab, BgkStage sa,
                                                            double *__restrict__ part) {
  constexpr int NP = NSP * NSP, BC = kBgkCells<NSP>;
  constexpr int PL = BC + BC / 16 + 17 > BC + BC / 64 + 65 ? BC + BC / 16 + 17 : BC + BC / 64 + 65;  // widest and tallest
  constexpr int NT = ((BC / 64 + 64) * NP + BC * NSP - 1) / (BC * NSP);  // halo values per thread
  static_assert(BC % 64 == 0, "the line is uniform over a wavefront");
  __shared__ double lds[2][NP * PL];
  const int BTX = 1 << g.tsh, BTY = BC >> g.tsh, RX = BTX + 1, NH = BTX + BTY;
  const int tiles_x = (g.nx + BTX - 1) / BTX, tiles = tiles_x * ((g.ny + BTY - 1) / BTY);
  // groups of a tile side by side on one XCD: they read the same factors Ea
  const int bid = xcd_tile(blockIdx.x, gridDim.x);
  const int grp = bid % g.ngrp, tile = bid / g.ngrp % tiles, mem = bid / g.ngrp / tiles;
  const int tid = threadIdx.x, line = __builtin_amdgcn_readfirstlane(tid / BC), c = tid % BC;
  const int i0 = (tile % tiles_x) * BTX, j0 = (tile / tiles_x) * BTY;
  const int ncx = min(BTX, g.nx - i0), ncy = min(BTY, g.ny - j0);
  const int tx = min(c & (BTX - 1), ncx - 1), ty = min(c >> g.tsh, ncy - 1);
  using OFF = unsigned;  // bytes
  auto at_cell = [&](int i, int j) { return (OFF)8 * ((OFF)i + (OFF)g.nx * (OFF)j); };
  const OFF kb = (OFF)(8 * g.cells);  // from one point's cells to the next one's
  // value at byte offset o of point k (uniform) of the plane at base
  auto get = [&](const double *base, OFF o, int k) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(plane_rsrc(base, 0xFFFFFFFFu), o,
                                                                           (int)(kb * (OFF)k), 0));
  };
  constexpr int kAuxNt = 2;
  auto put = [&](double *base, OFF o, int k, double v, auto nt) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(fr_u2, v), plane_rsrc(base, 0xFFFFFFFFu), o,
                                          (int)(kb * (OFF)k), decltype(nt)::value ? kAuxNt : 0);
  };
  const OFF own = at_cell(i0 + tx, j0 + ty);

  // halo values of this thread: point hp of the upwind row's cell i0 + h (h < BTX) or of the upwind
  // column's cell j0 + h - BTX, for a positive and another component (periodic wrap), and their
  // place in LDS but for the sign of the other direction
  OFF hat[NT][2];
  int hslot[NT][2], hstep[NT];
  bool hx[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = min(tid + t * BC * NSP, NH * NP - 1), h0 = n % NH, hp = n / NH;
    hx[t] = h0 >= BTX;
    const int h = hx[t] ? min(h0 - BTX, ncy - 1) : min(h0, ncx - 1);
    hstep[t] = hx[t] ? RX : 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int hi = hx[t] ? (s == 0 ? (i0 > 0 ? i0 - 1 : g.nx - 1) : (i0 + ncx < g.nx ? i0 + ncx : 0)) : i0 + h;
      const int hj = hx[t] ? j0 + h : (s == 0 ? (j0 > 0 ? j0 - 1 : g.ny - 1) : (j0 + ncy < g.ny ? j0 + ncy : 0));
      hat[t][s] = at_cell(hi, hj) + kb * (OFF)hp;
      hslot[t][s] = hp * PL + (hx[t] ? h * RX + (s == 0 ? 0 : ncx) : (s == 0 ? 0 : ncy) * RX + h);
    }
  }

  const long long mb = mem * g.mstride, lb = g.cells * (NSP * line);
  const double *const Ea = tab + (long long)mem * (g.nu + g.nv) * g.npts + lb;
  const double *const Eb = Ea + (long long)g.nu * g.npts;
  struct Vals {
    double w[NSP], u0[NSP], ea[NSP], h[NT];
    BgkVel e;
  } A, B;
  double eb[NSP];
  auto load = [&](int v, Vals &r) {
    r.e = vt[v];
    const double *const f = sa.u + mb + g.npts * v;
#pragma unroll
    for (int k = 0; k < NSP; ++k) r.w[k] = get(f + lb, own, k);
#pragma unroll
    for (int t = 0; t < NT; ++t) r.h[t] = get(f, (hx[t] ? r.e.sx : r.e.sy) == 0 ? hat[t][0] : hat[t][1], 0);
    const double *const ea = Ea + g.npts * r.e.a;
#pragma unroll
    for (int k = 0; k < NSP; ++k) r.ea[k] = get(ea, own, k);
    if constexpr (COMBINE) {
      const double *const f0 = sa.u0 + mb + g.npts * v + lb;
#pragma unroll
      for (int k = 0; k < NSP; ++k) r.u0[k] = get(f0, own, k);
    }
  };
  const int v0 = grp * g.per, v1 = min(v0 + g.per, g.nu * g.nv);
  const double itau = 1.0 / tau[mem];
  double m[NSP][4] = {};
  // operators of the current signs: they change a few times over a group
  double D[NP], nbx[NSP], dhx[NSP], Dy[NSP], nby[NSP], dhy = 0.0;
  int px = -1, py = -1, pb = -1;

  auto body = [&](int v, double *buf, const Vals &cur, Vals &nxt) {
    const int sx = cur.e.sx, sy = cur.e.sy;
    // own cells one place in from the halo column and row where those lie left and below
    const int at = (ty + 1 - sy) * RX + tx + 1 - sx;
#pragma unroll
    for (int k = 0; k < NSP; ++k) buf[(k + NSP * line) * PL + at] = cur.w[k];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int sn = hx[t] ? sx : sy, so = hx[t] ? sy : sx;
      buf[(sn == 0 ? hslot[t][0] : hslot[t][1]) + (so == 0 ? hstep[t] : 0)] = cur.h[t];
    }
    // before the next velocity's loads: the waits for these (now and then) then leave those alone
    if (cur.e.b != pb) {
      pb = cur.e.b;
#pragma unroll
      for (int k = 0; k < NSP; ++k) eb[k] = get(Eb + g.npts * pb, own, k);
    }
    load(min(v + 1, v1 - 1), nxt);
    if (sx != px) {
      px = sx;
#pragma unroll
      for (int q = 0; q < NP; ++q) D[q] = ops.D[sx][q];
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        nbx[q] = ops.nb[sx][q];
        dhx[q] = ops.dh[sx][q];
      }
    }
    if (sy != py) {
      py = sy;
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        Dy[q] = ops.D[sy][line * NSP + q];
        nby[q] = ops.nb[sy][q];
      }
      dhy = ops.dh[sy][line];
    }
    // barrier over LDS alone: the loads above stay in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int dx = sx == 0 ? -1 : 1, dy = sy == 0 ? -RX : RX;
    double nx = 0.0;
#pragma unroll
    for (int q = 0; q < NSP; ++q) nx += nbx[q] * buf[(q + NSP * line) * PL + at + dx];
    double *const o = sa.out + mb + g.npts * v + lb;
#pragma unroll
    for (int k = 0; k < NSP; ++k) {
      double X = dhx[k] * nx, ny = 0.0, Y = 0.0;
#pragma unroll
      for (int q = 0; q < NSP; ++q) {
        X += D[k * NSP + q] * cur.w[q];
        Y += Dy[q] * buf[(k + NSP * q) * PL + at];
        ny += nby[q] * buf[(k + NSP * q) * PL + at + dy];
      }
      Y += dhy * ny;
      double s = (eb[k] * cur.ea[k] - cur.w[k]) * itau - (cur.e.cx * X + cur.e.cy * Y);
      double t = sa.a1 * cur.w[k];
      if constexpr (COMBINE) t = sa.a0 * cur.u0[k] + t;
      s = t + sa.b * s;
      if constexpr (kBgkSums<NSP>) bgk_add(m[k], cur.e, s);
      put(o, own, k, s, std::true_type{});
    }
  };
  load(v0, A);
  for (int v = v0;;) {
    body(v, lds[0], A, B);
    if (++v == v1) break;
    body(v, lds[1], B, A);
    if (++v == v1) break;
  }
  if constexpr (kBgkSums<NSP>) {
    double *const o = part + ((long long)mem * g.ngrp + grp) * 4 * g.npts + lb;
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int k = 0; k < NSP; ++k) put(o + g.npts * n, own, k, m[k][n], std::false_type{});
  }
}

// ------------------------------------------------------------------ context
struct BgkCtx {
  int nx = 0, ny = 0, nsp = 0, nu = 0, nv = 0, nmem = 1;
  double dx = 1, dy = 1, gamma = 2.0;
  int num_cu = 256;
  HostOps ops;
  size_t len = 0;
  hipStream_t stream = nullptr;
  HostStaging staging;
  double *d_vel = nullptr;  // uv | vv | wu | wv
  BgkVel *d_vt = nullptr;
  double *d_tau = nullptr;
  double *d_cons = nullptr;  // moments of the last moments launch
  // sums of the velocity groups (large states): starts at d_cons, since a call forms them anew where it steps
  double *d_part = nullptr;
  double *d_tab = nullptr;  // Maxwellian factors Ea | Eb per member
  double *d_u = nullptr, *d_s1 = nullptr, *d_s2 = nullptr, *d_in = nullptr, *d_out = nullptr;

  long long bgk_tiles(int cells, int sh) const {
    const int tx = 1 << sh, ty = cells >> sh;
    return (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
  }

  BgkGeo geom;
  const BgkGeo &geo() const { return geom; }

  BgkGeo plan() const {
    BgkGeo g;
    g.nx = nx;
    g.ny = ny;
    g.nu = nu;
    g.nv = nv;
    g.nmem = nmem;
    g.iJx = 2.0 / dx;
    g.iJy = 2.0 / dy;
    g.cells = (long long)nx * ny;
    g.npts = g.cells * nsp * nsp;
    g.mstride = g.npts * nu * nv;
    g.gamma = gamma;
    // the tile that covers the grid with the fewest cells, the widest of equals
    const int bc = nsp <= 3 ? kBgkCells<3> : nsp == 4 ? kBgkCells<4> : kBgkCells<5>;
    long long best = 0;
    for (int sh = 6; sh >= 4; --sh) {
      const long long n = bgk_tiles(bc, sh);
      if (!best || n < best) best = n, g.tsh = sh;
    }
    // Groups: workgroups of one size in rounds of one per CU, so the time goes as rounds x
    // velocities per group; the fewer rounds the better beside that (128 x 128,
    // p = 2, three steps: 1 round 3.45 ms, 2 rounds 3.82, 3 rounds 3.96)
    const long long nvel = (long long)nu * nv;
    double cost = 0.0;
    for (long long n = 1; n <= std::max(1LL, nvel / 4); ++n) {
      const long long per = (nvel + n - 1) / n, rounds = (best * nmem * n + num_cu - 1) / num_cu;
      const double t = (double)(rounds * per) * (1.0 + 0.15 * (double)(rounds - 1));
      if (n == 1 || t < cost) cost = t, g.per = (int)per;
    }
    g.ngrp = (int)((nvel + g.per - 1) / g.per);
    return g;
  }

  template <int NSP>
  int launch_stage(const BgkStage &sa, hipStream_t st) const {
    BgkOps<NSP> o;
    for (int s = 0; s < 2; ++s) {
      const double *t = s ? ops.lr : ops.ll, *dh = s ? ops.dhr : ops.dhl;
      for (int k = 0; k < NSP; ++k) {
        o.nb[s][k] = s ? ops.ll[k] : ops.lr[k];
        o.dh[s][k] = dh[k];
        for (int q = 0; q < NSP; ++q)
          o.D[s][k * NSP + q] = (double)((long double)ops.dl[k + NSP * q] - (long double)t[q] * (long double)dh[k]);
      }
    }
    const BgkGeo &g = geo();
    const long long tiles = bgk_tiles(kBgkCells<NSP>, g.tsh);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles * g.ngrp * nmem)), dim3(kBgkCells<NSP> * NSP), 0, st, g, o, d_vt, d_tau,
                         d_tab, sa, d_part);
    };
    if (sa.a0 == 0.0)
      go(bgk_stage_kernel<NSP, false>);
    else
      go(bgk_stage_kernel<NSP, true>);
    FR_LAUNCHED("bgk_stage_kernel");
    return FR_OK;
  }

  // velocity sums of a state
  int launch_partial(const double *d_f, hipStream_t st) const {
    const BgkGeo &g = geo();
    hipLaunchKernelGGL(bgk_partial_kernel, dim3((unsigned)((g.npts + 255) / 256 * g.ngrp * nmem)), dim3(256), 0, st, g, d_f, d_vt, d_part);
    FR_LAUNCHED("bgk_partial_kernel");
    return FR_OK;
  }

  int launch_close(hipStream_t st) const {
    const BgkGeo &g = geo();
    hipLaunchKernelGGL(bgk_close_kernel, dim3((unsigned)((g.npts * nmem + 63) / 64)), dim3(64 * MQ), 0, st, g, d_part,
                       d_vel, d_vel + nu, d_tab);
    FR_LAUNCHED("bgk_close_kernel");
    return FR_OK;
  }

  // one stage of sa.u, whose velocity sums are in d_part; leaves those of the result there
  int stage_large(const BgkStage &sa, hipStream_t st) const {
    int rc = launch_close(st);
    if (rc) return rc;
    switch (nsp) {
      case 2: return launch_stage<2>(sa, st);
      case 3: return launch_stage<3>(sa, st);
      case 4: return launch_stage<4>(sa, st);
      default: rc = launch_stage<5>(sa, st);
    }
    return rc ? rc : launch_partial(sa.out, st);  // kBgkSums<5>
  }

  int stage(const BgkStage &sa, hipStream_t st) const { return large() ? stage_large(sa, st) : stage_cached(sa, st); }

  template <int NSP>
  int launch_rhs(const BgkStage &sa, hipStream_t st) const {
    BgkTileOps<NSP> o;
    for (int q = 0; q < NSP; ++q) {
      o.ll[q] = ops.ll[q];
      o.lr[q] = ops.lr[q];
      o.dhl[q] = ops.dhl[q];
      o.dhr[q] = ops.dhr[q];
    }
    for (int q = 0; q < NSP * NSP; ++q) o.dl[q] = ops.dl[q];
    const BgkGeo &g = geo();
    const long long tiles = (long long)((nx + BT - 1) / BT) * ((ny + BT - 1) / BT);
    const long long nb = tiles * nu * nv * nmem;
    hipLaunchKernelGGL(bgk_rhs_kernel<NSP>, dim3((unsigned)nb), dim3(BT * BT), 0, st, g, o, d_vel, d_vel + nu,
                       d_tau, d_tab, sa);
    FR_LAUNCHED("bgk_rhs_kernel");
    return FR_OK;
  }

  // moments kernel launch: nq wavefronts per group of 64 points, enough for about eight
  // wavefronts per SIMD; MQ / nq point groups per workgroup
  int launch_moments(const double *d_f, hipStream_t st) const {
    const BgkGeo &g = geo();
    const long long n = g.npts * nmem, groups = (n + 63) / 64;
    int nq = 1;
    while (nq < MQ && groups * nq < 8LL * 1024) nq *= 2;
    const long long nb = (groups + (MQ / nq) - 1) / (MQ / nq);
    hipLaunchKernelGGL(bgk_moments_kernel, dim3((unsigned)nb), dim3(64 * MQ), 0, st, g, d_f, d_vel, d_vel + nu,
                       d_vel + nu + nv, d_vel + 2 * nu + nv, d_cons, d_tab, nq);
    FR_LAUNCHED("bgk_moments_kernel");
    return FR_OK;
  }

  // whether the stage kernel serves: kBgkStream, bgk_fill, a velocity's plane of points below the 4 GiB that
  // its offsets reach, and points that the closure, with four threads for each, can launch (2^32 threads)
  bool large() const {
    const size_t bytes = len * sizeof(double);
    if (bytes <= kBgkStream || geom.npts >= (1LL << 29) || geom.npts * nmem >= (1LL << 30)) return false;
    if (nx > BT || ny > BT || (long long)nu * nv > kBgkFewVel) return true;
    const int bc = nsp <= 3 ? kBgkCells<3> : nsp == 4 ? kBgkCells<4> : kBgkCells<5>;
    const long long tiles = bgk_tiles(bc, geom.tsh);
    return (double)bytes * (double)geom.cells > (double)bgk_fill(nsp, tiles) * (double)(tiles * bc);
  }

  int stage_cached(const BgkStage &sa, hipStream_t st) const {
    const int rc = launch_moments(sa.u, st);
    if (rc) return rc;
    switch (nsp) {
      case 2: return launch_rhs<2>(sa, st);
      case 3: return launch_rhs<3>(sa, st);
      case 4: return launch_rhs<4>(sa, st);
      default: return launch_rhs<5>(sa, st);
    }
  }

  void release() {
    if (stream) (void)hipStreamSynchronize(stream);
    staging.release();
    double *bufs[] = {d_vel, d_tau, d_cons, d_tab, d_u, d_s1, d_s2, d_in, d_out};
    for (double *b : bufs)
      if (b) (void)hipFree(b);
    if (d_vt) (void)hipFree(d_vt);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

}  // namespace fr

using namespace fr;

struct fr_bgk_ctx : BgkCtx {};

extern "C" {

int fr_bgk_create(fr_bgk_ctx **out, const fr_bgk_desc *d) {
  FR_REQUIRE(out && d, FR_E_INVALID, "fr_bgk_create: null argument");
  *out = nullptr;
  FR_REQUIRE(d->nx >= 1 && d->ny >= 1 && d->nu >= 1 && d->nv >= 1 && d->nmem >= 1, FR_E_INVALID,
             "fr_bgk_create: sizes must be >= 1");
  FR_REQUIRE(d->deg >= 1 && d->deg <= 4, FR_E_UNSUPPORTED, "fr_bgk_create: degree must be in 1..4");
  FR_REQUIRE(d->dx > 0 && d->dy > 0 && d->gamma > 1.0, FR_E_INVALID, "fr_bgk_create: dx, dy > 0, gamma > 1");
  FR_REQUIRE(d->u && d->v && d->wu && d->wv && d->tau, FR_E_INVALID, "fr_bgk_create: null velocity grid or tau");
  for (int m = 0; m < d->nmem; ++m) FR_REQUIRE(d->tau[m] > 0.0, FR_E_INVALID, "fr_bgk_create: tau must be > 0");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(FR_E_HIP, "fr_bgk_create: no HIP device visible");
  fr_bgk_ctx *c = new (std::nothrow) fr_bgk_ctx();
  FR_REQUIRE(c, FR_E_NOMEM, "fr_bgk_create: out of host memory");
  c->nx = d->nx;
  c->ny = d->ny;
  c->nsp = d->deg + 1;
  c->nu = d->nu;
  c->nv = d->nv;
  c->nmem = d->nmem;
  c->dx = d->dx;
  c->dy = d->dy;
  c->gamma = d->gamma;
  int rc = no_throw("fr_bgk_create", [&] {
    return build_ops(d->deg, FR_CORR_RADAU, c->ops)
               ? (int)FR_OK
               : fail(FR_E_INVALID, "fr_bgk_create: operator construction failed");
  });
  if (rc) {
    delete c;
    return rc;
  }
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&c->num_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c->num_cu < 1)
    c->num_cu = 256;
  c->geom = c->plan();
  const BgkGeo &g = c->geom;
  c->len = (size_t)g.mstride * d->nmem;
  std::vector<double> vel;
  std::vector<BgkVel> vt;  // of the stage kernel alone
  rc = no_throw("fr_bgk_create", [&] {
    vel.insert(vel.end(), d->u, d->u + d->nu);
    vel.insert(vel.end(), d->v, d->v + d->nv);
    vel.insert(vel.end(), d->wu, d->wu + d->nu);
    vel.insert(vel.end(), d->wv, d->wv + d->nv);
    if (c->large()) vt.reserve((size_t)d->nu * d->nv);
    return (int)FR_OK;
  });
  if (rc) {
    delete c;
    return rc;
  }
  for (int b = 0; c->large() && b < d->nv; ++b)
    for (int a = 0; a < d->nu; ++a) {
      const double u = d->u[a], v = d->v[b], w = d->wu[a] * d->wv[b];
      vt.push_back({u * (2.0 / d->dx), v * (2.0 / d->dy), {w, w * u, w * v, w * 0.5 * (u * u + v * v)},
                    u > 0.0 ? 0 : 1, v > 0.0 ? 0 : 1, a, b});
    }
  hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc(&c->d_vel, vel.size() * sizeof(double));
  if (e == hipSuccess) e = hipMemcpy(c->d_vel, vel.data(), vel.size() * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess && c->large()) e = hipMalloc(&c->d_vt, vt.size() * sizeof(BgkVel));
  if (e == hipSuccess && c->large())
    e = hipMemcpy(c->d_vt, vt.data(), vt.size() * sizeof(BgkVel), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMalloc(&c->d_tau, d->nmem * sizeof(double));
  if (e == hipSuccess) e = hipMemcpy(c->d_tau, d->tau, d->nmem * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMalloc(&c->d_cons, (size_t)g.npts * 4 * (c->large() ? g.ngrp : 1) * d->nmem * sizeof(double));
  c->d_part = c->d_cons;
  if (e == hipSuccess) e = hipMalloc(&c->d_tab, (size_t)g.npts * (d->nu + d->nv) * d->nmem * sizeof(double));
  if (e == hipSuccess) e = hipMalloc(&c->d_u, c->len * sizeof(double));
  if (e != hipSuccess) {
    rc = hip_fail(e, "fr_bgk_create", __FILE__, __LINE__);
    c->release();
    delete c;
    return rc;
  }
  *out = c;
  return FR_OK;
}

int fr_bgk_destroy(fr_bgk_ctx *c) {
  if (!c) return FR_OK;
  c->release();
  delete c;
  return FR_OK;
}

size_t fr_bgk_state_len(const fr_bgk_ctx *c) { return c ? c->len : 0; }

int fr_bgk_rhs(fr_bgk_ctx *c, const double *f, double *df) {
  FR_REQUIRE(c && f && df, FR_E_INVALID, "fr_bgk_rhs: null argument");
  const size_t bytes = c->len * sizeof(double);
  if (!c->d_in) FR_HIP(hipMalloc(&c->d_in, bytes));
  if (!c->d_out) FR_HIP(hipMalloc(&c->d_out, bytes));
  FR_HIP(hipMemcpyAsync(c->d_in, f, bytes, hipMemcpyHostToDevice, c->stream));
  BgkStage sa{c->d_in, nullptr, c->d_out, 0.0, 0.0, 0.0, 1};
  int rc = c->stage_cached(sa, c->stream);
  if (rc) return rc;
  FR_HIP(hipMemcpyAsync(df, c->d_out, bytes, hipMemcpyDeviceToHost, c->stream));
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

int fr_bgk_set_state(fr_bgk_ctx *c, const double *f) {
  FR_REQUIRE(c && f, FR_E_INVALID, "fr_bgk_set_state: null argument");
  return copy_to_device(c->staging, c->d_u, f, c->len, c->stream);
}

int fr_bgk_set_state_dev(fr_bgk_ctx *c, const double *d_f) {
  FR_REQUIRE(c && d_f, FR_E_INVALID, "fr_bgk_set_state_dev: null argument");
  FR_HIP(hipMemcpyAsync(c->d_u, d_f, c->len * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

int fr_bgk_get_state(fr_bgk_ctx *c, double *f) {
  FR_REQUIRE(c && f, FR_E_INVALID, "fr_bgk_get_state: null argument");
  return copy_to_host(c->staging, f, c->d_u, c->len, c->stream);
}

// nsteps Shu-Osher SSP-RK3 steps of all members; each stage = closure + transport/relaxation
int fr_bgk_step(fr_bgk_ctx *c, double dt, int nsteps) {
  FR_REQUIRE(c && nsteps >= 0 && std::isfinite(dt), FR_E_INVALID, "fr_bgk_step: bad arguments");
  if (!c->d_s1) FR_HIP(hipMalloc(&c->d_s1, c->len * sizeof(double)));
  if (!c->d_s2) FR_HIP(hipMalloc(&c->d_s2, c->len * sizeof(double)));
  // A step goes from d_u to d_s1 (every stage writes every value) and the two swap, so no stage writes
  // an array it reads: the stage kernel's places outside the grid read the u^n of a cell whose
  // own thread may have stored its result already.
  int rc = nsteps > 0 && c->large() ? c->launch_partial(c->d_u, c->stream) : FR_OK;
  if (rc) return rc;
  for (int n = 0; n < nsteps; ++n) {
    double *const X = c->d_u, *const Y = c->d_s1;
    if ((rc = c->stage(BgkStage{X, X, Y, 0.0, 1.0, dt, 0}, c->stream))) return rc;
    if ((rc = c->stage(BgkStage{Y, X, c->d_s2, 0.75, 0.25, 0.25 * dt, 0}, c->stream))) return rc;
    if ((rc = c->stage(BgkStage{c->d_s2, X, Y, 1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0 * dt, 0}, c->stream))) return rc;
    std::swap(c->d_u, c->d_s1);
  }
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

// conserved moments (rho, rho U, rho V, E) of the device state at every solution point, host
// output w[member][c][pt]
int fr_bgk_moments(fr_bgk_ctx *c, double *w) {
  FR_REQUIRE(c && w, FR_E_INVALID, "fr_bgk_moments: null argument");
  int rc = c->launch_moments(c->d_u, c->stream);
  if (rc) return rc;
  const size_t bytes = (size_t)c->geo().npts * 4 * c->nmem * sizeof(double);
  FR_HIP(hipMemcpyAsync(w, c->d_cons, bytes, hipMemcpyDeviceToHost, c->stream));
  FR_HIP(hipStreamSynchronize(c->stream));
  return FR_OK;
}

// Gauss-Hermite rule for the weight exp(-x^2): nodes ascending, weights (host, native).
// The orthonormal Hermite functions p_j follow p_{j+1} = x sqrt(2/(j+1)) p_j - sqrt(j/(j+1)) p_{j-1},
// p_0 = pi^(-1/4), with p_n' = sqrt(2n) p_{n-1}.  All n zeros lie in |x| < sqrt(2n+1); a sign scan
// of p_n on a grid finer than the closest pair of zeros brackets each one, bisection narrows the
// bracket and Newton polishes it; the weight is 2 / p_n'(x)^2.
static void hermite_pn(int n, double x, double &pn, double &pn1) {
  double p1 = 0.7511255444649425, p0 = 0.0;  // pi^(-1/4), p_{-1}
  for (int j = 0; j < n; ++j) {
    const double p2 = x * std::sqrt(2.0 / (j + 1)) * p1 - std::sqrt((double)j / (j + 1)) * p0;
    p0 = p1;
    p1 = p2;
  }
  pn = p1;
  pn1 = p0;
}

int fr_gauss_hermite(int n, double *x, double *w) {
  FR_REQUIRE(n >= 1 && n <= 200 && x && w, FR_E_INVALID, "fr_gauss_hermite: bad arguments");
  const double R = std::sqrt(2.0 * n + 1.0);
  std::vector<double> lo, hi;
  for (int cells = 64 * n; (int)lo.size() != n; cells *= 2) {
    if (cells > (1 << 24)) return fail(FR_E_INVALID, "fr_gauss_hermite: zeros not separated");
    lo.clear();
    hi.clear();
    double xa = -R, pa, q;
    hermite_pn(n, xa, pa, q);
    for (int c = 1; c <= cells; ++c) {
      const double xb = -R + 2.0 * R * c / cells;
      double pb;
      hermite_pn(n, xb, pb, q);
      if ((pa < 0.0) != (pb < 0.0) || pb == 0.0) {
        lo.push_back(xa);
        hi.push_back(xb);
        if (pb == 0.0) {  // step past an exact zero so it is bracketed once
          xa = xb + 1e-300;
          hermite_pn(n, xa, pa, q);
          continue;
        }
      }
      xa = xb;
      pa = pb;
    }
  }
  for (int i = 0; i < n; ++i) {
    double a = lo[i], b = hi[i], pa, q;
    hermite_pn(n, a, pa, q);
    for (int it = 0; it < 200 && b - a > 1e-13 * std::max(1.0, std::fabs(a)); ++it) {
      const double m = 0.5 * (a + b);
      double pm;
      hermite_pn(n, m, pm, q);
      if ((pm < 0.0) == (pa < 0.0)) {
        a = m;
        pa = pm;
      } else {
        b = m;
      }
    }
    double z = 0.5 * (a + b), d = 0.0;
    for (int it = 0; it < 5; ++it) {
      double pn, pn1;
      hermite_pn(n, z, pn, pn1);
      d = std::sqrt(2.0 * n) * pn1;
      z -= pn / d;
    }
    double pn, pn1;
    hermite_pn(n, z, pn, pn1);
    d = std::sqrt(2.0 * n) * pn1;
    x[i] = z;
    w[i] = 2.0 / (d * d);
  }
  // symmetric rule: pair the nodes exactly
  for (int i = 0; i < n / 2; ++i) {
    const double z = 0.5 * (x[n - 1 - i] - x[i]), ww = 0.5 * (w[i] + w[n - 1 - i]);
    x[i] = -z;
    x[n - 1 - i] = z;
    w[i] = w[n - 1 - i] = ww;
  }
  if (n & 1) x[n / 2] = 0.0;
  return FR_OK;
}

}  // extern "C"
