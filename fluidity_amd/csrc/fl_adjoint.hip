// fl_adjoint.hip -- gfx950 kernels of the hand-written adjoint of the split
// MUSCL-Hancock + HLLC step (FP64).
//
// Forward: out_i = U_i + dtdh (G_{i-1/2} - G_{i+1/2}), G_{i+1/2} =
// HLLC(R_i, L_{i+1}), R_i / L_i the evolved face states of cell i from cells
// i-1..i+1 (solver/split_solver.hpp:138-162,
// reconstruction/muscl_reconstructor.hpp:99-172, flux_method/flux_hllc.hpp).
// Adjoint of one sweep, given lambda = dLoss/d out:
//  * sweep kernel, one lane per cell i of a line: recompute R_i, L_i and with
//    the next lane's L the flux G of face i+1/2, mu = dtdh (lambda_{i+1} -
//    lambda_i) (ghost cells carry no lambda), back-propagate mu through HLLC
//    to the face states, theirs of cell i (one of them from the lane before)
//    through the evolution to the cells i-1..i+1, and add to lambda what the
//    cells i-1..i+1 pass to cell i, also through ghost cells (mirror,
//    reflective flip; a periodic line is followed around its ends);
//  * the dt/dh and gamma adjoints are summed per workgroup, then over the
//    workgroups, in a fixed order, so the whole adjoint is deterministic.
// dt = cfl dh / max wavespeed couples the step to the state through the
// wavespeed of the cell holding the maximum (lowest index among ties); the
// step's finalize kernel adds that term.
#include "fl_adjoint.hpp"
#include "fl_adjoint_kernels.hpp"
#include "fl_sweep_tiles.hpp"

namespace fl {
namespace adj {

__device__ __forceinline__ int64_t ghost_index(int64_t i, int64_t n, int bc, bool& flip) {
  i = i < -4 ? -4 : (i > n + 3 ? n + 3 : i);
  flip = false;
  if (i >= 0 && i < n) return i;
  if (bc == kBcPeriodic) return i < 0 ? i + n : i - n;
  flip = (bc == kBcReflective);
  return i < 0 ? -i - 1 : 2 * n - 1 - i;
}

// State at (x, y) with the ghost rule of each dimension (reflective ghosts
// get the velocity flip of the forward sweep).
template <int ND>
__device__ __forceinline__ void load_state(const AGrid& g, int64_t x, int64_t y, double* u) {
  bool fx = false, fy = false;
  const int64_t xi = ghost_index(x, g.nx, g.bcx, fx);
  const int64_t yi = ND > 1 ? ghost_index(y, g.ny, g.bcy, fy) : 0;
  const double* p = g.U + (yi * g.nx + xi) * g.es;
#pragma unroll
  for (int k = 0; k < 2 + ND; ++k) u[k] = p[k * g.cs];
  if (fx) reflect<double, ND>(u, 0);
  if (ND > 1 && fy) reflect<double, ND>(u, 1);
}

// Pressure and velocities of every position within 4 ghost cells of the grid
// (ghost rule and reflective flip applied), on the padded grid P (x fastest,
// pad 4 in each dimension of the grid).
template <int ND>
__global__ void __launch_bounds__(256) prim_pad_kernel(AGrid g, Material<double> m,
                                                       double* __restrict__ P,
                                                       double* __restrict__ V0,
                                                       double* __restrict__ V1) {
  const int64_t px = g.nx + 8, py = ND > 1 ? g.ny + 8 : 1;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= px * py) return;
  const int64_t x = q % px - 4, y = ND > 1 ? q / px - 4 : 0;
  double u[2 + ND];
  load_state<ND>(g, x, y, u);
  const Prim<double, ND> w = prim_of<double, ND>(u, m);
  P[q] = w.p;
  V0[q] = w.vel[0];
  if (ND > 1) V1[q] = w.vel[ND - 1];
}

// chi_v of MHReconstructor::evolve (reconstruction/muscl_reconstructor.hpp:59-87,
// 106-118) -- the minimum over dimensions of chi about the cell and about its
// neighbour on the higher-pressure side -- for every position within one
// ghost cell of the grid, from the padded primitives.
template <int ND>
__global__ void __launch_bounds__(256) chi_pad_kernel(AGrid g, const double* __restrict__ P,
                                                      const double* __restrict__ V0,
                                                      const double* __restrict__ V1,
                                                      double* __restrict__ chi,
                                                      int* __restrict__ any) {
  const int64_t px = g.nx + 8;
  const int64_t cx = g.nx + 2, cy = ND > 1 ? g.ny + 2 : 1;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q == 0) *any = 0;  // the record flag, read by chi_gather_kernel
  if (q >= cx * cy) return;
  const int64_t x = q % cx - 1, y = ND > 1 ? q / cx - 1 : 0;
  auto at = [&](const double* A, int64_t xx, int64_t yy) {
    return A[(ND > 1 ? (yy + 4) * px : 0) + xx + 4];
  };
  const Material<double> no_shift{};  // the adjoint runs the reference's equations of state
  auto chi_d = [&](int64_t xx, int64_t yy, int d) {
    const int64_t dx = (d == 0), dy = (d == 1);
    const double* V = d == 0 ? V0 : V1;
    return chi_factor<double>(at(P, xx - 2 * dx, yy - 2 * dy), at(P, xx - dx, yy - dy),
                              at(P, xx + dx, yy + dy), at(P, xx + 2 * dx, yy + 2 * dy),
                              at(V, xx - dx, yy - dy), at(V, xx + dx, yy + dy), no_shift);
  };
  double c = DBL_MAX;
  for (int d = 0; d < ND; ++d) {
    const int64_t dx = (d == 0), dy = (d == 1);
    const int sign = signum(at(P, x + dx, y + dy) - at(P, x - dx, y - dy));
    c = smin(c, smin(chi_d(x, y, d), chi_d(x + sign * dx, y + sign * dy, d)));
  }
  chi[q] = c;
}

// ---- the flattening factor's adjoint ----------------------------------------
// chi_v of a cell (chi_pad_kernel) is the smallest of the flattening factors
// K_d(j) of the cell and of its neighbour on the higher-pressure side in each
// dimension d; where the selected factor is flattened and not clamped,
// K = 1 - (z - 0.75) / 0.1 with z = |p(j+1) - p(j-1)| / |p(j+2) - p(j-2)|
// along d carries the gradient (muscl_reconstructor.hpp:59-87); the
// flattening test, the neighbour and the minimum are branches.

// At a chi position q = (x, y) (of the grid padded by one cell) whose chi lies
// strictly between 0 and 1 (elsewhere the selected factor is clamped or not
// flattened and carries no gradient), G being the adjoint of chi that the
// position's face states passed back: which factor the minimum selected,
// rec_k = 4 d + (j - c along d) + 1 for K_d(j) (-1: none); and the adjoints
// of the pressures at j-2, j-1, j+1, j+2 along d (rec_v, 4 per position).
// *any is set when some position has a record.
template <int ND>
__device__ void chi_record(const AGrid& g, const double* __restrict__ P,
                           const double* __restrict__ V0, const double* __restrict__ V1, int64_t x,
                           int64_t y, int64_t q, double G, int* __restrict__ rec_k,
                           double* __restrict__ rec_v, int* __restrict__ any) {
  const int64_t px = g.nx + 8;
  auto at = [&](const double* A, int64_t xx, int64_t yy) {
    return A[(ND > 1 ? (yy + 4) * px : 0) + xx + 4];
  };
  const Material<double> no_shift{};
  auto chi_d = [&](int64_t xx, int64_t yy, int d) {
    const int64_t dx = (d == 0), dy = (d == 1);
    const double* V = d == 0 ? V0 : V1;
    return chi_factor<double>(at(P, xx - 2 * dx, yy - 2 * dy), at(P, xx - dx, yy - dy),
                              at(P, xx + dx, yy + dy), at(P, xx + 2 * dx, yy + 2 * dy),
                              at(V, xx - dx, yy - dy), at(V, xx + dx, yy + dy), no_shift);
  };
  int best = -1;
  {
    // the selection of chi_pad_kernel: smin(chi, smin(K(c), K(c + s)))
    double c = DBL_MAX;
    for (int d = 0; d < ND; ++d) {
      const int64_t dx = (d == 0), dy = (d == 1);
      const int sign = signum(at(P, x + dx, y + dy) - at(P, x - dx, y - dy));
      const double k0 = chi_d(x, y, d);
      const double k1 = chi_d(x + sign * dx, y + sign * dy, d);
      double mv = k0;
      int sel = 4 * d + 1;
      if (k1 < k0) {
        mv = k1;
        sel = 4 * d + sign + 1;
      }
      if (mv < c) {
        c = mv;
        best = sel;
      }
    }
  }
  if (best >= 0) {
    const int d = best / 4, jo = best % 4 - 1;
    const int64_t dx = (d == 0), dy = (d == 1);
    const int64_t jx = x + jo * dx, jy = y + jo * dy;
    const double* V = d == 0 ? V0 : V1;
    const double p_pp = at(P, jx - 2 * dx, jy - 2 * dy), p_p = at(P, jx - dx, jy - dy);
    const double p_n = at(P, jx + dx, jy + dy), p_nn = at(P, jx + 2 * dx, jy + 2 * dy);
    const double u_factor = at(V, jx - dx, jy - dy) - at(V, jx + dx, jy + dy);
    const double dp = fabs(p_n - p_p);
    const double pmin = smin(p_n, p_p);
    const bool flatten = u_factor > 0.0 && dv(dp, pmin) > 0.33;
    const double den = fabs(p_nn - p_pp);
    if (flatten && den > 0.0) {
      const double z = dv(dp, den);
      const double temp = 1.0 - dv(z - 0.75, 0.85 - 0.75);
      if (temp > 0.0 && temp < 1.0) {
        const double g_z = -G / (0.85 - 0.75);
        const double g_dp = g_z / den;
        const double g_den = -g_z * z / den;
        const double sn = (double)signum(p_n - p_p), snn = (double)signum(p_nn - p_pp);
        rec_v[4 * q + 0] = -g_den * snn;  // p(j-2)
        rec_v[4 * q + 1] = -g_dp * sn;    // p(j-1)
        rec_v[4 * q + 2] = g_dp * sn;     // p(j+1)
        rec_v[4 * q + 3] = g_den * snn;   // p(j+2)
        rec_k[q] = best;
        *any = 1;
        return;
      }
    }
  }
  rec_k[q] = -1;
}

// Adjoint of one sweep: a wave takes kAdjCells cells of a line along the sweep
// and three on either side, one a lane, and neighbours exchange in registers.
// PRIM: primitive-form limiting (a template parameter, so that the
// conservative-form kernel carries none of its code).
//
// FP64 arithmetic and its latency at two waves a SIMD bound it (2D: HLLC 182
// registers, FORCE 242, with primitive-form limiting 220 and 256, the latter
// with 28 to 30 spilled; HLLC at 512^2 at three a SIMD 26 us in x and 32 in y, at
// four, with spills, 38 and 44; workgroups of 8 waves 30 and 36, whose last round
// is a quarter full).
// With a thread per face, which evolved both cells beside it forward and back
// and passed its 16 contributions through memory to a kernel that gathered
// them, it took 33 us, the gather 9, the sums 5 and the flattening factors'
// records 4; now 24 us (x) and 28 (y) in all.  In the y sweep a wave's lanes run
// down a column: its loads touch a line each, which the columns of a workgroup
// share.  The waves of a workgroup take neighbouring lines, on a 1D grid
// neighbouring segments (four steps on 200000 cells and back, each recomputed
// in 64 lanes: 522 us with one wave of four at work, 392 with all).
//
// rec_k, rec_v and any receive the records of the flattening factors
// (chi_record) at the positions of the grid's lines, partials the workgroup's
// sums of the dt/dh and gamma adjoints.
template <int ND, int D, int FLUX, bool PRIM>
__global__ void __launch_bounds__(64 * kAdjWaves) __attribute__((amdgpu_waves_per_eu(2)))
sweep_adj_kernel(AGrid g, const double* __restrict__ lam, double* __restrict__ lam_in,
                 Material<double> m, int limiter, const StepRec* __restrict__ rec,
                 const double* __restrict__ chi_pad, const double* __restrict__ P,
                 const double* __restrict__ V0, const double* __restrict__ V1,
                 int* __restrict__ rec_k, double* __restrict__ rec_v, int* __restrict__ any,
                 double* __restrict__ partials) {
  constexpr int S = 2 + ND;
  constexpr int form = PRIM ? kFormPrim : kFormCons;
  const int64_t n = D == 0 ? g.nx : g.ny;          // cells along the sweep
  const int64_t lines = D == 0 ? g.ny : g.nx;
  const int bc = D == 0 ? g.bcx : g.bcy;
  const bool ring = bc == kBcPeriodic;
  // blocks go to the 8 XCDs in turn; each takes neighbouring groups of lines
  const int64_t total = gridDim.x, xcd = blockIdx.x % 8;
  const int64_t tile = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  const int64_t groups = (lines + kAdjWaves - 1) / kAdjWaves;
  const int t = (int)(threadIdx.x & 63);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // a workgroup's waves take neighbouring lines, or segments of the only one
  const int64_t seg = ND == 1 ? tile * kAdjWaves + w : tile / groups;
  const int64_t line_of = ND == 1 ? 0 : (tile % groups) * kAdjWaves + w;
  const bool live = ND == 1 ? seg * kAdjCells < n : line_of < lines;  // uniform over the wave
  const int64_t line = live ? line_of : lines - 1;
  const int64_t j = seg * kAdjCells - kAdjHalo + t;  // this lane's position
  // the cell it names, and whether it is one of the grid
  bool flip;
  const int64_t jc = ghost_index(j, n, bc, flip);
  const bool cell = ring || (j >= 0 && j < n);
  const int64_t xi = D == 0 ? jc : line, yi = D == 0 ? line : jc;
  const int64_t at = (yi * g.nx + xi) * g.es;
  // flattening factors exist for positions -1 .. n
  const int64_t jq = ring ? jc : (j < -1 ? -1 : (j > n ? n : j));
  const int64_t cxw = g.nx + 2;
  auto chi_at = [&](int64_t p) {
    const int64_t x = D == 0 ? p : line, y = D == 0 ? line : p;
    return (ND > 1 ? (y + 1) * cxw : 0) + x + 1;
  };
  double u0[S], la[S];
#pragma unroll
  for (int k = 0; k < S; ++k) u0[k] = g.U[at + k * g.cs];
#pragma unroll
  for (int k = 0; k < S; ++k) la[k] = lam[at + k * g.cs];
  const double chi = chi_pad[chi_at(jq)];
  const double dtdh = rec->dtdh;
  const double half_dtdh = 0.5 * dtdh;
  if (flip) reflect<double, ND>(u0, D);
#pragma unroll
  for (int k = 0; k < S; ++k) la[k] = cell ? la[k] : 0.0;

  // ---- forward: the face states of this cell, the flux of the face after it
  double R[S], L[S], G[S];
  {
    double um[S], up[S], Lc[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
      um[k] = below(u0[k]);
      up[k] = above(u0[k]);
    }
    evolve_faces<double, ND, D>(um, u0, up, chi, half_dtdh, limiter, form, m, R, Lc);
#pragma unroll
    for (int k = 0; k < S; ++k) L[k] = above(Lc[k]);
  }
  if constexpr (FLUX == kFluxHllc) hllc_flux<double, ND, D>(R, L, m, G);
  else force_flux<double, ND, D>(R, L, dtdh, 1.0 / dtdh, m, G);
  // ---- the face's adjoint; faces lie after positions -1 .. n - 1
  const bool face = ring || (j >= -1 && j < n);
  double mu[S], g_dtdh = 0.0, gR[S], gL[S];
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const double dl = above(la[k]) - la[k];
    mu[k] = dtdh * dl;
    g_dtdh += G[k] * dl;
    gR[k] = 0.0;
    gL[k] = 0.0;
  }
  GMat gm_face{0.0};
  if constexpr (FLUX == kFluxHllc) hllc_adj<ND, D>(R, L, m, mu, gR, gL, gm_face);
  else force_adj<ND, D>(R, L, dtdh, m, mu, gR, gL, g_dtdh, gm_face);
  // ---- the cell's adjoint, from the faces after and before it
  const bool state = ring || (j >= -1 && j <= n);
  GMat gm_cell{0.0};
  double g_half = 0.0, g_chi = 0.0, acc[S];
  {
    double um[S], up[S], gum[S], gup[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
      gR[k] = face ? gR[k] : 0.0;
      gL[k] = below(face ? gL[k] : 0.0);
      um[k] = below(u0[k]);
      up[k] = above(u0[k]);
      acc[k] = 0.0;
      gum[k] = 0.0;
      gup[k] = 0.0;
    }
    evolve_adj<ND, D>(um, u0, up, chi, half_dtdh, limiter, form, m, gR, gL, gum, acc, gup, g_half,
                      g_chi, gm_cell);
#pragma unroll
    for (int k = 0; k < S; ++k)
      acc[k] = (state ? acc[k] : 0.0) + above(state ? gum[k] : 0.0) + below(state ? gup[k] : 0.0);
  }
  // ---- what the ghost cells of the line's ends pass on to the cells they mirror
  if (!ring && (seg == 0 || (seg + 1) * kAdjCells >= n - 2)) {  // uniform
    const bool lo = j >= 0 && j <= 1, hi = j >= n - 2 && j < n;
    const int src_lo = lo ? t - (int)(2 * j + 1) : t;
    const int src_hi = hi ? t + (int)(2 * (n - j) - 1) : t;
    double add[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
      const double sgn = bc == kBcReflective && k == 2 + D ? -1.0 : 1.0;
      const double a = __shfl(acc[k], src_lo, 64), b = __shfl(acc[k], src_hi, 64);
      add[k] = (lo ? sgn * a : 0.0) + (hi ? sgn * b : 0.0);
    }
#pragma unroll
    for (int k = 0; k < S; ++k) acc[k] += add[k];
  }
  // ---- results: a segment's own cells, and at a line's ends its ghost cells
  const bool own = live && t >= kAdjHalo && t < kAdjHalo + kAdjCells && j < n;
  const bool before = live && j == -1, after = live && j == n && t > kAdjHalo &&
                                                t <= kAdjHalo + kAdjCells;
  if (own) {
#pragma unroll
    for (int k = 0; k < S; ++k) lam_in[at + k * g.cs] = la[k] + acc[k];
  }
  double s0 = 0.0, s1 = 0.0;
  if (own || (!ring && before)) {
    s0 += g_dtdh;
    s1 += gm_face.gamma;
  }
  if (own || (!ring && (before || after))) {
    s0 += 0.5 * g_half;
    s1 += gm_cell.gamma;
  }
  __shared__ double red[2][kAdjWaves];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s0 += __shfl_xor(s0, off, 64);
    s1 += __shfl_xor(s1, off, 64);
  }
  if (t == 0) {
    red[0][w] = s0;
    red[1][w] = s1;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double v = 0.0;
    for (int i = 0; i < kAdjWaves; ++i) v += red[threadIdx.x][i];
    partials[2 * blockIdx.x + threadIdx.x] = v;
  }
  if (own || before || after) {
    const int64_t q = chi_at(j);
    const double G = ring && !own ? 0.0 : g_chi;
    if (chi > 0.0 && chi < 1.0 && G != 0.0)
      chi_record<ND>(g, P, V0, V1, D == 0 ? j : line, D == 0 ? line : j, q, G, rec_k, rec_v, any);
    else
      rec_k[q] = -1;
  }
}

// Positions within 4 ghost cells of a line of n cells whose ghost rule maps
// to cell x (x itself first), at most 3.
__device__ __forceinline__ int alias_positions(int64_t x, int64_t n, int bc, int64_t* pos) {
  int k = 0;
  pos[k++] = x;
  int64_t cand[2];
  if (bc == kBcPeriodic) {
    cand[0] = x - n;
    cand[1] = x + n;
  } else {
    cand[0] = -x - 1;
    cand[1] = 2 * n - 1 - x;
  }
  for (int a = 0; a < 2; ++a) {
    const int64_t c = cand[a];
    if (c < -4 || c > n + 3 || (c >= 0 && c < n)) continue;
    bool flip;
    if (ghost_index(c, n, bc, flip) == x) pos[k++] = c;
  }
  return k;
}

// lambda += (dp/dU) times the pressure adjoints that the chi positions'
// selected factors pass to each cell (at the cell and at its ghost aliases,
// in a fixed order), and the gamma adjoint of the same terms (dp/dgamma)
// summed per workgroup into partials[2 b + 1] (partials[2 b] = 0).
// kPartialBlocks workgroups of 256 threads stride over the cells, so the sums
// have a fixed order; with no record at all (*any == 0) they only write
// zeros.
template <int ND, int D>
__global__ void __launch_bounds__(256) chi_gather_kernel(AGrid g, Material<double> m,
                                                         const int* __restrict__ rec_k,
                                                         const double* __restrict__ rec_v,
                                                         const int* __restrict__ any,
                                                         double* __restrict__ lam,
                                                         double* __restrict__ partials) {
  constexpr int S = 2 + ND;
  __shared__ double red[256];
  double acc = 0.0;
  const int64_t cx = g.nx + 2;
  if (*any) {
    for (int64_t cell = (int64_t)blockIdx.x * 256 + threadIdx.x; cell < g.nx * g.ny;
         cell += (int64_t)kPartialBlocks * 256) {
      const int64_t x = cell % g.nx, y = cell / g.nx;
      int64_t ax[3], ay[3] = {0, 0, 0};
      const int nax = alias_positions(x, g.nx, g.bcx, ax);
      const int nay = ND > 1 ? alias_positions(y, g.ny, g.bcy, ay) : 1;
      double gp = 0.0;
      for (int a = 0; a < nax; ++a)
        for (int b = 0; b < nay; ++b)
          for (int d = 0; d < ND; ++d) {
            const int64_t dx = (d == 0), dy = (d == 1);
            // a record at position c selecting K_d(c + jo) reaches the
            // pressure at c + jo + k, k in {-2, -1, 1, 2}: here t = jo + k
            for (int t = -3; t <= 3; ++t) {
              const int64_t qx = ax[a] - t * dx, qy = ay[b] - t * dy;
              // records lie on the grid's lines along D, and a cell past their ends
              if (D == 0 ? qx < -1 || qx > g.nx : qx < 0 || qx >= g.nx) continue;
              if (ND > 1 && (D == 1 ? qy < -1 || qy > g.ny : qy < 0 || qy >= g.ny)) continue;
              const int64_t qc = (ND > 1 ? (qy + 1) * cx : 0) + qx + 1;
              const int r = rec_k[qc];
              if (r < 0 || r / 4 != d) continue;
              const int k = t - (r % 4 - 1);
              if (k < -2 || k > 2 || k == 0) continue;
              gp += rec_v[4 * qc + (k < 0 ? k + 2 : k + 1)];
            }
          }
      if (gp != 0.0) {
        double u[S];
        const double* p = g.U + cell * g.es;
#pragma unroll
        for (int k = 0; k < S; ++k) u[k] = p[k * g.cs];
        // p = (gamma - 1) (E - rho |v|^2 / 2), v = m / rho
        const Prim<double, ND> w = prim_of<double, ND>(u, m);
        double v2 = 0.0;
#pragma unroll
        for (int i = 0; i < ND; ++i) v2 += w.vel[i] * w.vel[i];
        double* l = lam + cell * g.es;
        l[0] += gp * (m.gm1 * 0.5 * v2);
        l[1 * g.cs] += gp * m.gm1;
#pragma unroll
        for (int i = 0; i < ND; ++i) l[(2 + i) * g.cs] -= gp * (m.gm1 * w.vel[i]);
        acc += gp * (u[1] - 0.5 * u[0] * v2);
      }
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = 0.0;
    partials[2 * blockIdx.x + 1] = red[0];
  }
}

// Clears the argmax of n records.
__global__ void rec_clear_kernel(StepRec* rec, int64_t n) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) rec[k].argmax = ~0ull;
}

// Records a step's max wavespeed and dt/dh (its input g, the maximum in slot
// `slot`, its sweeps just run) and the lowest index of a cell whose wavespeed
// bits equal the maximum.
template <int ND>
__global__ void __launch_bounds__(256) record_kernel(AGrid g, Material<double> m,
                                                     const SimCtl* sim, int slot, StepRec* rec) {
  const unsigned long long target = sim->ws[slot];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    rec->maxws_bits = target;
    rec->dtdh = sim->c.dtdh;
  }
  unsigned long long best = ~0ull;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < g.nx * g.ny;
       i += (int64_t)gridDim.x * blockDim.x) {
    double u[2 + ND];
    const double* p = g.U + i * g.es;
#pragma unroll
    for (int k = 0; k < 2 + ND; ++k) u[k] = p[k * g.cs];
    const Prim<double, ND> w = prim_of<double, ND>(u, m);
    double ws = max_wavespeed<double, ND>(u, w, m);
    ws = ws == 0.0 ? 0.0 : ws;
    const unsigned long long b = (unsigned long long)__double_as_longlong(ws);
    if (b == target && (unsigned long long)i < best) best = (unsigned long long)i;
  }
  if (best != ~0ull) atomicMin(&rec->argmax, best);
}

// Sums the partials of the step's sweeps, turns the dt/dh adjoint
// into the max-wavespeed adjoint (d(dt/dh)/d maxws = -(dt/dh)/maxws), adds
// that cell's wavespeed adjoint into lambda_n and accumulates the gamma
// adjoint.  One workgroup of 256 threads.
template <int ND>
__global__ void __launch_bounds__(256) finalize_kernel(AGrid g, Material<double> m,
                                                       const StepRec* __restrict__ rec,
                                                       Partials parts,
                                                       double* __restrict__ lam_n,
                                                       double* __restrict__ acc) {
  __shared__ double s0[256], s1[256];
  double a0 = 0.0, a1 = 0.0;
  for (int i = 0; i < 4; ++i)
    for (int b = threadIdx.x; b < parts.n[i]; b += 256) {
      a0 += parts.p[i][2 * b];
      a1 += parts.p[i][2 * b + 1];
    }
  s0[threadIdx.x] = a0;
  s1[threadIdx.x] = a1;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s0[threadIdx.x] += s0[threadIdx.x + w];
      s1[threadIdx.x] += s1[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  const double g_dtdh = s0[0];
  const double maxws = __longlong_as_double((long long)rec->maxws_bits);
  const double g_maxws = -g_dtdh * rec->dtdh / maxws;
  GMat gm{0.0};
  const unsigned long long c = rec->argmax;
  if (c < (unsigned long long)(g.nx * g.ny)) {
    double u[2 + ND], gu[2 + ND];
    const double* p = g.U + (int64_t)c * g.es;
#pragma unroll
    for (int k = 0; k < 2 + ND; ++k) {
      u[k] = p[k * g.cs];
      gu[k] = 0.0;
    }
    wavespeed_adj<ND>(u, m, g_maxws, gu, gm);
    double* l = lam_n + (int64_t)c * g.es;
#pragma unroll
    for (int k = 0; k < 2 + ND; ++k) l[k * g.cs] += gu[k];
  }
  acc[0] += s1[0] + gm.gamma;
  acc[1] = g_dtdh;
}

__global__ void acc_clear_kernel(double* acc) {
  acc[0] = 0.0;
  acc[1] = 0.0;
}

#define FL_SWEEP_INST(ND, D, FLUX, PRIM)                                                     \
  template __global__ void sweep_adj_kernel<ND, D, FLUX, PRIM>(                               \
      AGrid, const double*, double*, Material<double>, int, const StepRec*, const double*,     \
      const double*, const double*, const double*, int*, double*, int*, double*);
#define FL_ADJ_INST(ND, D)                                                                  \
  FL_SWEEP_INST(ND, D, kFluxHllc, false)                                                     \
  FL_SWEEP_INST(ND, D, kFluxForce, false)                                                    \
  FL_SWEEP_INST(ND, D, kFluxHllc, true)                                                      \
  FL_SWEEP_INST(ND, D, kFluxForce, true)                                                     \
  template __global__ void chi_gather_kernel<ND, D>(AGrid, Material<double>, const int*,      \
                                                    const double*, const int*, double*, double*);

FL_ADJ_INST(1, 0)
FL_ADJ_INST(2, 0)
FL_ADJ_INST(2, 1)
template __global__ void prim_pad_kernel<1>(AGrid, Material<double>, double*, double*, double*);
template __global__ void prim_pad_kernel<2>(AGrid, Material<double>, double*, double*, double*);
template __global__ void chi_pad_kernel<1>(AGrid, const double*, const double*, const double*,
                                           double*, int*);
template __global__ void chi_pad_kernel<2>(AGrid, const double*, const double*, const double*,
                                           double*, int*);
template __global__ void record_kernel<1>(AGrid, Material<double>, const SimCtl*, int, StepRec*);
template __global__ void record_kernel<2>(AGrid, Material<double>, const SimCtl*, int, StepRec*);
template __global__ void finalize_kernel<1>(AGrid, Material<double>, const StepRec*,
                                            Partials, double*, double*);
template __global__ void finalize_kernel<2>(AGrid, Material<double>, const StepRec*,
                                            Partials, double*, double*);

}  // namespace adj
}  // namespace fl
