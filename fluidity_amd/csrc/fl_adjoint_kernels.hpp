// fl_adjoint_kernels.hpp -- argument blocks and declarations of the adjoint
// kernels (fl_adjoint.hip), shared with the C ABI host code.
#pragma once

#include "fl_kernels.hpp"

namespace fl {
namespace adj {

// An FP64 grid (state or adjoint field; both use the same strides).
struct AGrid {
  const double* U;
  int64_t es, cs;   // element and component strides
  int64_t nx, ny;
  int bcx, bcy;
};

// What the backward pass needs of one forward step.
struct StepRec {
  unsigned long long maxws_bits;  // max wavespeed of the step's input state
  double dtdh;                    // dt/dh the step's sweeps used
  unsigned long long argmax;      // lowest cell index attaining the maximum
  double pad;
};

constexpr int kPartialBlocks = 256;

// Waves of a sweep workgroup (a line each), the cells of a line that a wave
// takes, and those on either side that its lanes hold as well: the reverse of
// the cell before needs that of the face before it, whose left state is that
// of the cell before that.
constexpr int kAdjWaves = 4;
constexpr int kAdjHalo = 3;
constexpr int kAdjCells = 64 - 2 * kAdjHalo;

// (dt/dh, gamma) sums of a step, up to four lists of pairs.
struct Partials {
  const double* p[4];
  int n[4];
};

template <int ND>
__global__ void prim_pad_kernel(AGrid g, Material<double> m, double* P, double* V0, double* V1);
template <int ND>
__global__ void chi_pad_kernel(AGrid g, const double* P, const double* V0, const double* V1,
                               double* chi, int* any);
template <int ND, int D, int FLUX, bool PRIM>
__global__ void sweep_adj_kernel(AGrid g, const double* lam, double* lam_in, Material<double> m,
                                 int limiter, const StepRec* rec, const double* chi_pad,
                                 const double* P, const double* V0, const double* V1, int* rec_k,
                                 double* rec_v, int* any, double* partials);
template <int ND, int D>
__global__ void chi_gather_kernel(AGrid g, Material<double> m, const int* rec_k,
                                  const double* rec_v, const int* any, double* lam,
                                  double* partials);
__global__ void rec_clear_kernel(StepRec* rec, int64_t n);
template <int ND>
__global__ void record_kernel(AGrid g, Material<double> m, const SimCtl* sim, int slot,
                              StepRec* rec);
template <int ND>
__global__ void finalize_kernel(AGrid g, Material<double> m, const StepRec* rec,
                                Partials parts, double* lam_n, double* acc);
__global__ void acc_clear_kernel(double* acc);

}  // namespace adj
}  // namespace fl
