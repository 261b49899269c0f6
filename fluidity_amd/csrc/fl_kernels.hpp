// fl_kernels.hpp -- argument blocks shared by the gfx950 kernels and the
// host-side launch code of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fl_numerics.hpp"

namespace fl {

// Device-resident step control.  One instance drives a whole simulation so
// that the time-step loop never synchronises with the host: the control
// kernel turns the fused maximum wavespeed into dt and dt/dh exactly as
// Parameters::update_time_delta / dt_dh do (simulator/parameters.hpp:60-99)
// and advances run_time / iters (:67-71).
struct StepCtl {
  unsigned long long ws_bits[2];  // max wavespeed as bits, ping-pong by step parity
  double dt;
  double dtdh;
  double t;                       // run time
  long long iters;
  int active;                     // run_time < sim_time && iters < max_iters
  int pad;
};

// Device-resident control of fl_simulate's launched steps.  The first sweep of
// step k takes dt from the maximum itself (sweep_begin), so a step is its
// sweeps and nothing else: every workgroup reads t[k & 1], iters[k & 1] and
// the maximum ws[k % n] (n = 2 slots on 2D grids, 3 on 1D ones, where one
// sweep reads the maximum and reduces the next) and computes the same dt; the
// first workgroup writes the other halves, the block that the step's second
// sweep reads and the zero of a slot that nobody reads or reduces into in
// this sweep.
struct SimCtl {
  StepCtl c;         // dt, dtdh, active of the step; t and iters after it
  double t[2];       // run time before step k in t[k & 1]
  long long iters[2];
  // maximum wavespeeds as bits, on a cache line that no sweep reads dt from
  // while others reduce into it
  alignas(128) unsigned long long ws[3];
};

// Loop state of the persistent 1D step loop (persist1d_kernel) between its
// launches, and its timeout flag.
struct PersistCtl {
  unsigned long long ws;  // maximum wavespeed of the state as bits
  double t;
  long long iters;
  double dt;              // last step's
  int err;
  int pad;
};

template <typename T>
struct SweepArgs {
  const T* in;
  T* out;
  int64_t es;          // element stride (in T units): S for AoS, 1 for SoA
  int64_t cs;          // component stride: 1 for AoS, nx*ny for SoA
  int64_t rowb;        // bytes from one row to the next
  int64_t csb;         // component stride in bytes
  int64_t nx, ny;      // interior cells
  Material<T> mat;     // material in the sweep precision
  Material<double> mat64;  // FP64 material for the fused wavespeed
  int limiter, form;
  int bcx, bcy;
  int rows_per_block;  // row chunk marched by one workgroup
  int wide;            // 2D: both grids AoS, every cell at a multiple of 16 bytes
  T dtdh_host;         // used when ctl == nullptr
  const StepCtl* ctl;  // nullable: provides dtdh and the active flag
  // nullable: the first sweep of a step of fl_simulate, which turns the
  // maximum into dt (ctl unused)
  SimCtl* sim;
  int sim_half, sim_ws, sim_zero;  // k & 1, the slot read, the slot cleared
  int pad2;
  double cfl, dh, sim_time;
  long long max_iters;
  unsigned long long* ws_out;  // nullable: fused max wavespeed (bit pattern)
};

// Maximum workgroup width of the sweep kernels (LDS arrays are sized for it).
constexpr int kMaxBlock = 256;
constexpr int kMaxWaves = 8;  // waves of the widest workgroup (the cell-parallel sweeps')
constexpr int kHalo = 3;  // extra cells each side staged in LDS for chi

// Dynamic LDS of an x-sweep tile of B lanes over states of S components of
// tsize bytes: S + 3 rows of B + 2 kHalo staged columns, 2 S rows of B.
__host__ __device__ constexpr size_t x_tile_lds_bytes(int B, int S, int tsize) {
  return (size_t)((S + 3) * (B + 2 * kHalo) + 2 * S * B) * (size_t)tsize;
}

// Dynamic LDS of a y-sweep tile of B lanes (2D states, 4 components of tsize
// bytes): 3 rows of B + 2 kHalo columns, a ring of kYRing rows of 4 x B.
constexpr int kYRing = 5;
__host__ __device__ constexpr size_t y_tile_lds_bytes(int B, int tsize) {
  return (size_t)(3 * (B + 2 * kHalo) + kYRing * 4 * B) * (size_t)tsize;
}

// Cell-parallel 2D sweeps: kCellWaves waves per workgroup, one row of 64
// columns each.  LDS of FP size tsize: pressures and y velocities of
// kCellWaves + 6 rows, x velocities of kCellWaves rows (columns with their
// halo where the x direction reads it), one state per thread.
constexpr int kCellWaves = 8;
constexpr int kCellCols = 64 + 2 * kHalo;  // columns of a staged row with its halo
__host__ __device__ constexpr size_t cell_tile_lds_bytes(int tsize) {
  return (size_t)((kCellWaves + 6) * (kCellCols + 64) + kCellWaves * (kCellCols + 4 * 64)) *
         (size_t)tsize;
}
// Cells of one tile: 62 columns x kCellWaves rows (x sweep), 64 columns x
// kCellWaves - 2 rows (y sweep).
constexpr int kCellXCols = 62, kCellXRows = kCellWaves;
constexpr int kCellYCols = 64, kCellYRows = kCellWaves - 2;

// Blocks of a cell-parallel launch up to which each issues its atomicMax
// unseen (two rounds of the blocks the device holds).
constexpr unsigned kCellFewBlocks = 1024;

// Persistent 1D loop: cells of a wave's segment (4 lanes on either side hold
// the neighbours'), waves of a workgroup, workgroups and the words each
// publishes per step (the maximum, and 3 values of 4 cells at either end).
constexpr int kLineCells = 56;
constexpr int kPersistMaxWaves = 16;
constexpr int kPersistMaxGroups = 4 * 64;
constexpr int kPersistWords = 25;

// Standalone wavespeed max: at most kMaxWsBlocks workgroups of kMaxBlock
// threads, each thread loading kMaxWsUnroll cells per iteration.
constexpr int kMaxWsBlocks = 512;
constexpr int kMaxWsUnroll = 4;

}  // namespace fl

// Kernels defined in fl_sweep.hip (explicitly instantiated there).  WIDE:
// every grid of the launch is SweepArgs::wide.
namespace fl {
template <typename T, int ND, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void sweep_x_kernel(SweepArgs<T> a);
template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void sweep_y_kernel(SweepArgs<T> a);
template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void cell_x_kernel(SweepArgs<T> a0, SweepArgs<T> a1);
template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void cell_y_kernel(SweepArgs<T> a0, SweepArgs<T> a1);
template <typename T, int ND, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void sweep_x2_kernel(SweepArgs<T> a0, SweepArgs<T> a1);
template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
__global__ void sweep_y2_kernel(SweepArgs<T> a0, SweepArgs<T> a1);
template <typename T, int ND, bool FAST>
__global__ void max_wavespeed2_kernel(const T* in0, const T* in1, int64_t es0, int64_t cs0,
                                      int64_t es1, int64_t cs1, int64_t ncells,
                                      Material<double> m0, Material<double> m1,
                                      unsigned long long* dst);
template <typename T, int ND>
__global__ void max_wavespeed_kernel(const T* in, int64_t es, int64_t cs, int64_t ncells,
                                     Material<double> m64, unsigned long long* dst);
template <typename T, int S>
__global__ void component_sums_kernel(const T* in, int64_t es, int64_t cs, int64_t ncells,
                                      double* partial);
template <typename T, int ND>
__global__ void wavespeeds_kernel(const T* in, int64_t es, int64_t cs, int64_t ncells,
                                  Material<double> m64, double* ws);
__global__ void max_element_kernel(const double* v, int64_t n, unsigned long long* dst);
__global__ void zero_u64_kernel(unsigned long long* p);
__global__ void init_sim_kernel(SimCtl* sim);
// Counts that a two-material step clears for the next one (nullable).
struct MmCounts {
  int* p[4];
};
__global__ void mm_init_kernel(StepCtl* ctl, MmCounts counts);
__global__ void mm_control_kernel(StepCtl* ctl, double cfl, double dh, MmCounts counts);
template <typename T, int FLUX, bool FAST, bool VLC>
__global__ void persist1d_kernel(SweepArgs<T> a, PersistCtl* pc, unsigned long long* words,
                                 int nseg, double cfl, double dh, double sim_time,
                                 long long max_iters, long long nsteps, int first,
                                 unsigned int spin_limit);
__global__ void persist_init_kernel(PersistCtl* pc, unsigned long long* words, int count,
                                    int first);
}  // namespace fl
