// fl_levelset.hpp -- argument blocks and declarations of the level-set and
// ghost-fluid kernels (fl_levelset.hip), shared with the C ABI host code.
#pragma once

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

namespace fl {
namespace ls {

struct Grid {
  int64_t nx, ny;  // ny = 1 in 1D
  int nd;
  int pad;
};

// A conservative state grid: element stride and component stride in
// elements (AoS: es = S, cs = 1; SoA: es = 1, cs = cells).  f32: the grid
// holds floats (the FP32 bulk path); the level-set kernels compute in FP64
// and convert on load and store.
struct StateView {
  double* data;
  int64_t es, cs;
  int f32;
  int pad;
};

// Sweeps of an eikonal launch, its workgroups' threads and the tiles of each.
// A solve of two 384x192 level sets, 23 sweeps: 104 us of kernels with a launch
// a sweep, 60 with four to a launch on tiles of 32 x 16 cells.
constexpr int kEikSteps = 4;
constexpr int kEikThreads = 512;
constexpr int eik_tile_w(int nd) { return nd == 1 ? kEikThreads : 32; }
constexpr int eik_tile_h(int nd) { return kEikThreads / eik_tile_w(nd); }

// Bits of a tile: it holds a source; it is on the list.
constexpr unsigned kEikSource = 1u, kEikActive = 2u;

// Control words of the eikonal Jacobi loop.
struct EikCtl {
  int flags[3][kEikSteps];  // by launch % 3: sweep s of the launch changed a cell
  int done;
  int launches;   // launches that swept
  int appended;   // entries of the job's active-tile list
  int ntiles[2];  // those that a launch visits, by launch & 1
};

// One eikonal reinitialisation: the level set in, its two Jacobi distance
// buffers, per-cell info bytes, the tile flags, its loop control and the
// result.  Launches carry up to two jobs; blockIdx.z selects one.
struct EikJob {
  const double* phi;
  double* d[2];
  uint8_t* info;
  unsigned* tile;  // per tile: kEikSource | kEikActive
  int* list;       // the tiles a sweep visits, in no particular order
  EikCtl* ctl;
  double* out;
  uint8_t* band_mask;  // nullable
};
struct EikJobs {
  EikJob j[2];
};

struct Eos {
  double gamma, p_inf;
  int stiff;  // either stiffened gas (energy and sound speed with p_inf)
  int corr;   // corrected stiffened gas: pressure minus gamma p_inf
};

// Materials of an n-material step (n <= kMaxMat): level sets, states and
// equations of state, passed by value to the kernels that read all of them.
constexpr int kMaxMat = 8;
struct MatSet {
  int nmat;
  int pad;
  const double* phi[kMaxMat];
  StateView u[kMaxMat];
  Eos e[kMaxMat];
};
struct PhiSet {
  int nmat;
  int pad;
  double* phi[kMaxMat];
};

__global__ void masks_kernel(const double* phi, Grid g, double dh, uint8_t* masks);
template <int ND>
__global__ void gfm_star_n_kernel(MatSet ms, int m, Grid g, double dh, double* star,
                                  uint8_t* has_star, int* count_reset);
template <int ND>
__global__ void velocity_n_kernel(MatSet ms, int target, Grid g, double dh, double* V);
__global__ void project_n_kernel(PhiSet ps, int64_t count);
template <int ND>
__global__ void velocity_kernel(const double* phi0, const double* phi1, StateView u0,
                                StateView u1, int nmat, Grid g, double dh, int target, double* V);
__global__ void project2_kernel(double* phi0, double* phi1, int64_t count);
// One level set's RK3 stage: phi_n, the stage source, the speed and the output.
struct Rk3Job {
  const double* phi_n;
  const double* src;
  const double* V;
  double* out;
};
// Launched on (ceil(nx / 64), ceil(ny / (4 rows))) workgroups of 256 threads
// (rk3_stage2_kernel: z = 2, a level set each).
template <int ND, bool FAST>
__global__ void rk3_stage2_kernel(int stage, Rk3Job j0, Rk3Job j1, Grid g, int rows,
                                  const double* dt_dev, double h1);
template <int ND, bool FAST>
__global__ void rk3_first2_kernel(Rk3Job j0, Rk3Job j1, double* V0, double* V1, StateView u0,
                                  StateView u1, Grid g, int rows, const double* dt_dev, double dh,
                                  double h1);
template <int ND, bool FAST>
__global__ void rk3_last2_kernel(Rk3Job j0, Rk3Job j1, Grid g, int rows, const double* dt_dev,
                                 double h1);
template <int ND>
__global__ void rk3_stage_kernel(int stage, const double* phi_n, const double* src,
                                 const double* V, Grid g, double dt, const double* dt_dev,
                                 double h1, double* out);
template <int ND>
__global__ void eik_init_kernel(EikJobs jobs, Grid g, int64_t trows);
__global__ void eik_tile_act_kernel(EikJobs jobs, int64_t trows, int64_t segs, int tr_r,
                                    int segs_r);
// Workgroups per job of a sweep launch, which stride over the active tiles.
constexpr int kEikSweepGroups = 512;
template <int ND>
__global__ void eik_sweep_kernel(EikJobs jobs, Grid g, int64_t segs, double dh, double limit,
                                 int launch);
__global__ void eik_finish_kernel(EikJobs jobs, Grid g, double limit, double clamp);
template <int ND>
__global__ void gfm_star_kernel(const double* phi_m, const double* phi_o, StateView um,
                                StateView uo, Eos em, Eos eo, Grid g, double dh, double* star,
                                uint8_t* has_star, int* count_reset);
// Both materials of a two-material step in one pass each.
// One extrapolation job: a material's level set and state, its two Jacobi
// buffers (AoS), and its band list with the list's count.
struct ExtrapJob {
  const double* phi;
  StateView um;
  double* A;
  double* B;
  int* list;  // written by the band seed, read by the sweeps
  int* count;
};
constexpr int kExtrapBlocks = 128;  // workgroups per job of one sweep launch
// The cells of a material that take star states.
struct StarJob {
  int* list;
  int* count;
};

template <int ND>
__global__ void gfm_band_seed_kernel(const double* phi_m, double upper, StateView um,
                                     const double* star, const uint8_t* has_star, Grid g,
                                     double* A, double* B, int* list, int* count);
template <int ND>
__global__ void gfm_band_seed2_kernel(ExtrapJob j0, ExtrapJob j1, double upper,
                                      const double* star0, const double* star1,
                                      const uint8_t* has0, const uint8_t* has1, Grid g);
template <int ND>
__global__ void gfm_seed2_kernel(ExtrapJob j0, ExtrapJob j1, double upper, StarJob s0, StarJob s1,
                                 Grid g, double dh);
template <int ND>
__global__ void gfm_star_list_kernel(ExtrapJob j0, ExtrapJob j1, StarJob s0, StarJob s1, Eos e0,
                                     Eos e1, Grid g, double dh);
__global__ void count_clear_kernel(int* count);
template <int ND>
__global__ void gfm_extrap_kernel(ExtrapJob j0, ExtrapJob j1, Grid g, double dh, int sweep,
                                  int last);
template <int ND>
__global__ void combine_kernel(const double* phi0, StateView u0, StateView u1, Grid g,
                               StateView out);

}  // namespace ls
}  // namespace fl
