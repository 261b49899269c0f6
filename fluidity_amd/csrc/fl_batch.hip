// fl_batch.hip -- persistent kernels of the batched Euler step.
//
// A step of a batch is three launches, captured once in a hipGraph and
// replayed: the control kernel (one thread per problem: dt from the problem's
// fused maximum wavespeed, its run time and iteration count, as
// Parameters::update_time_delta / dt_dh / update_simulation_info,
// simulator/parameters.hpp:60-99), then one launch per sweep phase.  Phase 0
// runs the x sweep of every 2D problem and the whole step of every 1D problem;
// phase 1 runs the y sweep of every 2D problem.  Problems of very different
// sizes share a phase's list of tiles, largest problems first: cell-parallel
// tiles, one per workgroup, or marching tiles, which persistent workgroups
// take from a counter.  1D problems run register tiles (one segment a wave)
// beside the first and marching ones (eight segments in turn) beside the
// second.  Tile bodies are those of the single-grid sweeps
// (fl_sweep_tiles.hpp), so every problem's result is the single-grid result
// bit for bit.
#include "fl_batch.hpp"
#include "fl_sweep_tiles.hpp"

namespace fl {
namespace batch {

__global__ void init_kernel(StepCtl* ctls, int nprob) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nprob) return;
  StepCtl& c = ctls[i];
  c.ws_bits[0] = 0ull;
  c.ws_bits[1] = 0ull;
  c.dt = 0.0;
  c.dtdh = 0.0;
  c.t = 0.0;
  c.iters = 0;
  c.active = 1;
  c.pad = 0;
}

// The step's parity comes from each problem's own iteration count: the
// previous step's fused maximum sits in ws_bits[iters & 1] and this step's
// sweeps write ws_bits[(iters + 1) & 1].
__global__ void control_kernel(StepCtl* ctls, const Params* params, int nprob, Counters* cnt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    cnt->next[0] = 0;
    cnt->next[1] = 0;
  }
  if (i >= nprob) return;
  StepCtl& c = ctls[i];
  const Params p = params[i];
  const bool active = c.t < p.sim_time && c.iters < p.max_iters;
  if (active) {
    const int parity = (int)(c.iters & 1);
    const double maxws = __longlong_as_double((long long)c.ws_bits[parity]);
    const double dt = p.cfl * p.dh / maxws;
    c.dt = dt;
    c.dtdh = dt / p.dh;
    c.t += dt;
    c.iters += 1;
    c.ws_bits[parity ^ 1] = 0ull;
  }
  c.active = active ? 1 : 0;
}

// What control_kernel clears, before a timed phase.
__global__ void reset_counters_kernel(StepCtl* ctls, int nprob, Counters* cnt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    cnt->next[0] = 0;
    cnt->next[1] = 0;
  }
  if (i < nprob) ctls[i].ws_bits[(ctls[i].iters & 1) ^ 1] = 0ull;
}

// Sweep arguments of a problem in a phase (ND = 1 or 2: of which kind it is).
// timing != 0 runs every tile state -> work with a fixed dt/dh (launch-shape
// measurement; the states are not modified), the maximum of a step's last sweep
// into the slot that the next step's control clears: left out, register tiles
// of lines, an atomic each 448 cells, won phases that they are not the fastest
// in (512 problems in FP32 746 us a step against 650).
template <typename T, int ND, int PHASE>
__device__ __forceinline__ SweepArgs<T> phase_args(const Prob<T>& P, int timing, T timing_dtdh) {
  SweepArgs<T> a = P.x;
  // Known to the compiler, or the kernels keep sweep_begin and its registers: the
  // fast FP64 x phase then fits two waves per SIMD instead of three (200 planes
  // of 424^2 in marching tiles 1985 us a step against 1830), FP32 with it took
  // 1020 against 965.
  a.sim = nullptr;
  a.ws_out = nullptr;
  if (PHASE == 1) a.rows_per_block = P.rows_y;
  if (timing) {
    a.ctl = nullptr;
    a.dtdh_host = timing_dtdh;
    if (PHASE == 1 || ND == 1) a.ws_out = &P.ctl->ws_bits[(P.ctl->iters & 1) ^ 1];
  } else if (PHASE == 1) {
    a.in = P.x.out;
    a.out = const_cast<T*>(P.x.in);
    a.ws_out = &P.ctl->ws_bits[P.ctl->iters & 1];
  } else if (ND == 1) {
    const long long it = P.ctl->iters;  // already advanced by this step's control
    if ((it - 1) & 1) {                 // odd steps run work -> state
      a.in = P.x.out;
      a.out = const_cast<T*>(P.x.in);
    }
    a.ws_out = &P.ctl->ws_bits[it & 1];
  }
  return a;
}

// Persistent sweep phase: marching tiles, taken from the phase's counter.
// FAST: the fast FP64 numerics (FP32 has its own forms); VLC: every problem
// limits with van Leer in conservative form; WIDE: every 2D problem is
// SweepArgs::wide (fixed at compile time, as in the single-grid sweeps).
// The fast FP64 x phase is asked for three waves per SIMD, whose registers it is
// one or two short of where the limiter is chosen at run time.
template <typename T, int FLUX, int PHASE, bool FAST, bool VLC, bool WIDE>
__global__ void __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(
    sizeof(T) == 8 && FAST && PHASE == 0 ? 3 : SweepWaves<T>::value)))
phase_kernel(const Prob<T>* __restrict__ probs, const Tile* __restrict__ tiles, int ntiles,
             Counters* __restrict__ cnt, int timing, T timing_dtdh) {
  __shared__ int s_tile;
  for (;;) {
    if (threadIdx.x == 0) s_tile = atomicAdd(&cnt->next[PHASE], 1);
    __syncthreads();
    const int tile = __builtin_amdgcn_readfirstlane(s_tile);
    __syncthreads();
    if (tile >= ntiles) break;
    const Tile td = tiles[tile];
    const Prob<T>& P = probs[td.prob];
    if (PHASE == 1)
      sweep_y_tile<T, FLUX, FAST, VLC, WIDE>(phase_args<T, 2, 1>(P, timing, timing_dtdh), td.bx, td.by);
    else if (P.nd == 1)
      sweep_x_tile<T, 1, FLUX, FAST, VLC, false>(phase_args<T, 1, 0>(P, timing, timing_dtdh),
                                                 td.bx, 0);
    else
      sweep_x_tile<T, 2, FLUX, FAST, VLC, WIDE>(phase_args<T, 2, 0>(P, timing, timing_dtdh), td.bx,
                                          td.by);
    __syncthreads();  // the next tile reuses the LDS
  }
}

// Sweep phase of cell-parallel tiles, one per workgroup (32 lines of up to
// 65536 cells beside 16 planes of up to 1024^2: 275 -> 175 us a phase; a line
// marched eight segments of 254 cells one after the other, 120 us when alone).
template <typename T, int FLUX, int PHASE, bool FAST, bool VLC, bool WIDE>
__global__ void __launch_bounds__(64 * kCellWaves) __attribute__((amdgpu_waves_per_eu(4)))
cell_phase_kernel(const Prob<T>* __restrict__ probs, const Tile* __restrict__ tiles, int timing,
                  T timing_dtdh) {
  const Tile td = tiles[blockIdx.x];
  const Prob<T>& P = probs[td.prob];
  if (PHASE == 1)
    cell_y_tile<T, FLUX, FAST, VLC, WIDE>(phase_args<T, 2, 1>(P, timing, timing_dtdh), td.bx, td.by);
  else if (P.nd == 1)
    line_tile<T, FLUX, FAST, VLC>(phase_args<T, 1, 0>(P, timing, timing_dtdh), td.bx);
  else
    cell_x_tile<T, FLUX, FAST, VLC, WIDE>(phase_args<T, 2, 0>(P, timing, timing_dtdh), td.bx, td.by);
}

// 1D problems that ran an odd number of steps hold their result in the work
// buffer.  dir 0 copies it to the state buffer; dir 1 copies the state buffer
// back to the work buffer (after the work buffers were used as scratch).
// One workgroup per problem.
template <typename T>
__global__ void __launch_bounds__(256) finish_kernel(const Prob<T>* __restrict__ probs, int nprob,
                                                     int dir) {
  const int p = blockIdx.x;
  if (p >= nprob) return;
  const Prob<T>& P = probs[p];
  if (P.nd != 1 || !(P.ctl->iters & 1)) return;
  const int64_t n = P.x.nx;
  const T* src = dir == 0 ? P.x.out : P.x.in;
  T* dst = dir == 0 ? const_cast<T*>(P.x.in) : P.x.out;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    T u[3];
    load_cell<T, 3>(src, i, P.x.es, P.x.cs, u);
    store_cell<T, 3>(dst, i, P.x.es, P.x.cs, u);
  }
}

// FP64 sums of each conserved component of each problem's state (4 slots per
// problem, the fourth 0 in 1D).  One workgroup per problem; the order of
// additions is fixed, so the sums are reproducible.
template <typename T>
__global__ void __launch_bounds__(256) sums_kernel(const Prob<T>* __restrict__ probs, int nprob,
                                                   double* __restrict__ sums) {
  __shared__ double red[4][256];
  const int p = blockIdx.x;
  if (p >= nprob) return;
  const Prob<T>& P = probs[p];
  const int S = 2 + P.nd;
  const int64_t n = P.x.nx * P.x.ny;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const T* c = P.x.in + i * P.x.es;
    for (int k = 0; k < S; ++k) acc[k] += (double)c[k * P.x.cs];
  }
  for (int k = 0; k < 4; ++k) red[k][threadIdx.x] = acc[k];
  __syncthreads();
  if (threadIdx.x < 4) {
    double v = 0.0;
    for (int j = 0; j < (int)blockDim.x; ++j) v += red[threadIdx.x][j];
    sums[p * 4 + threadIdx.x] = v;
  }
}

#define FL_BATCH_PHASE(T, FLUX, PHASE, FAST, VLC, WIDE)                             \
  template __global__ void phase_kernel<T, FLUX, PHASE, FAST, VLC, WIDE>(        \
      const Prob<T>*, const Tile*, int, Counters*, int, T);                      \
  template __global__ void cell_phase_kernel<T, FLUX, PHASE, FAST, VLC, WIDE>(   \
      const Prob<T>*, const Tile*, int, T);
#define FL_BATCH_PHASES_W(T, FAST, VLC, WIDE)        \
  FL_BATCH_PHASE(T, kFluxHllc, 0, FAST, VLC, WIDE)   \
  FL_BATCH_PHASE(T, kFluxHllc, 1, FAST, VLC, WIDE)   \
  FL_BATCH_PHASE(T, kFluxForce, 0, FAST, VLC, WIDE)  \
  FL_BATCH_PHASE(T, kFluxForce, 1, FAST, VLC, WIDE)
#define FL_BATCH_PHASES(T, FAST, VLC)      \
  FL_BATCH_PHASES_W(T, FAST, VLC, false)   \
  FL_BATCH_PHASES_W(T, FAST, VLC, true)
#define FL_BATCH_INST(T)                                                                     \
  FL_BATCH_PHASES(T, false, false)                                                           \
  FL_BATCH_PHASES(T, false, true)                                                            \
  template __global__ void finish_kernel<T>(const Prob<T>*, int, int);                        \
  template __global__ void sums_kernel<T>(const Prob<T>*, int, double*);

FL_BATCH_INST(double)
FL_BATCH_INST(float)
// the fast FP64 numerics
FL_BATCH_PHASES(double, true, false)
FL_BATCH_PHASES(double, true, true)

}  // namespace batch
}  // namespace fl
