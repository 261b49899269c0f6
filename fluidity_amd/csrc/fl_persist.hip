// fl_persist.hip -- the step loop of a short 1D line in one launch.
//
// The reference's loop (simulator/simulator_impl.hpp:235-252) on a line of at
// most kPersistMaxCells cells.  A step there is latency: one cell's dependent
// arithmetic, and the exchange of the maximum wavespeed and of the segments'
// edges.  The line is cut into segments of at most kLineCells cells, one
// per wave; a lane holds its cell in registers for the whole loop, and four
// lanes on either side hold the neighbours' cells, so a step reads and writes
// no state.  Neighbours in a wave pass through DPP moves, waves of a workgroup
// through LDS, workgroups through words in device memory.
//
// Exchange between workgroups.  Before step k every workgroup publishes its
// maximum wavespeed and its four first and four last cells as 64-bit words,
// each a relaxed agent-scope atomic store (no fence, no counter), and polls
// the words of the others until none holds the value kEmpty; the maximum of
// all and the neighbours' cells then start the step.  A word is its own flag,
// so a step costs one store and one load through device memory; a barrier
// (atomic counter between release and acquire fences, then the loads of the
// state) cost three to four.  A step in FP64 HLLC: 100 cells 6.1 -> 2.3 us,
// 4096 cells 7.3 -> 4.6, 14000 cells 13.3 -> 5.1, 65536 cells 83 -> 6.6 (the
// barrier's counter took one atomic of 1058 workgroups).  Words go to
// the slots k % 3 in turn.  In step k, after its polls, a workgroup empties
// its words of slot (k + 2) % 3, which holds the publication of step k - 1:
// everyone has published k, so everyone is done with k - 1; and it waits for
// these stores before it publishes step k + 1, so whoever has seen that
// publication cannot take an old word of slot (k + 2) % 3 for a new one.
#include "fl_sweep_tiles.hpp"

namespace fl {

namespace {

constexpr int kPolls = kPersistMaxGroups / 64;  // maxima a lane polls
constexpr unsigned long long kEmpty = ~0ull;  // a NaN that no published word keeps

// Maximum over the wave, in every lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long max_dpp(unsigned long long v) {
  const unsigned lo =
      (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)v, (int)(unsigned)v, CTRL, ROWS, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(
      (int)(unsigned)(v >> 32), (int)(unsigned)(v >> 32), CTRL, ROWS, 0xf, false);
  const unsigned long long o = ((unsigned long long)hi << 32) | lo;
  return o > v ? o : v;
}
__device__ __forceinline__ unsigned long long wave_max_dpp(unsigned long long v) {
  v = max_dpp<0x111, 0xf>(v);  // row_shr:1
  v = max_dpp<0x112, 0xf>(v);  // row_shr:2
  v = max_dpp<0x114, 0xf>(v);  // row_shr:4
  v = max_dpp<0x118, 0xf>(v);  // row_shr:8
  v = max_dpp<0x142, 0xa>(v);  // row_bcast:15
  v = max_dpp<0x143, 0xc>(v);  // row_bcast:31
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}

// A state value as a published word and back (FP32 in the low half).
__device__ __forceinline__ unsigned long long word_of(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return b == kEmpty ? 0x7ff8000000000000ull : b;
}
__device__ __forceinline__ unsigned long long word_of(float v) { return __float_as_uint(v); }
__device__ __forceinline__ void of_word(unsigned long long w, double& v) {
  v = __longlong_as_double((long long)w);
}
__device__ __forceinline__ void of_word(unsigned long long w, float& v) {
  v = __uint_as_float((unsigned)w);
}

__device__ __forceinline__ void put(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long get(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

// The loop state of a line before its first launch, and every word empty.
__global__ void persist_init_kernel(PersistCtl* pc, unsigned long long* words, int count,
                                    int first) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < count) words[i] = kEmpty;
  if (i == 0) {
    pc->err = 0;
    if (first) {
      pc->ws = 0ull;
      pc->t = 0.0;
      pc->iters = 0;
      pc->dt = 0.0;
    }
  }
}

// Up to nsteps steps while run_time < sim_time and iters < max_iters, on the
// state a.in, which receives the result.  Launched on nseg / W workgroups of W
// waves, all resident (a cooperative launch where there is more than one);
// words: 3 slots of kPersistWords words of each workgroup.  first: the maximum
// wavespeed of the state is not known yet.  Every workgroup keeps run time and
// count itself: all see the same maximum.
template <typename T, int FLUX, bool FAST, bool VLC>
__global__ void __launch_bounds__(64 * kPersistMaxWaves)
persist1d_kernel(SweepArgs<T> a, PersistCtl* pc, unsigned long long* words, int nseg, double cfl,
                 double dh, double sim_time, long long max_iters, long long nsteps, int first,
                 unsigned int spin_limit) {
  constexpr int S = 3;
  constexpr bool F = UseFast<T, FAST>::value;
  const int limiter = VLC ? int(kLimVanLeer) : a.limiter;
  const int form = VLC ? int(kFormCons) : a.form;
  const int W = (int)(blockDim.x >> 6), G = (int)gridDim.x, b = (int)blockIdx.x;
  const int t = (int)(threadIdx.x & 63);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // by parity of the step: the waves' maxima and edges (first and last four cells)
  __shared__ unsigned long long s_max[2][kPersistMaxWaves];
  __shared__ T s_edge[2][kPersistMaxWaves][2][4][S];
  __shared__ unsigned long long s_all;
  __shared__ int s_ok;

  // this wave's cells [x0, x0 + m): lane 4 + i holds cell x0 + i
  const int n = (int)a.nx, seg = b * W + w;
  const int base = n / nseg, extra = n - base * nseg;
  const int x0 = seg * base + (seg < extra ? seg : extra);
  const int m = base + (seg < extra ? 1 : 0);
  const bool own = t >= 4 && t < 4 + m;
  const int side = t < 4 ? 0 : 1;                  // which neighbour a halo lane reads
  const int hc = t < 4 ? t : t - 4 - m;            // its cell of that neighbour's edge
  const bool halo = t < 4 || (t >= 4 + m && hc < 4);
  // the lane that a ghost cell of the line's ends mirrors (or wraps to, with
  // one segment); lanes past the halo repeat its last one
  const bool ring = a.bcx == kBcPeriodic && nseg > 1;
  const bool lo_end = seg == 0 && !ring, hi_end = seg == nseg - 1 && !ring;
  int src = t < 8 + m ? t : 7 + m;
  bool flip = false;
  if ((lo_end && src < 4) || (hi_end && src >= 4 + m)) {
    const int64_t g = map_ghost(x0 - 4 + src, n, a.bcx, flip);
    src = (int)g - (x0 - 4);
  }
  const bool ends = lo_end || hi_end;

  T u[S];
#pragma unroll
  for (int k = 0; k < S; ++k) u[k] = T(0);
  if (own) load_cell<T, S>(a.in, x0 + t - 4, a.es, a.cs, u);
  unsigned long long ws = 0ull;
  if (first) {
    if (own) ws = ws_bits(cell_wavespeed64<T, 1>(u, a.mat64));
  } else {
    ws = pc->ws;
  }
  double time = first ? 0.0 : pc->t, last_dt = first ? 0.0 : pc->dt;
  long long it = first ? 0 : pc->iters;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // a finished neighbour may store soon

  unsigned long long* const own_words = words + b;  // word i of slot s: [(s kPersistWords + i) G]
  int slot = 0;
  for (long long k = 0;; ++k) {
    const int par = (int)(k & 1);
    const int next2 = slot == 0 ? 2 : slot - 1;     // (slot + 2) % 3
    // ---- publish: edges (word 1 + 12 side + 3 cell + component), maximum (word 0)
    const unsigned long long wmax = wave_max_dpp(ws);
    if (t == 0) s_max[par][w] = wmax;
    const bool left = own && t < 8, right = own && t >= m;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      if (d == 0 ? left : right) {
        const int i = d == 0 ? t - 4 : t - m;
#pragma unroll
        for (int c = 0; c < S; ++c) {
          s_edge[par][w][d][i][c] = u[c];
          if (G > 1 && w == (d == 0 ? 0 : W - 1))
            put(own_words + (slot * kPersistWords + 1 + 12 * d + 3 * i + c) * G, word_of(u[c]));
        }
      }
    }
    __syncthreads();
    unsigned long long all = 0ull;
    for (int i = 0; i < W; ++i) all = s_max[par][i] > all ? s_max[par][i] : all;
    // ---- poll: the other workgroups' maxima (wave 0) and the edges beside this one
    const bool edge_lane = halo && ((side == 0 && w == 0 && !lo_end) ||
                                    (side == 1 && w == W - 1 && !hi_end));
    if (G > 1) {
      if (threadIdx.x == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied words of slot k + 1
        put(own_words + slot * kPersistWords * G, all == kEmpty ? 0x7ff8000000000000ull : all);
      }
      int ok = 1;
      if (w == 0 || w == W - 1) {
        const unsigned long long* const maxima = words + slot * kPersistWords * G;
        const int nb = side == 0 ? (b == 0 ? G - 1 : b - 1) : (b == G - 1 ? 0 : b + 1);
        const unsigned long long* const edge =
            words + (slot * kPersistWords + 1 + 12 * (1 - side) + 3 * (hc & 3)) * G + nb;
        unsigned int spins = 0;
        for (;;) {
          unsigned long long v[kPolls], e[S];
#pragma unroll
          for (int i = 0; i < kPolls; ++i)
            v[i] = (w == 0 && t + 64 * i < G) ? get(maxima + t + 64 * i) : 0ull;
#pragma unroll
          for (int c = 0; c < S; ++c) e[c] = edge_lane ? get(edge + c * G) : 0ull;
          bool wait = false;
          unsigned long long mx = 0ull;
#pragma unroll
          for (int i = 0; i < kPolls; ++i) {
            wait = wait || v[i] == kEmpty;
            mx = v[i] > mx ? v[i] : mx;
          }
#pragma unroll
          for (int c = 0; c < S; ++c) wait = wait || e[c] == kEmpty;
          if (!__any(wait)) {
            all = mx;
            if (edge_lane)
#pragma unroll
              for (int c = 0; c < S; ++c) of_word(e[c], u[c]);
            break;
          }
          if (++spins > spin_limit) {  // gives up: every workgroup then does
            ok = 0;
            break;
          }
        }
        if (w == 0) all = wave_max_dpp(all);
      }
      if (W > 1) {
        if (threadIdx.x == 0) {
          s_all = all;
          s_ok = 1;
        }
        __syncthreads();
        if (!ok) s_ok = 0;
        __syncthreads();
        all = s_all;
        ok = s_ok;
      }
      if (!ok) {
        if (t == 0) pc->err = 1;
        return;
      }
      if (w == 0 && t < kPersistWords) put(own_words + (next2 * kPersistWords + t) * G, kEmpty);
    }
    slot = slot == 2 ? 0 : slot + 1;
    // ---- the loop condition and dt (simulator/parameters.hpp:60-99)
    if (k >= nsteps || !(time < sim_time && it < max_iters)) {
      if (own) store_cell<T, S>(a.out, x0 + t - 4, a.es, a.cs, u);
      if (b == 0 && threadIdx.x == 0) {
        pc->ws = all;
        pc->t = time;
        pc->iters = it;
        pc->dt = last_dt;
      }
      return;
    }
    const double maxws = __longlong_as_double((long long)all);
    const double dt = cfl * dh / maxws;
    const double r64 = dt / dh;
    time += dt;
    it += 1;
    last_dt = dt;
    const T dtdh = (T)r64;
    const T half_dtdh = T(0.5) * dtdh;
    const T dhdt = T(1) / dtdh;
    // ---- the cells beside this wave's
    if (W > 1 && halo && !edge_lane) {
      // a neighbour wave's edge (the ends of the line are mirrored below)
      const int nw = side == 0 ? (w == 0 ? W - 1 : w - 1) : (w == W - 1 ? 0 : w + 1);
#pragma unroll
      for (int c = 0; c < S; ++c) u[c] = s_edge[par][nw][1 - side][hc][c];
    }
    if (G == 1 && W > 1 && edge_lane) {  // a periodic line in one workgroup
      const int nw = side == 0 ? W - 1 : 0;
#pragma unroll
      for (int c = 0; c < S; ++c) u[c] = s_edge[par][nw][1 - side][hc][c];
    }
    if (ends) {
#pragma unroll
      for (int c = 0; c < S; ++c) u[c] = __shfl(u[c], src, 64);
      if (a.bcx == kBcReflective && flip) reflect<T, 1>(u, 0);
    }
    // ---- the step
    T o[S];
    line_step<T, FLUX, F>(u, dtdh, half_dtdh, dhdt, limiter, form, a.mat, o);
    ws = 0ull;
    if (own) {
#pragma unroll
      for (int c = 0; c < S; ++c) u[c] = o[c];
      ws_fold<F, T, 1>(u, a, ws);
    }
  }
}

#define FL_PERSIST(T, FLUX, FAST, VLC)                                                          \
  template __global__ void persist1d_kernel<T, FLUX, FAST, VLC>(                                \
      SweepArgs<T>, PersistCtl*, unsigned long long*, int, double, double, double, long long,    \
      long long, int, unsigned int);
#define FL_PERSIST_ALL(T, FAST)             \
  FL_PERSIST(T, kFluxHllc, FAST, false)     \
  FL_PERSIST(T, kFluxHllc, FAST, true)      \
  FL_PERSIST(T, kFluxForce, FAST, false)    \
  FL_PERSIST(T, kFluxForce, FAST, true)     \
  FL_PERSIST(T, kFluxLaxFriedrichs, FAST, false) \
  FL_PERSIST(T, kFluxRichtmyer, FAST, false)
FL_PERSIST_ALL(double, false)
FL_PERSIST_ALL(double, true)
FL_PERSIST_ALL(float, false)

}  // namespace fl
