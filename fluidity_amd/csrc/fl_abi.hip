// fl_abi.hip -- host side of the C ABI declared in include/fluidity_amd.h.
//
// Validates arguments, builds the kernel argument blocks and launches the
// gfx950 kernels of fl_sweep.hip on the caller's stream.  No allocation
// happens outside fl_ctx_create.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "fl_abi_internal.hpp"

namespace {
thread_local std::string g_last_error;
}  // namespace

namespace fl {
namespace abi {

int fail(int status, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return status;
}

bool valid_block(int b) { return b >= 64 && b <= fl::kMaxBlock && (b % 64) == 0; }

int take_tuning(const fl_tuning* t, fl_tuning* tuning, int32_t* shape) {
  const int32_t block[2] = {t->x_block, t->y_block}, rows[2] = {t->x_rows, t->y_rows};
  int32_t* const block_out[2] = {&tuning->x_block, &tuning->y_block};
  int32_t* const rows_out[2] = {&tuning->x_rows, &tuning->y_rows};
  for (int d = 0; d < 2; ++d) {
    if (block[d] && !valid_block(block[d]))
      return fail(FL_ERR_ARGUMENT, "block widths must be multiples of 64 in [64, %d]",
                  fl::kMaxBlock);
    if (rows[d] != FL_ROWS_RULE && (rows[d] < -4096 || rows[d] > 4096))
      return fail(FL_ERR_ARGUMENT, "rows per workgroup must be in [1, 4096]");
  }
  for (int d = 0; d < 2; ++d) {
    if (block[d]) *block_out[d] = block[d];
    if (rows[d] == FL_ROWS_RULE) {
      shape[d] = kShapeRule;
    } else if (block[d] || rows[d]) {
      shape[d] = rows[d] < 0 ? kShapeCell : kShapeTuning;
      if (rows[d]) *rows_out[d] = abs(rows[d]);
    }
  }
  return FL_OK;
}

int resolve_tuning(const fl_tuning* t, fl_tuning* out, int32_t* shape) {
  *out = {256, 32, 256, 64};
  shape[0] = shape[1] = kShapeRule;
  return t ? take_tuning(t, out, shape) : FL_OK;
}

fl_tuning tuning_of(const fl_tuning& tuning, const int32_t* shape) {
  fl_tuning t = tuning;
  int32_t* const rows[2] = {&t.x_rows, &t.y_rows};
  for (int d = 0; d < 2; ++d) {
    if (shape[d] == kShapeRule) *rows[d] = FL_ROWS_RULE;
    if (shape[d] == kShapeCell) *rows[d] = -*rows[d];
  }
  return t;
}

int check_field(const fl_field* f, const char* name) {
  if (!f) return fail(FL_ERR_ARGUMENT, "%s is NULL", name);
  if (!f->data) return fail(FL_ERR_ARGUMENT, "%s->data is NULL", name);
  if (f->dtype != FL_F64 && f->dtype != FL_F32)
    return fail(FL_ERR_ARGUMENT, "%s->dtype %d is not FL_F64/FL_F32", name, f->dtype);
  if (f->layout != FL_LAYOUT_AOS && f->layout != FL_LAYOUT_SOA)
    return fail(FL_ERR_ARGUMENT, "%s->layout %d is not AoS/SoA", name, f->layout);
  if (f->ndim < 1 || f->ndim > 3)
    return fail(FL_ERR_ARGUMENT, "%s->ndim %d out of range", name, f->ndim);
  if (f->ndim == 3) return fail(FL_ERR_UNSUPPORTED, "%s: 3D grids are not supported", name);
  for (int d = 0; d < f->ndim; ++d)
    if (f->n[d] < 4)
      return fail(FL_ERR_ARGUMENT, "%s->n[%d] = %lld: need at least 4 cells (ghost pad)",
                  name, d, (long long)f->n[d]);
  if (f->ndim == 2 && f->n[1] > (int64_t)65535 * 4096)
    return fail(FL_ERR_ARGUMENT, "%s->n[1] too large", name);
  // the 2D sweeps address a row with 32-bit byte offsets (4 FP64 components)
  if (f->ndim == 2 && f->n[0] > ((int64_t)1 << 27))
    return fail(FL_ERR_ARGUMENT, "%s->n[0] = %lld: 2D rows hold at most 2^27 cells", name,
                (long long)f->n[0]);
  return FL_OK;
}

int check_pair(const fl_field* in, const fl_field* out) {
  int rc = check_field(in, "in");
  if (rc) return rc;
  rc = check_field(out, "out");
  if (rc) return rc;
  if (in->dtype != out->dtype || in->layout != out->layout || in->ndim != out->ndim)
    return fail(FL_ERR_ARGUMENT, "in and out differ in dtype/layout/ndim");
  for (int d = 0; d < in->ndim; ++d)
    if (in->n[d] != out->n[d]) return fail(FL_ERR_ARGUMENT, "in and out differ in shape");
  if (in->data == out->data)
    return fail(FL_ERR_ARGUMENT, "in and out alias: a sweep cannot update in place");
  return FL_OK;
}

int check_scheme(const fl_scheme* s, int ndim) {
  if (!s) return fail(FL_ERR_ARGUMENT, "scheme is NULL");
  if (s->limiter != FL_LIMITER_VAN_LEER && s->limiter != FL_LIMITER_SUPERBEE)
    return fail(FL_ERR_ARGUMENT, "scheme->limiter %d invalid", s->limiter);
  if (s->form != FL_FORM_CONSERVATIVE && s->form != FL_FORM_PRIMITIVE)
    return fail(FL_ERR_ARGUMENT, "scheme->form %d invalid", s->form);
  if (s->flux < FL_FLUX_HLLC || s->flux > FL_FLUX_RICHTMYER)
    return fail(FL_ERR_ARGUMENT, "scheme->flux %d invalid", s->flux);
  if (s->eos != FL_EOS_IDEAL && s->eos != FL_EOS_STIFF && s->eos != FL_EOS_STIFF_CORRECTED)
    return fail(FL_ERR_ARGUMENT, "scheme->eos %d invalid", s->eos);
  if (!(s->gamma > 1.0) || !isfinite(s->gamma))
    return fail(FL_ERR_ARGUMENT, "scheme->gamma %g must be finite and > 1", s->gamma);
  if (!isfinite(s->p_inf)) return fail(FL_ERR_ARGUMENT, "scheme->p_inf not finite");
  for (int d = 0; d < ndim; ++d)
    if (s->bc[d] < FL_BC_TRANSMISSIVE || s->bc[d] > FL_BC_PERIODIC)
      return fail(FL_ERR_ARGUMENT, "scheme->bc[%d] %d invalid", d, s->bc[d]);
  if (s->numerics != FL_NUMERICS_EXACT && s->numerics != FL_NUMERICS_FAST)
    return fail(FL_ERR_ARGUMENT, "scheme->numerics %d invalid", s->numerics);
  return FL_OK;
}

int require_exact(const fl_scheme* s, const char* what) {
  if (s->numerics != FL_NUMERICS_EXACT)
    return fail(FL_ERR_UNSUPPORTED, "%s runs the exact FP64 numerics only", what);
  return FL_OK;
}

void strides(const fl_field* f, int64_t& es, int64_t& cs) {
  const int S = 2 + f->ndim;
  const int64_t cells = f->n[0] * (f->ndim > 1 ? f->n[1] : 1);
  if (f->layout == FL_LAYOUT_AOS) {
    es = S;
    cs = 1;
  } else {
    es = 1;
    cs = cells;
  }
}

int64_t cell_count(const fl_field* f) { return f->n[0] * (f->ndim > 1 ? f->n[1] : 1); }

template <typename T>
fl::SweepArgs<T> make_args(const fl_context* ctx, const fl_field* in, const fl_field* out,
                           const fl_scheme* s, double dtdh, const fl::StepCtl* ctl,
                           unsigned long long* ws_out, int rows) {
  fl::SweepArgs<T> a;
  memset(&a, 0, sizeof(a));
  a.in = (const T*)in->data;
  a.out = (T*)out->data;
  strides(in, a.es, a.cs);
  a.nx = in->n[0];
  a.ny = in->ndim > 1 ? in->n[1] : 1;
  a.rowb = a.nx * a.es * (int64_t)sizeof(T);
  a.csb = a.cs * (int64_t)sizeof(T);
  a.mat = make_material<T>(s);
  a.mat64 = make_material<double>(s);
  a.limiter = s->limiter;
  a.form = s->form;
  a.bcx = s->bc[0];
  a.bcy = in->ndim > 1 ? s->bc[1] : 0;
  a.rows_per_block = rows;
  a.dtdh_host = (T)dtdh;
  a.ctl = ctl;
  a.ws_out = ws_out;
  a.wide = wide_cells(a);
  (void)ctx;
  return a;
}

// Rows per workgroup of a caller's tuning, halved (down to 4) while the launch would have fewer
// than kMinWaves waves (1.5 per SIMD of the 1024 on the device): small grids
// keep the machine filled whatever the tuning says.
constexpr int64_t kMinWaves = 1536;
int fit_rows(int rows, int64_t bands, int64_t ny, int block) {
  const int64_t waves = block / 64;
  while (rows > 4 && bands * ((ny + rows - 1) / rows) * waves < kMinWaves) rows /= 2;
  return rows;
}

// Kernels with van Leer in conservative form fixed at compile time exist for
// HLLC and FORCE.
template <int FLUX>
constexpr bool has_vlc() { return FLUX == fl::kFluxHllc || FLUX == fl::kFluxForce; }
inline bool is_vlc(int limiter, int form) {
  return FL_VLC_KERNELS && limiter == fl::kLimVanLeer && form == fl::kFormCons;
}

// The launch of one 2D sweep.
struct SweepShape {
  bool cell;  // the cell-parallel kernel (block and rows unused)
  int block;  // lanes per workgroup of the march
  int rows;   // rows per workgroup of the march
};

// Cells up to which the cell-parallel sweeps of one grid are the faster ones,
// and of the two grids of a launch together.  A step, cell-parallel against a
// round of marching tiles: FP64 exact 1200x1207 111 | 115 us, 1400^2 143 | 146,
// 1500x1507 165 | 158, 2048^2 298 | 274; fast 1200x1207 88 | 88, 1500x1507 125 |
// 118; FP32 1200x1207 61 | 61, 1400^2 77 | 76, 1500x1507 85 | 78, 2048^2 141 |
// 117.  (Two grids march at two waves per SIMD in FP64: their line is farther.)
constexpr int64_t kCellMax = 7 << 18;
template <typename T> constexpr int64_t kCellMaxTwo = 5 << 19;
template <> constexpr int64_t kCellMaxTwo<float> = 5 << 20;
// Cells up to which the autotuner tries them, and a caller's tuning gets them.
constexpr int64_t kCellTryMax = 10 << 20;

// Marching shape of a sweep by rule: tiles of one height that fill whole rounds
// of the workgroups that the device holds at once (`waves` per SIMD of 1024),
// so that the launch ends evenly, as tall as one round makes them but at most
// kRoundRows (6 warm-up rows in x, 8 in y come on top).  256 lanes, fewer where
// the columns leave a tenth of them idle.  Fixed numbers of waves (about 10500
// in x, 4096 in y) ended with a nearly empty round at some sizes: 1700x1707
// FP64 exact 212 us a step, in one round 197, FORCE in the fast numerics 156 and
// 124, FP32 124 and 91; 2600^2 421 and 434, FP32 200 and 169; 4096^2 fast 714 and
// 699, FP32 417 and 395.  Short wide grids need the wide workgroups for their
// number too: the atomics of the CFL maximum (10 ns each, one after the other)
// of 31250 workgroups of 64 lanes outlast the y sweep of 2000000 x 5 cells
// (FP32, 566 us a step against 313).
constexpr int64_t kRoundRows = 96;
SweepShape round_shape(int dim, int64_t nx, int64_t ny, int ngrids, int waves) {
  SweepShape best{false, 0, 0};
  double best_cost = 0.0;
  for (int B : {256, 128, 64}) {
    const int64_t cap = (int64_t)1024 * waves / (B / 64);
    const int64_t bands = ngrids * (dim ? (nx + B - 1) / B : (nx + B - 3) / (B - 2));
    const int64_t least = (bands * ((ny + kRoundRows - 1) / kRoundRows) + cap - 1) / cap;
    for (int64_t r = least; r < least + 4; ++r) {
      const int64_t tiles = std::min(r * cap / bands, std::min<int64_t>(ny, 65535));
      const int64_t rows = (ny + tiles - 1) / tiles;
      const int64_t rounds = (bands * ((ny + rows - 1) / rows) + cap - 1) / cap;
      const double cost = (double)(rounds * (rows + (dim ? 8 : 6)));
      if (!best.block || cost < (B < best.block ? 0.9 : 1.0) * best_cost) {
        best = {false, B, (int)rows};
        best_cost = cost;
      }
    }
  }
  return best;
}

// Launch shape of the sweep of dimension dim over ngrids grids of nx x ny
// cells.  By rule small grids go cell-parallel (a 64^2 FP64 sweep takes 7 us
// against 16 (x) and 21 us (y) marching) and larger ones march.
template <typename T>
SweepShape pick_shape(const fl_context* ctx, int dim, int64_t nx, int64_t ny, int ngrids) {
  const fl_tuning& tu = ctx->tuning;
  const bool few = nx * ny * ngrids <= (ngrids > 1 ? kCellMaxTwo<T> : kCellMax);
  // kShapeCell holds for one grid up to the size that it was measured at (a
  // 4096^2 sweep in the shapes tuned at 256^2: FP32 629 us cell-parallel, 535
  // marching); past it, and for two grids past the line, the tuning's march is
  // the fastest one of that measurement
  const int64_t measured = ctx->cell_cells[dim];
  const bool cell =
      ctx->shape[dim] == kShapeCell &&
      (few || (ngrids == 1 && nx * ny <= (measured ? measured : kCellTryMax)));
  if (ctx->shape[dim] != kShapeRule && !cell) {
    const int B = dim ? tu.y_block : tu.x_block;
    const int64_t bands = dim ? (nx + B - 1) / B : (nx + B - 3) / (B - 2);
    return {false, B, fit_rows(dim ? tu.y_rows : tu.x_rows, ngrids * bands, ny, B)};
  }
  if (cell || few) return {true, 0, 0};
  return round_shape(dim, nx, ny, ngrids, sizeof(T) == 4 ? 4 : ngrids > 1 ? 2 : 3);
}

// Workgroups of a sweep: the marching tiles over (x, y), or the cell-parallel
// ones in one dimension; z (march) or y (cell-parallel) counts the grids.
dim3 shape_grid(const SweepShape& sh, int dim, int64_t nx, int64_t ny, int ngrids) {
  if (sh.cell) {
    const int cols = dim ? fl::kCellYCols : fl::kCellXCols;
    const int rows = dim ? fl::kCellYRows : fl::kCellXRows;
    return dim3((unsigned)(((nx + cols - 1) / cols) * ((ny + rows - 1) / rows)), ngrids, 1);
  }
  const int B = sh.block;
  return dim3((unsigned)(dim ? (nx + B - 1) / B : (nx + B - 3) / (B - 2)),
              (unsigned)((ny + sh.rows - 1) / sh.rows), ngrids);
}

template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
void launch_flux_w(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a,
                   hipStream_t stream) {
  const int B = sh.block;
  if (sh.cell) {
    auto k = dim == 0 ? fl::cell_x_kernel<T, FLUX, FAST, VLC, WIDE>
                      : fl::cell_y_kernel<T, FLUX, FAST, VLC, WIDE>;
    hipLaunchKernelGGL(k, grid, dim3(64 * fl::kCellWaves), fl::cell_tile_lds_bytes(sizeof(T)),
                       stream, a, a);
  } else if (ndim == 1)
    hipLaunchKernelGGL((fl::sweep_x_kernel<T, 1, FLUX, FAST, VLC, false>), grid, dim3(B),
                       fl::x_tile_lds_bytes(B, 3, sizeof(T)), stream, a);
  else if (dim == 0)
    hipLaunchKernelGGL((fl::sweep_x_kernel<T, 2, FLUX, FAST, VLC, WIDE>), grid, dim3(B),
                       fl::x_tile_lds_bytes(B, 4, sizeof(T)), stream, a);
  else
    hipLaunchKernelGGL((fl::sweep_y_kernel<T, FLUX, FAST, VLC, WIDE>), grid, dim3(B),
                       fl::y_tile_lds_bytes(B, sizeof(T)), stream, a);
}

template <typename T, int FLUX, bool FAST, bool VLC>
void launch_flux_v(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a,
                   hipStream_t stream) {
  if (a.wide) launch_flux_w<T, FLUX, FAST, VLC, true>(ndim, dim, grid, sh, a, stream);
  else launch_flux_w<T, FLUX, FAST, VLC, false>(ndim, dim, grid, sh, a, stream);
}

// One sweep kernel of flux FLUX: the 1D sweep, or the x or y sweep of a 2D grid.
template <typename T, int FLUX, bool FAST>
void launch_flux(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a,
                 hipStream_t stream) {
  if constexpr (has_vlc<FLUX>()) {
    if (is_vlc(a.limiter, a.form)) {
      launch_flux_v<T, FLUX, FAST, true>(ndim, dim, grid, sh, a, stream);
      return;
    }
  }
  launch_flux_v<T, FLUX, FAST, false>(ndim, dim, grid, sh, a, stream);
}

// The fast FP64 numerics were requested (FP32 sweeps use them always).
inline bool fast_numerics(const fl_scheme* s) { return s->numerics == FL_NUMERICS_FAST; }

// Workgroups of B lanes of one sweep kernel that a CU holds at once.
template <typename T, int FLUX, bool FAST, bool VLC>
const void* sweep_kernel_2d(int dim) {
  return dim == 0 ? reinterpret_cast<const void*>(&fl::sweep_x_kernel<T, 2, FLUX, FAST, VLC, false>)
                  : reinterpret_cast<const void*>(&fl::sweep_y_kernel<T, FLUX, FAST, VLC, false>);
}

template <typename T, int FLUX, bool FAST>
int sweep_blocks_per_cu(int dim, int B, bool vlc) {
  const void* k = sweep_kernel_2d<T, FLUX, FAST, false>(dim);
  if constexpr (has_vlc<FLUX>())
    if (vlc) k = sweep_kernel_2d<T, FLUX, FAST, true>(dim);
  int n = 0;
  const size_t lds =
      dim == 0 ? fl::x_tile_lds_bytes(B, 4, sizeof(T)) : fl::y_tile_lds_bytes(B, sizeof(T));
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, B, lds) != hipSuccess) return 0;
  return n;
}

template <typename T, bool FAST>
int sweep_blocks_per_cu_f(int dim, int flux, int B, bool vlc) {
  switch (flux) {
    case FL_FLUX_HLLC: return sweep_blocks_per_cu<T, fl::kFluxHllc, FAST>(dim, B, vlc);
    case FL_FLUX_FORCE: return sweep_blocks_per_cu<T, fl::kFluxForce, FAST>(dim, B, vlc);
    case FL_FLUX_LAX_FRIEDRICHS:
      return sweep_blocks_per_cu<T, fl::kFluxLaxFriedrichs, FAST>(dim, B, vlc);
    default: return sweep_blocks_per_cu<T, fl::kFluxRichtmyer, FAST>(dim, B, vlc);
  }
}

template <typename T>
int sweep_blocks_per_cu_t(int dim, const fl_scheme* s, int B) {
  const bool vlc = is_vlc(s->limiter, s->form);
  if (std::is_same<T, double>::value && fast_numerics(s))
    return sweep_blocks_per_cu_f<T, true>(dim, s->flux, B, vlc);
  return sweep_blocks_per_cu_f<T, false>(dim, s->flux, B, vlc);
}

// Tile heights to time for one 2D sweep: the powers of two in `base`, and,
// for R = 1..16, the smallest height whose launch fits in R rounds of the
// workgroups the device holds at once (`slots`).  On a grid whose launch is
// a few rounds, one a little over a whole number of rounds leaves most of
// the machine idle in its last round.
std::vector<int> row_candidates(const int* base, int nbase, int64_t bands, int64_t ny,
                                int64_t slots) {
  std::vector<int> rows(base, base + nbase);
  for (int64_t R = 1; slots > 0 && R <= 16; ++R) {
    const int64_t chunks = R * slots / bands;
    if (chunks < 1) continue;
    const int64_t h = (ny + chunks - 1) / chunks;
    if (h >= 4 && h <= 128 && std::find(rows.begin(), rows.end(), (int)h) == rows.end())
      rows.push_back((int)h);
  }
  return rows;
}

template <typename T, bool FAST>
void launch_flux_t(int flux, int ndim, int dim, dim3 grid, const SweepShape& sh,
                   const fl::SweepArgs<T>& a, hipStream_t stream) {
  switch (flux) {
    case FL_FLUX_HLLC: launch_flux<T, fl::kFluxHllc, FAST>(ndim, dim, grid, sh, a, stream); break;
    case FL_FLUX_FORCE: launch_flux<T, fl::kFluxForce, FAST>(ndim, dim, grid, sh, a, stream); break;
    case FL_FLUX_LAX_FRIEDRICHS:
      launch_flux<T, fl::kFluxLaxFriedrichs, FAST>(ndim, dim, grid, sh, a, stream);
      break;
    default: launch_flux<T, fl::kFluxRichtmyer, FAST>(ndim, dim, grid, sh, a, stream); break;
  }
}

// begin (nullable): the sweep begins step k of a simulation.
struct SimBegin {
  fl::SimCtl* sim;
  const fl_sim_params* p;
  int64_t k;
};

template <typename T>
int launch_sweep_t(const fl_context* ctx, const fl_field* in, const fl_field* out, int dim,
                   const fl_scheme* s, double dtdh, const fl::StepCtl* ctl,
                   unsigned long long* ws_out, const SimBegin* begin, hipStream_t stream) {
  dim3 grid;
  SweepShape sh{false, ctx->tuning.x_block, 1};
  if (in->ndim == 1) {
    grid = dim3((unsigned)((in->n[0] + (sh.block - 3)) / (sh.block - 2)), 1, 1);
  } else {
    sh = pick_shape<T>(ctx, dim, in->n[0], in->n[1], 1);
    grid = shape_grid(sh, dim, in->n[0], in->n[1], 1);
  }
  fl::SweepArgs<T> a = make_args<T>(ctx, in, out, s, dtdh, ctl, ws_out, sh.rows);
  if (begin) {
    const int n = sim_slots(in->ndim);
    a.sim = begin->sim;
    a.sim_half = (int)(begin->k & 1);
    a.sim_ws = (int)(begin->k % n);
    a.sim_zero = (int)((begin->k + n - 1) % n);
    a.cfl = begin->p->cfl;
    a.dh = begin->p->dh;
    a.sim_time = begin->p->sim_time;
    a.max_iters = (long long)begin->p->max_iters;
  }
  if (std::is_same<T, double>::value && fast_numerics(s))
    launch_flux_t<T, true>(s->flux, in->ndim, dim, grid, sh, a, stream);
  else
    launch_flux_t<T, false>(s->flux, in->ndim, dim, grid, sh, a, stream);
  FL_HIP(hipGetLastError());
  return FL_OK;
}

int launch_sweep(const fl_context* ctx, const fl_field* in, const fl_field* out, int dim,
                 const fl_scheme* s, double dtdh, const fl::StepCtl* ctl,
                 unsigned long long* ws_out, hipStream_t stream) {
  if (in->dtype == FL_F64)
    return launch_sweep_t<double>(ctx, in, out, dim, s, dtdh, ctl, ws_out, nullptr, stream);
  return launch_sweep_t<float>(ctx, in, out, dim, s, dtdh, ctl, ws_out, nullptr, stream);
}

int launch_sim_step(const fl_context* ctx, const fl_field* state, const fl_field* work,
                    const fl_scheme* s, const fl_sim_params* p, fl::SimCtl* sim, int64_t k,
                    hipStream_t stream) {
  if (state->ndim == 1)
    return (k & 1) ? launch_sim_step(ctx, work, nullptr, state, s, p, sim, k, stream)
                   : launch_sim_step(ctx, state, nullptr, work, s, p, sim, k, stream);
  return launch_sim_step(ctx, state, work, state, s, p, sim, k, stream);
}

int launch_sim_step(const fl_context* ctx, const fl_field* in, const fl_field* mid,
                    const fl_field* out, const fl_scheme* s, const fl_sim_params* p,
                    fl::SimCtl* sim, int64_t k, hipStream_t stream) {
  const SimBegin begin = {sim, p, k};
  const bool one = in->ndim == 1;
  unsigned long long* next = &sim->ws[(k + 1) % sim_slots(in->ndim)];
  const int rc = in->dtype == FL_F64
                     ? launch_sweep_t<double>(ctx, in, one ? out : mid, 0, s, 1.0, nullptr,
                                              one ? next : nullptr, &begin, stream)
                     : launch_sweep_t<float>(ctx, in, one ? out : mid, 0, s, 1.0, nullptr,
                                             one ? next : nullptr, &begin, stream);
  if (rc || one) return rc;
  return launch_sweep(ctx, mid, out, 1, s, 1.0, &sim->c, next, stream);
}

// Both materials' sweeps of dimension `dim` in one launch: in[m] -> out[m]
// with scheme s[m].  The two grids share shape, layout and dtype; the flux
// methods must be equal (the launch instantiates one), else each grid is
// swept on its own.
template <typename T, int FLUX, bool FAST, bool VLC, bool WIDE>
void launch_flux2_w(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a0,
                    const fl::SweepArgs<T>& a1, hipStream_t stream) {
  const int B = sh.block;
  if (sh.cell) {
    auto k = dim == 0 ? fl::cell_x_kernel<T, FLUX, FAST, VLC, WIDE>
                      : fl::cell_y_kernel<T, FLUX, FAST, VLC, WIDE>;
    hipLaunchKernelGGL(k, grid, dim3(64 * fl::kCellWaves), fl::cell_tile_lds_bytes(sizeof(T)),
                       stream, a0, a1);
  } else if (ndim == 1)
    hipLaunchKernelGGL((fl::sweep_x2_kernel<T, 1, FLUX, FAST, VLC, false>), grid, dim3(B),
                       fl::x_tile_lds_bytes(B, 3, sizeof(T)), stream, a0, a1);
  else if (dim == 0)
    hipLaunchKernelGGL((fl::sweep_x2_kernel<T, 2, FLUX, FAST, VLC, WIDE>), grid, dim3(B),
                       fl::x_tile_lds_bytes(B, 4, sizeof(T)), stream, a0, a1);
  else
    hipLaunchKernelGGL((fl::sweep_y2_kernel<T, FLUX, FAST, VLC, WIDE>), grid, dim3(B),
                       fl::y_tile_lds_bytes(B, sizeof(T)), stream, a0, a1);
}

template <typename T, int FLUX, bool FAST, bool VLC>
void launch_flux2_v(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a0,
                    const fl::SweepArgs<T>& a1, hipStream_t stream) {
  if (a0.wide && a1.wide)
    launch_flux2_w<T, FLUX, FAST, VLC, true>(ndim, dim, grid, sh, a0, a1, stream);
  else
    launch_flux2_w<T, FLUX, FAST, VLC, false>(ndim, dim, grid, sh, a0, a1, stream);
}

// fast: the fast FP64 numerics (FP64 only; the FP32 kernels have their own)
template <typename T, int FLUX>
void launch_flux2(int ndim, int dim, dim3 grid, const SweepShape& sh, const fl::SweepArgs<T>& a0,
                  const fl::SweepArgs<T>& a1, bool fast, hipStream_t stream) {
  const bool vlc = has_vlc<FLUX>() && is_vlc(a0.limiter, a0.form) && is_vlc(a1.limiter, a1.form);
  if constexpr (std::is_same<T, double>::value) {
    if (fast) {
      if constexpr (has_vlc<FLUX>())
        if (vlc) return launch_flux2_v<T, FLUX, true, true>(ndim, dim, grid, sh, a0, a1, stream);
      return launch_flux2_v<T, FLUX, true, false>(ndim, dim, grid, sh, a0, a1, stream);
    }
  }
  if constexpr (has_vlc<FLUX>())
    if (vlc) return launch_flux2_v<T, FLUX, false, true>(ndim, dim, grid, sh, a0, a1, stream);
  launch_flux2_v<T, FLUX, false, false>(ndim, dim, grid, sh, a0, a1, stream);
}

template <typename T>
int launch_sweep2_t(const fl_context* ctx, const fl_field* const in[2],
                    const fl_field* const out[2], int dim, const fl_scheme* const s[2],
                    double dtdh, hipStream_t stream, const fl::StepCtl* ctl) {
  const fl_field* f = in[0];
  dim3 grid;
  SweepShape sh{false, ctx->tuning.x_block, 1};
  if (f->ndim == 1) {
    grid = dim3((unsigned)((f->n[0] + (sh.block - 3)) / (sh.block - 2)), 1, 2);
  } else {
    // the cells of both grids count towards filling the machine
    sh = pick_shape<T>(ctx, dim, f->n[0], f->n[1], 2);
    grid = shape_grid(sh, dim, f->n[0], f->n[1], 2);
  }
  const fl::SweepArgs<T> a0 = make_args<T>(ctx, in[0], out[0], s[0], dtdh, ctl, nullptr, sh.rows);
  const fl::SweepArgs<T> a1 = make_args<T>(ctx, in[1], out[1], s[1], dtdh, ctl, nullptr, sh.rows);
  const bool fast = fast_numerics(s[0]);
  switch (s[0]->flux) {
    case FL_FLUX_HLLC:
      launch_flux2<T, fl::kFluxHllc>(f->ndim, dim, grid, sh, a0, a1, fast, stream);
      break;
    case FL_FLUX_FORCE:
      launch_flux2<T, fl::kFluxForce>(f->ndim, dim, grid, sh, a0, a1, fast, stream);
      break;
    case FL_FLUX_LAX_FRIEDRICHS:
      launch_flux2<T, fl::kFluxLaxFriedrichs>(f->ndim, dim, grid, sh, a0, a1, fast, stream);
      break;
    default:
      launch_flux2<T, fl::kFluxRichtmyer>(f->ndim, dim, grid, sh, a0, a1, fast, stream);
      break;
  }
  FL_HIP(hipGetLastError());
  return FL_OK;
}

int launch_sweep2(const fl_context* ctx, const fl_field* const in[2], const fl_field* const out[2],
                  int dim, const fl_scheme* const s[2], double dtdh, hipStream_t stream,
                  const fl::StepCtl* ctl) {
  // one launch instantiates one flux method and one form of the numerics
  if (s[0]->flux != s[1]->flux ||
      (in[0]->dtype == FL_F64 && fast_numerics(s[0]) != fast_numerics(s[1]))) {
    for (int m = 0; m < 2; ++m) {
      const int rc = launch_sweep(ctx, in[m], out[m], dim, s[m], dtdh, ctl, nullptr, stream);
      if (rc) return rc;
    }
    return FL_OK;
  }
  if (in[0]->dtype == FL_F64)
    return launch_sweep2_t<double>(ctx, in, out, dim, s, dtdh, stream, ctl);
  return launch_sweep2_t<float>(ctx, in, out, dim, s, dtdh, stream, ctl);
}

int launch_max_ws2(const fl_field* f0, const fl_field* f1, const fl_scheme* s0,
                   const fl_scheme* s1, unsigned long long* dst, hipStream_t stream) {
  int64_t es0, cs0, es1, cs1;
  strides(f0, es0, cs0);
  strides(f1, es1, cs1);
  const int64_t n = cell_count(f0);
  const int B = fl::kMaxBlock;
  int64_t blocks = (n + B - 1) / B;
  if (blocks > fl::kMaxWsBlocks) blocks = fl::kMaxWsBlocks;
  if (blocks < 1) blocks = 1;
  const fl::Material<double> m0 = make_material<double>(s0), m1 = make_material<double>(s1);
  const dim3 grid((unsigned)blocks);
  if (f0->dtype == FL_F64) {
    // the fast forms when both materials ask for the fast numerics
    const bool fast = fast_numerics(s0) && fast_numerics(s1);
    auto k = f0->ndim == 1 ? (fast ? fl::max_wavespeed2_kernel<double, 1, true>
                                   : fl::max_wavespeed2_kernel<double, 1, false>)
                           : (fast ? fl::max_wavespeed2_kernel<double, 2, true>
                                   : fl::max_wavespeed2_kernel<double, 2, false>);
    hipLaunchKernelGGL(k, grid, dim3(B), 0, stream, (const double*)f0->data,
                       (const double*)f1->data, es0, cs0, es1, cs1, n, m0, m1, dst);
  } else {
    if (f0->ndim == 1)
      hipLaunchKernelGGL((fl::max_wavespeed2_kernel<float, 1, false>), grid, dim3(B), 0, stream,
                         (const float*)f0->data, (const float*)f1->data, es0, cs0, es1, cs1,
                         n, m0, m1, dst);
    else
      hipLaunchKernelGGL((fl::max_wavespeed2_kernel<float, 2, false>), grid, dim3(B), 0, stream,
                         (const float*)f0->data, (const float*)f1->data, es0, cs0, es1, cs1,
                         n, m0, m1, dst);
  }
  FL_HIP(hipGetLastError());
  return FL_OK;
}

int launch_max_ws(const fl_field* f, const fl_scheme* s, unsigned long long* dst,
                  hipStream_t stream) {
  int64_t es, cs;
  strides(f, es, cs);
  const int64_t n = cell_count(f);
  const fl::Material<double> m64 = make_material<double>(s);
  const int B = fl::kMaxBlock;
  int64_t blocks = (n + B - 1) / B;
  if (blocks > fl::kMaxWsBlocks) blocks = fl::kMaxWsBlocks;
  if (blocks < 1) blocks = 1;
  dim3 grid((unsigned)blocks);
  if (f->dtype == FL_F64) {
    if (f->ndim == 1)
      hipLaunchKernelGGL((fl::max_wavespeed_kernel<double, 1>), grid, dim3(B), 0, stream,
                         (const double*)f->data, es, cs, n, m64, dst);
    else
      hipLaunchKernelGGL((fl::max_wavespeed_kernel<double, 2>), grid, dim3(B), 0, stream,
                         (const double*)f->data, es, cs, n, m64, dst);
  } else {
    if (f->ndim == 1)
      hipLaunchKernelGGL((fl::max_wavespeed_kernel<float, 1>), grid, dim3(B), 0, stream,
                         (const float*)f->data, es, cs, n, m64, dst);
    else
      hipLaunchKernelGGL((fl::max_wavespeed_kernel<float, 2>), grid, dim3(B), 0, stream,
                         (const float*)f->data, es, cs, n, m64, dst);
  }
  FL_HIP(hipGetLastError());
  return FL_OK;
}

double bits_to_double(unsigned long long b) {
  double d;
  memcpy(&d, &b, sizeof(d));
  return d;
}

}  // namespace abi
}  // namespace fl

using namespace fl::abi;

// ---- persistent 1D step loop -------------------------------------------------

namespace {

// Longer lines take the launched sweeps: past a workgroup of 16 waves on every
// CU a step is more arithmetic than exchange.
constexpr int64_t kPersistMaxCells =
    (int64_t)fl::kLineCells * fl::kPersistMaxWaves * fl::kPersistMaxGroups;
constexpr int64_t kPersistChunk = 1 << 16;     // steps per launch (then the host looks)
// Polls before a workgroup gives up (each is a load from device memory: a
// fraction of a second in all, against a few microseconds per step).
constexpr unsigned int kPersistSpin = 1u << 18;

template <typename T, int FLUX, bool FAST>
const void* persist_kernel_ptr(bool vlc) {
  if constexpr (has_vlc<FLUX>())
    if (vlc) return reinterpret_cast<const void*>(&fl::persist1d_kernel<T, FLUX, FAST, true>);
  return reinterpret_cast<const void*>(&fl::persist1d_kernel<T, FLUX, FAST, false>);
}

template <typename T, bool FAST>
const void* persist_kernel_for(int flux, bool vlc) {
  switch (flux) {
    case FL_FLUX_HLLC: return persist_kernel_ptr<T, fl::kFluxHllc, FAST>(vlc);
    case FL_FLUX_FORCE: return persist_kernel_ptr<T, fl::kFluxForce, FAST>(vlc);
    case FL_FLUX_LAX_FRIEDRICHS: return persist_kernel_ptr<T, fl::kFluxLaxFriedrichs, FAST>(vlc);
    default: return persist_kernel_ptr<T, fl::kFluxRichtmyer, FAST>(vlc);
  }
}

// Launch of the persistent loop on a line: its segments (one per wave) and
// the waves of a workgroup.  groups 0: it does not apply (long lines, or more
// workgroups than the device holds at once).
struct PersistShape {
  const void* kernel;
  int segments, waves, groups;
};

// Up to 8 segments share one workgroup, whose waves exchange through LDS
// alone; more go four to a workgroup, one per SIMD (4096 cells: 4.8 us a step,
// with one or two to a workgroup 5.1 and 4.8, with eight 5.3), or as many as
// leave one workgroup per CU to poll.
PersistShape persist_shape(const fl_field* f, const fl_scheme* s) {
  PersistShape sh = {nullptr, 0, 0, 0};
  if (f->ndim != 1 || f->n[0] > kPersistMaxCells) return sh;
  const bool vlc = is_vlc(s->limiter, s->form);
  sh.kernel = f->dtype == FL_F32 ? persist_kernel_for<float, false>(s->flux, vlc)
              : fast_numerics(s) ? persist_kernel_for<double, true>(s->flux, vlc)
                                 : persist_kernel_for<double, false>(s->flux, vlc);
  int nseg = (int)((f->n[0] + fl::kLineCells - 1) / fl::kLineCells);
  const int spread = (nseg + fl::kPersistMaxGroups - 1) / fl::kPersistMaxGroups;
  const int waves = nseg <= 8 ? nseg : std::max(4, spread);
  const int groups = (nseg + waves - 1) / waves;
  nseg = groups * waves;
  if (groups > 1) {
    int per_cu = 0, dev = 0, cus = 0, coop = 0;
    if (groups > fl::kPersistMaxGroups || hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess ||
        !coop ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, sh.kernel, 64 * waves, 0) !=
            hipSuccess ||
        groups > per_cu * cus)
      return sh;
  }
  sh.segments = nseg;
  sh.waves = waves;
  sh.groups = groups;
  return sh;
}

// fl_simulate on a short 1D line: the step loop in launches of up to
// kPersistChunk steps each.
template <typename T>
int simulate_persist1d(fl_context* c, fl_field* state, const fl_scheme* s, const fl_sim_params* p,
                       const PersistShape& sh, fl_sim_result* result, hipStream_t st) {
  fl::SweepArgs<T> a = make_args<T>(c, state, state, s, 0.0, nullptr, nullptr, 1);
  double cfl = p->cfl, dh = p->dh, sim_time = p->sim_time;
  long long max_iters = (long long)p->max_iters, nsteps = kPersistChunk;
  int nseg = sh.segments, first = 1;
  unsigned int spin = kPersistSpin;
  const int count = sh.groups > 1 ? 3 * fl::kPersistWords * sh.groups : 1;
  for (;; first = 0) {
    hipLaunchKernelGGL(fl::persist_init_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256),
                       0, st, c->pctl, c->words, count, first);
    void* args[] = {&a, &c->pctl, &c->words, &nseg, &cfl, &dh, &sim_time, &max_iters, &nsteps,
                    &first, &spin};
    if (sh.groups > 1)
      FL_HIP(hipLaunchCooperativeKernel(sh.kernel, dim3(sh.groups), dim3(64 * sh.waves), args, 0,
                                        st));
    else
      FL_HIP(hipLaunchKernel(sh.kernel, dim3(1), dim3(64 * sh.waves), args, 0, st));
    const long long before = first ? 0 : c->host_pctl->iters;
    FL_HIP(hipMemcpyAsync(c->host_pctl, c->pctl, sizeof(fl::PersistCtl), hipMemcpyDeviceToHost,
                          st));
    FL_HIP(hipStreamSynchronize(st));
    const fl::PersistCtl& h = *c->host_pctl;
    if (h.err)
      return fail(FL_ERR_HIP, "persistent step loop: an exchange timed out after step %lld",
                  before);
    // ended by its condition, or after the launch's steps
    if (h.iters - before < nsteps || h.iters >= max_iters) break;
  }
  const fl::PersistCtl h = *c->host_pctl;
  const double final_ws = bits_to_double(h.ws);
  if (result) {
    result->run_time = h.t;
    result->iters = h.iters;
    result->last_dt = h.dt;
    result->max_wavespeed = final_ws;
  }
  if (!(final_ws > 0.0) || isnan(final_ws))
    return fail(FL_ERR_NUMERIC, "max wavespeed %g after %lld steps (NaN or vacuum)", final_ws,
                (long long)h.iters);
  return FL_OK;
}

}  // namespace

namespace {

void drop_sim_graphs(fl_context* c) {
  for (int g = 0; g < 2; ++g) {
    if (c->sim_exec[g]) (void)hipGraphExecDestroy(c->sim_exec[g]);
    if (c->sim_graph[g]) (void)hipGraphDestroy(c->sim_graph[g]);
    c->sim_exec[g] = nullptr;
    c->sim_graph[g] = nullptr;
  }
}

}  // namespace

extern "C" {

const char* fl_status_string(int status) {
  switch (status) {
    case FL_OK: return "ok";
    case FL_ERR_ARGUMENT: return "invalid argument";
    case FL_ERR_UNSUPPORTED: return "unsupported";
    case FL_ERR_HIP: return "HIP runtime error";
    case FL_ERR_NUMERIC: return "numeric failure";
    default: return "unknown status";
  }
}

const char* fl_last_error(void) { return g_last_error.c_str(); }

const char* fl_version(void) { return "fluidity_amd 0.1 (gfx950)"; }

int fl_ctx_create(int device, fl_context** out) {
  if (!out) return fail(FL_ERR_ARGUMENT, "ctx out-pointer is NULL");
  *out = nullptr;
  int count = 0;
  FL_HIP(hipGetDeviceCount(&count));
  if (device < 0 || device >= count)
    return fail(FL_ERR_ARGUMENT, "device %d out of range (%d devices)", device, count);
  DeviceGuard g(device);
  fl_context* c = new fl_context();
  memset(c, 0, sizeof(*c));
  c->device = device;
  (void)resolve_tuning(nullptr, &c->tuning, c->shape);
  c->use_graphs = 1;
  // one block on the device and one pinned, each part on 256 bytes of its own
  size_t dev = 0, host = 0;
  auto part = [](size_t& at, size_t bytes) {
    const size_t a = at;
    at += (bytes + 255) & ~(size_t)255;
    return a;
  };
  const size_t sums = sizeof(double) * kSumBlocks * 4;
  const size_t ctl = part(dev, sizeof(fl::StepCtl)), ws_tmp = part(dev, sizeof(unsigned long long)),
               sim = part(dev, sizeof(fl::SimCtl)), eik = part(dev, 2 * sizeof(fl::ls::EikCtl)),
               pctl = part(dev, sizeof(fl::PersistCtl)), partial = part(dev, sums),
               words = part(dev, sizeof(unsigned long long) * 3 * fl::kPersistWords *
                                     fl::kPersistMaxGroups);
  const size_t host_ctl = part(host, sizeof(fl::StepCtl)), host_sim = part(host, sizeof(fl::SimCtl)),
               host_eik = part(host, 2 * sizeof(fl::ls::EikCtl)),
               host_pctl = part(host, sizeof(fl::PersistCtl)), host_partial = part(host, sums);
  hipError_t e = hipMalloc((void**)&c->dev_block, dev);
  if (e == hipSuccess) e = hipHostMalloc((void**)&c->host_block, host, 0);
  if (e == hipSuccess) e = hipStreamCreate(&c->cap_stream);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&c->step_ev, hipEventDisableTiming);
  if (e != hipSuccess) {
    fl_ctx_destroy(c);
    return fail(FL_ERR_HIP, "context allocation failed: %s", hipGetErrorString(e));
  }
  c->ctl = (fl::StepCtl*)(c->dev_block + ctl);
  c->ws_tmp = (unsigned long long*)(c->dev_block + ws_tmp);
  c->sim = (fl::SimCtl*)(c->dev_block + sim);
  c->eik = (fl::ls::EikCtl*)(c->dev_block + eik);
  c->pctl = (fl::PersistCtl*)(c->dev_block + pctl);
  c->partial = (double*)(c->dev_block + partial);
  c->words = (unsigned long long*)(c->dev_block + words);
  c->host_ctl = (fl::StepCtl*)(c->host_block + host_ctl);
  c->host_sim = (fl::SimCtl*)(c->host_block + host_sim);
  c->host_eik = (fl::ls::EikCtl*)(c->host_block + host_eik);
  c->host_pctl = (fl::PersistCtl*)(c->host_block + host_pctl);
  c->host_partial = (double*)(c->host_block + host_partial);
  *out = c;
  return FL_OK;
}

int fl_ctx_destroy(fl_context* c) {
  if (!c) return FL_OK;
  DeviceGuard g(c->device);
  drop_sim_graphs(c);
  if (c->cap_stream) (void)hipStreamDestroy(c->cap_stream);
  if (c->step_ev) (void)hipEventDestroy(c->step_ev);
  if (c->dev_block) (void)hipFree(c->dev_block);
  if (c->host_block) (void)hipHostFree(c->host_block);
  delete c;
  return FL_OK;
}

int fl_ctx_set_tuning(fl_context* c, const fl_tuning* t) {
  if (!c || !t) return fail(FL_ERR_ARGUMENT, "NULL context or tuning");
  const int rc = take_tuning(t, &c->tuning, c->shape);
  if (rc) return rc;
  if (t->x_block || t->x_rows) c->cell_cells[0] = 0;
  if (t->y_block || t->y_rows) c->cell_cells[1] = 0;
  return FL_OK;
}

int fl_ctx_get_tuning(const fl_context* c, fl_tuning* t) {
  if (!c || !t) return fail(FL_ERR_ARGUMENT, "NULL context or tuning");
  *t = tuning_of(c->tuning, c->shape);
  return FL_OK;
}

int fl_ctx_autotune(fl_context* c, const fl_field* in, const fl_field* work,
                    const fl_scheme* s, int reps, fl_tuning* chosen, void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  int rc = check_pair(in, work);
  if (rc) return rc;
  if ((rc = check_scheme(s, in->ndim))) return rc;
  if (reps < 1 || reps > 100) return fail(FL_ERR_ARGUMENT, "reps %d out of [1, 100]", reps);
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  static const int widths[] = {64, 128, 256};
  static const int xrows[] = {8, 16, 32, 64};
  static const int yrows[] = {16, 32, 64, 128};
  int cus = 0;
  FL_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
  hipEvent_t e0, e1;
  FL_HIP(hipEventCreate(&e0));
  FL_HIP(hipEventCreate(&e1));
  const fl_tuning saved = c->tuning;
  const int32_t saved_shape[2] = {c->shape[0], c->shape[1]};
  const int64_t saved_cells[2] = {c->cell_cells[0], c->cell_cells[1]};
  fl_tuning best = c->tuning;
  // the sweep with the context's current shape: milliseconds over reps launches
  // (on a line with the maximum that its steps reduce: 200000 cells are 3226
  // workgroups of 64 lanes, whose atomics are most of the 58 us of a step, in
  // 256 lanes 32)
  auto timed = [&](int dim, float* total) -> int {
    int err = FL_OK;
    *total = 0.0f;
    for (int r = 0; r <= reps && !err; ++r) {  // r = 0 warms up
      if (hipEventRecord(e0, st) != hipSuccess) err = fail(FL_ERR_HIP, "hipEventRecord");
      if (!err)
        err = launch_sweep(c, in, work, dim, s, 1e-3, nullptr, in->ndim == 1 ? c->ws_tmp : nullptr,
                           st);
      if (!err && hipEventRecord(e1, st) != hipSuccess) err = fail(FL_ERR_HIP, "hipEventRecord");
      if (!err && hipEventSynchronize(e1) != hipSuccess) err = fail(FL_ERR_HIP, "hipEventSynchronize");
      float ms = 0.0f;
      if (!err) (void)hipEventElapsedTime(&ms, e0, e1);
      if (r > 0) *total += ms;
    }
    return err;
  };
  for (int dim = 0; dim < in->ndim && !rc; ++dim) {
    float best_ms = 1e30f;
    if (in->ndim == 2) c->shape[dim] = kShapeTuning;
    for (int w : widths) {
      std::vector<int> rows(1, 0);  // 1D: the height is unused
      if (in->ndim == 2) {
        const int64_t nx = in->n[0], ny = in->n[1];
        const int64_t bands = dim ? (nx + w - 1) / w : (nx + w - 3) / (w - 2);
        const int per_cu = in->dtype == FL_F64 ? sweep_blocks_per_cu_t<double>(dim, s, w)
                                               : sweep_blocks_per_cu_t<float>(dim, s, w);
        rows = row_candidates(dim ? yrows : xrows, 4, bands, ny, (int64_t)per_cu * cus);
      }
      for (size_t k = 0; k < rows.size() && !rc; ++k) {
        fl_tuning t = best;
        if (dim == 0) {
          t.x_block = w;
          if (rows[k]) t.x_rows = rows[k];
        } else {
          t.y_block = w;
          t.y_rows = rows[k];
        }
        c->tuning = t;
        float total = 0.0f;
        rc = timed(dim, &total);
        if (!rc && total < best_ms) {
          best_ms = total;
          best = t;
        }
      }
    }
    // the cell-parallel kernel, on grids where it can be the faster one
    if (in->ndim == 2 && !rc && in->n[0] * in->n[1] <= kCellTryMax) {
      float total = 0.0f;
      c->shape[dim] = kShapeCell;
      c->cell_cells[dim] = in->n[0] * in->n[1];
      rc = timed(dim, &total);
      // the best of many marching shapes is a lucky one when they are about
      // equal, the more so where a sweep takes 20 us (512^2: 22 against 17 us
      // in the steps after it)
      const bool small = in->n[0] * in->n[1] <= (1 << 20);
      if (!rc && total >= (small ? 1.25f : 1.05f) * best_ms) c->shape[dim] = kShapeTuning;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  c->tuning = rc ? saved : best;
  for (int d = 0; rc && d < 2; ++d) {
    c->shape[d] = saved_shape[d];
    c->cell_cells[d] = saved_cells[d];
  }
  if (!rc && chosen) *chosen = tuning_of(c->tuning, c->shape);
  return rc;
}

int fl_split_sweep(fl_context* c, const fl_field* in, const fl_field* out, int dim,
                   const fl_scheme* s, double dtdh, void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  int rc = check_pair(in, out);
  if (rc) return rc;
  rc = check_scheme(s, in->ndim);
  if (rc) return rc;
  if (dim < 0 || dim >= in->ndim) return fail(FL_ERR_ARGUMENT, "dim %d out of range", dim);
  if (!(dtdh > 0.0) || !isfinite(dtdh)) return fail(FL_ERR_ARGUMENT, "dtdh %g must be > 0", dtdh);
  DeviceGuard g(c->device);
  return launch_sweep(c, in, out, dim, s, dtdh, nullptr, nullptr, (hipStream_t)stream);
}

int fl_split_solve(fl_context* c, fl_field* in, fl_field* out, const fl_scheme* s, double dtdh,
                   void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  int rc = check_pair(in, out);
  if (rc) return rc;
  rc = check_scheme(s, in->ndim);
  if (rc) return rc;
  if (!(dtdh > 0.0) || !isfinite(dtdh)) return fail(FL_ERR_ARGUMENT, "dtdh %g must be > 0", dtdh);
  DeviceGuard g(c->device);
  for (int d = 0; d < in->ndim; ++d) {
    rc = launch_sweep(c, in, out, d, s, dtdh, nullptr, nullptr, (hipStream_t)stream);
    if (rc) return rc;
    if (in->ndim != 1 && d < in->ndim - 1) {  // solver/cuda/split_solver.cuh:75-78
      void* tmp = in->data;
      in->data = out->data;
      out->data = tmp;
    }
  }
  return FL_OK;
}

int fl_split_step(fl_context* c, fl_field* in, fl_field* out, const fl_scheme* s, double dtdh,
                  double* max_wavespeed, void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  int rc = check_pair(in, out);
  if (rc) return rc;
  rc = check_scheme(s, in->ndim);
  if (rc) return rc;
  if (!(dtdh > 0.0) || !isfinite(dtdh)) return fail(FL_ERR_ARGUMENT, "dtdh %g must be > 0", dtdh);
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  if (max_wavespeed) hipLaunchKernelGGL(fl::zero_u64_kernel, dim3(1), dim3(1), 0, st, c->ws_tmp);
  for (int d = 0; d < in->ndim; ++d) {
    // the last sweep writes the final states and reduces their wavespeeds
    unsigned long long* ws = (max_wavespeed && d == in->ndim - 1) ? c->ws_tmp : nullptr;
    rc = launch_sweep(c, in, out, d, s, dtdh, nullptr, ws, st);
    if (rc) return rc;
    if (in->ndim != 1 && d < in->ndim - 1) {  // solver/cuda/split_solver.cuh:75-78
      void* tmp = in->data;
      in->data = out->data;
      out->data = tmp;
    }
  }
  if (max_wavespeed) {
    FL_HIP(hipMemcpyAsync(&c->host_ctl->ws_bits[0], c->ws_tmp, sizeof(unsigned long long),
                          hipMemcpyDeviceToHost, st));
    FL_HIP(hipStreamSynchronize(st));
    *max_wavespeed = bits_to_double(c->host_ctl->ws_bits[0]);
  }
  return FL_OK;
}

int fl_max_wavespeed(fl_context* c, const fl_field* in, const fl_scheme* s, double* result,
                     void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  if (!result) return fail(FL_ERR_ARGUMENT, "result is NULL");
  int rc = check_field(in, "in");
  if (rc) return rc;
  rc = check_scheme(s, in->ndim);
  if (rc) return rc;
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(fl::zero_u64_kernel, dim3(1), dim3(1), 0, st, c->ws_tmp);
  rc = launch_max_ws(in, s, c->ws_tmp, st);
  if (rc) return rc;
  FL_HIP(hipMemcpyAsync(&c->host_ctl->ws_bits[0], c->ws_tmp, sizeof(unsigned long long),
                        hipMemcpyDeviceToHost, st));
  FL_HIP(hipStreamSynchronize(st));
  *result = bits_to_double(c->host_ctl->ws_bits[0]);
  return FL_OK;
}

int fl_set_wavespeeds(fl_context* c, const fl_field* in, const fl_scheme* s, double* ws,
                      void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  if (!ws) return fail(FL_ERR_ARGUMENT, "wavespeeds is NULL");
  int rc = check_field(in, "in");
  if (rc) return rc;
  rc = check_scheme(s, in->ndim);
  if (rc) return rc;
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  int64_t es, cs;
  strides(in, es, cs);
  const int64_t n = cell_count(in);
  const fl::Material<double> m64 = make_material<double>(s);
  const int B = fl::kMaxBlock;
  int64_t blocks = (n + B - 1) / B;
  if (blocks > 8192) blocks = 8192;
  const dim3 grid((unsigned)blocks);
  if (in->dtype == FL_F64) {
    if (in->ndim == 1)
      hipLaunchKernelGGL((fl::wavespeeds_kernel<double, 1>), grid, dim3(B), 0, st,
                         (const double*)in->data, es, cs, n, m64, ws);
    else
      hipLaunchKernelGGL((fl::wavespeeds_kernel<double, 2>), grid, dim3(B), 0, st,
                         (const double*)in->data, es, cs, n, m64, ws);
  } else {
    if (in->ndim == 1)
      hipLaunchKernelGGL((fl::wavespeeds_kernel<float, 1>), grid, dim3(B), 0, st,
                         (const float*)in->data, es, cs, n, m64, ws);
    else
      hipLaunchKernelGGL((fl::wavespeeds_kernel<float, 2>), grid, dim3(B), 0, st,
                         (const float*)in->data, es, cs, n, m64, ws);
  }
  FL_HIP(hipGetLastError());
  return FL_OK;
}

int fl_max_element(fl_context* c, const double* first, int64_t count, double* result,
                   void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  if (!first || !result) return fail(FL_ERR_ARGUMENT, "first or result is NULL");
  if (count <= 0) return fail(FL_ERR_ARGUMENT, "count must be > 0 (got %lld)", (long long)count);
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  const int B = fl::kMaxBlock;
  int64_t blocks = (count + B - 1) / B;
  if (blocks > fl::kMaxWsBlocks) blocks = fl::kMaxWsBlocks;
  hipLaunchKernelGGL(fl::zero_u64_kernel, dim3(1), dim3(1), 0, st, c->ws_tmp);
  hipLaunchKernelGGL(fl::max_element_kernel, dim3((unsigned)blocks), dim3(B), 0, st, first, count,
                     c->ws_tmp);
  FL_HIP(hipGetLastError());
  FL_HIP(hipMemcpyAsync(&c->host_ctl->ws_bits[0], c->ws_tmp, sizeof(unsigned long long),
                        hipMemcpyDeviceToHost, st));
  FL_HIP(hipStreamSynchronize(st));
  const unsigned long long k = c->host_ctl->ws_bits[0];
  if (k == ~0ull) {
    *result = NAN;
  } else {
    // invert the order-preserving key of the max_element kernel
    const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    *result = bits_to_double(b);
  }
  return FL_OK;
}

int fl_ctx_set_graphs(fl_context* c, int enable) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  c->use_graphs = enable ? 1 : 0;
  return FL_OK;
}

int fl_simulate(fl_context* c, fl_field* state, fl_field* work, const fl_scheme* s,
                const fl_sim_params* p, fl_sim_result* result, void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  int rc = check_pair(state, work);
  if (rc) return rc;
  rc = check_scheme(s, state->ndim);
  if (rc) return rc;
  if (!p) return fail(FL_ERR_ARGUMENT, "params is NULL");
  if (!(p->cfl > 0.0) || !isfinite(p->cfl)) return fail(FL_ERR_ARGUMENT, "cfl must be > 0");
  if (!(p->dh > 0.0) || !isfinite(p->dh)) return fail(FL_ERR_ARGUMENT, "dh must be > 0");
  if (p->max_iters < 0) return fail(FL_ERR_ARGUMENT, "max_iters must be >= 0");
  if (isnan(p->sim_time)) return fail(FL_ERR_ARGUMENT, "sim_time is NaN");
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;

  if (c->use_graphs && p->max_iters > 0) {  // (no step: its launch alone is 20 us more)
    const PersistShape sh = persist_shape(state, s);
    if (sh.groups > 0) {
      if (state->dtype == FL_F64)
        return simulate_persist1d<double>(c, state, s, p, sh, result, st);
      return simulate_persist1d<float>(c, state, s, p, sh, result, st);
    }
  }

  hipLaunchKernelGGL(fl::init_sim_kernel, dim3(1), dim3(1), 0, st, c->sim);
  rc = launch_max_ws(state, s, &c->sim->ws[0], st);
  if (rc) return rc;

  // Steps are launched in batches; between batches the host reads the control
  // words once to stop when the loop condition fails.  With graphs on, a run
  // of kSimGraphSteps steps and the steps that a loop of max_iters leaves over
  // are captured and replayed (one host launch per graph, about 1 us less per
  // kernel on the device): at once for loops of kSimGraphMin steps or more,
  // from the second call of the same loop on for shorter ones, which cost
  // less than their capture.  A step past the stop condition does nothing.
  constexpr int kSimGraphSteps = 18;  // a multiple of both slot cycles (2 and 3)
  constexpr int64_t kSimGraphMin = 4 * kSimGraphSteps;
  constexpr int64_t kBatch = 14 * kSimGraphSteps;
  const int64_t left_over = p->max_iters % kSimGraphSteps;
  int64_t launched = 0;
  bool graphs = false;
  if (c->use_graphs) {
    SimGraphKey key;
    memset(&key, 0, sizeof(key));
    key.a = state->data;
    key.b = work->data;
    key.dtype = state->dtype;
    key.layout = state->layout;
    key.ndim = state->ndim;
    for (int d = 0; d < 3; ++d) key.n[d] = state->n[d];
    key.scheme = *s;
    key.cfl = p->cfl;
    key.dh = p->dh;
    key.sim_time = p->sim_time;
    key.max_iters = p->max_iters;
    key.tuning = c->tuning;
    for (int d = 0; d < 2; ++d) {
      key.shape[d] = c->shape[d];
      key.cell_cells[d] = c->cell_cells[d];
    }
    const bool again = memcmp(&key, &c->sim_key, sizeof(key)) == 0;
    if (!again) {
      drop_sim_graphs(c);
      c->sim_key = key;
    }
    graphs = again || p->max_iters >= kSimGraphMin;
    const int64_t steps[2] = {p->max_iters >= kSimGraphSteps ? kSimGraphSteps : 0, left_over};
    for (int g = 0; graphs && g < 2; ++g) {
      if (c->sim_exec[g] || !steps[g]) continue;
      FL_HIP(hipStreamBeginCapture(c->cap_stream, hipStreamCaptureModeThreadLocal));
      for (int64_t k = 0; k < steps[g] && !rc; ++k)
        rc = launch_sim_step(c, state, work, s, p, c->sim, k, c->cap_stream);
      hipGraph_t gr = nullptr;
      const hipError_t e = hipStreamEndCapture(c->cap_stream, &gr);
      if (rc) {
        if (gr) (void)hipGraphDestroy(gr);
        return rc;
      }
      if (e != hipSuccess)
        return fail(FL_ERR_HIP, "step graph capture failed: %s", hipGetErrorString(e));
      c->sim_graph[g] = gr;
      FL_HIP(hipGraphInstantiate(&c->sim_exec[g], gr, nullptr, nullptr, 0));
    }
  }
  do {
    const int64_t nb = std::min<int64_t>(p->max_iters - launched, kBatch);
    int64_t k = 0;
    if (graphs) {
      for (; k + kSimGraphSteps <= nb; k += kSimGraphSteps)
        FL_HIP(hipGraphLaunch(c->sim_exec[0], st));
      if (nb - k == left_over && left_over) {
        FL_HIP(hipGraphLaunch(c->sim_exec[1], st));
        k = nb;
      }
    }
    for (; k < nb; ++k)
      if ((rc = launch_sim_step(c, state, work, s, p, c->sim, launched + k, st))) return rc;
    launched += nb;
    FL_HIP(hipMemcpyAsync(c->host_sim, c->sim, sizeof(fl::SimCtl), hipMemcpyDeviceToHost, st));
    FL_HIP(hipStreamSynchronize(st));
  } while (launched < p->max_iters && c->host_sim->c.active);
  const fl::SimCtl hs = *c->host_sim;
  const fl::StepCtl hc = hs.c;
  if (state->ndim == 1 && (hc.iters & 1)) {
    const int64_t bytes = cell_count(state) * 3 * (state->dtype == FL_F64 ? 8 : 4);
    FL_HIP(hipMemcpyAsync(state->data, work->data, (size_t)bytes, hipMemcpyDeviceToDevice, st));
    FL_HIP(hipStreamSynchronize(st));
  }
  const double final_ws = bits_to_double(hs.ws[hc.iters % sim_slots(state->ndim)]);
  if (result) {
    result->run_time = hc.t;
    result->iters = hc.iters;
    result->last_dt = hc.dt;
    result->max_wavespeed = final_ws;
  }
  if (!(final_ws > 0.0) || isnan(final_ws))
    return fail(FL_ERR_NUMERIC, "max wavespeed %g after %lld steps (NaN or vacuum)", final_ws,
                (long long)hc.iters);
  return FL_OK;
}

int fl_conservation_sums(fl_context* c, const fl_field* in, double* sums, void* stream) {
  if (!c) return fail(FL_ERR_ARGUMENT, "context is NULL");
  if (!sums) return fail(FL_ERR_ARGUMENT, "sums is NULL");
  int rc = check_field(in, "in");
  if (rc) return rc;
  DeviceGuard g(c->device);
  hipStream_t st = (hipStream_t)stream;
  int64_t es, cs;
  strides(in, es, cs);
  const int64_t n = cell_count(in);
  const int S = 2 + in->ndim;
  int64_t blocks = (n + 255) / 256;
  if (blocks > kSumBlocks) blocks = kSumBlocks;
  dim3 grid((unsigned)blocks);
  if (in->dtype == FL_F64) {
    if (S == 3)
      hipLaunchKernelGGL((fl::component_sums_kernel<double, 3>), grid, dim3(256), 0, st,
                         (const double*)in->data, es, cs, n, c->partial);
    else
      hipLaunchKernelGGL((fl::component_sums_kernel<double, 4>), grid, dim3(256), 0, st,
                         (const double*)in->data, es, cs, n, c->partial);
  } else {
    if (S == 3)
      hipLaunchKernelGGL((fl::component_sums_kernel<float, 3>), grid, dim3(256), 0, st,
                         (const float*)in->data, es, cs, n, c->partial);
    else
      hipLaunchKernelGGL((fl::component_sums_kernel<float, 4>), grid, dim3(256), 0, st,
                         (const float*)in->data, es, cs, n, c->partial);
  }
  FL_HIP(hipGetLastError());
  FL_HIP(hipMemcpyAsync(c->host_partial, c->partial, sizeof(double) * blocks * S,
                        hipMemcpyDeviceToHost, st));
  FL_HIP(hipStreamSynchronize(st));
  for (int k = 0; k < S; ++k) {
    double v = 0.0;
    for (int64_t b = 0; b < blocks; ++b) v += c->host_partial[b * S + k];
    sums[k] = v;
  }
  return FL_OK;
}

}  // extern "C"
