// fused.hip -- the whole 3-D hydro step of one grid in one HBM pass.
//
// k_fused runs the tile march of fused_core.h over one grid: one block per
// (column tile, z chunk), with the tiles of each XCD contiguous; on 2-D
// grids (nz = 1), k_fused2d marches row strips along y (march2d.h).  k_cfl
// gives the first step's CFL limit.  The file is compiled three times:
// EVH_FUSED_PREC=64 (FP64, fast arithmetic), EVH_FUSED_PREC=32 (FP32-mixed)
// and EVH_FUSED_EXACT=1 (FP64 with the reference's arithmetic, compiled
// without FMA contraction).
#include "fused_core.h"
#include "march2d.h"

#ifndef EVH_FUSED_PREC
#define EVH_FUSED_PREC 64
#endif
#ifndef EVH_FUSED_EXACT
#define EVH_FUSED_EXACT 0
#endif
#if EVH_FUSED_EXACT && EVH_FUSED_PREC != 64
#error "the exact form is FP64"
#endif
constexpr bool kExact = EVH_FUSED_EXACT != 0;
// the exact build's kernel has a name of its own, so that profiles keep the
// two FP64 forms apart
#if EVH_FUSED_EXACT
#define K_FUSED k_fused_exact
#define K_FUSED2D k_fused2d_exact
#else
#define K_FUSED k_fused
#define K_FUSED2D k_fused2d
#endif

namespace evh {
namespace {

using core::Geo;

// WPE: waves per SIMD the register allocation must leave room for
// (512 / WPE VGPRs per lane).
// SLAB: a z-slab whose ghost planes may come from halo buffers.
template <typename T, typename S, int SOLVER, int LIMITER, int TX, int TY, int WPE, bool SLAB>
__global__ void __launch_bounds__((core::TileShape<TX, TY>::NT)) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    K_FUSED(KParams P, Geo G, const S *__restrict__ qin, S *__restrict__ qout, StepCtl C, S *__restrict__ tout) {
  __shared__ core::Smem<T, TX, TY> sm;
  const int lin = xcd_tile(blockIdx.x, G.ntiles);
  double dt;
  if (!step_begin(P, C, dt) || lin < 0) return;  // no step, or a padding block (whole blocks, before any barrier)
  core::march<T, S, SOLVER, LIMITER, TX, TY, kExact, SLAB>(P, G, qin, qout, 0, 0, dt, C.st, C.lim, lin, sm, tout);
}

// 2-D grids (nz = 1): row strips marching along y (march2d.h)
template <typename T, typename S, int SOLVER, int LIMITER, int WPE>
__global__ void __launch_bounds__(core2d::NL) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    K_FUSED2D(KParams P, core2d::Geo2 G, const S *__restrict__ qin, S *__restrict__ qout, StepCtl C,
              S *__restrict__ tout) {
  __shared__ core2d::Smem2<T> sm;
  const int lin = xcd_tile(blockIdx.x, G.ntiles);
  double dt;
  if (!step_begin(P, C, dt) || lin < 0) return;  // no step, or a padding block (whole blocks, before any barrier)
  core2d::march2d<T, S, SOLVER, LIMITER, kExact>(P, G, qin, qout, dt, C.st, C.lim, lin, sm, tout);
}

// primitive + CFL min over q without materialising w (first step, after
// uploads): exact IEEE arithmetic, so the first dt equals the reference's.
template <typename S>
__global__ void __launch_bounds__(256) k_cfl(KParams P, Geo G, const S *__restrict__ q, Status *st) {
  double vmin = 1e6;
  for (long long c = blockIdx.x * 256LL + threadIdx.x; c < G.n; c += (long long)gridDim.x * 256) {
    double qc[6], wc[5];
#pragma unroll
    for (int m = 0; m < 6; m++) qc[m] = double(q[m * G.n + c]);
    const int e = q2w(P, qc, wc);
    if (e) report_next(st, e, (unsigned long long)c);
    vmin = min_limit(vmin, cfl_cell(P, wc));
  }
  block_min_pos<256>(&st->vmin_bits, vmin);
}

Geo make_geo(const evh_ctx *h, int tx, int ty) {
  Geo g;
  g.nx = h->grid.nx;
  g.ny = h->grid.ny;
  g.nz = h->grid.nz;
  g.n = h->grid.n();
  g.tiles_x = (g.nx + tx - 1) / tx;
  g.tiles_y = (g.ny + ty - 1) / ty;
  g.zchunk = h->zchunk > 0 ? h->zchunk
                           : march_chunk(h->cfg.precision == EVH_FP32_MIXED ? kMarch32 : kMarch64,
                                         (long long)g.tiles_x * g.tiles_y, g.nz, 128);
  if (g.zchunk > g.nz) g.zchunk = g.nz;
  g.nchunks = (g.nz + g.zchunk - 1) / g.zchunk;
  g.ntiles = g.tiles_x * g.tiles_y * g.nchunks;
  g.zlo = h->zslab[0] ? h->zhalo[0] : nullptr;
  g.zhi = h->zslab[1] ? h->zhalo[1] : nullptr;
  return g;
}

template <typename T, typename S, int SOLVER, int LIMITER, int TX, int TY, int WPE, bool SLAB = false>
void launch_ty(evh_ctx *h, const StepCtl &c) {
  const Geo g = make_geo(h, TX, TY);
  const int blocks = xcd_blocks(g.ntiles);
  hipLaunchKernelGGL((K_FUSED<T, S, SOLVER, LIMITER, TX, TY, WPE, SLAB>), dim3(blocks), dim3((core::TileShape<TX, TY>::NT)), 0,
                     h->stream, h->kp, g, (const S *)h->qbuf[h->cur], (S *)h->qbuf[1 - h->cur], c,
                     (S *)h->tbuf);
}

// the 2-D form: strips of 252 columns, chunks of up to 64 rows (the z chunk
// of the tuning, when set), WPE waves per SIMD
template <typename T, typename S, int SOLVER, int LIMITER, int WPE>
void launch_2d(evh_ctx *h, const StepCtl &c) {
  core2d::Geo2 g;
  g.nx = h->grid.nx;
  g.ny = h->grid.ny;
  g.n = h->grid.n();
  g.strips = (g.nx + core2d::NC - 1) / core2d::NC;
  g.ychunk = h->zchunk > 0 ? h->zchunk : march_chunk(sizeof(T) == 4 ? kMarch2d32 : kMarch2d64, g.strips, g.ny, 64);
  if (g.ychunk > g.ny) g.ychunk = g.ny;
  g.nchunks = (g.ny + g.ychunk - 1) / g.ychunk;
  g.ntiles = g.strips * g.nchunks;
  hipLaunchKernelGGL((K_FUSED2D<T, S, SOLVER, LIMITER, WPE>), dim3(xcd_blocks(g.ntiles)), dim3(core2d::NL), 0,
                     h->stream, h->kp, g, (const S *)h->qbuf[h->cur], (S *)h->qbuf[1 - h->cur], c,
                     (S *)h->tbuf);
}

// The register budget is 2 waves per SIMD in FP64 (a column's values take
// about 220 of the 256 registers it leaves; 168 for 3 waves spill 64: 12.4 ms
// against 5.8 at 512^3) and 4 in FP32.  2-D grids take the row-strip march in
// its one shape.
template <typename T, typename S, int SOLVER, int LIMITER>
void launch_fused_t(evh_ctx *h, const StepCtl &c) {
  constexpr int W = sizeof(T) == 8 ? 2 : 4;
  const int nx = h->grid.nx, ny = h->grid.ny;
  if (h->grid.nz == 1) {
    // 2-D: FP64 at 3 waves per SIMD (its row carry in LDS: 3% faster than 2
    // waves at 8192^2), FP32 at 4
    launch_2d<T, S, SOLVER, LIMITER, sizeof(T) == 8 ? 3 : 4>(h, c);
    return;
  }
  const bool slab = h->zslab[0] || h->zslab[1];  // with halo buffers: tile height 12 (the z chunk is the tuning's)
  if (!slab && h->tile_ty == 8) {
    launch_ty<T, S, SOLVER, LIMITER, 16, 8, W>(h, c);
    return;
  }
  if constexpr (sizeof(T) == 4) {
    if (wide_tile(tiles_of(nx, ny, 32, 6), tiles_of(nx, ny, 16, 12))) {
      if (slab) launch_ty<T, S, SOLVER, LIMITER, 32, 6, W, true>(h, c);
      else launch_ty<T, S, SOLVER, LIMITER, 32, 6, W>(h, c);
      return;
    }
  }
  if (slab) launch_ty<T, S, SOLVER, LIMITER, 16, 12, W, true>(h, c);
  else launch_ty<T, S, SOLVER, LIMITER, 16, 12, W>(h, c);
}

template <typename T, typename S>
hipError_t launch_fused_prec(evh_ctx *h, const StepCtl &c) {
  const int s = h->kp.solver, l = h->kp.limiter;
  if (s == 1 && l == 1) launch_fused_t<T, S, 1, 1>(h, c);
  else if (s == 1 && l == 2) launch_fused_t<T, S, 1, 2>(h, c);
  else if (s == 1 && l == 3) launch_fused_t<T, S, 1, 3>(h, c);
  else if (s == 2 && l == 1) launch_fused_t<T, S, 2, 1>(h, c);
  else if (s == 2 && l == 2) launch_fused_t<T, S, 2, 2>(h, c);
  else if (s == 2 && l == 3) launch_fused_t<T, S, 2, 3>(h, c);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace

#if EVH_FUSED_PREC == 64 && !EVH_FUSED_EXACT
// 3-D grids, and 2-D grids (nz = 1) in the march's 2-D form
bool fused_supported(const evh_config &c) { return c.nx >= 2 && c.ny >= 2 && c.nz >= 1; }

hipError_t launch_cfl(evh_ctx *h) {
  const Geo g = make_geo(h, 16, 12);
  long long b = (g.n + 255) / 256;
  if (b > 2048) b = 2048;
  if (h->cfg.precision == EVH_FP32_MIXED)
    hipLaunchKernelGGL(k_cfl<float>, dim3((int)b), dim3(256), 0, h->stream, h->kp, g, (const float *)h->qbuf[h->cur],
                       h->st);
  else
    hipLaunchKernelGGL(k_cfl<double>, dim3((int)b), dim3(256), 0, h->stream, h->kp, g,
                       (const double *)h->qbuf[h->cur], h->st);
  return hipGetLastError();
}
#endif

#if EVH_FUSED_EXACT
hipError_t launch_fused_exact(evh_ctx *h, const StepCtl &c) { return launch_fused_prec<double, double>(h, c); }
#elif EVH_FUSED_PREC == 32
hipError_t launch_fused_f32(evh_ctx *h, const StepCtl &c) { return launch_fused_prec<float, float>(h, c); }
#else
hipError_t launch_fused_f64(evh_ctx *h, const StepCtl &c) { return launch_fused_prec<double, double>(h, c); }

hipError_t launch_fused_step(evh_ctx *h, const StepCtl &c) {
  if (h->cfg.precision == EVH_FP32_MIXED) return launch_fused_f32(h, c);
  if (h->mode == EVH_MODE_FUSED_EXACT) return launch_fused_exact(h, c);
  return launch_fused_f64(h, c);
}
#endif

}  // namespace evh
