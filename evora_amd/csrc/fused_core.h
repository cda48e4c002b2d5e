// fused_core.h -- the tile march of the fused hydro step, shared by the
// single-grid kernel (fused.hip) and the batched persistent kernel
// (batch.hip).
//
// A block owns a TX x TY column tile of one box and marches up a chunk of z
// planes, reading q^n once and writing q^{n+1} once; w, evo and s never
// exist in HBM.  The interior waves (TX TY / 64 of them) own the tile's
// columns one to one; the last wave (the "ring wave") owns the 2 (TX + TY)
// columns of the first halo ring, one or two per lane, and loads the second
// ring and the four corners, so every interior lane does useful work in every
// stage.  The two roles run loops of their own with the same barriers.  Per
// plane k:
//   S1  w of plane k goes to LDS with both halo rings.
//   S2  primitive (comp.f90:26-85) of plane k+1, with the ghost cells of
//       `bound` (boundary.f90) folded into the load index (a column's x-y
//       offset is formed once per march; the ring wave forms its own ahead,
//       in S3, and its second-ring cells' here); limited slopes in x, y, z
//       and the predictor evo (muscl.f90:45-169) of plane k; the x/y face states go to LDS per face; the interior
//       lanes solve their z face k-1/2 (riemann.f90) and finish plane k-1
//       as (q + dtx*(Fx) + dty*(Fy)) + dtz*(Fz), the reference's x, y, z
//       order (muscl.f90:191-272, integration :287), store it, and take the
//       CFL limit of its new state for the next hydrostep
//       (timestep.f90:26-57; CflMin).
//   S3  x and y faces of plane k: interior lane (i,j) solves its left and
//       bottom faces, the ring wave the TY right-edge and TX top-edge faces
//       in one solve.  Each flux overwrites the two states it came from.
//   S4  q(k) + dtx*(Fx) + dty*(Fy) of plane k, carried in registers with the
//       z flux and the top z state to S2 of plane k+1.
// Template parameters: T compute type, S storage type of q (double/double
// for the FP64 form, float/float for the FP32-mixed form), SOLVER, LIMITER,
// TX x TY the tile.  2-D grids march along y instead (march2d.h).
//
// What bounds it: FP64, the issue of vector instructions (a wave64 FP64
// instruction takes about 5 cycles of its SIMD, and the SIMDs that hold
// interior waves only have one to issue 98% of the time); FP32-mixed, the
// L1's requests to L2 for the ring.  512^3 HLLC blast, FP64: 6.36 ms with both
// roles in one loop (219 VGPRs) and the carry in LDS; 5.49 ms (24.4 G cell
// updates/s) with a loop per role, so that neither holds the other's values
// (the carry in registers, 32 of 135 LDS operations per plane gone, 46 KB of
// LDS instead of 72), third-order reciprocals and roots, the star flux from
// its jump conditions, the predictor from shared factors, and the limit from
// q.  FP32-mixed: 3.33 -> 2.62 ms (51 G), with its constants in scalar
// registers (16 B/lane of spills gone) and the 32 x 6 tile.
#pragma once

#include "evh_internal.h"
#include "physics_fast.h"

namespace evh {
namespace core {

template <int TX_, int TY_>
struct TileShape {
  static constexpr int TX = TX_, TY = TY_;
  static constexpr int NI = TX * TY;              // interior lanes
  static constexpr int NT = NI + 64;              // + the ring wave
  static constexpr int NR1 = 2 * TX + 2 * TY;     // first-ring columns
  static constexpr int NP = (NR1 + 4 + 63) / 64;  // columns and corners per ring lane
  static constexpr int EW = TX + 4;               // extended plane pitch (x from -2 to TX+1)
  static constexpr int EA = EW * (TY + 4);        // extended plane area
  static constexpr int NFX = (TX + 1) * TY;       // x faces of a plane
  static constexpr int NFY = TX * (TY + 1);       // y faces of a plane
  static_assert(NI % 64 == 0, "interior lanes must fill whole wavefronts");
  static_assert(TX + TY <= 64, "the edge faces must fit one wavefront");
  __device__ static __forceinline__ int eidx(int x, int y) { return (x + 2) + EW * (y + 2); }
};

struct Geo {
  int nx, ny, nz;
  long long n;
  int zchunk;
  int tiles_x, tiles_y, nchunks;
  int ntiles;  // tiles_x * tiles_y * nchunks
  // a z-slab of a grid decomposed along z: the two ghost planes below (zlo)
  // and above (zhi) come from the neighbouring slabs, [6][2][ny][nx] in the
  // storage type; null: the z rules of bound
  const void *zlo, *zhi;
};

// mixed form: FP64 pressure recovery where the flow is fast
template <typename T>
struct Prim;

template <>
struct Prim<double> {
  __device__ static __forceinline__ int q2w(const KParams &P, double q[6], double w[5], double &rinv) {
    return fast::q2w(P, q, w, rinv);
  }
};

template <>
struct Prim<float> {
  // 0.5 m^2 / rho in FP64, an IEEE quotient
  __device__ static __forceinline__ double kin64(const float q[6]) {
    const double r = q[0];
    return fm::div_cr(0.5 * (double(q[1]) * q[1] + double(q[2]) * q[2] + double(q[3]) * q[3]), r, fm::rcp(r));
  }
  // FP32 recovery, except where the subtraction E - kin cancels: there
  // (kin/E above the Mach threshold) p = g1 (E - kin) is evaluated in FP64.
  // With dualenergy on, the entropy branch (kin/E > de_thresh1,
  // comp.f90:61-64) recovers p = S rho**g1 and E = kin + p/g1 in FP64.
  __device__ static __forceinline__ int q2w(const KParams &P, float q[6], float w[5], float &rinv) {
    rinv = fm::rcp(q[0]);
    w[0] = q[0];
    w[1] = q[1] * rinv;
    w[2] = q[2] * rinv;
    w[3] = q[3] * rinv;
    const float m2 = fm::fma(q[3], q[3], fm::fma(q[2], q[2], q[1] * q[1]));
    const float kin = 0.5f * m2 * rinv;
    const bool fast_flow = kin > P.f.kin_frac64 * q[4];
    float pr;
    if (P.dualenergy && kin * fm::rcp(q[4]) > P.f.de_thresh1) {
      const double r64 = double(q[0]);
      const double k64 = kin64(q);
      // (the Newton form of the power: this rare branch must not raise the
      // register count of the whole FP32 kernel)
      const double p64 = double(q[5]) * fast::pow_g1<false>(P, r64);
      q[4] = float(k64 + p64 * P.g1inv);
      pr = float(p64);
    } else {
      if (fast_flow) {
        pr = float(P.g1 * (double(q[4]) - kin64(q)));
      } else {
        pr = P.f.g1 * (q[4] - kin);
      }
      if (P.dualenergy) q[5] = pr * fast::rpow_g1(P, q[0]);
    }
    w[4] = pr;
    return (pr <= 0.f) ? kErrNegPressure : kOk;
  }
};

// Arithmetic of the march.  Phys<false> is the fast form (physics_fast.h:
// refined hardware reciprocals and roots, cube-root powers, fused operations
// in the predictor, the Riemann solvers and the update; in FP64 the primitive
// recovery and the sum of a face state keep the reference's roundings, with
// IEEE quotients from shared reciprocals).
// Phys<true> is the reference's own arithmetic (physics.h: IEEE division
// and square root, the reference's operation order; its translation unit is
// compiled without FMA contraction), so that every face state, flux and
// update is the one the reference forms, bit for bit except where the
// entropy takes a power (device pow against the host libm).
template <bool EXACT>
struct Phys;

template <>
struct Phys<false> {
  template <typename T>
  __device__ static __forceinline__ int q2w(const KParams &P, T q[6], T w[5], T &rinv) {
    return Prim<T>::q2w(P, q, w, rinv);
  }
  template <int LIMITER, typename T>
  __device__ static __forceinline__ T slope3(T wl, T wc, T wr) {
    return fast::slope3<LIMITER>(wl, wc, wr);
  }
  template <typename T>
  __device__ static __forceinline__ T mad(T a, T b, T c) {
    return fm::fma(a, b, c);
  }
  template <int LIMITER, typename T>
  __device__ static __forceinline__ T slope2(T dwl, T dwr) {
    return fast::slope2<LIMITER>(dwl, dwr);
  }
  template <typename T>
  using Evo = fast::EvoFactors<T>;
  template <typename T>
  __device__ static __forceinline__ void evo3d(const fast::EvoFactors<T> &F, const KParams &P, const T w[5], T rinv, const T sx[5],
                                               const T sy[5], const T sz[5], T ev[5]) {
    fast::evo3d(F, P, w, rinv, sx, sy, sz, ev);
  }
  template <typename T>
  __device__ static __forceinline__ void evo2d(const fast::EvoFactors<T> &F, const KParams &P, const T w[5], T rinv, const T sx[5],
                                               const T sy[5], T ev[5]) {
    fast::evo2d(F, P, w, rinv, sx, sy, ev);
  }
  template <int SOLVER, int DIR, typename T>
  __device__ static __forceinline__ int riemann(const KParams &P, const T wl[5], const T wr[5], T f[6]) {
    return fast::riemann<SOLVER, DIR>(P, wl, wr, f);
  }
  template <typename T>
  __device__ static __forceinline__ double cfl_cell(const KParams &P, const T w[5], T rinv) {
    return fast::cfl_cell(P, w, rinv);
  }
  // temperature p / rho * temp0 (for thermal conduction)
  template <typename T>
  __device__ static __forceinline__ T temp(const KParams &P, const T w[5], T rinv) {
    return w[4] * rinv * consts(P, T()).temp0;
  }
};

// The reference's HLL and HLLC (riemann.f90:47-153) with its expressions
// and operation order (physics.h), written branch-free like the fast forms:
// the side is selected first and one flux / state / star state is formed.
// Every quotient is the IEEE one, formed as fm::div_cr from the refined
// reciprocal of its divisor (several quotients by one density share it),
// and every square root as fm::sqrt_pos: the sequences the compiler emits
// for IEEE division and square root, without their range scaling, so the
// results are the IEEE ones for the normal operands of the hydro step.  The
// entropy components take p / rho**g1 from the fast power (fastmath.h); they
// are the only ones a power enters, and the device and host powers differ
// in the last bits in any case.
namespace exact_bf {
template <int DIR>
__device__ __forceinline__ void flux(const KParams &P, const double w[5], double sq, double f[6]) {
  const double u2 = w[1] * w[1] + w[2] * w[2] + w[3] * w[3];
  const double ud = w[DIR];
  f[0] = w[0] * ud;
#pragma unroll
  for (int i = 1; i <= 3; i++) f[i] = (i == DIR) ? (w[0] * (ud * ud) + w[4]) : (w[0] * ud * w[i]);
  f[4] = ud * (0.5 * w[0] * u2 + P.gg1 * w[4]);
  f[5] = ud * sq;
}
// state (riemann.f90:207-239); p/g1 from the correctly rounded 1/g1 (g1inv)
__device__ __forceinline__ void state(const KParams &P, const double w[5], double sq, double q[6]) {
  q[0] = w[0];
  q[1] = w[0] * w[1];
  q[2] = w[0] * w[2];
  q[3] = w[0] * w[3];
  const double u2 = (w[1] * w[1]) + (w[2] * w[2]) + (w[3] * w[3]);
  q[4] = 0.5 * w[0] * u2 + fm::div_cr(w[4], P.g1, P.g1inv);
  q[5] = sq;
}
// sqrt(g p / rho) with y the refined reciprocal of rho
__device__ __forceinline__ double sound(const KParams &P, double rho, double p, double y) {
  return fm::sqrt_pos(fm::div_cr(P.g * p, rho, y));
}
// predictor terms (muscl.f90:100-104) and evo (muscl.f90:68,86,106-107); s(5)/rho
// is the IEEE quotient from the correctly rounded rinv
template <int D>
__device__ __forceinline__ void predictor_dir(const KParams &P, const double w[5], double rinv, const double s[5],
                                              double a[5]) {
#pragma unroll
  for (int i = 0; i < 5; i++) a[i] = w[D + 1] * s[i];
  a[4] = a[4] + P.g * w[4] * s[D + 1];
  a[D + 1] = a[D + 1] + fm::div_cr(s[4], w[0], rinv);
}
struct EvoFactors {
  double dt2;
  __device__ EvoFactors(const KParams &, double dt) : dt2(-0.5 * dt) {}
};
__device__ __forceinline__ void evo3d(const EvoFactors &F, const KParams &P, const double w[5], double rinv,
                                      const double sx[5], const double sy[5], const double sz[5], double ev[5]) {
  double a1[5], a2[5], a3[5];
  predictor_dir<0>(P, w, rinv, sx, a1);
  predictor_dir<1>(P, w, rinv, sy, a2);
  predictor_dir<2>(P, w, rinv, sz, a3);
#pragma unroll
  for (int m = 0; m < 5; m++) ev[m] = F.dt2 * (a1[m] * P.dxinv + a2[m] * P.dyinv + a3[m] * P.dzinv);
}
__device__ __forceinline__ void evo2d(const EvoFactors &F, const KParams &P, const double w[5], double rinv,
                                      const double sx[5], const double sy[5], double ev[5]) {
  double a1[5], a2[5];
  predictor_dir<0>(P, w, rinv, sx, a1);
  predictor_dir<1>(P, w, rinv, sy, a2);
#pragma unroll
  for (int m = 0; m < 5; m++) ev[m] = F.dt2 * (a1[m] * P.dxinv + a2[m] * P.dyinv);
}
template <int DIR>
__device__ __forceinline__ int hll(const KParams &P, const double wl[5], const double wr[5], double f[6]) {
  int code = (wl[4] <= 0.0 || wr[4] <= 0.0) ? kErrRiemannPressure : kOk;
  const double al = sound(P, wl[0], wl[4], fm::rcp(wl[0]));
  const double ar = sound(P, wr[0], wr[4], fm::rcp(wr[0]));
  const double sl = dmin(wl[DIR] - al, wr[DIR] - ar);
  const double sr = dmax(wl[DIR] + al, wr[DIR] + ar);
  const bool left = 0.0 < sl, right = 0.0 > sr, mid = sl <= 0.0 && 0.0 <= sr;
  if (!left && !right && !mid && !code) code = kErrHll;
  const double sql = wl[4] * fast::rpow_g1(P, wl[0]);
  const double sqr = wr[4] * fast::rpow_g1(P, wr[0]);
  double fl[6], fr[6], ql[6], qr[6];
  flux<DIR>(P, wl, sql, fl);
  flux<DIR>(P, wr, sqr, fr);
  state(P, wl, sql, ql);
  state(P, wr, sqr, qr);
  const double den = sr - sl;
  const double yd = fm::rcp(den);
#pragma unroll
  for (int i = 0; i < 6; i++) {
    const double fm_ = fm::div_cr(sr * fl[i] - sl * fr[i] + sl * sr * (qr[i] - ql[i]), den, yd);
    f[i] = left ? fl[i] : (right ? fr[i] : fm_);
  }
  return code;
}
template <int DIR>
__device__ __forceinline__ int hllc(const KParams &P, const double wl[5], const double wr[5], double f[6]) {
  int code = (wl[4] <= 0.0 || wr[4] <= 0.0) ? kErrRiemannPressure : kOk;
  const double yl = fm::rcp(wl[0]), yr = fm::rcp(wr[0]);
  const double al = sound(P, wl[0], wl[4], yl);
  const double ar = sound(P, wr[0], wr[4], yr);
  const double sl = dmin(wl[DIR] - al, wr[DIR] - ar);
  const double sr = dmax(wl[DIR] + al, wr[DIR] + ar);
  const double facl = wl[0] * (sl - wl[DIR]);
  const double facr = wr[0] * (sr - wr[DIR]);
  const double fd = facl - facr;
  const double sm = fm::div_cr(wr[4] - wl[4] + facl * wl[DIR] - facr * wr[DIR], fd, fm::rcp(fd));
  const int br = (0.0 < sl) ? 0
               : (0.0 > sr) ? 1
               : (sl < 0.0 && 0.0 < sm) ? 2
               : (sm <= 0.0 && 0.0 < sr) ? 3 : -1;
  if (br < 0 && !code) code = kErrHllc;
  const bool right = br == 1 || br == 3;
  double w[5];
#pragma unroll
  for (int i = 0; i < 5; i++) w[i] = right ? wr[i] : wl[i];
  const double y = right ? yr : yl;
  const double sq = w[4] * fast::rpow_g1(P, w[0]);
  flux<DIR>(P, w, sq, f);
  // star state (statex, riemann.f90:241-288) and f + s (qx - q)
  const double s = right ? sr : sl;
  const double ud = w[DIR];
  double q[6], qx[6];
  state(P, w, sq, q);
  const double ssm = s - sm;
  qx[0] = fm::div_cr(w[0] * (s - ud), ssm, fm::rcp(ssm));
#pragma unroll
  for (int i = 1; i <= 3; i++) qx[i] = ((i == DIR) ? sm : w[i]) * qx[0];
  const double energy = q[4];  // 0.5 rho u2 + p/g1, formed as in state
  const double rsu = w[0] * (s - ud);
  qx[4] = qx[0] * (fm::div_cr(energy, w[0], y) + (sm - ud) * (sm + fm::div_cr(w[4], rsu, fm::rcp(rsu))));
  qx[5] = qx[0] * fm::div_cr(sq, w[0], y);
  const bool star = br >= 2;
#pragma unroll
  for (int i = 0; i < 6; i++) f[i] = star ? f[i] + s * (qx[i] - q[i]) : f[i];
  return code;
}
}  // namespace exact_bf

template <>
struct Phys<true> {
  // q2w + pressure (comp.f90:26-85): the fast form's FP64 primitive already
  // forms every value as the reference does (IEEE quotients by rho from one
  // reciprocal), and returns the correctly rounded 1/rho; the dual-energy
  // branches take their powers from the fast form
  __device__ static __forceinline__ int q2w(const KParams &P, double q[6], double w[5], double &rinv) {
    return fast::q2w(P, q, w, rinv);
  }
  template <int LIMITER>
  __device__ static __forceinline__ double slope3(double wl, double wc, double wr) {
    return evh::slope3<LIMITER>(wl, wc, wr);
  }
  __device__ static __forceinline__ double mad(double a, double b, double c) { return a * b + c; }
  template <int LIMITER>
  __device__ static __forceinline__ double slope2(double dwl, double dwr) {
    return evh::limited_slope<LIMITER>(dwl, dwr);
  }
  template <typename T>
  using Evo = exact_bf::EvoFactors;
  __device__ static __forceinline__ void evo3d(const exact_bf::EvoFactors &F, const KParams &P, const double w[5],
                                               double rinv, const double sx[5], const double sy[5],
                                               const double sz[5], double ev[5]) {
    exact_bf::evo3d(F, P, w, rinv, sx, sy, sz, ev);
  }
  __device__ static __forceinline__ void evo2d(const exact_bf::EvoFactors &F, const KParams &P, const double w[5],
                                               double rinv, const double sx[5], const double sy[5], double ev[5]) {
    exact_bf::evo2d(F, P, w, rinv, sx, sy, ev);
  }
  template <int SOLVER, int DIR>
  __device__ static __forceinline__ int riemann(const KParams &P, const double wl[5], const double wr[5], double f[6]) {
    if (SOLVER == 1) return exact_bf::hll<DIR>(P, wl, wr, f);
    return exact_bf::hllc<DIR>(P, wl, wr, f);
  }
  // timestep.f90:39-44 for one cell
  __device__ static __forceinline__ double cfl_cell(const KParams &P, const double w[5], double rinv) {
    const double a = exact_bf::sound(P, w[0], w[4], rinv);
    const double sx = fabs(w[1]) + a, sy = fabs(w[2]) + a, sz = fabs(w[3]) + a;
    const double vx = fm::div_cr(P.dx, sx, fm::rcp(sx));
    const double vy = fm::div_cr(P.dy, sy, fm::rcp(sy));
    const double vz = fm::div_cr(P.dz, sz, fm::rcp(sz));
    return dmin(dmin(vx, vy), vz);
  }
  __device__ static __forceinline__ double temp(const KParams &P, const double w[5], double rinv) {
    return fm::div_cr(w[4], w[0], rinv) * P.temp0;
  }
};

// Ghost-mapped offsets (the index rules of `bound`) of column (gx, gy) and
// of plane gz, clamped into the ghost layers: partial tiles in x and y, and
// in z the prefetch of plane nz + 2 after the last plane (never used; it
// would fall outside the grid for nz = 2).  A column's offset is fixed for
// the whole march, so only the plane's is formed per plane.
// A column's offset takes more than 31 bits: a plane of more than 2^31 cells fits
// the 288 GB (FP32-mixed with nz = 2: both buffers take 96 bytes per cell of
// it).  64 bits cost less than an unsigned, which the addresses extend at each
// load: 24 boxes FP32-mixed, 10 steps 9.39 ms against 9.44 (9.34 with an int).
using Col = long long;
__host__ __device__ __forceinline__ Col col_offset(const KParams &P, const Geo &G, int gx, int gy) {
  const bool per = P.boundtype == 2;
  const int cx = gx < -2 ? -2 : (gx > G.nx + 1 ? G.nx + 1 : gx);
  const int cy = gy < -2 ? -2 : (gy > G.ny + 1 ? G.ny + 1 : gy);
  return Col(ghost_src(cx, G.nx, per)) + Col(G.nx) * Col(ghost_src(cy, G.ny, per));
}
__device__ __forceinline__ long long plane_offset(const KParams &P, const Geo &G, int gz) {
  const int cz = gz < -2 ? -2 : (gz > G.nz + 1 ? G.nz + 1 : gz);
  return (long long)G.nx * G.ny * ghost_src(cz, G.nz, P.boundtype == 2);
}

// raw q of the column at offset c of the plane at offset `plane` (the same in
// all lanes)
template <typename S>
__device__ __forceinline__ void fetch_at(const Geo &G, const S *__restrict__ q, long long plane, Col c, S raw[6]) {
#pragma unroll
  for (int m = 0; m < 6; m++) raw[m] = (q + (m * G.n + plane))[c];
}

// raw q of column offset c in plane gz (clamped as plane_offset does).
// Inside the grid, and on a side without a neighbour, that is q with the
// ghost rules of bound; in a z-slab (SLAB) the ghost planes beyond the slab
// are the neighbour's planes in the halo buffer of that side, [6][2][ny][nx]
// (the planes communicate receives, parallel.f90:317-381).  Whole grids take
// the kernels without the test.
template <bool SLAB, typename S>
__device__ __forceinline__ void fetch_plane(const KParams &P, const Geo &G, const S *__restrict__ q, int gz,
                                            Col c, S raw[6]) {
  if constexpr (SLAB) {
    const long long pl = (long long)G.nx * G.ny;
    const S *h = nullptr;
    if (gz < 0 && G.zlo) h = (const S *)G.zlo + pl * (gz < -2 ? 0 : gz + 2);
    else if (gz >= G.nz && G.zhi) h = (const S *)G.zhi + pl * (gz > G.nz ? 1 : 0);
    if (h) {
#pragma unroll
      for (int m = 0; m < 6; m++) raw[m] = (h + m * 2 * pl)[c];
      return;
    }
  }
  fetch_at(G, q, plane_offset(P, G, gz), c, raw);
}

// A copy of v in a register of its own.  Without it the compiler lets the
// prefetched value and its copy share a register, loads the next plane
// elsewhere and moves it back at the end of the iteration, which waits for
// the load (and for the stores before it) there instead of a plane later.
template <typename S>
__device__ __forceinline__ S own_copy(S v) {
  asm("" : "+v"(v));
  return v;
}

// primitive of a fetched cell; wall: a ghost column beyond the reflecting
// upper x (boundary.f90:57-64)
template <bool EXACT, typename S, typename T>
__device__ __forceinline__ void prim_cell(const KParams &P, bool wall, const S raw[6], T qc[6], T wc[5], T &rinv) {
#pragma unroll
  for (int m = 0; m < 6; m++) qc[m] = T(own_copy(raw[m]));
  Phys<EXACT>::q2w(P, qc, wc, rinv);
  if (wall) {
    wc[1] = -wc[1];
    wc[2] = -wc[2];
    wc[3] = -wc[3];
  }
}

template <typename T, int EA>
__device__ __forceinline__ void store_w(T (*W)[EA], int slot, const T w[5]) {
#pragma unroll
  for (int m = 0; m < 5; m++) W[m][slot] = w[m];
}

// ---- the CFL minimum of the new state
// The running minimum of one lane, min_c 1 / max_d (|u_d| + a) / dx_d.  Every
// cell counts: a test of 16 operations that told which cells cannot set the
// minimum spared most of a field that varies from cell to cell, but none of a
// uniform medium, whose cells all have its largest speed, and cost more there:
// 256^3 shock and cloud FP64 0.784 ms with it, 0.741 without; FP32-mixed 0.390,
// 0.371; 512^3 blast in 1% noise 5.43, 5.46; FP32-mixed 2.51, 2.58.
//
// Where p comes from E by a margin above its rounding (and p > 0, so that
// nothing is to be reported) the FP64 fast form takes the limit from q without
// the primitive: rho / max_d (|m_d| + a rho) / dx_d with (a rho)^2 = g g1/2
// (2 rho E - m^2), 28 operations for 47.  Six roundings, those of the square
// halved by its root: against 80 bits, over gas at rest and in motion in 2-D
// and 3-D, rms 0.9e-16 (times E/p, as with p = g1 (E - kin)), where the
// primitive's arithmetic gives 1.0e-16 and the reciprocal of a speed from q,
// without the residuals of root and quotient, 1.2e-16.  A lane without cells
// gives 1e6.
template <typename T, bool EXACT>
struct CflMin {
  double v = 1e6;
  __device__ __forceinline__ void add(const KParams &P, const T w[5], T rinv) {
    v = min_limit(v, Phys<EXACT>::cfl_cell(P, w, rinv));
  }
  // from q; false where it takes the primitive (and for NaN)
  __device__ __forceinline__ bool add(const KParams &P, const T q[6]) {
    if constexpr (!EXACT && sizeof(T) == 8) {
      const double m2 = fm::fma(q[3], q[3], fm::fma(q[2], q[2], q[1] * q[1]));
      const double x = fm::fma(q[4] + q[4], q[0], -m2);
      // x > 0 says rho E > 0; x that has over- or underflown takes the primitive
      if (!(x > fm::fma(P.calm, m2, 1e-290) && x < 1e300 * q[0])) return false;
      const double ar = fm::sqrt_near(P.ggm * x);
      const double sx = (fm::fabs(q[1]) + ar) * P.dxinv;
      const double sy = (fm::fabs(q[2]) + ar) * P.dyinv;
      const double sz = (fm::fabs(q[3]) + ar) * P.dzinv;
      const double s = dmax(dmax(sx, sy), sz);
      v = min_limit(v, fm::div_cr(q[0], s, fm::rcp(s)));
      return true;
    } else {
      return false;
    }
  }
  // the wave's minimum, in every lane
  __device__ __forceinline__ double wave_min() {
    for (int off = 32; off > 0; off >>= 1) v = min_limits(v, __shfl_xor(v, off));
    return v;
  }
};

// LDS of one block
template <typename T, int TX, int TY>
struct Smem {
  using TS = TileShape<TX, TY>;
  T W[5][TS::EA];    // w of plane k, both halo rings
  T XB[10][TS::NFX]; // x face (fi, j), fi = 0..TX: [0,5) left state, [5,10) right state; then flux
  T YB[10][TS::NFY]; // y face (i, fj), fj = 0..TY
  double vmin[TS::NI / 64];  // the interior waves' CFL minima
};

// the first Riemann error (err, in plane err_k) and the first negative
// pressure of the new state (nerr, nerr_k) a lane sees; reported once after
// the march, with the lane's own column (gx, gy)
struct LaneErrors {
  int err = 0, err_k = 0, nerr = 0, nerr_k = 0;
};

// The tile's place: columns from (x0, y0), output planes z0 <= k < z1.
struct Place {
  int x0, y0, z0, z1;
};

// ---- the interior waves of the march: lane tid owns column tid of the tile
template <typename T, typename S, int SOLVER, int LIMITER, int TX, int TY, bool EXACT, bool SLAB>
__device__ __forceinline__ void march_columns(const KParams &P, const Geo &G, const Place &L,
                                              const S *__restrict__ qin, S *__restrict__ qout, double dt,
                                              Smem<T, TX, TY> &sm, S *__restrict__ tout, const Status *lim, CflMin<T, EXACT> &cfl,
                                              LaneErrors &er, int tid) {
  using TS = TileShape<TX, TY>;
  constexpr int EW = TS::EW;
  auto &W = sm.W;
  auto &XB = sm.XB;
  auto &YB = sm.YB;
  const int cx = tid % TX, cy = tid / TX;
  const int gx = L.x0 + cx, gy = L.y0 + cy;
  const bool inside = gx < G.nx && gy < G.ny;
  const bool wall = P.boundtype == 3 && gx >= G.nx;
  const int me = TS::eidx(cx, cy);
  const int fxl = cx + (TX + 1) * cy, fyb = cx + TX * cy;  // the left x face and the bottom y face
  const int z0 = L.z0, z1 = L.z1;

  const typename Phys<EXACT>::template Evo<T> evof(P, dt);
  const T dtx = uniform(T(dt * P.dxinv)), dty = uniform(T(dt * P.dyinv)), dtz = uniform(T(dt * P.dzinv));

  // w of planes k and k+1 and (wm) of plane k-1 or, where the limiter takes
  // one-sided differences only, its difference from plane k; qc, qn: the (dual-energy corrected) q of planes
  // k and k+1, the base of the update, kept in registers so that q is read
  // from HBM once; pre: the raw q of the plane after, loaded one plane ahead,
  // so that no wave stalls on memory right after issuing a load
  T wm[5], wc[5], wp[5], qc[6], qn[6];
  T rc, rp;
  S pre[6];
  const Col own_xy = col_offset(P, G, gx, gy);
  {
    S ra[6], rb[6];  // all three planes in flight together
    fetch_plane<SLAB>(P, G, qin, z0 - 2, own_xy, ra);
    fetch_plane<SLAB>(P, G, qin, z0 - 1, own_xy, rb);
    fetch_plane<SLAB>(P, G, qin, z0, own_xy, pre);
    prim_cell<EXACT>(P, wall, ra, qn, wm, rc);
    prim_cell<EXACT>(P, wall, rb, qn, wc, rc);
  }
  constexpr bool kDiff = LIMITER != 2;
  if constexpr (kDiff) {
#pragma unroll
    for (int m = 0; m < 5; m++) wm[m] = wc[m] - wm[m];
  }
#pragma unroll
  for (int m = 0; m < 6; m++) qc[m] = T(0);
  // carried from plane k-1: its partial update, the flux of its bottom z
  // face and its top z state
  T part[6], fzb[6], zrp[5];
#pragma unroll
  for (int m = 0; m < 6; m++) { part[m] = T(0); fzb[m] = T(0); }
#pragma unroll
  for (int m = 0; m < 5; m++) zrp[m] = T(0);

  for (int k = z0 - 1; k <= z1; k++) {
    const bool out_plane = k >= z0 && k < z1;
    // ---- S1: w of plane k to LDS
    store_w(W, me, wc);
    __syncthreads();

    // ---- S2: primitive of plane k+1; slopes, predictor and face states of
    // plane k
    prim_cell<EXACT>(P, wall, pre, qn, wp, rp);
    fetch_plane<SLAB>(P, G, qin, k + 2, own_xy, pre);
    T sx[5], sy[5], sz[5], ev[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      sx[m] = Phys<EXACT>::template slope3<LIMITER>(W[m][me - 1], wc[m], W[m][me + 1]);
      sy[m] = Phys<EXACT>::template slope3<LIMITER>(W[m][me - EW], wc[m], W[m][me + EW]);
      if constexpr (kDiff) {
        const T dz = wp[m] - wc[m];
        sz[m] = Phys<EXACT>::template slope2<LIMITER>(wm[m], dz);
        wm[m] = dz;
      } else {
        sz[m] = Phys<EXACT>::template slope3<LIMITER>(wm[m], wc[m], wp[m]);
        wm[m] = wc[m];
      }
    }
    if (P.secondorder) {
      Phys<EXACT>::evo3d(evof, P, wc, rc, sx, sy, sz, ev);
    } else {
#pragma unroll
      for (int m = 0; m < 5; m++) { ev[m] = T(0); sx[m] = T(0); sy[m] = T(0); sz[m] = T(0); }
    }
    {
      T zl[5], zr[5];
#pragma unroll
      for (int m = 0; m < 5; m++) {
        XB[5 + m][fxl] = fast::face_state(wc[m], T(-0.5), sx[m], ev[m]);   // right state of the left face
        XB[m][fxl + 1] = fast::face_state(wc[m], T(0.5), sx[m], ev[m]);   // left state of the right face
        YB[5 + m][fyb] = fast::face_state(wc[m], T(-0.5), sy[m], ev[m]);
        YB[m][fyb + TX] = fast::face_state(wc[m], T(0.5), sy[m], ev[m]);
        zl[m] = fast::face_state(wc[m], T(-0.5), sz[m], ev[m]);
        zr[m] = fast::face_state(wc[m], T(0.5), sz[m], ev[m]);
      }
      // z face k-1/2 and the end of plane k-1; the scheduling barrier keeps
      // this solve apart from the x/y solves
      __builtin_amdgcn_sched_barrier(0);
      if (k >= z0) {
        T fz[6];
        const int e = Phys<EXACT>::template riemann<SOLVER, 3>(P, zrp, zl, fz);
        if (e && inside && !er.err) { er.err = e; er.err_k = k; }
        if (k - 1 >= z0) {
          T o[6];
#pragma unroll
          for (int m = 0; m < 6; m++) o[m] = Phys<EXACT>::mad(dtz, fzb[m] - fz[m], part[m]);
          const long long op = (long long)G.nx * G.ny * (k - 1);  // the plane; own_xy is the cell's place in it
          if (inside) {
#pragma unroll
            for (int m = 0; m < 6; m++) (qout + (m * G.n + op))[own_xy] = S(o[m]);
          }
          // the limits (and temperature) of the new state, where they are wanted
          if (inside && (tout || (lim && !cfl.add(P, o)))) {
            T wn[5], rn;
            const int ep = Phys<EXACT>::q2w(P, o, wn, rn);
            if (ep && !er.nerr) { er.nerr = ep; er.nerr_k = k - 1; }
            if (lim) cfl.add(P, wn, rn);
            if (tout) (tout + op)[own_xy] = S(Phys<EXACT>::temp(P, wn, rn));
          }
        }
#pragma unroll
        for (int m = 0; m < 6; m++) fzb[m] = fz[m];
      }
#pragma unroll
      for (int m = 0; m < 5; m++) zrp[m] = zr[m];
    }
    __syncthreads();

    // ---- S3: the left x face and the bottom y face of plane k, as one
    // straight-line block so that the two solves interleave
    if (out_plane) {
      T xl[5], xr[5], fx[6], yl[5], yr[5], fy[6];
#pragma unroll
      for (int m = 0; m < 5; m++) {
        xl[m] = XB[m][fxl];
        xr[m] = XB[5 + m][fxl];
        yl[m] = YB[m][fyb];
        yr[m] = YB[5 + m][fyb];
      }
      const int ex = Phys<EXACT>::template riemann<SOLVER, 1>(P, xl, xr, fx);
      const int ey = Phys<EXACT>::template riemann<SOLVER, 2>(P, yl, yr, fy);
      // faces of cells outside the box (partial tiles) do not count
      const int e = (gy < G.ny && gx <= G.nx && ex) ? ex : ((gx < G.nx && gy <= G.ny) ? ey : 0);
      const bool take = e && !er.err;
      er.err = take ? e : er.err;
      er.err_k = take ? k : er.err_k;
#pragma unroll
      for (int m = 0; m < 6; m++) {
        XB[m][fxl] = fx[m];
        YB[m][fyb] = fy[m];
      }
    }
    __syncthreads();

    // ---- S4: x/y differences of plane k
    if (out_plane) {
#pragma unroll
      for (int m = 0; m < 6; m++) part[m] = Phys<EXACT>::mad(dtx, XB[m][fxl] - XB[m][fxl + 1], qc[m]);
#pragma unroll
      for (int m = 0; m < 6; m++) part[m] = Phys<EXACT>::mad(dty, YB[m][fyb] - YB[m][fyb + TX], part[m]);
    }
    // rotate the column window
#pragma unroll
    for (int m = 0; m < 5; m++) wc[m] = wp[m];
    rc = rp;
#pragma unroll
    for (int m = 0; m < 6; m++) qc[m] = qn[m];
  }
}

// ---- the ring wave of the march: lane `lane` owns first-ring columns (or
// corners) lane, lane + 64, ... and the second-ring cell beyond each.  The
// same barriers as march_columns.
template <typename T, typename S, int SOLVER, int LIMITER, int TX, int TY, bool EXACT, bool SLAB>
__device__ __forceinline__ void march_ring(const KParams &P, const Geo &G, const Place &L, const S *__restrict__ qin,
                                           double dt, Smem<T, TX, TY> &sm, LaneErrors &er, int lane) {
  using TS = TileShape<TX, TY>;
  constexpr int EW = TS::EW, NP = TS::NP;
  auto &W = sm.W;
  const int z0 = L.z0, z1 = L.z1;
  const typename Phys<EXACT>::template Evo<T> evof(P, dt);

  // per column: the state's place (the face it belongs to), the slots of its
  // w and of its second-ring cell, its q offsets
  bool owns[NP], second[NP], wall[NP], wall2[NP], isx[NP];
  T half[NP], *out[NP];
  int ostride[NP], me[NP], slot2[NP];
  Col own_xy[NP], r2_xy[NP];
  T wm[NP][5], wc[NP][5], wp[NP][5], rc[NP], rp[NP], rw2[NP][5], tq[6], tr;
  S pre[NP][6], pre2[NP][6];
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int c = lane + 64 * p;
    int cx, cy, r2x, r2y;
    owns[p] = c < TS::NR1;
    second[p] = c < TS::NR1 + 4;
    isx[p] = c < 2 * TY;
    half[p] = T(0.5);
    if (c < TY) {  // left of the tile: the left state of the left-edge faces
      cx = -1; cy = c; r2x = -2; r2y = c;
      out[p] = &sm.XB[0][(TX + 1) * cy];
    } else if (c < 2 * TY) {  // right: the right state of the right-edge faces
      cx = TX; cy = c - TY; r2x = TX + 1; r2y = cy;
      out[p] = &sm.XB[5][TX + (TX + 1) * cy];
      half[p] = T(-0.5);
    } else if (c < 2 * TY + TX) {  // below
      cx = c - 2 * TY; cy = -1; r2x = cx; r2y = -2;
      out[p] = &sm.YB[0][cx];
    } else if (c < TS::NR1) {  // above
      cx = c - 2 * TY - TX; cy = TY; r2x = cx; r2y = TY + 1;
      out[p] = &sm.YB[5][cx + TX * TY];
      half[p] = T(-0.5);
    } else {  // the four corners of the first ring; lanes without a job load one too
      cx = (c & 1) ? TX : -1;
      cy = (c & 2) ? TY : -1;
      r2x = cx;
      r2y = cy;
      out[p] = &sm.XB[0][0];
    }
    ostride[p] = isx[p] ? TS::NFX : TS::NFY;
    me[p] = TS::eidx(cx, cy);
    slot2[p] = TS::eidx(r2x, r2y);
    own_xy[p] = col_offset(P, G, L.x0 + cx, L.y0 + cy);
    r2_xy[p] = col_offset(P, G, L.x0 + r2x, L.y0 + r2y);
    wall[p] = P.boundtype == 3 && L.x0 + cx >= G.nx;
    wall2[p] = P.boundtype == 3 && L.x0 + r2x >= G.nx;
    S ra[6], rb[6], rd[6], r2[6];
    fetch_plane<SLAB>(P, G, qin, z0 - 2, own_xy[p], ra);
    fetch_plane<SLAB>(P, G, qin, z0 - 1, own_xy[p], rb);
    fetch_plane<SLAB>(P, G, qin, z0 - 1, r2_xy[p], r2);
    fetch_plane<SLAB>(P, G, qin, z0, own_xy[p], rd);
    fetch_plane<SLAB>(P, G, qin, z0, r2_xy[p], pre2[p]);
    fetch_plane<SLAB>(P, G, qin, z0 + 1, own_xy[p], pre[p]);
    prim_cell<EXACT>(P, wall[p], ra, tq, wm[p], tr);
    prim_cell<EXACT>(P, wall[p], rb, tq, wc[p], rc[p]);
    prim_cell<EXACT>(P, wall2[p], r2, tq, rw2[p], tr);
    prim_cell<EXACT>(P, wall[p], rd, tq, wp[p], rp[p]);
  }

  for (int k = z0 - 1; k <= z1; k++) {
    const bool out_plane = k >= z0 && k < z1;
    // ---- S1
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (owns[p]) store_w(W, me[p], wc[p]);
      if (second[p]) store_w(W, slot2[p], rw2[p]);
    }
    __syncthreads();

    // ---- S2: the face state of each column
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (owns[p]) {
        T sx[5], sy[5], sz[5], ev[5];
        const int i = me[p];
#pragma unroll
        for (int m = 0; m < 5; m++) {
          sx[m] = Phys<EXACT>::template slope3<LIMITER>(W[m][i - 1], wc[p][m], W[m][i + 1]);
          sy[m] = Phys<EXACT>::template slope3<LIMITER>(W[m][i - EW], wc[p][m], W[m][i + EW]);
          sz[m] = Phys<EXACT>::template slope3<LIMITER>(wm[p][m], wc[p][m], wp[p][m]);
        }
        if (P.secondorder) {
          Phys<EXACT>::evo3d(evof, P, wc[p], rc[p], sx, sy, sz, ev);
        } else {
#pragma unroll
          for (int m = 0; m < 5; m++) { ev[m] = T(0); sx[m] = T(0); sy[m] = T(0); }
        }
#pragma unroll
        for (int m = 0; m < 5; m++) out[p][m * ostride[p]] = fast::face_state(wc[p][m], half[p], isx[p] ? sx[m] : sy[m], ev[m]);
      }
      // the second ring's w of plane k+1
      prim_cell<EXACT>(P, wall2[p], pre2[p], tq, rw2[p], tr);
      fetch_plane<SLAB>(P, G, qin, k + 2, r2_xy[p], pre2[p]);
    }
    __syncthreads();

    // ---- S3: the TY right-edge x faces (lanes 0..TY-1) and the TX top-edge
    // y faces (lanes TY..TY+TX-1) in one solve, so that the wave does not run
    // two: a y face is the x face of the states with u and v exchanged.  The
    // solvers are bit-symmetric under that exchange: |u|^2 is formed
    // symmetrically and every other term by its role.
    if (out_plane && lane < TY + TX) {
      const bool isy = lane >= TY;
      T *fb = isy ? &sm.YB[0][(lane - TY) + TX * TY] : &sm.XB[0][TX + (TX + 1) * lane];
      const int st_ = isy ? TS::NFY : TS::NFX;
      T wl[5], wr[5], f[6];
#pragma unroll
      for (int m = 0; m < 5; m++) { wl[m] = fb[m * st_]; wr[m] = fb[(5 + m) * st_]; }
      const T l1 = wl[1], r1 = wr[1];
      wl[1] = isy ? wl[2] : wl[1];
      wl[2] = isy ? l1 : wl[2];
      wr[1] = isy ? wr[2] : wr[1];
      wr[2] = isy ? r1 : wr[2];
      const int e = Phys<EXACT>::template riemann<SOLVER, 1>(P, wl, wr, f);
      const T f1 = f[1];
      f[1] = isy ? f[2] : f[1];
      f[2] = isy ? f1 : f[2];
      const bool counts = isy ? (L.x0 + lane - TY < G.nx && L.y0 + TY <= G.ny)
                              : (L.x0 + TX <= G.nx && L.y0 + lane < G.ny);
      if (e && !er.err && counts) { er.err = e; er.err_k = k; }
#pragma unroll
      for (int m = 0; m < 6; m++) fb[m * st_] = f[m];
    }
    // rotate the column windows and form the primitive of plane k+2 here, where
    // the interior waves run two solves: S1 comes between two barriers, and
    // the ring wave's primitives there made every wave wait (512^3 FP64: 6.19
    // against 5.54 ms with the second ring's in S1 too)
#pragma unroll
    for (int p = 0; p < NP; p++) {
#pragma unroll
      for (int m = 0; m < 5; m++) { wm[p][m] = wc[p][m]; wc[p][m] = wp[p][m]; }
      rc[p] = rp[p];
      prim_cell<EXACT>(P, wall[p], pre[p], tq, wp[p], rp[p]);
      fetch_plane<SLAB>(P, G, qin, k + 3, own_xy[p], pre[p]);
    }
    __syncthreads();
  }
}

// One tile `lin` (x fastest, then y, then z chunk) of the box whose q starts
// at element qoff of qin_all/qout_all.  st takes the step's errors, lim (unless
// null) the CFL minimum and the negative pressures of the new state; errors carry the box
// index above bit 40 of the cell.
// With tout (single box only), the temperature of each new cell is stored
// there too, for the conduction pass that follows the sweep.  SLAB: the grid
// is a z-slab whose ghost planes may come from halo buffers (Geo::zlo, zhi).
// The two roles run loops of their own, so that neither holds the other's
// values in registers.
template <typename T, typename S, int SOLVER, int LIMITER, int TX, int TY, bool EXACT, bool SLAB = false>
__device__ __forceinline__ void march(const KParams &P, const Geo &G, const S *__restrict__ qin_all,
                                      S *__restrict__ qout_all, long long qoff, int box, double dt, Status *st,
                                      Status *lim, int lin, Smem<T, TX, TY> &sm,
                                      S *__restrict__ tout = nullptr) {
  using TS = TileShape<TX, TY>;
  constexpr int NI = TS::NI;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tid = (int)(threadIdx.x & 63) + 64 * wave;
  const int tile = lin % (G.tiles_x * G.tiles_y);
  const int chunk = lin / (G.tiles_x * G.tiles_y);
  Place L;
  L.x0 = (tile % G.tiles_x) * TX;
  L.y0 = (tile / G.tiles_x) * TY;
  L.z0 = chunk * G.zchunk;
  L.z1 = min(L.z0 + G.zchunk, G.nz);
  const S *__restrict__ qin = qin_all + qoff;
  S *__restrict__ qout = qout_all + qoff;

  LaneErrors er;
  int gx, gy;  // the lane's own column, which locates its errors
  if (wave < NI / 64) {
    CflMin<T, EXACT> cfl;
    march_columns<T, S, SOLVER, LIMITER, TX, TY, EXACT, SLAB>(P, G, L, qin, qout, dt, sm, tout, lim, cfl, er, tid);
    const double v = cfl.wave_min();
    if ((tid & 63) == 0) sm.vmin[wave] = v;
    gx = L.x0 + tid % TX;
    gy = L.y0 + tid / TX;
  } else {
    const int lane = tid - NI;
    march_ring<T, S, SOLVER, LIMITER, TX, TY, EXACT, SLAB>(P, G, L, qin, dt, sm, er, lane);
    // its last faces are the right-edge x faces, then the top-edge y faces
    gx = L.x0 + (lane < TY ? TX : lane - TY);
    gy = L.y0 + (lane < TY ? lane : TY);
  }
  // one atomic per block: the waves of all blocks meet at one address
  __syncthreads();
  if (lim && threadIdx.x == 0) {
    double v = sm.vmin[0];
#pragma unroll
    for (int i = 1; i < NI / 64; i++) v = min_limits(v, sm.vmin[i]);
    atomic_min_pos(&lim->vmin_bits, v);
  }
  if (er.err || er.nerr) {  // clamped into the box
    const unsigned long long tag = (unsigned long long)box << 40;  // box index above the cell index
    const long long ex = min(max(gx, 0), G.nx - 1), ey = min(max(gy, 0), G.ny - 1);
    if (er.err) report(st, er.err, tag | (unsigned long long)(ex + G.nx * (ey + (long long)G.ny * er.err_k)));
    if (lim && er.nerr) report_next(lim, er.nerr, tag | (unsigned long long)(ex + G.nx * (ey + (long long)G.ny * er.nerr_k)));
  }
}

}  // namespace core
}  // namespace evh
