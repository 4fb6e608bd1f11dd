// advdiff.hpp -- the advection-diffusion strip of the full-grid stencil kernels.
#pragma once

#include <type_traits>

#include "device_util.hpp"

namespace cup2d {

constexpr int BC_KILL_FAC = 100;  // Definitions.h:38

// Launch shape of the full-grid stencil kernels (chosen by a sweep over
// RY in {8,16,32}, TX in {128,256}, unroll in {2,4,8}): rows per workgroup,
// widest column strip, unroll depth of the row march.
constexpr int STENCIL_RY = 8, STENCIL_TX = 256;
// Columns per strip, a power of two; the last strip of a row may be ragged
// (its lanes past NX clamp their loads and store nothing).  Taking only
// widths that divide NX left grids such as 2016 x 992 with strips of 32: half
// a wave, and an eighth of the loads in flight per workgroup (advDiff 19.7 ->
// 15.1 us, projection 18.1 -> 15.4 us there).
static inline int strip_width(int NX) {
  int t = 32;
  while (t < STENCIL_TX && t < NX) t <<= 1;
  return t;
}
static inline int strips_x(int NX) { return (NX + strip_width(NX) - 1) / strip_width(NX); }
static inline bool ragged(int NX) { return NX % strip_width(NX) != 0; }
// fn(RAGGED, STREAM, T{}) as compile-time values: whether the grid's last
// strips (of the given width) are ragged, whether its stores are streamed, and
// the planes' type
template <typename F>
inline void strip_dispatch(const cup2d_ctx* c, int width, F&& fn) {
  const bool rg = c->g.NX % width != 0;
  if (c->f32) {
    if (rg) fn(std::true_type{}, std::false_type{}, float{});
    else fn(std::false_type{}, std::false_type{}, float{});
  } else if (c->stream_stores) {
    if (rg) fn(std::true_type{}, std::true_type{}, double{});
    else fn(std::false_type{}, std::true_type{}, double{});
  } else {
    if (rg) fn(std::true_type{}, std::false_type{}, double{});
    else fn(std::false_type{}, std::false_type{}, double{});
  }
}

// the statement with RAGGED = whether the grid's last strips are ragged
#define CUP2D_RAGGED_DISPATCH(NX, ...)  \
  do {                                  \
    if (ragged(NX)) {                   \
      constexpr bool RAGGED = true;     \
      __VA_ARGS__;                      \
    } else {                            \
      constexpr bool RAGGED = false;    \
      __VA_ARGS__;                      \
    }                                   \
  } while (0)

// The lanes of a strip workgroup's wave whose left / right neighbour column
// lies outside the wave (the other wave, or the next strip).
struct WaveEdges {
  bool w, e;
  __device__ WaveEdges() {
    const int lane = threadIdx.x & 63;
    const int last = (blockDim.x < 64 ? (int)blockDim.x : 64) - 1;
    w = lane == 0;
    e = lane == last;
  }
};

// ------------------------------------------------------------- advDiff
// advDiff.cpp:14-34 (stencil), :47-55 (factors), :68-79 (faded lab).  Each
// workgroup also writes its share of the boundary flux
// IF = sum_E u - sum_W u + sum_N v - sum_S v (advDiff.cpp:93-102).
// T: the velocity planes' type; the stencil is evaluated in T (FP32 at
// FP32 precision), the factors are formed in double and rounded once.
// STREAM: the stores are non-temporal (cup2d_ctx::stream_stores).
template <int RY, bool RAGGED, bool STREAM, typename T>
__device__ inline void advdiff_strip(const T* __restrict__ u, const T* __restrict__ v,
                                     T* __restrict__ uo, T* __restrict__ vo,
                                     const Grid& g, const StepState* __restrict__ st,
                                     double* __restrict__ fluxpart, int bx, int by, int gx, int gy,
                                     double* lds) {
  const int NX = g.NX, NY = g.NY;
  const int xr = bx * blockDim.x + threadIdx.x;
  const bool in = !RAGGED || xr < NX;
  const int x = in ? xr : NX - 1;
  const int y0 = by * RY;
  const double dt = st->dt, h = g.h;
  const double dUINF0 = st->uinf[0], dUINF1 = st->uinf[1];
  const T UINF0 = (T)dUINF0, UINF1 = (T)dUINF1;
  const T dfac = (T)((g.nu / h) * (dt / h)), afac = (T)(-0.5 * dt / h);
  const double norUinf = dmax(dmax(fabs(dUINF0), fabs(dUINF1)), 2.220446049250313e-16);
  const double tW = dmax(dUINF0, 0.0) / norUinf, tS = dmax(dUINF1, 0.0) / norUinf;
  const double tE = dmin(dUINF0, 0.0) / norUinf, tN = dmin(dUINF1, 0.0) / norUinf;
  const T fadeW = (T)(1 - tW * tW / BC_KILL_FAC), fadeS = (T)(1 - tS * tS / BC_KILL_FAC);
  const T fadeE = (T)(1 - tE * tE / BC_KILL_FAC), fadeN = (T)(1 - tN * tN / BC_KILL_FAC);

  // All loads of the strip are issued first (clamped indices, so every load
  // is unconditional), then the rows are computed with selects of the
  // boundary values: the wave keeps the whole strip's loads in flight.
  // The x neighbours come from the adjacent lanes (lane_from_left/right);
  // only the wave's edge lanes load theirs (uH, vH: the west column for
  // lane 0, the east one for the last lane).
  const size_t i0 = (size_t)y0 * NX + x;
  const bool hasW = x > 0, hasE = x + 1 < NX;
  const size_t dW = hasW ? 1 : 0, dE = hasE ? 1 : 0;
  const WaveEdges we;
  T uC[RY + 2], vC[RY + 2], uH[RY], vH[RY];
  {
    const size_t is = y0 > 0 ? i0 - NX : i0;
    uC[0] = u[is];
    vC[0] = v[is];
#pragma unroll
    for (int iy = 0; iy <= RY; ++iy) {
      const size_t i = y0 + iy < NY ? i0 + (size_t)iy * NX : i0 + (size_t)(iy - 1) * NX;
      uC[iy + 1] = u[i];
      vC[iy + 1] = v[i];
    }
    if (we.w || we.e) {
      const size_t dh = we.w ? (size_t)0 - dW : dE;
#pragma unroll
      for (int iy = 0; iy < RY; ++iy) {
        const size_t i = i0 + (size_t)iy * NX + dh;
        uH[iy] = u[i];
        vH[iy] = v[i];
      }
    }
  }
  T uc = uC[1], vc = vC[1];
  T us = y0 == 0 ? uc * fadeS : uC[0];
  T vs = y0 == 0 ? vc * fadeS : vC[0];
  double flux = 0;
#pragma unroll
  for (int iy = 0; iy < RY; ++iy) {
    const int y = y0 + iy;
    const bool hasN = y + 1 < NY;
    const T un = hasN ? uC[iy + 2] : uc * fadeN, vn = hasN ? vC[iy + 2] : vc * fadeN;
    // (the shifts run before the selects: every lane takes part in them)
    const T sul = lane_from_left(uc), svl = lane_from_left(vc);
    const T sur = lane_from_right(uc), svr = lane_from_right(vc);
    const T ul = we.w ? uH[iy] : sul, vl = we.w ? vH[iy] : svl;
    const T ur = we.e ? uH[iy] : sur, vr = we.e ? vH[iy] : svr;
    const T uw = hasW ? ul : uc * fadeW, vw = hasW ? vl : vc * fadeW;
    const T ue = hasE ? ur : uc * fadeE, ve = hasE ? vr : vc * fadeE;
    const T dUadv = (uc + UINF0) * (ue - uw) + (vc + UINF1) * (un - us);
    const T dUdif = ue + un + uw + us - 4 * uc;
    const T dVadv = (uc + UINF0) * (ve - vw) + (vc + UINF1) * (vn - vs);
    const T dVdif = ve + vn + vw + vs - 4 * vc;
    const T u1 = uc + (afac * dUadv + dfac * dUdif);
    const T v1 = vc + (afac * dVadv + dfac * dVdif);
    const size_t idx = i0 + (size_t)iy * NX;
    if (in) {
      if constexpr (STREAM) {
        __builtin_nontemporal_store(u1, uo + idx);
        __builtin_nontemporal_store(v1, vo + idx);
      } else {
        uo[idx] = u1;
        vo[idx] = v1;
      }
    }
    // selects, not branches, so the row loop stays one basic block
    flux = x == 0 ? flux - u1 : flux;
    flux = x == NX - 1 ? flux + u1 : flux;
    flux = y == 0 ? flux - v1 : flux;
    flux = y == NY - 1 ? flux + v1 : flux;
    us = uc; vs = vc;
    uc = un; vc = vn;
  }
  const int e = edge_index(bx, by, gx, gy);
  if (e < 0) return;
  if (!in) flux = 0;
  flux = block_sum_dyn(flux, lds);
  if (threadIdx.x == 0) fluxpart[e] = flux;
}

}  // namespace cup2d
