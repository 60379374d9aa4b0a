// Multilayer shallow-water model: fused RHS + RK-stage kernel, boundary
// conditions and the C ABI entry points (somaxhip_swm_*).
//
// Reference: somax/_src/models/swm/multilayer.py -- vector_field (:150-201),
// apply_boundary_conditions (:203-223) and the wall helpers (:383-410).
// Staggering: arrays of one shape (Ny, Nx); h[j,i] at the cell centre, u[j,i]
// on its east face, v[j,i] on its north face, X point [j,i] at its north-east
// corner.  Intermediate fields are evaluated wherever their stencil lies in
// the array; tendencies are written on the interior and are zero on the ghost
// ring, except wind (top layer) and bottom drag (bottom layer), which act on
// the full arrays.
//
// One kernel evaluates the RHS and the RK stage combination, one workgroup per
// tile and layer: it stages h, u, v of its layer (boundary condition applied on
// load, 1-cell halo) through LDS; each thread forms the cumulative pressure
// gradient sum_{l<=k} g'_l (h_l[e] - h_l[w]) of its points in registers, the
// layers above read from global memory in layer order, so the hydrostatic
// coupling costs no extra pass and the differences of h are exact in FP32 (the
// cumulative pressure itself is ~g*H, four orders of magnitude above its
// cell-to-cell change).

#include <cstring>
#include <new>
#include <string>
#include <utility>
#include <vector>

#include "somaxhip.h"
#include "common.h"
#include "kernels.h"

namespace somax {

constexpr int SWM_MAX_LAYERS = 8;
// A multi-stage call carries the thickness as its deviation from the rest
// thickness; its first and last stage read and write the caller's full thickness.
constexpr int SWM_TOTAL_IN = 1, SWM_TOTAL_START = 2, SWM_TOTAL_OUT = 4;

struct SwmArgs {
  const float* hs;  // stage state (raw; BC applied on load when apply_bc)
  const float* us;
  const float* vs;
  const float* hn;  // step start state (nullable: out = c1*s + c2*rhs)
  const float* un;
  const float* vn;
  float* ho;
  float* uo;
  float* vo;
  int Nx, Ny, nl;
  long plane;
  float gprime[SWM_MAX_LAYERS];
  float hoff[SWM_MAX_LAYERS];  // thickness = stored h + hoff[k] (rest thickness when h holds deviations)
  const float* f_row;     // Ny
  const float* wind_row;  // Ny
  float wind_coef;        // tau0 / H[0]
  float nu, kappa;
  float idx, idy, idx2, idy2;
  float c1, c2;
  int bc;        // SOMAXHIP_BC_*
  int apply_bc;  // 1: RHS of BC(stage state)
  // Tsit5: next stage state of the three fields, n floats apart (ho, uo, vo are
  // then nullable together)
  NextState<float> next;
  long n;
  int tiles;  // tile workgroups of a layer (the rest take the ghost ring)
  int total;  // SWM_TOTAL_*: which thicknesses are stored in full although hoff is set
};

namespace {

constexpr int STX = 64;        // tile width
constexpr int SWV = 4;         // waves per workgroup (rows wv, wv + SWV, .. of the tile each)
constexpr int SRW = 1;         // rows per wave (2: 16.2 us a stage against 14.0 at 512^2 x 2, 7.6 against 5.4 at 64^2 x 3)
constexpr int SNT = 64 * SWV;  // threads per workgroup

enum { F_H = 0, F_U = 1, F_V = 2 };

// Value of field `f` at (gy, gx) after the boundary condition, from the raw
// array `p` (0 outside the array).  Sources are interior points, so the
// mapping reads nothing the condition itself would change.
__device__ inline float bc_value(const float* p, int f, int gy, int gx, int Ny, int Nx, int bc, int apply) {
  if (gy < 0 || gy >= Ny || gx < 0 || gx >= Nx) return 0.0f;
  if (!apply) return p[(long)gy * Nx + gx];
  int sy = gy, sx = gx;
  if (bc == SOMAXHIP_BC_PERIODIC || bc == SOMAXHIP_BC_CHANNEL) {
    sx = gx == 0 ? Nx - 2 : (gx == Nx - 1 ? 1 : gx);
  }
  if (bc == SOMAXHIP_BC_PERIODIC) {
    sy = gy == 0 ? Ny - 2 : (gy == Ny - 1 ? 1 : gy);
  } else {
    // wall rules on the rows (wall and channel)
    if (f == F_V) {
      if (gy == 0 || gy == Ny - 2 || gy == Ny - 1) return 0.0f;
    } else {
      sy = gy == 0 ? 1 : (gy == Ny - 1 ? Ny - 2 : gy);
    }
    if (bc == SOMAXHIP_BC_WALL) {
      if (f == F_U) {
        if (gx == 0 || gx == Nx - 2 || gx == Nx - 1) return 0.0f;
      } else {
        sx = gx == 0 ? 1 : (gx == Nx - 1 ? Nx - 2 : gx);
      }
    }
  }
  return p[(long)sy * Nx + sx];
}


// Source index of row gy (or column gx) for each field after the boundary
// condition; -1 where the condition sets the value to 0 or outside the array.
// The conditions are separable: a row rule and a column rule per field.
struct BcAxis {
  int h, u, v;
};
__device__ inline BcAxis bc_rows(int gy, int Ny, int bc, int apply) {
  if (gy < 0 || gy >= Ny) return {-1, -1, -1};
  if (!apply) return {gy, gy, gy};
  if (bc == SOMAXHIP_BC_PERIODIC) {
    const int s = gy == 0 ? Ny - 2 : (gy == Ny - 1 ? 1 : gy);
    return {s, s, s};
  }
  const int s = gy == 0 ? 1 : (gy == Ny - 1 ? Ny - 2 : gy);  // zero gradient / free slip
  const int sv = (gy == 0 || gy == Ny - 2 || gy == Ny - 1) ? -1 : gy;  // no normal flow
  return {s, s, sv};
}
__device__ inline BcAxis bc_cols(int gx, int Nx, int bc, int apply) {
  if (gx < 0 || gx >= Nx) return {-1, -1, -1};
  if (!apply) return {gx, gx, gx};
  if (bc == SOMAXHIP_BC_PERIODIC || bc == SOMAXHIP_BC_CHANNEL) {
    const int s = gx == 0 ? Nx - 2 : (gx == Nx - 1 ? 1 : gx);
    return {s, s, s};
  }
  const int s = gx == 0 ? 1 : (gx == Nx - 1 ? Nx - 2 : gx);
  const int su = (gx == 0 || gx == Nx - 2 || gx == Nx - 1) ? -1 : gx;
  return {s, su, s};
}

// Linear block -> tile, each XCD taking a contiguous run of the T tiles in
// row-major order (vertically adjacent tiles share their halo rows in L2).
__device__ inline void swm_tile(int b, int T, int tiles_x, int& ty, int& tx) {
  const int xcd = b & 7, slot = b >> 3;
  const int per = T >> 3, extra = T & 7;
  const int t = xcd * per + (xcd < extra ? xcd : extra) + slot;
  ty = t / tiles_x;
  tx = t - ty * tiles_x;
}

// What an output point needs beside its derivative: the step-start values and,
// with NEXT, the terms of the next stage state.
struct SwmPoint {
  float n[3], y[3], k[5][3];
};
template <bool NEXT>
__device__ __forceinline__ void swm_point_fetch(const SwmArgs& a, long idx, float hstart, SwmPoint& f) {
  f.n[0] = a.hn ? a.hn[idx] - hstart : 0.0f;
  f.n[1] = a.hn ? a.un[idx] : 0.0f;
  f.n[2] = a.hn ? a.vn[idx] : 0.0f;
  if constexpr (NEXT) {
#pragma unroll
    for (int c = 0; c < 3; ++c) f.y[c] = a.next.y[c * a.n + idx];
#pragma unroll
    for (int j = 0; j < 5; ++j)
      if (j < a.next.nk) {
#pragma unroll
        for (int c = 0; c < 3; ++c) f.k[j][c] = a.next.k[j][c * a.n + idx];
      }
  }
}
// Stage combination of the raw stage values s and the derivatives d at idx
// (the form of the quasi-geostrophic stage's), with the next stage state (NEXT).
template <bool NEXT>
__device__ __forceinline__ void swm_point_store(const SwmArgs& a, long idx, const float (&s)[3], const float (&d)[3],
                                                float hout, const SwmPoint& f) {
  float o[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    o[c] = a.hn ? f.n[c] + a.c1 * (s[c] - f.n[c]) + a.c2 * d[c] : a.c1 * s[c] + a.c2 * d[c];
  if (!NEXT || a.ho) {
    a.ho[idx] = o[0] + hout;
    a.uo[idx] = o[1];
    a.vo[idx] = o[2];
  }
  if constexpr (NEXT) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double t = (double)f.y[c];
#pragma unroll
      for (int j = 0; j < 5; ++j)
        if (j < a.next.nk) t += a.next.w[j] * (double)f.k[j][c];
      t += a.next.wl * (double)o[c];
      a.next.out[c * a.n + idx] = (float)t;
    }
  }
}

}  // namespace

// PV (zeta + f_X) / h_X at X point (gy, gx) (rows and columns up to N-2) from the
// global arrays of one layer, each value read through the boundary condition when
// `apply` (the same mapping as the tile loads).  Used only for the X points past
// the last row / column that the energy-enstrophy flux needs (their periodic
// images).  No load depends on a test, so they issue together.
__device__ __forceinline__ float pv_global(const SwmArgs& a, const float* h, const float* u, const float* v, float hk,
                                           float hin, int gy, int gx) {
  const BcAxis r0 = bc_rows(gy, a.Ny, a.bc, a.apply_bc), r1 = bc_rows(gy + 1, a.Ny, a.bc, a.apply_bc);
  const BcAxis c0 = bc_cols(gx, a.Nx, a.bc, a.apply_bc), c1 = bc_cols(gx + 1, a.Nx, a.bc, a.apply_bc);
  auto at = [&](const float* p, int r, int c) {
    const float x = p[max(r, 0) * a.Nx + max(c, 0)];
    return r < 0 || c < 0 ? 0.0f : x;
  };
  const float v1 = at(v, r0.v, c1.v), v0 = at(v, r0.v, c0.v), u1 = at(u, r1.u, c0.u), u0 = at(u, r0.u, c0.u);
  const float h00 = at(h, r0.h, c0.h) - hin, h01 = at(h, r0.h, c1.h) - hin;
  const float h10 = at(h, r1.h, c0.h) - hin, h11 = at(h, r1.h, c1.h) - hin;
  const float f0 = a.f_row[gy], f1 = a.f_row[gy + 1];
  const float zeta = (v1 - v0) * a.idx - (u1 - u0) * a.idy;
  const float hx = hk + 0.25f * (h00 + h01 + h10 + h11);
  return (zeta + 0.5f * (f0 + f1)) * __builtin_amdgcn_rcpf(hx);
}

// EEN: the energy-enstrophy-conserving (triad) vorticity flux instead of the
// reference's average form.  Its stencil reaches the X points one row and
// one column further north / east, so the tile carries a 2-cell halo on those
// sides and the tile's PV is formed once into LDS.  X points past the last
// row / column take the value of their periodic image (row / column 1) in a
// periodic direction and 0 beside a wall.
//
// What bounds it: at 512^2 x 2 the traffic of three fields in, three step-start
// fields and three out (19 MB, 3.7 us at the rate of a large copy) and the length of
// a workgroup's chain of loads, LDS and stores.  All loads are issued together, the
// periodic images' with the tile's (they were a chain of dependent loads after the
// barrier in every tile of the last column): 16 -> 10.3 us a stage at 512^2 x 2
// (energy-enstrophy, channel); 64^2 x 3 with Tsit5's combination 8.3 -> 5.3.
// Tiles cover the interior block (rows and columns 1 .. N-2); the workgroups past
// the `tiles` ones take the ghost ring, a point per thread.  A tile none of whose
// loads the boundary condition moves (`edge` false) loads without tests, and its
// raw values are the tile's.
template <bool EEN, bool NEXT>
__global__ __launch_bounds__(SNT, NEXT ? 4 : 8) void swm_stage_kernel(SwmArgs a) {
  constexpr int STY = SWV * SRW;              // tile height
  constexpr int PW = EEN ? STX + 3 : STX + 2;  // LDS pitch
  constexpr int PH = EEN ? STY + 3 : STY + 2;  // LDS rows
  constexpr int QW = STX + 2;                // X points of the tile and its 1-point halo
  constexpr int QH = STY + 2;
  __shared__ float sf[3][PH * PW];  // h, u, v
  __shared__ float sfx[STY + 2];    // Coriolis at the corner rows y0-1 .. y0+STY
  __shared__ float sq[EEN ? QH * QW : 1];
  const float* sh = sf[0];
  const float* su = sf[1];
  const float* sv = sf[2];

  const int tid = threadIdx.x;
  const int tx = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int Nx = a.Nx, Ny = a.Ny;
  const int k = blockIdx.y;  // one workgroup per tile and layer
  const long off = (long)k * a.plane;
  const float* hs = a.hs + off;
  const float* us = a.us + off;
  const float* vs = a.vs + off;
  const bool top = k == 0, bottom = k == a.nl - 1;
  const float hk = a.hoff[k];
  const float hin = a.total & SWM_TOTAL_IN ? hk : 0.0f, hstart = a.total & SWM_TOTAL_START ? hk : 0.0f;
  const float hout = a.total & SWM_TOTAL_OUT ? hk : 0.0f;

  if ((int)blockIdx.x >= a.tiles) {
    // ghost ring: row 0, row Ny-1, then the two columns; no flux, only the wind
    // and the drag on the boundary condition's velocities
    const int i = ((int)blockIdx.x - a.tiles) * SNT + tid;
    if (i >= 2 * Nx + 2 * (Ny - 2)) return;
    const int e = i - 2 * Nx;
    const int gy = i < Nx ? 0 : (i < 2 * Nx ? Ny - 1 : 1 + (e >> 1));
    const int gx = i < Nx ? i : (i < 2 * Nx ? i - Nx : ((e & 1) ? Nx - 1 : 0));
    const long idx = off + (long)gy * Nx + gx;
    const float s[3] = {a.hs[idx] - hin, a.us[idx], a.vs[idx]};
    SwmPoint pt;
    swm_point_fetch<NEXT>(a, idx, hstart, pt);
    float d[3] = {0.0f, 0.0f, 0.0f};
    if (top) d[1] += a.wind_coef * a.wind_row[gy];
    if (bottom) {
      d[1] -= a.kappa * bc_value(us, F_U, gy, gx, Ny, Nx, a.bc, a.apply_bc);
      d[2] -= a.kappa * bc_value(vs, F_V, gy, gx, Ny, Nx, a.bc, a.apply_bc);
    }
    swm_point_store<NEXT>(a, idx, s, d, hout, pt);
    return;
  }

  int tyi, txi;
  swm_tile(blockIdx.x, a.tiles, (Nx - 2 + STX - 1) / STX, tyi, txi);
  const int x0 = 1 + txi * STX;
  const int y0 = 1 + tyi * STY;
  // the tile reads columns x0-1 .. x0-2+PW and rows y0-1 .. y0-2+PH; the
  // conditions change columns 0, N-2 and N-1 (and rows likewise)
  const bool edge = x0 < 2 || y0 < 2 || x0 - 2 + PW > Nx - 3 || y0 - 2 + PH > Ny - 3;

  // Every load of the workgroup is issued before the first LDS store, so that one
  // memory latency covers them: the tile (64 columns by rows wv, wv + SWV, .., then
  // the columns past the 64th, one element a thread; in-plane offsets fit in 32
  // bits: a plane is below 2^31 cells), this thread's own points, and the
  // thickness of the layers above.
  constexpr int NR = (PH + SWV - 1) / SWV;
  constexpr int TAIL = PW - STX;
  static_assert(3 * PH * TAIL <= SNT, "one tail element per thread");
  float t[NR][3], tail = 0.0f;
  const int tf = tid / (PH * TAIL), tr = tid / TAIL - tf * PH, tc = tid % TAIL;  // field, row, column of the tail
  const bool tail_in = tid < 3 * PH * TAIL;
  float raw[SRW][3];
  const int ox = min(x0 + tx, Nx - 2);  // output column (clamped: a point outside stores nothing)
  if (edge) {
    const BcAxis cm = bc_cols(x0 - 1 + tx, Nx, a.bc, a.apply_bc);
    const int ch = max(cm.h, 0), cu = max(cm.u, 0);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int r = wv + SWV * j;
      const BcAxis rm = bc_rows(y0 - 1 + r, Ny, a.bc, a.apply_bc);
      const int rh = max(rm.h, 0) * Nx, rv = max(rm.v, 0) * Nx;
      t[j][0] = hs[rh + ch];
      t[j][1] = us[rh + cu];
      t[j][2] = vs[rv + ch];
      if (rm.h < 0 || cm.h < 0) t[j][0] = 0.0f;
      if (rm.h < 0 || cm.u < 0) t[j][1] = 0.0f;
      if (rm.v < 0 || cm.h < 0) t[j][2] = 0.0f;
    }
    if (tail_in) {
      const BcAxis tm = bc_cols(x0 - 1 + STX + tc, Nx, a.bc, a.apply_bc);
      const BcAxis rm = bc_rows(y0 - 1 + tr, Ny, a.bc, a.apply_bc);
      const int c = tf == 1 ? tm.u : tm.h, r = tf == 2 ? rm.v : rm.h;
      if (c >= 0 && r >= 0) tail = (tf == 0 ? hs : (tf == 1 ? us : vs))[r * Nx + c];
    }
#pragma unroll
    for (int r = 0; r < SRW; ++r) {
      const int o = min(y0 + wv + SWV * r, Ny - 2) * Nx + ox;
      raw[r][0] = hs[o];
      raw[r][1] = us[o];
      raw[r][2] = vs[o];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      // (rows past the tile's: clamped, not stored)
      const int o = min(y0 - 1 + wv + SWV * j, Ny - 1) * Nx + x0 - 1 + tx;
      t[j][0] = hs[o];
      t[j][1] = us[o];
      t[j][2] = vs[o];
    }
    if (tail_in) tail = (tf == 0 ? hs : (tf == 1 ? us : vs))[(y0 - 1 + tr) * Nx + x0 - 1 + STX + tc];
  }
  SwmPoint pt[SRW];
  float wind_r[SRW];
#pragma unroll
  for (int r = 0; r < SRW; ++r) {
    const int gy = min(y0 + wv + SWV * r, Ny - 2);
    swm_point_fetch<NEXT>(a, off + (gy * Nx + ox), hstart, pt[r]);
    wind_r[r] = a.wind_row[gy];
  }
  // Coriolis at the corner rows y0-1 .. y0+STY
  const int fy = y0 - 1 + tid;
  const bool f_in = tid <= STY + 1 && fy + 1 < Ny;
  float f0 = 0.0f, f1 = 0.0f;
  if (f_in) {
    f0 = a.f_row[fy];
    f1 = a.f_row[fy + 1];
  }
  // The pressure gradient of layer k sums g'_j times the thickness differences
  // of the layers j <= k at this thread's points (U and V): those of the layers
  // above come straight from global memory through the boundary condition (the
  // values the tile loads would hold), added in layer order, so the sums equal a
  // layer loop's.  Two layers at a time: their loads are in flight together.
  float dpx[SRW], dpy[SRW];
#pragma unroll
  for (int r = 0; r < SRW; ++r) {
    dpx[r] = dpy[r] = 0.0f;
    const int gy = min(y0 + wv + SWV * r, Ny - 2);
    // (interior points: the map of every neighbour is an element)
    const int r0 = bc_rows(gy, Ny, a.bc, a.apply_bc).h * Nx, r1 = bc_rows(gy + 1, Ny, a.bc, a.apply_bc).h * Nx;
    const int c0 = bc_cols(ox, Nx, a.bc, a.apply_bc).h, c1 = bc_cols(ox + 1, Nx, a.bc, a.apply_bc).h;
    for (int j0 = 0; j0 < k; j0 += 2) {
      float h00[2], h01[2], h10[2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (j0 + b < k) {
          const float* hj = a.hs + (long)(j0 + b) * a.plane;
          h00[b] = hj[r0 + c0];
          h01[b] = hj[r0 + c1];
          h10[b] = hj[r1 + c0];
        }
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (j0 + b < k) {
          const float hj = a.total & SWM_TOTAL_IN ? a.hoff[j0 + b] : 0.0f;
          const float c00 = h00[b] - hj;
          dpx[r] += a.gprime[j0 + b] * ((h01[b] - hj) - c00);
          dpy[r] += a.gprime[j0 + b] * ((h10[b] - hj) - c00);
        }
    }
  }
  if (EEN && edge) {
    // X points past the last row / column: their periodic images, or 0 beside a
    // wall; the column's by threads 0.., the row's by threads 64..
    const bool xper = a.bc != SOMAXHIP_BC_WALL, yper = a.bc == SOMAXHIP_BC_PERIODIC;
    const int cx = Nx - 1 - (x0 - 1), cy = Ny - 1 - (y0 - 1);  // their tile column and row
    int xr = -1, xc = -1;
    if (tid < QH) {
      xr = tid;
      xc = cx;
    } else if (tid >= 64 && tid < 64 + QW) {
      xr = cy;
      xc = tid - 64;
    }
    // (the corner is the column's; nothing past it is read)
    if (xr >= 0 && xr < QH && xr <= cy && xc < QW && xc <= cx && (xc == cx ? tid < QH : xr == cy)) {
      const int gy = y0 - 1 + xr, gx = x0 - 1 + xc;
      const bool zero = (xc == cx && !xper) || (xr == cy && !yper);
      const float qv = pv_global(a, hs, us, vs, hk, hin, xr == cy ? 1 : gy, xc == cx ? 1 : gx);
      sq[xr * QW + xc] = zero ? 0.0f : qv;
    }
  }
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int r = wv + SWV * j;
    if (r < PH) {
#pragma unroll
      for (int c = 0; c < 3; ++c) sf[c][r * PW + tx] = c == 0 ? t[j][c] - hin : t[j][c];
    }
  }
  if (tail_in) sf[tf][tr * PW + STX + tc] = tf == 0 ? tail - hin : tail;
  if (tid <= STY + 1) sfx[tid] = f_in ? 0.5f * (f0 + f1) : 0.0f;
  __syncthreads();
  const float gp = a.gprime[k];
  if (EEN) {
    // PV of the tile's X points (rows y0-1 .. y0+STY, columns x0-1 .. x0+STX);
    // X point (y0-1+xr, x0-1+xc) reads tile rows xr, xr+1 and columns xc, xc+1
    for (int i = tid; i < QH * QW; i += SNT) {
      const int xr = i / QW, xc = i - xr * QW;
      const int gy = y0 - 1 + xr, gx = x0 - 1 + xc;
      if (edge && (gy > Ny - 2 || gx > Nx - 2)) continue;  // an image (above), or never read
      const int c = xr * PW + xc;
      const float zeta = (sv[c + 1] - sv[c]) * a.idx - (su[c + PW] - su[c]) * a.idy;
      const float hx = hk + 0.25f * (sh[c] + sh[c + 1] + sh[c + PW] + sh[c + PW + 1]);
      sq[i] = (zeta + sfx[xr]) * __builtin_amdgcn_rcpf(hx);
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < SRW; ++r) {
    const int ly = wv + SWV * r;
    const int gy = y0 + ly, gx = x0 + tx;
    if (gy > Ny - 2 || gx > Nx - 2) continue;
    const int c = (ly + 1) * PW + tx + 1;  // LDS index of (gy, gx)
#define H(dj, di) sh[c + (dj) * PW + (di)]
#define U(dj, di) su[c + (dj) * PW + (di)]
#define V(dj, di) sv[c + (dj) * PW + (di)]
    float dh = 0.0f, du = 0.0f, dv = 0.0f;
    dpx[r] += gp * (H(0, 1) - H(0, 0));
    dpy[r] += gp * (H(1, 0) - H(0, 0));
    // mass: upwind fluxes on the four faces of the cell
    const float fe = U(0, 0) * (hk + (U(0, 0) > 0.0f ? H(0, 0) : H(0, 1)));
    const float fw = U(0, -1) * (hk + (U(0, -1) > 0.0f ? H(0, -1) : H(0, 0)));
    const float gn = V(0, 0) * (hk + (V(0, 0) > 0.0f ? H(0, 0) : H(1, 0)));
    const float gs = V(-1, 0) * (hk + (V(-1, 0) > 0.0f ? H(-1, 0) : H(0, 0)));
    dh = -((fe - fw) * a.idx + (gn - gs) * a.idy);
    auto vh = [&](int dj, int di) { return (hk + 0.5f * (H(dj, di) + H(dj + 1, di))) * V(dj, di); };
    auto uh = [&](int dj, int di) { return (hk + 0.5f * (H(dj, di) + H(dj, di + 1))) * U(dj, di); };
    auto ke = [&](int dj, int di) {
      return 0.25f * (U(dj, di) * U(dj, di) + U(dj, di - 1) * U(dj, di - 1) + V(dj, di) * V(dj, di) +
                      V(dj - 1, di) * V(dj - 1, di));
    };
    float fu, fv;
    if (EEN) {
      // triads (three corners of a cell, /12) at the corner each U / V pair shares
      auto Q = [&](int dj, int di) { return sq[(ly + 1 + dj) * QW + tx + 1 + di]; };
      const float q00 = Q(0, 0), q0m = Q(0, -1), qm0 = Q(-1, 0), qmm = Q(-1, -1);
      const float q01 = Q(0, 1), qm1 = Q(-1, 1), q10 = Q(1, 0), q1m = Q(1, -1);
      const float t_ne = q0m + q00 + qm0;  // cell (gy, gx): NE triad
      const float t_se = q00 + qm0 + qmm;  //                SE triad
      const float t_nw = qmm + q0m + q00;  //                NW triad
      const float t_nw_e = qm0 + q00 + q01;  // cell (gy, gx+1): NW triad
      const float t_sw_e = qm1 + qm0 + q00;  //                  SW triad
      const float t_sw_n = q00 + q0m + q1m;  // cell (gy+1, gx): SW triad
      const float t_se_n = q10 + q00 + q0m;  //                  SE triad
      constexpr float r12 = 1.0f / 12.0f;
      fu = r12 * (t_ne * vh(0, 0) + t_nw_e * vh(0, 1) + t_se * vh(-1, 0) + t_sw_e * vh(-1, 1));
      fv = -r12 * (t_sw_n * uh(1, -1) + t_se_n * uh(1, 0) + t_nw * uh(0, -1) + t_ne * uh(0, 0));
    } else {
      // PV at X points (dj, di) relative to (gy, gx)
      auto q = [&](int dj, int di) {
        const float zeta = (V(dj, di + 1) - V(dj, di)) * a.idx - (U(dj + 1, di) - U(dj, di)) * a.idy;
        const float hx = hk + 0.25f * (H(dj, di) + H(dj, di + 1) + H(dj + 1, di) + H(dj + 1, di + 1));
        return (zeta + sfx[ly + 1 + dj]) * __builtin_amdgcn_rcpf(hx);
      };
      const float q00 = q(0, 0);
      const float qU = 0.5f * (q00 + q(-1, 0));
      const float vhU = 0.25f * (vh(0, 0) + vh(0, 1) + vh(-1, 0) + vh(-1, 1));
      const float qV = 0.5f * (q00 + q(0, -1));
      const float uhV = 0.25f * (uh(0, 0) + uh(0, -1) + uh(1, 0) + uh(1, -1));
      fu = qU * vhU;
      fv = -qV * uhV;
    }
    const float ke0 = ke(0, 0);
    du = fu - ((ke(0, 1) - ke0) + dpx[r]) * a.idx;
    dv = fv - ((ke(1, 0) - ke0) + dpy[r]) * a.idy;
    if (a.nu != 0.0f) {
      du += a.nu * ((U(0, 1) - 2.0f * U(0, 0) + U(0, -1)) * a.idx2 + (U(1, 0) - 2.0f * U(0, 0) + U(-1, 0)) * a.idy2);
      dv += a.nu * ((V(0, 1) - 2.0f * V(0, 0) + V(0, -1)) * a.idx2 + (V(1, 0) - 2.0f * V(0, 0) + V(-1, 0)) * a.idy2);
    }
    if (top) du += a.wind_coef * wind_r[r];
    if (bottom) {
      du -= a.kappa * U(0, 0);
      dv -= a.kappa * V(0, 0);
    }
#undef H
#undef U
#undef V
    const float d[3] = {dh, du, dv};
    float s[3];
#pragma unroll
    for (int f = 0; f < 3; ++f) s[f] = edge ? raw[r][f] : sf[f][c];
    if (edge) s[0] -= hin;  // (the tile's are shifted)
    swm_point_store<NEXT>(a, off + (long)gy * Nx + gx, s, d, hout, pt[r]);
  }
}

// out = BC(in) for the three fields of every layer (apply_boundary_conditions).
__global__ __launch_bounds__(256) void swm_bc_kernel(const float* h, const float* u, const float* v, float* ho,
                                                     float* uo, float* vo, int Ny, int Nx, long plane, int bc) {
  const int gx = blockIdx.x * 256 + threadIdx.x;
  const int gy = blockIdx.y;
  const long off = (long)blockIdx.z * plane;
  if (gx >= Nx) return;
  const long i = off + (long)gy * Nx + gx;
  ho[i] = bc_value(h + off, F_H, gy, gx, Ny, Nx, bc, 1);
  uo[i] = bc_value(u + off, F_U, gy, gx, Ny, Nx, bc, 1);
  vo[i] = bc_value(v + off, F_V, gy, gx, Ny, Nx, bc, 1);
}

// Diagnostics (multilayer.py:225-255): PV and relative vorticity at X points,
// kinetic energy at T points (each where its stencil lies in the array), and
// per layer the FP64 sums over the interior of KE + 0.5 g' h^2 (energy) and
// 0.5 q^2 h_X (potential enstrophy); partial sums per block, reduced later
// in a fixed order.
__global__ __launch_bounds__(256) void swm_diag_kernel(const float* h, const float* u, const float* v, float* qo,
                                                       float* zo, float* keo, int Nx, int Ny, long plane,
                                                       const float* f_row, SwmArgs g, double* partial) {
  __shared__ double sa[256], sb[256];
  const int x = blockIdx.x * 256 + threadIdx.x;
  const int y = blockIdx.y;
  const int k = blockIdx.z;
  double e = 0.0, en = 0.0;
  if (x < Nx) {
    const long s = k * plane + (long)y * Nx + x;
    const float* H = h + s;
    const float* U = u + s;
    const float* V = v + s;
    float qv = 0.0f, zv = 0.0f, hx = 0.0f;
    if (y <= Ny - 2 && x <= Nx - 2) {
      zv = (V[1] - V[0]) * g.idx - (U[Nx] - U[0]) * g.idy;
      hx = 0.25f * (H[0] + H[1] + H[Nx] + H[Nx + 1]);
      qv = (zv + 0.5f * (f_row[y] + f_row[y + 1])) / hx;
    }
    float kv = 0.0f;
    if (y >= 1 && x >= 1) kv = 0.25f * (U[0] * U[0] + U[-1] * U[-1] + V[0] * V[0] + V[-Nx] * V[-Nx]);
    if (qo) qo[s] = qv;
    if (zo) zo[s] = zv;
    if (keo) keo[s] = kv;
    if (y >= 1 && y <= Ny - 2 && x >= 1 && x <= Nx - 2) {
      const double hv = H[0];
      e = (double)kv + 0.5 * (double)g.gprime[k] * hv * hv;
      en = 0.5 * (double)qv * (double)qv * (double)hx;
    }
  }
  const int t = threadIdx.x;
  sa[t] = e;
  sb[t] = en;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
      sa[t] += sa[t + w];
      sb[t] += sb[t + w];
    }
    __syncthreads();
  }
  if (t == 0) {
    const long blk = (long)k * gridDim.y * gridDim.x + (long)y * gridDim.x + blockIdx.x;
    partial[2 * blk] = sa[0];
    partial[2 * blk + 1] = sb[0];
  }
}

// The state entering (sign -1) or leaving (sign +1) a Tsit5 call: ho[k] = h[k] +
// sign H[k] over every point of nl planes (total thickness <-> deviation from the
// rest thickness; exact in FP32 while |h - H| <= H), uo = u and vo = v.
struct SwmMove {
  const float *h, *u, *v;
  float *ho, *uo, *vo;
  long plane;
  float sign;
  float hoff[SWM_MAX_LAYERS];
};
__global__ __launch_bounds__(256) void swm_move_kernel(SwmMove a) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int k = blockIdx.y;
  if (i >= a.plane) return;
  const long e = k * a.plane + i;
  const float h = a.h[e], u = a.u[e], v = a.v[e];
  a.ho[e] = h + a.sign * a.hoff[k];
  a.uo[e] = u;
  a.vo[e] = v;
}

}  // namespace somax

using namespace somax;

struct somaxhip_swm_plan_s {
  int nx = 0, ny = 0, nl = 0, Nx = 0, Ny = 0, bc = 0;
  int vflux = SOMAXHIP_VFLUX_AVERAGE;
  double dx = 0.0, dy = 0.0;
  std::vector<float> gprime;
  std::vector<float> Hk;
  double H0 = 1.0;
  float* f_row = nullptr;
  float* wind_row = nullptr;
  long plane = 0;
  size_t ws_bytes = 0;
  ~somaxhip_swm_plan_s() {
    if (f_row) (void)hipFree(f_row);
    if (wind_row) (void)hipFree(wind_row);
  }
};

namespace {

// Stage launches bracketed by event pairs; the pairs are read after the
// whole step so that no host synchronisation sits between launches.
struct SwmProf {
  somaxhip_kernel_stat* stats;
  int max_stats;
  int n;
  hipError_t err;
  std::vector<hipEvent_t> ev;  // e0, e1 per launch
  std::vector<double> bytes;   // algorithmic bytes per launch
};
thread_local SwmProf* g_swm_prof = nullptr;

void swm_move(somaxhip_swm_plan p, const float* h, const float* u, const float* v, float* ho, float* uo, float* vo,
              float sign, hipStream_t st) {
  SwmMove m{h, u, v, ho, uo, vo, p->plane, sign, {}};
  for (int k = 0; k < p->nl; ++k) m.hoff[k] = p->Hk[k];
  hipLaunchKernelGGL(swm_move_kernel, dim3((unsigned)((p->plane + 255) / 256), p->nl, 1), dim3(256), 0, st, m);
}

void swm_launch(somaxhip_swm_plan p, SwmArgs& a, hipStream_t st) {
  const int sty = SWV * SRW;
  a.tiles = ((p->Nx - 2 + STX - 1) / STX) * ((p->Ny - 2 + sty - 1) / sty);
  const int ring = 2 * p->Nx + 2 * (p->Ny - 2);
  const dim3 grid((unsigned)(a.tiles + (ring + SNT - 1) / SNT), (unsigned)p->nl, 1);
  const bool een = p->vflux == SOMAXHIP_VFLUX_ENERGY_ENSTROPHY;
  if (a.next.out) {
    if (een) hipLaunchKernelGGL((swm_stage_kernel<true, true>), grid, dim3(SNT), 0, st, a);
    else hipLaunchKernelGGL((swm_stage_kernel<false, true>), grid, dim3(SNT), 0, st, a);
  } else {
    if (een) hipLaunchKernelGGL((swm_stage_kernel<true, false>), grid, dim3(SNT), 0, st, a);
    else hipLaunchKernelGGL((swm_stage_kernel<false, false>), grid, dim3(SNT), 0, st, a);
  }
}

void swm_stage(somaxhip_swm_plan p, const float* hs, const float* us, const float* vs, const float* hn,
               const float* un, const float* vn, float* ho, float* uo, float* vo, const somaxhip_swm_params* prm,
               float c1, float c2, int apply_bc, bool deviation, hipStream_t st,
               const NextState<float>* next = nullptr, int total = 0) {
  SwmArgs a{};
  a.total = total;
  a.hs = hs;
  a.us = us;
  a.vs = vs;
  a.hn = hn;
  a.un = un;
  a.vn = vn;
  a.ho = ho;
  a.uo = uo;
  a.vo = vo;
  a.Nx = p->Nx;
  a.Ny = p->Ny;
  a.nl = p->nl;
  a.plane = p->plane;
  for (int k = 0; k < p->nl; ++k) {
    a.gprime[k] = p->gprime[k];
    a.hoff[k] = deviation ? p->Hk[k] : 0.0f;
  }
  a.f_row = p->f_row;
  a.wind_row = p->wind_row;
  a.wind_coef = (float)(prm->tau0 / p->H0);
  a.nu = (float)prm->nu;
  a.kappa = (float)prm->kappa;
  a.idx = (float)(1.0 / p->dx);
  a.idy = (float)(1.0 / p->dy);
  a.idx2 = (float)(1.0 / (p->dx * p->dx));
  a.idy2 = (float)(1.0 / (p->dy * p->dy));
  a.c1 = c1;
  a.c2 = c2;
  a.bc = p->bc;
  a.apply_bc = apply_bc;
  if (next) {
    a.next = *next;
    a.n = (long)p->nl * p->plane;
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (g_swm_prof) {
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, st);
  }
  swm_launch(p, a, st);
  if (g_swm_prof) {
    (void)hipEventRecord(e1, st);
    SwmProf& pr = *g_swm_prof;
    pr.ev.push_back(e0);
    pr.ev.push_back(e1);
    // algorithmic bytes: read the stage state (3 fields), the step start
    // state when combined, write 3 fields; interior cells
    const double cells = (double)p->nl * p->nx * p->ny;
    pr.bytes.push_back(cells * 4.0 * 3.0 * (hn ? 3.0 : 2.0));
  }
}

int check_plan(somaxhip_swm_plan p, const char* who) {
  if (!p) {
    set_error(std::string(who) + ": null plan");
    return SOMAXHIP_ERR_ARG;
  }
  return SOMAXHIP_OK;
}

}  // namespace

extern "C" {

int somaxhip_swm_plan_create(const somaxhip_swm_desc* d, somaxhip_swm_plan* out) {
  if (!d || !out) {
    set_error("somaxhip_swm_plan_create: null argument");
    return SOMAXHIP_ERR_ARG;
  }
  *out = nullptr;
  if (d->nx < 2 || d->ny < 2 || d->nl < 1 || d->nl > SWM_MAX_LAYERS || !(d->dx > 0) || !(d->dy > 0)) {
    set_error("somaxhip_swm_plan_create: need nx, ny >= 2, 1 <= nl <= 8, dx, dy > 0");
    return SOMAXHIP_ERR_ARG;
  }
  if ((long)(d->nx + 2) * (d->ny + 2) > 0x7fffffffL) {
    set_error("somaxhip_swm_plan_create: a plane of (nx + 2) * (ny + 2) cells must be below 2^31");
    return SOMAXHIP_ERR_ARG;
  }
  if (!d->g_prime || !d->H || !d->f_row || !d->wind_row) {
    set_error("somaxhip_swm_plan_create: a required table pointer is null");
    return SOMAXHIP_ERR_ARG;
  }
  if (d->bc != SOMAXHIP_BC_PERIODIC && d->bc != SOMAXHIP_BC_WALL && d->bc != SOMAXHIP_BC_CHANNEL) {
    set_error("somaxhip_swm_plan_create: unknown boundary condition");
    return SOMAXHIP_ERR_ARG;
  }
  if (!(d->H[0] > 0)) {
    set_error("somaxhip_swm_plan_create: H[0] must be positive");
    return SOMAXHIP_ERR_ARG;
  }
  if (d->vorticity_flux != SOMAXHIP_VFLUX_AVERAGE && d->vorticity_flux != SOMAXHIP_VFLUX_ENERGY_ENSTROPHY) {
    set_error("somaxhip_swm_plan_create: unknown vorticity flux");
    return SOMAXHIP_ERR_ARG;
  }
  somaxhip_swm_plan p = new (std::nothrow) somaxhip_swm_plan_s();
  if (!p) {
    set_error("somaxhip_swm_plan_create: out of host memory");
    return SOMAXHIP_ERR_ALLOC;
  }
  p->nx = d->nx;
  p->ny = d->ny;
  p->nl = d->nl;
  p->Nx = d->nx + 2;
  p->Ny = d->ny + 2;
  p->dx = d->dx;
  p->dy = d->dy;
  p->bc = d->bc;
  p->vflux = d->vorticity_flux;
  p->H0 = d->H[0];
  for (int k = 0; k < d->nl; ++k) {
    p->gprime.push_back((float)d->g_prime[k]);
    p->Hk.push_back((float)d->H[k]);
  }
  p->plane = (long)p->Ny * p->Nx;
  std::vector<float> f(p->Ny), w(p->Ny);
  for (int j = 0; j < p->Ny; ++j) {
    f[j] = (float)d->f_row[j];
    w[j] = (float)d->wind_row[j];
  }
  hipError_t e = hipMalloc(&p->f_row, p->Ny * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&p->wind_row, p->Ny * sizeof(float));
  if (e == hipSuccess) e = hipMemcpy(p->f_row, f.data(), p->Ny * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(p->wind_row, w.data(), p->Ny * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    set_error(std::string("somaxhip_swm_plan_create: ") + hipGetErrorString(e));
    delete p;
    return SOMAXHIP_ERR_ALLOC;
  }
  // workspace: thickness deviation of the step start and two stage states
  p->ws_bytes = (size_t)7 * p->nl * p->plane * sizeof(float);
  *out = p;
  return SOMAXHIP_OK;
}

int somaxhip_swm_plan_destroy(somaxhip_swm_plan p) {
  delete p;
  return SOMAXHIP_OK;
}

size_t somaxhip_swm_workspace_bytes(somaxhip_swm_plan p) { return p ? p->ws_bytes : 0; }

int somaxhip_swm_rhs(somaxhip_swm_plan p, const float* h, const float* u, const float* v, float* dh, float* du,
                     float* dv, const somaxhip_swm_params* prm, int apply_bc, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_swm_rhs");
  if (rc) return rc;
  if (!h || !u || !v || !dh || !du || !dv || !prm) {
    set_error("somaxhip_swm_rhs: null field or params");
    return SOMAXHIP_ERR_ARG;
  }
  swm_stage(p, h, u, v, nullptr, nullptr, nullptr, dh, du, dv, prm, 0.0f, 1.0f, apply_bc ? 1 : 0, false,
            reinterpret_cast<hipStream_t>(stream));
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

int somaxhip_swm_apply_bc(somaxhip_swm_plan p, const float* h, const float* u, const float* v, float* ho, float* uo,
                          float* vo, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_swm_apply_bc");
  if (rc) return rc;
  if (!h || !u || !v || !ho || !uo || !vo) {
    set_error("somaxhip_swm_apply_bc: null field");
    return SOMAXHIP_ERR_ARG;
  }
  if (ho == h || uo == u || vo == v) {
    set_error("somaxhip_swm_apply_bc: output must not alias the input");
    return SOMAXHIP_ERR_ARG;
  }
  dim3 grid((p->Nx + 255) / 256, p->Ny, p->nl);
  hipLaunchKernelGGL(swm_bc_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), h, u, v, ho, uo, vo,
                     p->Ny, p->Nx, p->plane, p->bc);
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

int somaxhip_swm_diagnose(somaxhip_swm_plan p, const float* h, const float* u, const float* v, float* q, float* zeta,
                          float* ke, double* energy_enstrophy, void* ws, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_swm_diagnose");
  if (rc) return rc;
  if (!h || !u || !v || !energy_enstrophy || !ws) {
    set_error("somaxhip_swm_diagnose: null field, output or workspace");
    return SOMAXHIP_ERR_ARG;
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  SwmArgs g{};
  for (int k = 0; k < p->nl; ++k) g.gprime[k] = p->gprime[k];
  g.idx = (float)(1.0 / p->dx);
  g.idy = (float)(1.0 / p->dy);
  const int bx = (p->Nx + 255) / 256;
  double* partial = static_cast<double*>(ws);  // 2 * nl * Ny * bx doubles, well inside the workspace
  hipLaunchKernelGGL(swm_diag_kernel, dim3(bx, p->Ny, p->nl), dim3(256), 0, st, h, u, v, q, zeta, ke, p->Nx, p->Ny,
                     p->plane, p->f_row, g, partial);
  launch_pair_reduce(partial, bx * p->Ny, p->nl, p->dx * p->dy, energy_enstrophy, st);
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

int somaxhip_swm_step(somaxhip_swm_plan p, float* h, float* u, float* v, int nsteps, double dt,
                      const somaxhip_swm_params* prm, void* ws, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_swm_step");
  if (rc) return rc;
  if (!h || !u || !v || !prm || !ws || nsteps < 0) {
    set_error("somaxhip_swm_step: null field, params or workspace, or negative nsteps");
    return SOMAXHIP_ERR_ARG;
  }
  if (nsteps == 0) return SOMAXHIP_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const long n = (long)p->nl * p->plane;
  float* w = static_cast<float*>(ws);
  float *e0 = w, *e1 = w + n, *u1 = w + 2 * n, *v1 = w + 3 * n, *e2 = w + 4 * n, *u2 = w + 5 * n, *v2 = w + 6 * n;
  // The thickness is carried as its deviation from the rest thickness during
  // the call (e0 between steps): FP32 total thickness (~500 m) keeps only ~3e-5 m
  // of the interface signal (~1 m) whose differences drive the pressure gradient.
  // The stages that read or write the caller's h convert it as they go (as launches
  // of their own the two conversions took 7.5 of 40 us at 512^2 x 2).
  const float s = (float)dt;
  for (int k = 0; k < nsteps; ++k) {
    const bool first = k == 0, last = k == nsteps - 1;
    const float* hn = first ? h : e0;
    const int start = first ? SWM_TOTAL_START : 0;
    swm_stage(p, hn, u, v, nullptr, nullptr, nullptr, e1, u1, v1, prm, 1.0f, s, 1, true, st, nullptr,
              first ? SWM_TOTAL_IN : 0);
    swm_stage(p, e1, u1, v1, hn, u, v, e2, u2, v2, prm, 0.25f, 0.25f * s, 1, true, st, nullptr, start);
    swm_stage(p, e2, u2, v2, hn, u, v, last ? h : e0, u, v, prm, 2.0f / 3.0f, 2.0f / 3.0f * s, 1, true, st, nullptr,
              start | (last ? SWM_TOTAL_OUT : 0));
  }
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

size_t somaxhip_swm_tsit5_workspace_bytes(somaxhip_swm_plan p) {
  return p ? (size_t)9 * 3 * p->nl * p->plane * sizeof(float) : 0;
}

// Tsit5 on (h, u, v), as somaxhip_qg_step_tsit5: six evaluations per step, each
// stage kernel forming the next stage state; thickness carried as its deviation
// from the rest thickness.  tws: Y0 (step start), K0..K4 and two stage states,
// each the three fields back to back.
int somaxhip_swm_step_tsit5(somaxhip_swm_plan p, float* h, float* u, float* v, int nsteps, double dt,
                            const somaxhip_swm_params* prm, void* tws, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_swm_step_tsit5");
  if (rc) return rc;
  if (!h || !u || !v || !prm || !tws || nsteps < 0) {
    set_error("somaxhip_swm_step_tsit5: null field, params or Tsit5 workspace, or negative nsteps");
    return SOMAXHIP_ERR_ARG;
  }
  if (nsteps == 0) return SOMAXHIP_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const long n = (long)p->nl * p->plane;
  float* Y0 = static_cast<float*>(tws);
  float* K = Y0 + 3 * n;
  float* Y[2] = {K + 15 * n, K + 18 * n};
  swm_move(p, h, u, v, Y0, Y0 + n, Y0 + 2 * n, -1.0f, st);
  for (int s = 0; s < nsteps; ++s) {
    for (int i = 0; i < 6; ++i) {
      const float* in = i ? Y[(i - 1) & 1] : Y0;
      float* k = i < 5 ? K + 3 * i * n : nullptr;
      NextState<float> next{};
      next.y = Y0;
      next.nk = i;
      for (int j = 0; j < i; ++j) {
        next.k[j] = K + 3 * j * n;
        next.w[j] = dt * TSIT5_A[i + 1][j];
      }
      next.wl = dt * TSIT5_A[i + 1][i];
      next.out = i < 5 ? Y[i & 1] : Y0;
      swm_stage(p, in, in + n, in + 2 * n, nullptr, nullptr, nullptr, k, k ? k + n : nullptr, k ? k + 2 * n : nullptr,
                prm, 0.0f, 1.0f, 1, true, st, &next);
    }
  }
  swm_move(p, Y0, Y0 + n, Y0 + 2 * n, h, u, v, 1.0f, st);
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

size_t somaxhip_rqg_workspace_bytes(somaxhip_swm_plan p) {
  return p ? (size_t)11 * 3 * p->nl * p->plane * sizeof(float) : 0;
}

// ReparameterizedQG time stepping: y' = f(y) with f = RHS(P(BC(y))) (the
// projection inside apply_boundary_conditions, reparameterized.py:186-189),
// Tsit5 or SSP-RK3 in Butcher form, thickness carried as the
// deviation eta.  tws: Y0, Y, K0..K5, one spare, B (after the BC), Pj (projected).
int somaxhip_rqg_step(somaxhip_swm_plan p, somaxhip_qg_plan qp, int solver, double f0, const double* H,
                      const double* M, float* h, float* u, float* v, int nsteps, double dt,
                      const somaxhip_swm_params* prm, void* qg_ws, void* tws, somaxhip_stream_t stream) {
  int rc = check_plan(p, "somaxhip_rqg_step");
  if (rc) return rc;
  if (!qp || !H || !M || !h || !u || !v || !prm || !qg_ws || !tws || nsteps < 0 ||
      (solver != SOMAXHIP_SOLVER_SSPRK3 && solver != SOMAXHIP_SOLVER_TSIT5)) {
    set_error("somaxhip_rqg_step: null argument, negative nsteps or unknown solver");
    return SOMAXHIP_ERR_ARG;
  }
  if (qg_plan_f64(qp)) {
    set_error("somaxhip_rqg_step: the QG plan computes in FP64; the projection takes an FP32 / BF16 plan");
    return SOMAXHIP_ERR_ARG;
  }
  if (nsteps == 0) return SOMAXHIP_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const long n = (long)p->nl * p->plane;
  float* Y0 = static_cast<float*>(tws);
  float* Y = Y0 + 3 * n;
  float* K[6];
  for (int i = 0; i < 6; ++i) K[i] = Y + (i + 1) * 3 * n;
  float* B = Y + 8 * 3 * n;
  float* Pj = B + 3 * n;
  swm_move(p, h, u, v, Y0, Y0 + n, Y0 + 2 * n, -1.0f, st);
  int err = SOMAXHIP_OK;
  auto f = [&](const float* y, float* k) {
    hipLaunchKernelGGL(swm_bc_kernel, dim3((p->Nx + 255) / 256, p->Ny, p->nl), dim3(256), 0, st, y, y + n,
                       y + 2 * n, B, B + n, B + 2 * n, p->Ny, p->Nx, p->plane, p->bc);
    const int r = somaxhip_qg_project(qp, f0, H, M, B, B + n, B + 2 * n, 1, Pj, Pj + n, Pj + 2 * n, nullptr, qg_ws,
                                      stream);
    if (r && !err) err = r;
    swm_stage(p, Pj, Pj + n, Pj + 2 * n, nullptr, nullptr, nullptr, k, k + n, k + 2 * n, prm, 0.0f, 1.0f, 0, true,
              st);
  };
  auto comb = [&](const double* w, int nk, float* out) {
    LinComb c{};
    c.y = Y0;
    c.nk = nk;
    for (int j = 0; j < nk; ++j) {
      c.k[j] = K[j];
      c.w[j] = dt * w[j];
    }
    c.n = 3 * n;
    c.out = out;
    launch_lincomb(c, st);
  };
  if (solver == SOMAXHIP_SOLVER_TSIT5) {
    for (int s = 0; s < nsteps && !err; ++s)
      for (int i = 0; i < 6; ++i) {
        f(i ? Y : Y0, K[i]);
        comb(TSIT5_A[i + 1], i + 1, i < 5 ? Y : Y0);  // row 6: the new state, in place
      }
  } else {
    // SSP-RK3 in Butcher form: c = (0, 1, 1/2), b = (1/6, 1/6, 2/3)
    static const double a1[1] = {1.0}, a2[2] = {0.25, 0.25}, b3[3] = {1.0 / 6.0, 1.0 / 6.0, 2.0 / 3.0};
    for (int s = 0; s < nsteps && !err; ++s) {
      f(Y0, K[0]);
      comb(a1, 1, Y);
      f(Y, K[1]);
      comb(a2, 2, Y);
      f(Y, K[2]);
      comb(b3, 3, Y0);
    }
  }
  if (err) return err;
  swm_move(p, Y0, Y0 + n, Y0 + 2 * n, h, u, v, 1.0f, st);
  SOMAX_HIP_CHECK(hipGetLastError());
  return SOMAXHIP_OK;
}

int somaxhip_swm_step_profile(somaxhip_swm_plan p, float* h, float* u, float* v, int nsteps, double dt,
                              const somaxhip_swm_params* prm, void* ws, somaxhip_stream_t stream,
                              somaxhip_kernel_stat* stats, int max_stats, int* nstats) {
  if (!stats || !nstats || max_stats < 1) {
    set_error("somaxhip_swm_step_profile: null stats");
    return SOMAXHIP_ERR_ARG;
  }
  SwmProf prof{stats, max_stats, 0, hipSuccess, {}, {}};
  g_swm_prof = &prof;
  const int rc = somaxhip_swm_step(p, h, u, v, nsteps, dt, prm, ws, stream);
  g_swm_prof = nullptr;
  hipError_t e = hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream));
  std::memset(&stats[0], 0, sizeof(stats[0]));
  std::strncpy(stats[0].name, "swm_stage", sizeof(stats[0].name) - 1);
  for (size_t i = 0; i < prof.bytes.size(); ++i) {
    float ms = 0.0f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, prof.ev[2 * i], prof.ev[2 * i + 1]);
    stats[0].launches += 1;
    stats[0].total_ms += ms;
    stats[0].bytes += prof.bytes[i];
  }
  for (hipEvent_t ev : prof.ev) (void)hipEventDestroy(ev);
  *nstats = 1;
  if (rc) return rc;
  SOMAX_HIP_CHECK(e);
  return SOMAXHIP_OK;
}

}  // extern "C"
