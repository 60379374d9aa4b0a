// Direct Helmholtz inversion in FP64 for small and middle-sized grids (gfx950).
//
// psi = Cm2l (lap_h - lambda)^-1 Cl2m q of one batch in three launches, every
// sum and every intermediate in FP64 (v_mfma_f64_16x16x4), q and psi in the
// state's own type:
//   forward   layer -> mode projection, both mirror folds and the x transform
//   spectral  y transform, division by the Helmholtz symbol, y transform back
//   inverse   x transform back, unfolding, mass correction, mode -> layer mix
// (the first two in one launch on the smallest planes, direct_front)
//
// Why: below about 600 points a side the transforms are a few MFLOP to a
// GFLOP, and what costs time is the number of launches and the chain inside
// each, not the matrix rate.  FP64 needs no split operands, no refinement
// solve and no flushes, and three launches replace 6 (FP32, six-product) or
// 12 (mixed).  Measured (us, one inversion in a replayed graph; FP32 transforms of
// 128 x 128 tiles -> direct): 64^2 x 1 62 -> 10.7, 128^2 x 3 93 -> 18.2, 256^2 x 3
// 98 -> 33.5, 512^2 x 3 143 -> 72 (64 x 64 tiles: about as fast).  Per
// launch at 64^2: 5 to 7 us, of which 1.5 are a launch's own and each dependent trip
// to the Infinity Cache is 1 (the L2s start a kernel empty); at 512^2 x 3:
// forward 21, spectral 30, inverse 24, against 5.6, 11.2 and 5.6 at the FP64
// matrix rate (the 257th row of every folded extent costs a tile of 16, and 204
// spectral workgroups leave a fifth of the chip idle).
//
// Mirror folds: S[N-1-n][a] = (-1)^a S[n][a] for any N, so a DST-I splits by
// output parity into two products of half the length, and a plane into four
// independent blocks (px, py).  Folded position j < h = ceil(N/2) stands for
// the pair (phys, N-1-phys), phys = j + 1 and the ghost pair last
// (fold_phys), so an input with a zero ghost ring contracts over h - 1; the
// middle of an odd N pairs with itself and counts once.
//
// Fragment order: every operand of a product is stored as the MFMA reads it,
// element [lane] of k-step s (four k) of a tile of 16 indices at s * 64 +
// lane, lane = (k % 4) * 16 + index % 16; loads are 512 contiguous bytes a
// wave.  The 16 x 16 result (row = lane / 16 + 4 r, column = lane % 16) of one
// product *is* four k-steps of the next product's operand, row = k and column
// = index, so results are stored without any shuffle.  Extents are padded to
// 16 with zeros in the tables, which makes every padded result zero.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <new>
#include <type_traits>
#include <utility>
#include <vector>

#include "common.h"
#include "kernels.h"

namespace somax {

namespace {

typedef double double4m __attribute__((ext_vector_type(4)));

struct DirectArgs {
  const void* q;
  void* psi;
  int Nx, Ny, hx, hy;  // points and folded extents ceil(N / 2)
  int ntx, nty;        // tiles of 16 per folded extent
  int P, M, nlmax;
  long plane;
  int apply_bc;
  int split;           // forward: workgroups that share one data tile
  // member and plane tables (null with one member: planes 0 .. P-1)
  const int* mfirst;
  const int* mnl;
  const int* member;
  const int* layer;
  const unsigned char* mask;  // ghost ring of psi set to 0 (one member: mask0)
  int mask0;
  const double* cl2m;  // [M][8][8]
  const double* cm2l;
  const double* lam;   // per plane
  // per axis: forward and inverse operators in fragment order (parity stride
  // 256 nt^2), eigenvalues per parity (16 nt each) and column sums (even parity)
  const double *fx, *gx, *fy, *gy, *lamx, *lamy, *cx, *cy;
  double* T;  // [P][py][px] blocks of 256 ntx nty
  double* V;
  // mass correction (homsol null: none), as in LayerArgs
  const void* homsol;
  const double* hmean;
  double inv_count;
  double* partial;  // [P][ntx] sums of the modal psi
  float* psi_wall;  // wall psi per plane (FP32 states)
  double* alpha;    // per-plane multipliers (FP64 states)
};

template <int G>
struct DirectTable {
  BlockTable t;
  DirectArgs a[G];
};
// Batch c and its block l in XCD-contiguous order (-1: padding block).
template <int G>
__device__ inline int direct_block(const DirectTable<G>& g, int& c) {
  if (G == 1) {
    c = 0;
    return xcd_order(blockIdx.x, gridDim.x);
  }
  int l;
  if (!table_class(g.t, blockIdx.x, c, l)) return -1;
  return xcd_order(l, g.t.count[c]);
}

__device__ inline double4m mfma64(double a, double b, double4m c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// A fragment stream from global memory: four batches of four k-steps in
// flight (1024 matrix cycles, about one trip to the Infinity Cache).  `p` is
// this lane's element of step 0.
typedef double Ring[4][4];
__device__ __forceinline__ void ring_load(Ring& v, int i, const double* p, int b) {
  const double* q = p + b * 256;
#pragma unroll
  for (int t = 0; t < 4; ++t) v[i][t] = q[t * 64];
}
// The first four of nb batches (fewer: the last one again, so that the number
// of loads in flight does not depend on nb).
__device__ __forceinline__ void ring_start(Ring& v, const double* p, int nb) {
#pragma unroll
  for (int i = 0; i < 4; ++i) ring_load(v, i, p, i < nb ? i : nb - 1);
}
// Runs batch(b, i, whole) over nb batches, ring slot i = b % 4, refilling a
// slot by load(i, b + 4) as soon as it is used; whole: certainly not the last
// batch.  Loads stay ahead of the next batch's products by the scheduling
// barrier.
template <class Batch, class Load>
__device__ __forceinline__ void ring_run(int nb, Batch batch, Load load) {
  int b = 0;
  for (; b + 8 <= nb; b += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      batch(b + i, i, std::true_type{});
      load(i, b + i + 4);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (b + i < nb) batch(b + i, i, std::false_type{});
    if (b + i + 4 < nb) load(i, b + i + 4);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (b + i + 4 < nb) batch(b + i + 4, i, std::false_type{});
}

// acc += sum over ns k-steps (whole batches: the padding is zero) of the
// stream p, started in v, and an LDS operand (this lane's element of step s at
// l[s * SL]); LA: the LDS operand is the A side.
template <bool LA, int SL>
__device__ __forceinline__ void product(Ring& v, const double* p, const double* l, int ns, double4m& acc) {
  const int nb = (ns + 3) >> 2;
  double x[2][4];  // the LDS operand one batch ahead
  auto read = [&](int i, int b) {
    const int at = 4 * (b < nb ? b : nb - 1);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[i][t] = l[(at + t) * SL];
  };
  read(0, 0);
  ring_run(
      nb,
      [&](int b, int i, auto whole) {
        read((i + 1) & 1, b + 1);
        const double(&y)[4] = x[i & 1];
        acc = LA ? mfma64(y[0], v[i][0], acc) : mfma64(v[i][0], y[0], acc);
        // extents of a power of two plus one end on a batch of one step
        if (decltype(whole)::value || 4 * b + 1 < ns) {
#pragma unroll
          for (int t = 1; t < 4; ++t) acc = LA ? mfma64(y[t], v[i][t], acc) : mfma64(v[i][t], y[t], acc);
        }
      },
      [&](int i, int b) { ring_load(v, i, p, b); });
}

__host__ __device__ inline int direct_k(int h, int apply_bc) { return apply_bc ? h - 1 : h; }
// LDS pitch (doubles) of the forward kernel's data rows: = 2 mod 4, so the 16
// rows of a fragment read fall on distinct banks; a whole number of batches of
// 16 entries before the pad.
__host__ __device__ inline int direct_pitch(int K) { return ((K + 15) & ~15) + 2; }

// Forward: workgroup = one tile of 16 folded rows of one plane (and a share of
// the output tiles).  Its threads project the four mirror points of every
// folded point to the plane's mode and leave the four parity sums in LDS; the
// two waves of each parity (px, py) then multiply its rows by the x operator.
template <class R, int NL, int G>
__global__ __launch_bounds__(512) void direct_forward_kernel(DirectTable<G> g) {
  extern __shared__ __attribute__((aligned(16))) double sd[];
  int c;
  const int l = direct_block<G>(g, c);
  if (l < 0) return;
  const DirectArgs& a = g.a[c];
  const int part = l % a.split;
  const int rest = l / a.split;
  const int yt = rest % a.nty, z = rest / a.nty;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int K = direct_k(a.hx, a.apply_bc);
  const int pitch = direct_pitch(K), kpad = pitch - 2;
  const int par = wave & 3, px = par & 1;
  const double* Bx = a.fx + px * 256L * a.ntx * a.ntx + lane;
  const int ns = (K + 3) / 4;
  int t = part + a.split * (wave >> 2);
  const double* B = Bx + (long)t * 256 * a.ntx;
  Ring v;
  if (t < a.ntx) ring_start(v, B, (ns + 3) >> 2);

  int m = 0, first = 0, nl = a.P, mode = z;
  if (a.mfirst) {
    m = a.member[z];
    first = a.mfirst[m];
    nl = a.mnl[m];
    mode = a.layer[z];
  }
  const double* cl = a.cl2m + m * 64 + mode * MAX_LAYERS;
  const R* q = static_cast<const R*>(a.q) + (long)first * a.plane;
  const int Nx = a.Nx, Ny = a.Ny;
  const bool bc = a.apply_bc != 0;
  // EB points of a thread at a time, all their loads before the first sum
  auto project = [&](auto eb) {
    constexpr int EB = decltype(eb)::value;
    for (int e0 = tid; e0 < 16 * kpad; e0 += 512 * EB) {
      int yy[EB], jj[EB], x[EB], y[EB];
      bool live[EB];
      double u[EB][4];
#pragma unroll
      for (int b = 0; b < EB; ++b) {
        const int e = e0 + 512 * b;
        yy[b] = e / kpad;
        jj[b] = e - yy[b] * kpad;
        const int jy = yt * 16 + yy[b];
        live[b] = yy[b] < 16 && jj[b] < K && jy < a.hy && !(bc && jy == a.hy - 1);
        x[b] = live[b] ? fold_phys(jj[b], a.hx) : 0;
        y[b] = live[b] ? fold_phys(jy, a.hy) : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) u[b][i] = 0.0;
      }
      for (int k0 = 0; k0 < nl; k0 += NL) {
        // (layers past the last read it again and are left out of the sum)
        R r[EB][NL][4];
#pragma unroll
        for (int b = 0; b < EB; ++b)
#pragma unroll
          for (int k = 0; k < NL; ++k) {
            const R* p = q + (k0 + k < nl ? k0 + k : nl - 1) * a.plane;
            const int r0 = y[b] * Nx, r1 = (Ny - 1 - y[b]) * Nx, xm = Nx - 1 - x[b];
            r[b][k][0] = p[r0 + x[b]];
            r[b][k][1] = p[r0 + xm];
            r[b][k][2] = p[r1 + x[b]];
            r[b][k][3] = p[r1 + xm];
          }
#pragma unroll
        for (int k = 0; k < NL; ++k)
          if (k0 + k < nl) {
            const double w = cl[k0 + k];
#pragma unroll
            for (int b = 0; b < EB; ++b)
#pragma unroll
              for (int i = 0; i < 4; ++i) u[b][i] += w * (double)r[b][k][i];
          }
      }
#pragma unroll
      for (int b = 0; b < EB; ++b) {
        if (yy[b] >= 16) continue;
        double* v = u[b];
        if (2 * x[b] == Nx - 1) v[1] = v[3] = 0.0;  // the middle of an odd line counts once
        if (2 * y[b] == Ny - 1) v[2] = v[3] = 0.0;
        const double p0 = v[0] + v[1], m0 = v[0] - v[1], p1 = v[2] + v[3], m1 = v[2] - v[3];
        double* o = sd + yy[b] * pitch + jj[b];
        o[0] = live[b] ? p0 + p1 : 0.0;  // [py][px]
        o[16 * pitch] = live[b] ? m0 + m1 : 0.0;
        o[32 * pitch] = live[b] ? p0 - p1 : 0.0;
        o[48 * pitch] = live[b] ? m0 - m1 : 0.0;
      }
    }
  };
  if (16 * kpad <= 512) project(std::integral_constant<int, 1>{});
  else project(std::integral_constant<int, (NL <= 2 ? 4 : 2)>{});
  __syncthreads();
  const double* A = sd + par * 16 * pitch + (lane & 15) * pitch + (lane >> 4);
  double* T = a.T + ((long)(z * 4 + par) * a.ntx) * (256L * a.nty) + yt * 256 + lane;
  for (; t < a.ntx; t += 2 * a.split) {
    double4m acc = {0.0, 0.0, 0.0, 0.0};
    product<true, 4>(v, B, A, ns, acc);
    const int next = t + 2 * a.split;
    if (next < a.ntx) {
      B = Bx + (long)next * 256 * a.ntx;
      ring_start(v, B, (ns + 3) >> 2);
    }
    double* o = T + (long)t * (256L * a.nty);
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r * 64] = acc[r];
  }
}

// The y products and the division of 16 x-modes of one parity block.
struct Spectral {
  Ring v;                     // the start of this wave's first y tile, O
  Ring g;                     // and of its first tile of the way back
  const double *F, *Gy, *ly, *cy;  // this lane's y operators, eigenvalues and column sums
  double lyv[4], cyv[4];           // the latter two of the next tile
  const double* O;
  long zb;
  int ns, t0;
  bool sums;
  double lx, cxv;
};
__device__ __forceinline__ void spectral_tile(Spectral& s, int t) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    s.lyv[r] = s.ly[t * 16 + 4 * r];
    s.cyv[r] = s.sums ? s.cy[t * 16 + 4 * r] : 0.0;
  }
}
__device__ __forceinline__ void spectral_start(Spectral& s, const DirectArgs& a, int z, int py, int px, int xt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  s.zb = (long)(z * 4 + py * 2 + px) * (256L * a.ntx * a.nty);
  s.ns = (a.hy + 3) / 4;
  const long ypar = py * 256L * a.nty * a.nty;
  s.F = a.fy + ypar + lane;
  s.Gy = a.gy + ypar + lane;
  s.t0 = wave < a.nty ? wave : a.nty - 1;
  s.O = s.F + (long)s.t0 * 256 * a.nty;
  // (waves without a tile load nothing: their streams would cost L1 time, 64 KB a
  // ring and workgroup; measured 128^2 x 3 two Tsit5 steps 308 -> 301 us)
  if (wave < a.nty) ring_start(s.v, s.O, (s.ns + 3) >> 2);
  s.lx = a.lamx[px * 16 * a.ntx + xt * 16 + (lane & 15)] - a.lam[z];
  s.ly = a.lamy + py * 16 * a.nty + (lane >> 4);
  s.sums = a.homsol && px == 0 && py == 0;
  s.cxv = s.sums ? a.cx[xt * 16 + (lane & 15)] : 0.0;
  s.cy = a.cy + (lane >> 4);
}
// From the modes' data Ts (fragment order) to V; W: the same space for the quotient.
// EARLY: at most one tile a wave, its eigenvalues read before (spectral_tile) and
// the ring of its way back started before the first product.
template <int NW, bool EARLY>
__device__ __forceinline__ void spectral_run(Spectral& s, const DirectArgs& a, int z, int xt, const double* Ts,
                                             double* W, double* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double total = 0.0;
  Ring& g = EARLY ? s.g : s.v;
  if (EARLY && wave < a.nty) ring_start(s.g, s.Gy + (long)s.t0 * 256 * a.nty, (s.ns + 3) >> 2);
  for (int t = wave; t < a.nty; t += NW) {
    double4m acc = {0.0, 0.0, 0.0, 0.0};
    if (!EARLY) spectral_tile(s, t);
    product<false, 64>(s.v, s.O, Ts + lane, s.ns, acc);
    // next: this wave's next tile, else its first tile of the way back
    if (!EARLY) {
      s.O = t + NW < a.nty ? s.F + (long)(t + NW) * 256 * a.nty : s.Gy + (long)s.t0 * 256 * a.nty;
      ring_start(s.v, s.O, (s.ns + 3) >> 2);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double w = acc[r] / (s.lx + s.lyv[r]);
      W[(t * 4 + r) * 64 + lane] = w;
      total += w * s.cxv * s.cyv[r];
    }
  }
  if (s.sums) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o);
    if (lane == 0) red[wave] = total;
  }
  __syncthreads();
  if (s.sums && tid == 0) {
    double w = 0.0;
    for (int i = 0; i < NW; ++i) w += red[i];
    a.partial[(long)z * a.ntx + xt] = w;
  }
  double* V = a.V + s.zb + xt * 256 + lane;
  if (EARLY) s.O = s.Gy + (long)s.t0 * 256 * a.nty;
  for (int t = wave; t < a.nty; t += NW) {
    double4m acc = {0.0, 0.0, 0.0, 0.0};
    product<true, 64>(g, s.O, W + lane, s.ns, acc);
    if (t + NW < a.nty) {
      s.O = s.Gy + (long)(t + NW) * 256 * a.nty;
      ring_start(g, s.O, (s.ns + 3) >> 2);
    }
    double* o = V + (long)t * (256L * a.ntx);
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r * 64] = acc[r];
  }
}

// Spectral: workgroup = 16 x-modes of one parity block of one plane.  The y
// transform's result stays in LDS (fragment order) between the two products.
template <int NW, int G>
__global__ __launch_bounds__(64 * NW) void direct_spectral_kernel(DirectTable<G> g) {
  extern __shared__ __attribute__((aligned(16))) double sd[];
  __shared__ double red[NW];
  int c;
  const int l = direct_block<G>(g, c);
  if (l < 0) return;
  const DirectArgs& a = g.a[c];
  // py slowest, so an XCD mostly reads one parity's y operators
  const int xt = l % a.ntx;
  int rest = l / a.ntx;
  const int px = rest & 1;
  rest >>= 1;
  const int z = rest % a.P, py = rest / a.P;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double* T = a.T + ((long)(z * 4 + py * 2 + px) * a.ntx + xt) * (256L * a.nty);
  double* W = sd;                 // [4 nty k-steps of iy][64]
  double* Ts = sd + 256 * a.nty;  // the x-modes' data, staged once for all waves
  Spectral s;
  spectral_start(s, a, z, py, px, xt);
  // straight into LDS, 1 KiB a wave and instruction
  for (int e = wave; e < 2 * a.nty; e += NW)
    __builtin_amdgcn_global_load_lds(T + e * 128 + lane * 2, Ts + e * 128, 16, 0, 0);
  __syncthreads();
  spectral_run<NW, false>(s, a, z, xt, Ts, W, red);
}

// Forward and spectral in one, for planes of a few tiles: workgroup = 16 x-modes of
// one parity block of one plane.  It projects and folds the whole plane to its
// parity (every workgroup of a plane again: a few loads a thread), takes its 16
// modes of the x product from LDS to LDS, and goes on as the spectral kernel.  The
// same sums in the same order.  Bound by the chain of loads and short products, of
// which it saves one launch and one trip through memory: at 64^2 x 1 an inversion
// in a replayed graph 12.3 -> 10.5 us, an FP64 step of three 60.6 -> 52.5 (with the
// ring of the way back started late, by waves without a tile too: 11.3, 55.9).
template <class R, int NL>
__global__ __launch_bounds__(512) void direct_front_kernel(DirectTable<1> g) {
  constexpr int NW = 8;
  extern __shared__ __attribute__((aligned(16))) double sd[];
  __shared__ double red[NW];
  const DirectArgs& a = g.a[0];
  const int l = xcd_order(blockIdx.x, gridDim.x);
  const int xt = l % a.ntx;
  int rest = l / a.ntx;
  const int px = rest & 1;
  rest >>= 1;
  const int z = rest % a.P, py = rest / a.P;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int K = direct_k(a.hx, a.apply_bc), rows = direct_k(a.hy, a.apply_bc);
  const int pitch = direct_pitch(K), kpad = pitch - 2, nsx = (K + 3) / 4;
  double* X = sd;  // [16 nty][pitch]
  double* Ts = sd + 16 * a.nty * pitch;
  double* W = Ts + 256 * a.nty;
  const double* B = a.fx + px * 256L * a.ntx * a.ntx + (long)xt * 256 * a.ntx + lane;
  Ring vx;
  if (wave < a.nty) ring_start(vx, B, (nsx + 3) >> 2);
  Spectral sp;
  spectral_start(sp, a, z, py, px, xt);
  spectral_tile(sp, sp.t0);

  int m = 0, first = 0, nl = a.P, mode = z;
  if (a.mfirst) {
    m = a.member[z];
    first = a.mfirst[m];
    nl = a.mnl[m];
    mode = a.layer[z];
  }
  const double* cl = a.cl2m + m * 64 + mode * MAX_LAYERS;
  const R* q = static_cast<const R*>(a.q) + (long)first * a.plane;
  const int Nx = a.Nx, Ny = a.Ny;
  // EB points of a thread at a time, all their loads before the first sum
  constexpr int EB = NL <= 2 ? 4 : 2;
  for (int e0 = tid; e0 < rows * kpad; e0 += 512 * EB) {
    int x[EB], y[EB], at[EB];
    bool live[EB];
    double u[EB][4];
#pragma unroll
    for (int b = 0; b < EB; ++b) {
      const int e = min(e0 + 512 * b, rows * kpad - 1);  // (past the end: the last point again)
      const int jy = e / kpad, jj = e - jy * kpad;
      live[b] = jj < K;
      x[b] = fold_phys(live[b] ? jj : 0, a.hx);
      y[b] = fold_phys(jy, a.hy);
      at[b] = jy * pitch + jj;
#pragma unroll
      for (int i = 0; i < 4; ++i) u[b][i] = 0.0;
    }
    for (int k0 = 0; k0 < nl; k0 += NL) {
      // (layers past the last read it again and are left out of the sum)
      R r[EB][NL][4];
#pragma unroll
      for (int b = 0; b < EB; ++b)
#pragma unroll
        for (int k = 0; k < NL; ++k) {
          const R* p = q + (k0 + k < nl ? k0 + k : nl - 1) * a.plane;
          const int r0 = y[b] * Nx, r1 = (Ny - 1 - y[b]) * Nx, xm = Nx - 1 - x[b];
          r[b][k][0] = p[r0 + x[b]];
          r[b][k][1] = p[r0 + xm];
          r[b][k][2] = p[r1 + x[b]];
          r[b][k][3] = p[r1 + xm];
        }
#pragma unroll
      for (int k = 0; k < NL; ++k)
        if (k0 + k < nl) {
          const double w = cl[k0 + k];
#pragma unroll
          for (int b = 0; b < EB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) u[b][i] += w * (double)r[b][k][i];
        }
    }
#pragma unroll
    for (int b = 0; b < EB; ++b) {
      double* s = u[b];
      if (2 * x[b] == Nx - 1) s[1] = s[3] = 0.0;  // the middle of an odd line counts once
      if (2 * y[b] == Ny - 1) s[2] = s[3] = 0.0;
      const double c0 = px ? s[0] - s[1] : s[0] + s[1], c1 = px ? s[2] - s[3] : s[2] + s[3];
      X[at[b]] = live[b] ? (py ? c0 - c1 : c0 + c1) : 0.0;
    }
  }
  for (int e = rows * pitch + tid; e < 16 * a.nty * pitch; e += 512) X[e] = 0.0;
  __syncthreads();
  if (wave < a.nty) {  // one tile a wave: at most 65 folded points (direct_front)
    double4m acc = {0.0, 0.0, 0.0, 0.0};
    product<true, 4>(vx, B, X + (wave * 16 + (lane & 15)) * pitch + (lane >> 4), nsx, acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) Ts[wave * 256 + r * 64 + lane] = acc[r];
  }
  __syncthreads();
  spectral_run<NW, true>(sp, a, z, xt, Ts, W, red);
}

// Inverse: workgroup = 16 x 16 XT folded points (four mirror images of each) of
// one member.  Wave (mode, py, px) computes one parity block of one mode; the
// blocks meet in LDS, where they are unfolded, corrected and mixed to layers.
// XT = 2 halves what a wave streams per product (the data of 16 rows serves two
// tiles of columns).
template <class R, int NMODE, int XT, int G>
__global__ __launch_bounds__(256 * NMODE) void direct_inverse_kernel(DirectTable<G> g) {
  extern __shared__ __attribute__((aligned(16))) double sd[];  // [mode][py px][16][CP]
  __shared__ double salpha[MAX_LAYERS];
  __shared__ double scm[64];
  constexpr int CP = 16 * XT + 1;
  int c;
  const int l = direct_block<G>(g, c);
  if (l < 0) return;
  const DirectArgs& a = g.a[c];
  const int nbx = (a.ntx + XT - 1) / XT;
  const int xt = (l % nbx) * XT;
  const int rest = l / nbx;
  const int yt = rest % a.nty, m = rest / a.nty;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int first = 0, nl = a.P;
  bool mask = a.mask0 != 0;
  if (a.mfirst) {
    first = a.mfirst[m];
    nl = a.mnl[m];
    mask = a.mask[m] != 0;
  }
  const int par = wave & 3, px = par & 1;
  const long blk = 256L * a.ntx * a.nty;
  const double* B[XT];  // (a tile past the last streams it again)
#pragma unroll
  for (int j = 0; j < XT; ++j)
    B[j] = a.gx + px * 256L * a.ntx * a.ntx + (long)(xt + j < a.ntx ? xt + j : a.ntx - 1) * 256 * a.ntx + lane;
  const double* A = a.V + (long)(first * 4 + par) * blk + (long)yt * (256L * a.ntx) + lane;
  const int ns = (a.hx + 3) / 4;
  int k = wave >> 2;
  A += (k < nl ? k : nl - 1) * 4 * blk;
  const int nb = (ns + 3) >> 2;
  Ring va, vb[XT];
  auto start = [&] {
    ring_start(va, A, nb);
#pragma unroll
    for (int j = 0; j < XT; ++j) ring_start(vb[j], B[j], nb);
  };
  start();
  if (tid < 64) scm[tid] = a.cm2l[m * 64 + tid];
  // this thread's points of the unfolding (column j * 16 + xx of each tile) and
  // the first modes' homogeneous solutions there
  const int Nx = a.Nx, Ny = a.Ny;
  const int yy = (tid >> 4) & 15, xx = tid & 15;
  const int jy = yt * 16 + yy;
  const int y = jy < a.hy ? fold_phys(jy, a.hy) : 0, ym = Ny - 1 - y;
  bool live[XT];
  int at[XT][4];  // a plane is below 2^31 points
#pragma unroll
  for (int j = 0; j < XT; ++j) {
    const int jx = (xt + j) * 16 + xx;
    live[j] = jy < a.hy && jx < a.hx;
    const int x = live[j] ? fold_phys(jx, a.hx) : 0, xm = Nx - 1 - x;
    at[j][0] = y * Nx + x;
    at[j][1] = y * Nx + xm;
    at[j][2] = ym * Nx + x;
    at[j][3] = ym * Nx + xm;
  }
  const R* hom = static_cast<const R*>(a.homsol) + (long)first * a.plane;
  constexpr int NH = XT == 1 && NMODE * sizeof(R) <= 24 ? NMODE : 0;  // modes fetched early (registers)
  R hv[NH ? NH : 1][4];
  if (a.homsol) {
#pragma unroll
    for (int p = 0; p < NH; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) hv[p][i] = hom[(p < nl ? p : nl - 1) * a.plane + at[0][i]];
    if (tid < nl) {
      const double* p = a.partial + (long)(first + tid) * a.ntx;
      double s = 0.0;
#pragma unroll 4
      for (int i = 0; i < a.ntx; ++i) s += p[i];
      const double hm = a.hmean[first + tid];
      salpha[tid] = hm != 0.0 ? -(s * a.inv_count) / hm : 0.0;
    }
  }
  for (; k < nl; k += NMODE) {
    double4m acc[XT];
#pragma unroll
    for (int j = 0; j < XT; ++j) acc[j] = double4m{0.0, 0.0, 0.0, 0.0};
    ring_run(
        nb,
        [&](int b, int i, auto whole) {
#pragma unroll
          for (int j = 0; j < XT; ++j) acc[j] = mfma64(va[i][0], vb[j][i][0], acc[j]);
          if (decltype(whole)::value || 4 * b + 1 < ns) {
#pragma unroll
            for (int t = 1; t < 4; ++t)
#pragma unroll
              for (int j = 0; j < XT; ++j) acc[j] = mfma64(va[i][t], vb[j][i][t], acc[j]);
          }
        },
        [&](int i, int b) {
          ring_load(va, i, A, b);
#pragma unroll
          for (int j = 0; j < XT; ++j) ring_load(vb[j], i, B[j], b);
        });
    if (k + NMODE < nl) {
      A += NMODE * 4 * blk;
      start();
    }
    double* o = sd + ((k * 4 + par) * 16 + (lane >> 4)) * CP + (lane & 15);
#pragma unroll
    for (int j = 0; j < XT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[4 * r * CP + 16 * j] = acc[j][r];
  }
  __syncthreads();
  if (a.homsol && l == m * nbx * a.nty && tid < nl) {
    double w = 0.0;
    for (int p = 0; p < nl; ++p) w += scm[tid * MAX_LAYERS + p] * salpha[p];
    if (a.psi_wall) a.psi_wall[first + tid] = (float)w;
    if (a.alpha) a.alpha[first + tid] = salpha[tid];
  }
  R* psi = static_cast<R*>(a.psi) + (long)first * a.plane;
  for (int kl = tid >> 8; kl < nl; kl += NMODE)
#pragma unroll
    for (int j = 0; j < XT; ++j) {
      if (!live[j]) continue;
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      auto add = [&](int p, const R* h) {
        const double w = scm[kl * MAX_LAYERS + p];
        const double* e = sd + (p * 4 * 16 + yy) * CP + 16 * j + xx;
        const double e00 = e[0], e01 = e[16 * CP], e10 = e[32 * CP], e11 = e[48 * CP];  // [py][px]
        const double sp = e00 + e01, sm = e00 - e01, tp = e10 + e11, tm = e10 - e11;
        double u[4] = {sp + tp, sm + tm, sp - tp, sm - tm};
        if (a.homsol) {
#pragma unroll
          for (int i = 0; i < 4; ++i) u[i] += salpha[p] * (double)h[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += w * u[i];
      };
#pragma unroll
      for (int p = 0; p < NH; ++p)
        if (p < nl) add(p, hv[p]);
      for (int p = NH; p < nl; ++p) {
        R h[4] = {};
        if (a.homsol) {
#pragma unroll
          for (int i = 0; i < 4; ++i) h[i] = hom[p * a.plane + at[j][i]];
        }
        add(p, h);
      }
      // the ghost pair of either axis
      const bool zero = mask && (y == 0 || at[j][0] == y * Nx);
#pragma unroll
      for (int i = 0; i < 4; ++i) psi[kl * a.plane + at[j][i]] = zero ? (R)0 : (R)v[i];
    }
}

constexpr int DIRECT_LDS = 157 * 1024;
// The spectral kernel's loads into LDS take 16 bytes a lane; a caller's workspace
// need not be aligned to more than a double.
constexpr size_t DIRECT_ALIGN = 16;
size_t forward_lds(const DirectArgs& a) {
  return (size_t)64 * direct_pitch(direct_k(a.hx, a.apply_bc)) * sizeof(double);
}
size_t front_lds(const DirectArgs& a) {
  return (size_t)a.nty * (16 * direct_pitch(direct_k(a.hx, a.apply_bc)) + 512) * sizeof(double);
}
// The forward and spectral kernels in one launch (direct_front_kernel) while that
// saves more than its repeated folds cost.  A workgroup loads rows x row x layers
// points four times (rows of at least 32 points: shorter ones cost as much).
// us of an inversion in a replayed graph, two launches -> one: 16^2 x 1 10.5 -> 8.3,
// 64^2 x 1 12.3 -> 10.5, 64^2 x 7 21.4 -> 19.9, 126^2 x 2 (8064) 14.9 -> 14.3; but 126^2 x 3
// (12096) 16.0 -> 17.3, 30 x 120 x 6 (11520) 19.2 -> 19.6.  Up to 64 points a side every wave has at most one
// tile, and its ring holds the tile's whole stream or, at 65 folded points, all but
// the last step (160^2 x 1: 16.8 -> 18.2).  And one workgroup per CU, as a full chip pays for every
// repeat (steps of ensembles: 64^2, 240 workgroups 98 -> 93, 288 108 -> 120; 32^2, 192
// 103 -> 95, 384 104 -> 112).
bool direct_front(const DirectArgs& a) {
  const int K = direct_k(a.hx, a.apply_bc), rows = direct_k(a.hy, a.apply_bc);
  return K <= 64 && rows <= 64 && rows * std::max(direct_pitch(K) - 2, 32) * a.nlmax <= 8192 &&
         a.P * 4 * a.ntx <= 256;
}
size_t spectral_lds(const DirectArgs& a) { return (size_t)512 * a.nty * sizeof(double); }
// Column tiles per workgroup of the inverse kernel: two where a fold has more
// than eight tiles (measured at 512^2 x 3: 30 -> 23 us) and the registers of a
// workgroup of up to three modes hold the second stream.
int inverse_xt(int ntx, int nlmax) { return ntx > 8 && nlmax <= 3 ? 2 : 1; }
size_t inverse_lds(const DirectArgs& a, int xt) { return (size_t)a.nlmax * 4 * 16 * (16 * xt + 1) * sizeof(double); }

template <class K>
hipError_t raise_lds(K kernel, int bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
template <class R, int G>
hipError_t prepare_kernels() {
  hipError_t e = raise_lds(direct_forward_kernel<R, 1, G>, DIRECT_LDS);
  if (G == 1) {
    if (e == hipSuccess) e = raise_lds(direct_front_kernel<R, 1>, DIRECT_LDS);
    if (e == hipSuccess) e = raise_lds(direct_front_kernel<R, 2>, DIRECT_LDS);
    if (e == hipSuccess) e = raise_lds(direct_front_kernel<R, 3>, DIRECT_LDS);
    if (e == hipSuccess) e = raise_lds(direct_front_kernel<R, 4>, DIRECT_LDS);
  }
  if (e == hipSuccess) e = raise_lds(direct_forward_kernel<R, 2, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_forward_kernel<R, 3, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_forward_kernel<R, 4, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_spectral_kernel<4, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_spectral_kernel<8, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 1, 1, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 2, 1, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 3, 1, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 4, 1, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 1, 2, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 2, 2, G>, DIRECT_LDS);
  if (e == hipSuccess) e = raise_lds(direct_inverse_kernel<R, 3, 2, G>, DIRECT_LDS);
  return e;
}
hipError_t prepare_direct() {
  static OncePerDevice once;
  return once([] {
    hipError_t e = prepare_kernels<float, 1>();
    if (e == hipSuccess) e = prepare_kernels<float, MAX_GROUP>();
    if (e == hipSuccess) e = prepare_kernels<double, 1>();
    return e;
  });
}

template <class R, int G>
void launch_forward(DirectTable<G>& g, int blocks, size_t lds, int nlmax, hipStream_t st) {
  if (nlmax == 1) hipLaunchKernelGGL((direct_forward_kernel<R, 1, G>), dim3(blocks), dim3(512), lds, st, g);
  else if (nlmax == 2) hipLaunchKernelGGL((direct_forward_kernel<R, 2, G>), dim3(blocks), dim3(512), lds, st, g);
  else if (nlmax == 3) hipLaunchKernelGGL((direct_forward_kernel<R, 3, G>), dim3(blocks), dim3(512), lds, st, g);
  else hipLaunchKernelGGL((direct_forward_kernel<R, 4, G>), dim3(blocks), dim3(512), lds, st, g);
}
template <class R>
void launch_front(DirectTable<1>& g, hipStream_t st) {
  const DirectArgs& a = g.a[0];
  const dim3 blocks(a.P * 4 * a.ntx), threads(512);
  const size_t lds = front_lds(a);
  if (a.nlmax == 1) hipLaunchKernelGGL((direct_front_kernel<R, 1>), blocks, threads, lds, st, g);
  else if (a.nlmax == 2) hipLaunchKernelGGL((direct_front_kernel<R, 2>), blocks, threads, lds, st, g);
  else if (a.nlmax == 3) hipLaunchKernelGGL((direct_front_kernel<R, 3>), blocks, threads, lds, st, g);
  else hipLaunchKernelGGL((direct_front_kernel<R, 4>), blocks, threads, lds, st, g);
}
template <int G>
void launch_spectral(DirectTable<G>& g, int blocks, size_t lds, int nty, hipStream_t st) {
  if (nty > 4) hipLaunchKernelGGL((direct_spectral_kernel<8, G>), dim3(blocks), dim3(512), lds, st, g);
  else hipLaunchKernelGGL((direct_spectral_kernel<4, G>), dim3(blocks), dim3(256), lds, st, g);
}
template <class R, int XT, int G>
void launch_inverse(DirectTable<G>& g, int blocks, size_t lds, int nlmax, hipStream_t st) {
  if (nlmax == 1) hipLaunchKernelGGL((direct_inverse_kernel<R, 1, XT, G>), dim3(blocks), dim3(256), lds, st, g);
  else if (nlmax == 2) hipLaunchKernelGGL((direct_inverse_kernel<R, 2, XT, G>), dim3(blocks), dim3(512), lds, st, g);
  else if (nlmax == 3) hipLaunchKernelGGL((direct_inverse_kernel<R, 3, XT, G>), dim3(blocks), dim3(768), lds, st, g);
  else hipLaunchKernelGGL((direct_inverse_kernel<R, 4, 1, G>), dim3(blocks), dim3(1024), lds, st, g);
}

// One axis on the host: operators in fragment order, eigenvalues, column sums.
struct AxisTables {
  std::vector<double> f, g, lam, c;
};
AxisTables axis_tables(int N, double d) {
  const int h = (N + 1) / 2, nt = (h + 15) / 16, hp = 16 * nt;
  AxisTables t;
  t.f.assign(2 * (size_t)hp * hp, 0.0);
  t.g.assign(2 * (size_t)hp * hp, 0.0);
  // padded modes: a symbol that no Helmholtz parameter, of either sign, brings to 0 (0 / 0
  // there would reach every point through the next product)
  t.lam.assign(2 * (size_t)hp, -std::numeric_limits<double>::infinity());
  t.c.assign(hp, 0.0);
  // S[n][k] = sqrt(2/(N+1)) sin(pi (n+1)(k+1)/(N+1)); angles reduced in
  // integers to [0, 2(N+1)), one sine per residue
  const long period = 2L * (N + 1);
  std::vector<double> sn(period);
  const double c = std::sqrt(2.0 / (N + 1));
  for (long r = 0; r < period; ++r) {
    // exact symmetries of the sine: arguments in [0, pi/2]
    long u = r % (N + 1);
    if (2 * u > N + 1) u = N + 1 - u;
    const double v = c * std::sin(M_PI * (double)u / (double)(N + 1));
    sn[r] = r > N + 1 ? -v : v;
  }
  sn[N + 1] = 0.0;
  auto S = [&](int a, int n) { return sn[((long)(a + 1) * (n + 1)) % period]; };
  auto frag = [&](int idx, int k) {  // tile of 16 indices, k-step, lane
    return (size_t)(idx / 16) * 16 * hp + (size_t)(k / 4) * 64 + (k % 4) * 16 + idx % 16;
  };
  for (int p = 0; p < 2; ++p) {
    const int hm = p == 0 ? h : N / 2;  // modes of this parity
    for (int i = 0; i < hm; ++i) {
      for (int j = 0; j < h; ++j) {
        const double v = S(2 * i + p, fold_phys(j, h));
        t.f[p * (size_t)hp * hp + frag(i, j)] = v;
        t.g[p * (size_t)hp * hp + frag(j, i)] = v;
      }
      const double s = std::sin(0.5 * M_PI * (2 * i + p + 1) / (double)(N + 1));
      t.lam[p * (size_t)hp + i] = -4.0 * s * s / (d * d);
      if (p == 0) {
        double sum = 0.0;
        for (int n = 0; n < N; ++n) sum += S(2 * i, n);
        t.c[i] = sum;
      }
    }
  }
  return t;
}

}  // namespace

struct Direct {
  DirectArgs a{};
  void* mem = nullptr;
  ~Direct() { (void)hipFree(mem); }
};

bool direct_fits(int Nx, int Ny) {
  const int hx = (Nx + 1) / 2, hy = (Ny + 1) / 2;
  return hx <= DIRECT_MAX_H && hy <= DIRECT_MAX_H;
}

size_t direct_bytes(int Nx, int Ny, int P) {
  const size_t ntx = ((Nx + 1) / 2 + 15) / 16, nty = ((Ny + 1) / 2 + 15) / 16;
  return ((size_t)P * 2 * 4 * 256 * ntx * nty + (size_t)P * ntx) * sizeof(double) + DIRECT_ALIGN;
}

void direct_destroy(Direct* d) { delete d; }

Direct* direct_create(const DirectDesc& s, hipError_t* err) {
  std::unique_ptr<Direct> d(new (std::nothrow) Direct());
  *err = hipErrorOutOfMemory;
  if (!d) return nullptr;
  DirectArgs& a = d->a;
  a.Nx = s.Nx;
  a.Ny = s.Ny;
  a.hx = (s.Nx + 1) / 2;
  a.hy = (s.Ny + 1) / 2;
  a.ntx = (a.hx + 15) / 16;
  a.nty = (a.hy + 15) / 16;
  a.plane = (long)s.Nx * s.Ny;
  a.M = (int)s.nl.size();
  a.nlmax = *std::max_element(s.nl.begin(), s.nl.end());
  std::vector<int> first, member, layer;
  for (int m = 0; m < a.M; ++m) {
    first.push_back((int)member.size());
    for (int k = 0; k < s.nl[m]; ++k) {
      member.push_back(m);
      layer.push_back(k);
    }
  }
  a.P = (int)member.size();
  a.mask0 = s.mask[0];
  const bool same = s.Nx == s.Ny && s.dx == s.dy;  // one set of tables serves both axes
  const AxisTables tx = axis_tables(s.Nx, s.dx), ty = same ? AxisTables{} : axis_tables(s.Ny, s.dy);
  // every table in one allocation and one copy
  std::vector<char> host;
  std::vector<std::pair<const void**, size_t>> at;
  auto put = [&](auto** out, const auto& v) {
    const size_t o = (host.size() + 255) / 256 * 256, bytes = v.size() * sizeof(v[0]);
    host.resize(o + bytes);
    std::memcpy(host.data() + o, v.data(), bytes);
    at.emplace_back(reinterpret_cast<const void**>(out), o);
  };
  put(&a.fx, tx.f);
  put(&a.gx, tx.g);
  put(&a.lamx, tx.lam);
  put(&a.cx, tx.c);
  if (!same) {
    put(&a.fy, ty.f);
    put(&a.gy, ty.g);
    put(&a.lamy, ty.lam);
    put(&a.cy, ty.c);
  }
  put(&a.cl2m, s.cl2m);
  put(&a.cm2l, s.cm2l);
  put(&a.lam, s.lam);
  if (a.M > 1) {
    put(&a.mfirst, first);
    put(&a.mnl, s.nl);
    put(&a.member, member);
    put(&a.layer, layer);
    put(&a.mask, s.mask);
  }
  hipError_t e = hipMalloc(&d->mem, host.size());
  if (e == hipSuccess) e = hipMemcpy(d->mem, host.data(), host.size(), hipMemcpyHostToDevice);
  for (const auto& p : at) *p.first = static_cast<char*>(d->mem) + p.second;
  if (same) {
    a.fy = a.fx;
    a.gy = a.gx;
    a.lamy = a.lamx;
    a.cy = a.cx;
  }
  if (e == hipSuccess) e = prepare_direct();
  // Forward: split the output tiles of a data tile over workgroups until the
  // launch has about one per CU (each share repeats the projection).
  a.split = std::min(a.ntx, std::max(1, 256 / (a.P * a.nty)));
  *err = e;
  return e == hipSuccess ? d.release() : nullptr;
}

namespace {
DirectArgs call_args(const DirectCall& c) {
  DirectArgs a = c.d->a;
  a.q = c.q;
  a.psi = c.psi;
  a.apply_bc = c.apply_bc ? 1 : 0;
  const size_t blocks = (size_t)a.P * 4 * 256 * a.ntx * a.nty;
  const uintptr_t at = reinterpret_cast<uintptr_t>(c.buf);
  a.T = reinterpret_cast<double*>((at + DIRECT_ALIGN - 1) / DIRECT_ALIGN * DIRECT_ALIGN);
  a.V = a.T + blocks;
  a.partial = a.V + blocks;
  a.homsol = c.homsol;
  a.hmean = c.hmean;
  a.inv_count = 1.0 / (double)a.plane;
  a.psi_wall = c.psi_wall;
  a.alpha = c.alpha;
  return a;
}

template <class R, int G>
void run(const DirectCall* c, int n, hipStream_t st, const DirectPhase& phase) {
  DirectTable<G> g{};
  int blocks[3] = {0, 0, 0}, nty = 0, ntx = 0, nlmax = 0;
  for (int i = 0; i < n; ++i) {
    nty = std::max(nty, c[i].d->a.nty);
    ntx = std::max(ntx, c[i].d->a.ntx);
    nlmax = std::max(nlmax, c[i].d->a.nlmax);
  }
  const int xt = inverse_xt(ntx, nlmax);
  size_t lds[3] = {0, 0, 0};
  BlockTable t[3] = {};
  for (int i = 0; i < n; ++i) {
    const DirectArgs& a = g.a[i] = call_args(c[i]);
    const int count[3] = {a.P * a.nty * a.split, a.P * 4 * a.ntx, a.M * ((a.ntx + xt - 1) / xt) * a.nty};
    const size_t need[3] = {forward_lds(a), spectral_lds(a), inverse_lds(a, xt)};
    for (int k = 0; k < 3; ++k) {
      table_add(t[k], count[k], 1, 1);
      blocks[k] = G == 1 ? count[k] : t[k].start[t[k].n];
      lds[k] = std::max(lds[k], need[k]);
    }
  }
  bool front = false;
  if constexpr (G == 1) {
    front = direct_front(g.a[0]);
    if (front) phase(3, [&] { launch_front<R>(g, st); });
  }
  if (!front) {
    phase(0, [&] {
      g.t = t[0];
      launch_forward<R, G>(g, blocks[0], lds[0], nlmax, st);
    });
    phase(1, [&] {
      g.t = t[1];
      launch_spectral<G>(g, blocks[1], lds[1], nty, st);
    });
  }
  phase(2, [&] {
    g.t = t[2];
    if (xt == 2) launch_inverse<R, 2, G>(g, blocks[2], lds[2], nlmax, st);
    else launch_inverse<R, 1, G>(g, blocks[2], lds[2], nlmax, st);
  });
}
}  // namespace

void launch_direct(const DirectCall& c, hipStream_t st, const DirectPhase& phase) {
  if (c.f64) run<double, 1>(&c, 1, st, phase);
  else run<float, 1>(&c, 1, st, phase);
}
void launch_direct_group(const DirectCall* c, int n, hipStream_t st, const DirectPhase& phase) {
  run<float, MAX_GROUP>(c, n, st, phase);
}

}  // namespace somax
