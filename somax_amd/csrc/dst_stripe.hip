// Three transforms of a solve in one launch (gfx950).
//
// A solve multiplies every plane by four sine operands (dst_gemm.hip):
//   F1: T[ix][y] = sum_x Sx[ix][x] X[y][x]
//   F2: W[ix][j] = sum_y T[ix][y] Sy[j][y] / (lamx[ix] + lamy[j] - lambda)
//   I1: V[y][ix] = sum_j Sy[y][j] W[ix][j]
//   I2: out[y][x] = sum_ix V[y][ix] Sx[x][ix]
// Row ix of T, W and V needs no other row ix, so a workgroup that owns a stripe
// of 32 of them runs F1, F2 and I1 from LDS to LDS and only V leaves the CU.
// On planes of a few hundred points the launches it replaces are chains of
// latencies (6.5 to 11 us each, of which the products take under one): start,
// arguments, first loads, k-loop, stores.
//
// Each wave owns one 32 x 32 output tile of every product: its rows of the
// operand that sweeps (X, Sy or Sy^T) go from global memory straight into its
// registers, the next product's while the current one's results are written; the stripe is read from LDS by all waves.
// Three barriers in all.  What bounds it: on small planes that chain, 8 us at 66^2
// (three launches: 24); at 257^2 the sweeps, each workgroup reading every operand
// once (1 MB, mixed) at the rate of its L1.  Measured, three launches and stripes
// (us): the launches themselves at 129^2 x 12 planes 24.6 -> 13.1, the correction's
// 22 -> 12.5; a right-hand side, mixed, 64^2 x 3 53 -> 39, 128^2 x 3 69 -> 52, 256^2
// x 3 82 -> 60, 512^2 x 3 115 -> 99; six products 256^2 x 3 49 -> 38, 512^2 x 3 76
// -> 70; an SSP-RK3 step of 3-layer mixed ensembles, 128^2 x 16 394 -> 275, x 96 978
// -> 900, 256^2 x 48 1611 -> 1547, 512^2 x 16 2049 -> 2023: no number of planes was
// slower.  The sweeps are kept in the order of the fragments (frag_row): read from
// row-major rows they cost four times the L1's time.
//
// Every output's chain of products, the FP64 sums of its
// windows and the dot products of the one or two rows past a multiple of 128 are
// those of dst_gemm.hip, so both forms give the same bits.

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace somax {
namespace {

constexpr int SR = 32;  // rows of a stripe
__host__ __device__ constexpr int pieces_of(int np) { return np == 1 ? 1 : (np == 3 ? 2 : 3); }
__host__ __device__ constexpr int round32(int v) { return (v + 31) & ~31; }
// LDS pitch of a stripe's rows (elements): 16 bytes past a multiple of 64, so the
// b128 reads of 8 consecutive rows fall on distinct banks.
__host__ __device__ constexpr int stripe_pitch(int K) { return round32(K) + 8; }

// One product of the solve: the operand that sweeps.
struct StripeOp {
  const uint16_t* B;    // in fragment order, k padded to ldb
  const uint16_t* row;  // row-major, pitch ldb (X: null)
  long ldb, b_piece;
  long b_plane, b_var;  // elements between batch planes; between parity variants
  int b_par;            // parity choosing the variant: 0 = x, 1 = y
  int K, R;             // contraction; sweep extent
  int cut;              // its part in tiles (R, or R - 1 or 2: the rest are dots)
};
struct StripeArgs {
  StripeOp op[3];
  const uint16_t* S;  // the sine operand of F1
  long lds, s_piece, s_var;
  int s_par;
  int R, cut;  // extent of ix; its part in stripes
  const float *lamA, *lamB, *lam;
  int lam_var, lamB_var;
  const unsigned char* hp;
  uint64_t hp_bits;
  int np_lo, np_hi;
  uint16_t* O;  // V
  long ldo, o_piece, o_batch;
  int pad;  // V's columns [R, pad) are zero
  int fold_P, stripes;
};

// The sweeping rows of a wave's tile: chunks of two k-tiles (four k16 steps, a
// window of the FP64 sums), DEPTH of them in registers: D, the chunks of the
// launch's longest contraction, as far as the registers go.
template <int NP, int D>
struct Sweep {
  static constexpr int NPC = pieces_of(NP);
  static constexpr int DEPTH = NP == 6 ? 2 : D;
  bf16x8 v[DEPTH][4][NPC];
};
// chunk c of nk k-tiles into slot i (steps past the last repeat it, so that the
// number of loads in flight is known)
template <int NP, int D>
__device__ __forceinline__ void sweep_load(Sweep<NP, D>& w, int i, const uint16_t* p, long piece, int c, int nk) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int step = min(4 * c + s, 2 * nk - 1);
#pragma unroll
    for (int q = 0; q < Sweep<NP, D>::NPC; ++q)
      w.v[i][s][q] = *reinterpret_cast<const bf16x8*>(p + q * piece + step * 512);
  }
}
template <int NP, int D>
__device__ __forceinline__ void sweep_start(Sweep<NP, D>& w, const uint16_t* p, long piece, int nk) {
#pragma unroll
  for (int i = 0; i < Sweep<NP, D>::DEPTH; ++i) sweep_load(w, i, p, piece, i, nk);
}

// acc (+ sum) += the tile's products over nk k-tiles; l: this lane's stripe row
// in LDS, lpiece its piece stride.  SA: the sweeping operand is the A side.
template <bool SA, int NP, int D>
__device__ __forceinline__ void sweep_run(Sweep<NP, D>& w, const uint16_t* p, long piece, int nk, const uint16_t* l,
                                          int lpiece, floatx16& acc, double (&sum)[16]) {
  constexpr int NPC = Sweep<NP, D>::NPC, DEPTH = Sweep<NP, D>::DEPTH;
  const int nch = (nk + 1) >> 1;
  for (int c0 = 0; c0 < nch; c0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int c = c0 + d;
      if (c >= nch) break;
      floatx16 t = acc;
      if (NP == 6) t = floatx16{};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s >= 2 && 2 * c + 1 >= nk) break;
        bf16x8 f[NPC];
#pragma unroll
        for (int q = 0; q < NPC; ++q) f[q] = *reinterpret_cast<const bf16x8*>(l + q * lpiece + (4 * c + s) * 16);
        const auto& g = w.v[d][s];
        auto mul = [&](int pa, int pb) {
          t = SA ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(g[pa], f[pb], t, 0, 0, 0)
                 : __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[pa], g[pb], t, 0, 0, 0);
        };
        mul(0, 0);
        if constexpr (NP >= 3) {
          mul(0, 1);
          mul(1, 0);
        }
        if constexpr (NP >= 6) {
          mul(0, 2);
          mul(1, 1);
          mul(2, 0);
        }
      }
      if (NP == 6 && c < nch - 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] += (double)t[r];
      } else {
        acc = t;
      }
      if (c + DEPTH < nch) {
        sweep_load(w, d, p, piece, c + DEPTH, nk);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// Eight operand values from their pieces, summed as dst_gemm.hip's fringe does.
template <int NPC, class acc_t>
__device__ __forceinline__ void join(const u32x4 (&w)[NPC], acc_t (&v)[8]) {
  auto lo = [](uint32_t u) { return __builtin_bit_cast(float, u << 16); };
  auto hi = [](uint32_t u) { return __builtin_bit_cast(float, u & 0xffff0000u); };
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[2 * e] = (acc_t)lo(w[0][e]);
    v[2 * e + 1] = (acc_t)hi(w[0][e]);
#pragma unroll
    for (int q = 1; q < NPC; ++q) {
      v[2 * e] += (acc_t)lo(w[q][e]);
      v[2 * e + 1] += (acc_t)hi(w[q][e]);
    }
  }
}

// Eight lanes share a dot product along k, lane l the chunks of eight k at 64 j + 8 l
// in order of j; their sums meet in a tree (dot_sum).  acc += v . f
template <class acc_t>
__device__ __forceinline__ void dot8(const acc_t (&v)[8], const acc_t* f, acc_t& acc) {
#pragma unroll
  for (int e = 0; e < 8; ++e) acc += v[e] * f[e];
}
template <class acc_t>
__device__ __forceinline__ float dot_sum(acc_t t) {
  t += __shfl_xor(t, 1);
  t += __shfl_xor(t, 2);
  t += __shfl_xor(t, 4);
  return (float)t;
}
template <int NPC>
using dot_t = typename std::conditional<NPC == 3, double, float>::type;
// Lane groups are counted from the last wave, whose tile is the first to be missing.
template <int NT>
__device__ __forceinline__ int dot_group() {
  return NT / 8 - 1 - ((int)threadIdx.x >> 3);
}

// The dots of a main stripe: its 32 rows by the one or two sweeping rows past the
// tiles, one a lane group.  The sweeping row is fetched a product ahead (three
// pieces: when it is used, the registers are taken).
constexpr int DOT_CHUNKS = (STRIPE_MAX_N + 63) / 64;
template <int NPC>
struct EdgeDot {
  u32x4 raw[DOT_CHUNKS][NPC];
};
template <int NPC, bool FRAG, int J0, int J1>
__device__ __forceinline__ void edge_load(EdgeDot<NPC>& d, const StripeOp& o, const uint16_t* B, int row) {
  const uint16_t* b = B + (FRAG ? frag_row(row, o.ldb) : row * o.ldb);
  const int klast = ((o.K + 7) & ~7) - 8;
#pragma unroll
  for (int j = J0; j < J1; ++j) {
    const int k1 = min(64 * j + ((int)threadIdx.x & 7) * 8, klast);  // (past the end: not used)
    const int k0 = FRAG ? frag_col(k1) : k1;
#pragma unroll
    for (int q = 0; q < NPC; ++q) d.raw[j][q] = *reinterpret_cast<const u32x4*>(b + q * o.b_piece + k0);
  }
}
template <int NPC, int NT, bool FRAG>
__device__ __forceinline__ void edge_fetch(EdgeDot<NPC>& d, const StripeOp& o, const uint16_t* B) {
  const int row = o.cut + dot_group<NT>() / SR;
  if (NPC < 3 && row < o.R) edge_load<NPC, FRAG, 0, DOT_CHUNKS>(d, o, B, row);
}
template <int NPC, int NT, bool FRAG, class Store>
__device__ __forceinline__ void edge_dots(EdgeDot<NPC>& d, const StripeOp& o, const uint16_t* B, const uint16_t* l,
                                          int pitch, int lpiece, Store store) {
  const int g = dot_group<NT>(), r = g & (SR - 1), row = o.cut + g / SR, l8 = threadIdx.x & 7;
  if (row < o.R) {  // (whole lane groups)
    dot_t<NPC> acc = 0;
    if constexpr (NPC == 3) edge_load<NPC, FRAG, 0, 3>(d, o, B, row);
#pragma unroll
    for (int j = 0; j < DOT_CHUNKS; ++j) {
      if constexpr (NPC == 3)
        if (j == 3) edge_load<NPC, FRAG, 3, DOT_CHUNKS>(d, o, B, row);
      const int k0 = 64 * j + l8 * 8;
      if (k0 < o.K) {
        u32x4 fw[NPC];
#pragma unroll
        for (int q = 0; q < NPC; ++q) fw[q] = *reinterpret_cast<const u32x4*>(l + q * lpiece + r * pitch + k0);
        dot_t<NPC> v[8], f[8];
        join(fw, f);
        join(d.raw[j], v);
        dot8(v, f, acc);
      }
    }
    const float v = dot_sum(acc);
    if (l8 == 0) store(r, row, v);
  }
}

// The dots of the one or two rows ix past the stripes (nr; f: their values, ldf apart)
// by all sweeping rows.  A wave takes 32 sweeping rows, whose fragments its lanes
// read as they lie: lane (row, half) holds the chunks of the lanes 2 i + half of
// eight, i = step mod 4, so the tree of dot_sum is one exchange and three sums.
template <int NPC, int NT, bool ROWS, class Store>
__device__ __forceinline__ void rest_dots(const StripeOp& o, const uint16_t* F, const uint16_t* rowm, int nr,
                                          const dot_t<NPC>* f, int ldf, Store store) {
  using acc_t = dot_t<NPC>;
  constexpr int SB = 8;  // steps in flight
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, steps = (o.K + 15) >> 4;
  // the sweeping rows past its tiles, eight lanes a dot (fetched first)
  const int g = dot_group<NT>(), re = nr == 1 ? 0 : g & 1, erow = o.cut + (nr == 1 ? g : g >> 1);
  EdgeDot<NPC> d;
  if (erow < o.R) {
    if (ROWS) edge_load<NPC, false, 0, DOT_CHUNKS>(d, o, rowm, erow);
    else edge_load<NPC, true, 0, DOT_CHUNKS>(d, o, F, erow);
  }
  for (int t = wave; 32 * t < o.cut; t += NT / 64) {
    const uint16_t* p = F + t * 32 * o.ldb + lane * 8;
    acc_t acc[2][4] = {};
    for (int s0 = 0; s0 < steps; s0 += SB) {
      u32x4 raw[SB][NPC];
#pragma unroll
      for (int i = 0; i < SB; ++i) {
        const int s = min(s0 + i, steps - 1);  // (past the end: not used)
#pragma unroll
        for (int q = 0; q < NPC; ++q) raw[i][q] = *reinterpret_cast<const u32x4*>(p + q * o.b_piece + s * 512);
      }
#pragma unroll
      for (int i = 0; i < SB; ++i) {
        const int k0 = 16 * (s0 + i) + 8 * half;
        if (k0 < o.K) {
          acc_t v[8];
          join(raw[i], v);
          dot8(v, f + k0, acc[0][i & 3]);
          if (nr > 1) dot8(v, f + ldf + k0, acc[1][i & 3]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (r < nr) {
        acc_t s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = acc[r][i] + __shfl_xor(acc[r][i], 32);
        const int row = 32 * t + (lane & 31);
        if (half == 0 && row < o.R) store(r, row, (float)((s[0] + s[1]) + (s[2] + s[3])));
      }
  }
  if (erow < o.R) {
    acc_t acc = 0;
#pragma unroll
    for (int j = 0; j < DOT_CHUNKS; ++j) {
      const int k0 = 64 * j + ((int)threadIdx.x & 7) * 8;
      if (k0 < o.K) {
        acc_t v[8];
        join(d.raw[j], v);
        dot8(v, f + re * ldf + k0, acc);
      }
    }
    const float v = dot_sum(acc);
    if ((threadIdx.x & 7) == 0) store(re, erow, v);
  }
}

// v as NPC bf16 pieces at o, `piece` elements apart
template <int NPC>
__device__ __forceinline__ void put_pieces(uint16_t* o, long piece, float v) {
#pragma unroll
  for (int q = 0; q < NPC; ++q) {
    const uint16_t b = bf16_rne(v);
    o[q * piece] = b;
    v = v - bf16_bits_to_f32(b);
  }
}
// v as the sum of its NPC pieces
template <int NPC>
__device__ __forceinline__ dot_t<NPC> joined(float v) {
  dot_t<NPC> s = 0;
#pragma unroll
  for (int q = 0; q < NPC; ++q) {
    const float b = bf16_bits_to_f32(bf16_rne(v));
    s = q == 0 ? (dot_t<NPC>)b : s + (dot_t<NPC>)b;
    v = v - b;
  }
  return s;
}
// row of register r of a 32 x 32 accumulator (its column: lane & 31)
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Zeros the columns [R, round32(R)) of the nr rows of a stripe of NPC pieces.
template <int NPC, int NT>
__device__ __forceinline__ void zero_tail(uint16_t* l, int pitch, int lpiece, int nr, int R) {
  const int n = round32(R) - R;
  for (int e = threadIdx.x; e < NPC * nr * n; e += NT) {
    const int q = e / (nr * n), rest = e - q * (nr * n), r = rest / n;
    l[q * lpiece + r * pitch + R + rest - r * n] = 0;
  }
}

struct Place {  // what a workgroup owns
  long z;
  int ix0, nr;     // its rows ix
  bool rest;       // the rows past the stripes: dots only
  int px, py, m;   // parities and mode of the plane
};

// F2's results, I1 and its stores, NP products.
template <int NPF, int NP, int NT, int D>
__device__ __forceinline__ void stripe_inverse(const StripeArgs& a, const Place& w, bool tile1, const floatx16& acc2,
                                               const double (&sum2)[16], EdgeDot<pieces_of(NPF)>& ef,
                                               const uint16_t* T, uint16_t* W,
                                               const float* la, float lb, float lamz) {
  constexpr int NPC = pieces_of(NP);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const StripeOp& f = a.op[1];
  const StripeOp& o = a.op[2];
  const int pT = stripe_pitch(f.K), pW = stripe_pitch(o.K), lW = SR * pW;
  const long vo = (o.b_par ? w.py : w.px) * o.b_var, vf = (f.b_par ? w.py : w.px) * f.b_var;
  const uint16_t* B = o.B + vo;
  const uint16_t* Bo = o.row + vo;
  const int nk = (o.K + 31) / 32;
  const int row0 = 32 * wave;
  const bool tile = row0 < o.cut;
  const uint16_t* p = B + row0 * o.ldb + lane * 8;
  Sweep<NP, D> sw;
  if (tile) sweep_start(sw, p, o.b_piece, nk);
  EdgeDot<NPC> eo;
  if (o.cut < o.R) edge_fetch<NPC, NT, false>(eo, o, Bo);
  if (tile1) {
    const int col = row0 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = acc_row(r, lane);
      float v = NPF == 6 ? (float)(sum2[r] + (double)acc2[r]) : acc2[r];
      const float q = v / ((la[row] - lamz) + lb);
      put_pieces<NPC>(W + row * pW + col, lW, col < f.R ? q : 0.0f);
    }
  }
  if (f.cut < f.R) {
    const float* lamB = a.lamB + w.py * a.lamB_var;
    edge_dots<pieces_of(NPF), NT, false>(ef, f, f.row + vf, T, pT, SR * pT, [&](int r, int s, float v) {
      put_pieces<NPC>(W + r * pW + s, lW, v / (la[r] + lamB[s] - lamz));
    });
    zero_tail<NPC, NT>(W, pW, lW, SR, f.R);
  }
  __syncthreads();
  uint16_t* O = a.O + w.z * a.o_batch + w.ix0;
  if (tile) {
    floatx16 acc = {};
    double sum[16] = {};
    sweep_run<true>(sw, p, o.b_piece, nk, W + (lane & 31) * pW + (lane >> 5) * 8, lW, acc, sum);
    const int col = lane & 31;
    const bool in = w.ix0 + col < a.R;
    if (w.ix0 + col < a.pad) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = row0 + acc_row(r, lane);
        const float v = NP == 6 ? (float)(sum[r] + (double)acc[r]) : acc[r];
        if (row < o.cut) put_pieces<NPC>(O + (long)row * a.ldo + col, a.o_piece, in ? v : 0.0f);
      }
    }
  }
  if (o.cut < o.R)
    edge_dots<NPC, NT, false>(eo, o, Bo, W, pW, lW, [&](int r, int s, float v) {
      if (w.ix0 + r < a.pad) put_pieces<NPC>(O + (long)s * a.ldo + r, a.o_piece, w.ix0 + r < a.R ? v : 0.0f);
    });
}

// The one or two rows ix past the stripes, by dots: F2 and I1 (NP products) from
// their row of T, two rows of doubles apart from it that of W.
template <int NPF, int NP, int NT>
__device__ __forceinline__ void rest_inverse(const StripeArgs& a, const Place& w, const dot_t<pieces_of(NPF)>* T,
                                             double* Wd, const float* la, float lamz) {
  constexpr int NPC = pieces_of(NP);
  const StripeOp& f = a.op[1];
  const StripeOp& o = a.op[2];
  const int lT = round32(f.K), lW = round32(o.K);
  const long vf = (f.b_par ? w.py : w.px) * f.b_var, vo = (o.b_par ? w.py : w.px) * o.b_var;
  const float* lamB = a.lamB + w.py * a.lamB_var;
  dot_t<NPC>* W = reinterpret_cast<dot_t<NPC>*>(Wd);
  rest_dots<pieces_of(NPF), NT, true>(f, f.B + vf, f.row + vf, w.nr, T, lT, [&](int r, int s, float v) {
    W[r * lW + s] = joined<NPC>(v / (la[r] + lamB[s] - lamz));
  });
  for (int e = threadIdx.x; e < w.nr * (lW - f.R); e += NT) W[e % w.nr * lW + f.R + e / w.nr] = 0;
  __syncthreads();
  uint16_t* O = a.O + w.z * a.o_batch + w.ix0;
  rest_dots<NPC, NT, true>(o, o.B + vo, o.row + vo, w.nr, W, lW,
                     [&](int r, int s, float v) { put_pieces<NPC>(O + (long)s * a.ldo + r, a.o_piece, v); });
  const int n = a.pad - a.R;  // zero columns of every row
  for (int e = threadIdx.x; e < n * o.R; e += NT) {
    const int s = e / n;
    put_pieces<NPC>(O + (long)s * a.ldo + w.nr + (e - s * n), a.o_piece, 0.0f);
  }
}

// The stripe of Sx into LDS.
template <int NPC, int NT>
__device__ __forceinline__ void stage_stripe(const StripeArgs& a, const Place& w, uint16_t* S0) {
  const StripeOp& o = a.op[0];
  const int tid = threadIdx.x, p0 = stripe_pitch(o.K), l0 = SR * p0;
  const uint16_t* S = a.S + (a.s_par ? w.py : w.px) * a.s_var + (long)w.ix0 * a.lds;
  const int c8 = round32(o.K) / 8, n = NPC * w.nr * c8;
  constexpr int LB = 4;
  for (int e0 = tid; e0 < n; e0 += LB * NT) {
    u32x4 v[LB];
    int at[LB];
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int e = min(e0 + i * NT, n - 1);
      const int q = e / (w.nr * c8), rest = e - q * (w.nr * c8), r = rest / c8, k = (rest - r * c8) * 8;
      v[i] = *reinterpret_cast<const u32x4*>(S + q * a.s_piece + (long)r * a.lds + k);
      at[i] = q * l0 + r * p0 + k;
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) *reinterpret_cast<u32x4*>(S0 + at[i]) = v[i];
  }
}

// NPF: products of F1 and F2; NPI: most products of I1 (a mode with fewer runs
// three); NT: 64 threads for each of the most 32-row tiles of a sweep; D: the most
// chunks of a contraction.
template <int NPF, int NPI, int NT, int D>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void dst_stripe_kernel(StripeArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  __shared__ float la[SR];
  constexpr int NPC = pieces_of(NPF);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  Place w;
  {
    // each XCD takes a contiguous run of stripes (a plane's share its sweeps)
    const int T = gridDim.x, b = blockIdx.x, xcd = b & 7, per = T >> 3, extra = T & 7;
    const int t = xcd * per + min(xcd, extra) + (b >> 3);
    const int z = t / a.stripes, s = t - z * a.stripes;
    w.z = z;
    w.ix0 = min(SR * s, a.cut);
    w.rest = SR * s >= a.cut;
    w.nr = w.rest ? a.R - a.cut : SR;
    int blk = 0;
    w.m = z;
    if (a.fold_P) {
      blk = z / a.fold_P;
      w.m = z - blk * a.fold_P;
    }
    w.px = blk & 1;
    w.py = blk >> 1;
  }
  const StripeOp& o = a.op[0];
  const StripeOp& f = a.op[1];
  const int p0 = stripe_pitch(o.K), pT = stripe_pitch(f.K);
  const int l0 = SR * p0, lT = SR * pT;
  uint16_t* S0 = lds;  // the stripe of Sx, later of W
  uint16_t* T = lds + std::max(NPC * l0, pieces_of(NPI) * SR * stripe_pitch(a.op[2].K));

  const float lamz = a.lam[w.m];
  const bool lo = a.hp ? a.hp[w.m] != 0 : ((a.hp_bits >> w.m) & 1) != 0;
  const int np = lo ? a.np_lo : a.np_hi;
  const uint16_t* B = o.B + w.z * o.b_plane;
  const float* lam_a = a.lamA + w.px * a.lam_var;
  if (w.rest) {
    // rows of values (not pieces): Sx, T, W, each two rows of doubles at most
    using acc_t = dot_t<NPC>;
    const int lS = round32(o.K), lF = round32(f.K);
    double* base = reinterpret_cast<double*>(lds);
    acc_t* fS = reinterpret_cast<acc_t*>(base);
    acc_t* fT = reinterpret_cast<acc_t*>(base + 2 * lS);
    const float la_mine = lam_a[min(w.ix0 + (tid & (SR - 1)), a.R - 1)];
    const uint16_t* S = a.S + (a.s_par ? w.py : w.px) * a.s_var + (long)w.ix0 * a.lds;
    for (int e = tid; e < w.nr * (lS / 8); e += NT) {
      const int r = e / (lS / 8), k = (e - r * (lS / 8)) * 8;
      u32x4 raw[NPC];
#pragma unroll
      for (int q = 0; q < NPC; ++q) raw[q] = *reinterpret_cast<const u32x4*>(S + q * a.s_piece + (long)r * a.lds + k);
      acc_t v[8];
      join(raw, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) fS[r * lS + k + i] = v[i];
    }
    if (tid < SR) la[tid] = la_mine;
    __syncthreads();
    rest_dots<NPC, NT, false>(o, B, nullptr, w.nr, fS, lS, [&](int r, int s, float v) { fT[r * lF + s] = joined<NPC>(v); });
    for (int e = tid; e < w.nr * (lF - o.R); e += NT) fT[e % w.nr * lF + o.R + e / w.nr] = 0;
    __syncthreads();
    double* fW = base + 2 * lS + 2 * lF;
    if (NPI == 1) rest_inverse<NPF, 1, NT>(a, w, fT, fW, la, lamz);
    else if (NPI == 3 || np == 3) rest_inverse<NPF, 3, NT>(a, w, fT, fW, la, lamz);
    else rest_inverse<NPF, 6, NT>(a, w, fT, fW, la, lamz);
    return;
  }

  // F1's sweep, then the stripe of Sx
  const int row0 = 32 * wave;
  const uint16_t* p = B + row0 * o.ldb + lane * 8;
  const int nk0 = (o.K + 31) / 32;
  const bool tile0 = row0 < o.cut;
  Sweep<NPF, D> sw;
  if (tile0) sweep_start(sw, p, o.b_piece, nk0);
  EdgeDot<NPC> eo, ef;
  if (o.cut < o.R) edge_fetch<NPC, NT, true>(eo, o, B);
  const int colB = row0 + (lane & 31);  // this lane's column of a tile of F1 or F2
  const float lb = a.lamB[w.py * a.lamB_var + min(colB, f.R - 1)];
  const float la_mine = lam_a[min(w.ix0 + (tid & (SR - 1)), a.R - 1)];
  stage_stripe<NPC, NT>(a, w, S0);
  if (tid < SR) la[tid] = la_mine;
  __syncthreads();
  // F1
  const int nk1 = (f.K + 31) / 32;
  const uint16_t* Bf = f.B + (f.b_par ? w.py : w.px) * f.b_var;
  const uint16_t* pf = Bf + row0 * f.ldb + lane * 8;
  Sweep<NPF, D> sf;
  const bool tile1 = row0 < f.cut;
  floatx16 acc = {};
  double sum[16] = {};
  if (tile0) sweep_run<false>(sw, p, o.b_piece, nk0, S0 + (lane & 31) * p0 + (lane >> 5) * 8, l0, acc, sum);
  if (tile1) sweep_start(sf, pf, f.b_piece, nk1);
  if (f.cut < f.R) edge_fetch<NPC, NT, false>(ef, f, f.row + (f.b_par ? w.py : w.px) * f.b_var);
  if (tile0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = NPF == 6 ? (float)(sum[r] + (double)acc[r]) : acc[r];
      put_pieces<NPC>(T + acc_row(r, lane) * pT + colB, lT, colB < o.R ? v : 0.0f);
    }
  }
  if (o.cut < o.R) {
    edge_dots<NPC, NT, true>(eo, o, B, S0, p0, l0,
                       [&](int r, int s, float v) { put_pieces<NPC>(T + r * pT + s, lT, v); });
    zero_tail<NPC, NT>(T, pT, lT, SR, o.R);
  }
  __syncthreads();

  // F2
  acc = floatx16{};
#pragma unroll
  for (int r = 0; r < 16; ++r) sum[r] = 0.0;
  if (tile1) sweep_run<false>(sf, pf, f.b_piece, nk1, T + (lane & 31) * pT + (lane >> 5) * 8, lT, acc, sum);
  if (NPI == 1) stripe_inverse<NPF, 1, NT, D>(a, w, tile1, acc, sum, ef, T, S0, la, lb, lamz);
  else if (NPI == 3 || np == 3) stripe_inverse<NPF, 3, NT, D>(a, w, tile1, acc, sum, ef, T, S0, la, lb, lamz);
  else stripe_inverse<NPF, 6, NT, D>(a, w, tile1, acc, sum, ef, T, S0, la, lb, lamz);
}

// dst: the rows x ld (multiples of 32) matrices of src in fragment order.
__global__ __launch_bounds__(256) void fragment_order_kernel(const uint16_t* src, uint16_t* dst, long rows, long ld,
                                                             long n) {
  const long e = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (e >= n) return;
  const long m = e / (rows * ld), at = e - m * rows * ld;
  const long frag = at / 512;
  const int l = (int)(at - frag * 512) / 8;
  const long tile = frag / (ld / 16), step = frag - tile * (ld / 16);
  *reinterpret_cast<u32x4*>(dst + e) =
      *reinterpret_cast<const u32x4*>(src + m * rows * ld + (tile * 32 + (l & 31)) * ld + step * 16 + (l >> 5) * 8);
}

int most_products(const GemmArgs& g) { return std::max(g.np_lo, g.np_hi); }
size_t stripe_lds(const GemmArgs& f1, const GemmArgs& f2, const GemmArgs& i1) {
  const int pf = pieces_of(most_products(f1)), pi = pieces_of(most_products(i1));
  return (size_t)SR * 2 *
         (std::max(pf * stripe_pitch(f1.K), pi * stripe_pitch(i1.K)) + pf * stripe_pitch(f2.K));
}
int tiles_of(int cut) { return (cut + 31) / 32; }

template <int NPF, int NPI>
void launch(const StripeArgs& a, int waves, int nk, int blocks, size_t lds, hipStream_t st) {
  // (with rows past the tiles, four more waves for their dots)
  if (waves <= 4 && nk <= 4)
    hipLaunchKernelGGL((dst_stripe_kernel<NPF, NPI, 256, 2>), dim3(blocks), dim3(256), lds, st, a);
  else if (nk <= 6)
    hipLaunchKernelGGL((dst_stripe_kernel<NPF, NPI, 512, 3>), dim3(blocks), dim3(512), lds, st, a);
  else
    hipLaunchKernelGGL((dst_stripe_kernel<NPF, NPI, 512, 4>), dim3(blocks), dim3(512), lds, st, a);
}
constexpr size_t STRIPE_LDS_MAX = 128 * 1024;
template <int NPF, int NPI>
hipError_t raise() {
  for (const void* f : {reinterpret_cast<const void*>(dst_stripe_kernel<NPF, NPI, 256, 2>),
                        reinterpret_cast<const void*>(dst_stripe_kernel<NPF, NPI, 512, 3>),
                        reinterpret_cast<const void*>(dst_stripe_kernel<NPF, NPI, 512, 4>)}) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, STRIPE_LDS_MAX);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
}  // namespace

hipError_t launch_fragment_order(const uint16_t* src, uint16_t* dst, long rows, long ld, int matrices, hipStream_t st) {
  const long n = rows * ld * matrices;
  hipLaunchKernelGGL(fragment_order_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, st, src, dst, rows, ld,
                     n);
  return hipGetLastError();
}

hipError_t prepare_dst_stripe() {
  static OncePerDevice once;
  return once([] {
    hipError_t e = raise<3, 1>();
    if (e == hipSuccess) e = raise<3, 6>();
    if (e == hipSuccess) e = raise<6, 6>();
    return e;
  });
}

bool dst_stripe_fits(const GemmArgs& f1, const GemmArgs& f2, const GemmArgs& i1) {
  if (f1.Xf || !f2.Sfrag || !i1.Sfrag) return false;
  const int npf = most_products(f1), npi = most_products(i1);
  const bool kinds = f1.np_lo == f1.np_hi && ((npf == 3 && npi == 1) || (npf == 3 && npi == 6) || (npf == 6 && npi == 6));
  // every six-product transform with its FP64 windows, the others without
  const bool sums = (npf != 6 || (f1.acc64 && f2.acc64)) && (npi != 6 || i1.acc64);
  const GemmCut c1 = gemm_cut(f1.RA, f1.RB, f1.K, 1), c2 = gemm_cut(f2.RA, f2.RB, f2.K, 1),
                c3 = gemm_cut(i1.RA, i1.RB, i1.K, 1);
  const int tiles = std::max(tiles_of(c1.bm), std::max(tiles_of(c2.bm), tiles_of(c3.am)));
  return kinds && sums && c1.am == c2.am && c1.am == c3.bm && tiles <= 8 && stripe_lds(f1, f2, i1) <= STRIPE_LDS_MAX;
}

void launch_dst_stripe(const GemmArgs& f1, const GemmArgs& f2, const GemmArgs& i1, int batch, hipStream_t st) {
  StripeArgs a{};
  const GemmCut c1 = gemm_cut(f1.RA, f1.RB, f1.K, 1), c2 = gemm_cut(f2.RA, f2.RB, f2.K, 1),
                c3 = gemm_cut(i1.RA, i1.RB, i1.K, 1);
  a.op[0] = StripeOp{f1.Xb, nullptr, round32(f1.K), f1.x_piece, f1.x_batch, 0, 0, f1.K, f1.RB, c1.bm};
  a.op[1] = StripeOp{f2.Sfrag, f2.Sb, f2.lds, f2.s_piece, 0, f2.s_var, f2.s_par, f2.K, f2.RB, c2.bm};
  a.op[2] = StripeOp{i1.Sfrag, i1.Sb, i1.lds, i1.s_piece, 0, i1.s_var, i1.s_par, i1.K, i1.RA, c3.am};
  a.S = f1.Sb;
  a.lds = f1.lds;
  a.s_piece = f1.s_piece;
  a.s_var = f1.s_var;
  a.s_par = f1.s_par;
  a.R = f1.RA;
  a.cut = c1.am;
  a.lamA = f2.lamA;
  a.lamB = f2.lamB;
  a.lam = f2.lam;
  a.lam_var = f2.lam_var;
  a.lamB_var = f2.lamB_var;
  a.hp = i1.hp;
  a.hp_bits = i1.hp_bits;
  a.np_lo = i1.np_lo;
  a.np_hi = i1.np_hi;
  a.O = i1.Ob;
  a.ldo = i1.ldo;
  a.o_piece = i1.o_piece;
  a.o_batch = i1.o_batch;
  a.pad = i1.RBpad;
  a.fold_P = f1.fold_P;
  a.stripes = tiles_of(c1.am) + (c1.am < f1.RA ? 1 : 0);
  const int waves = std::max(tiles_of(c1.bm), std::max(tiles_of(c2.bm), tiles_of(c3.am)));
  const int nk = (std::max(f1.K, std::max(f2.K, i1.K)) + 31) / 32;
  const int blocks = a.stripes * batch;
  const size_t lds = stripe_lds(f1, f2, i1);
  const int npf = most_products(f1), npi = most_products(i1);
  if (npf == 6) launch<6, 6>(a, waves, nk, blocks, lds, st);
  else if (npi == 6) launch<3, 6>(a, waves, nk, blocks, lds, st);
  else launch<3, 1>(a, waves, nk, blocks, lds, st);
}

}  // namespace somax
