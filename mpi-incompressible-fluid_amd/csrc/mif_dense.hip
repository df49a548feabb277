// mif_dense.hip -- transform passes as matrix products on the matrix cores,
// for line lengths without a specialised kernel in mif_fft_pow2.hip.
//
// A line length such as 95, 101 or 191 intervals has a large prime factor,
// and a Stockham transform spends R operations per element in a radix-R
// stage by direct sums.  Here a whole pass is a product with the transform's
// matrix, halved by its symmetry: with R = n (periodic) or R = n - 1 (node
// Neumann), e_j = x_j + x_{R-j} and o_j = x_j - x_{R-j} (j <= R/2),
//   periodic, forward   r_k = sum_j e_j cos(2 pi j k / n)
//                       i_k = -sum_j o_j sin(2 pi j k / n)
//   Neumann, forward    Y_{2q}   = sum_j w_j e_j cos(2 pi j q / R)
//                       Y_{2q+1} = sum_j w_j o_j cos(pi j (2q + 1) / R)
// (w_0 = 1, else 2), and the inverse runs the other way, x_j = a_j + b_j and
// x_{R-j} = a_j - b_j with a from the even part (r_k or Y_{2q}) and b from
// the odd part.  That is n multiply-adds per element and pass, on
// V_MFMA_*_16X16X4 tiles: 16 lines by 16 coefficients, K = 4.  A periodic line
// of even length folds once more about n/4: with h = n/2, the terms of even
// and odd k are sums over e_j + e_{h-j}, e_j - e_{h-j}, o_j - o_{h-j} and
// o_j + o_{h-j} (j <= h/2), four parts of a quarter of the line each and n/2
// multiply-adds per element (kQuadMin).
//
// Slot order, scaling, the fused divergence, unpack and defect passes are
// those of mif_fft_pow2.hip.
//
// Measured against the mixed-radix kernel (x / y / z pass, us): 128^3 nodes
// between walls, FP64 406 / 407 / 806 -> 17 / 16 / 26; 201^3, FP64 150 / 164 /
// 294 -> 65 / 59 / 111, FP32 115 / 132 / 234 -> 42 / 41 / 77; 256^3, FP64 629 /
// 645 / 1220 -> 116 / 109 / 208; 480 x 480 x 199 points, periodic, FP64 661 /
// 675 / 13572 -> 531 / 516 / 538.  It was faster at every length measured,
// smooth or not, 2 to 24 points with 256 on the other axes (whole solve, walls
// / periodic, FP64: 2 points 167 -> 42 / 39 -> 28 us, 16 points 226 -> 56 / 81
// -> 43; up to 8 times in FP32) and 20 to 481 on all, so every line whose row
// tiles in two parts one workgroup's 16 waves can hold takes it: up to 512 wall
// nodes or 511 periodic points (dense_plan).  Longer ones stay with mif_fft.hip,
// also the even periodic ones that four parts would hold.
// At 256 nodes the products take 4.3 GFLOP per pass (about 55 us at the FP64
// rate) and the memory 60 us: the two phases of a workgroup overlap only
// through the other three workgroups of its CU.
//
// Work split: a workgroup owns 16 lines; each wave owns one of the H / 16 row
// tiles (H = R/2 + 1, or n/4 + 1) of every part's matrix, for all lines (on x
// there may be waves beyond those, launch_dense_pass).  The folded lines sit
// in LDS, the matrices are read fragment by fragment from global memory (they
// are shared by all workgroups and stay in L2; a fragment is one 16-byte load
// per lane in FP64).
#include <algorithm>
#include <cmath>
#include <vector>

#include "mif_kernels.h"

namespace mif {

namespace dense {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mm;
template <>
struct Mm<double> {
  typedef d4 acc;
  typedef double frag __attribute__((ext_vector_type(2)));
  __device__ static inline acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of element r of a lane's accumulator (its column is lane % 16)
  __device__ static inline int row(int r, int lane) { return (lane >> 4) + 4 * r; }
  static constexpr int kPadX = 2;
  static constexpr bool kBlocked = false;
};
template <>
struct Mm<float> {
  typedef f4 acc;
  typedef float frag __attribute__((ext_vector_type(2)));
  __device__ static inline acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int r, int lane) { return 4 * (lane >> 4) + r; }
  static constexpr int kPadX = 4;
  static constexpr bool kBlocked = true;
};

// Lines of a workgroup: one MFMA tile.  Two tiles per workgroup (half the
// matrix reads, half the workgroups in flight) measured slower at every size:
// 181^3 FP64 z pass 78.9 -> 96.7 us, 301 x 301 x 200 y pass 152 -> 168 us,
// 64^3 8.8 -> 12.4 us.
constexpr int NL = 16;

// What the x pass loads or stores instead of its buffer (FusedIO).
enum { IO_PLAIN = 0, IO_FIELD = 1, IO_FIELD_DC = 2, IO_DEFECT = 3, IO_PACK = 4 };

}  // namespace dense

// MODE 0: forward, 1: inverse, 2: forward + scale + inverse (axis 2).
// QUAD: four parts (a periodic line of even length), else two.
template <typename T, int AXIS, int MODE, int IO, typename TV, bool QUAD>
__global__ void __launch_bounds__(1024) k_dense(DGrid g, DensePlan P, const T* __restrict__ M, SpectralScale sc,
                                               T* __restrict__ B, long bp0, long bplane, FusedIO io) {
  using namespace dense;
  using Op = Mm<T>;
  using Acc = typename Op::acc;
  using Frag = typename Op::frag;
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NP = QUAD ? 4 : 2;
  const int H = P.H, KS = P.KS, KP = 8 * P.KS, n = P.n, R = P.R, h = n >> 1;
  const bool periodic = P.periodic;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nthr = blockDim.x, W = nthr >> 6;
  const int n0 = g.npts[0], n1 = g.npts[1], n2 = g.npts[2];
  // the parts: [row][line] on the strided axes, [line][row] on x
  const int px = KP + Op::kPadX;
  const int half = AXIS == 0 ? NL * px : KP * NL;
  T* const Eo = (T*)smem;
  auto at = [&](int k, int l) -> int {
    return AXIS == 0 ? l * px + k : k * NL + l;
  };
  int bx, by;
  {
    const int tile = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    bx = tile % gridDim.x;
    by = tile / gridDim.x;
  }
  const long ms = AXIS == 0 ? 1 : (AXIS == 1 ? bp0 : bplane);
  // element j of the physical line and its mirror image; self: it has none
  auto self = [&](int j) -> bool { return 2 * j == R || (periodic && j == 0); };
  // spectral slot of row r of part p (-1: none)
  auto slot = [&](int p, int r) -> int {
    if constexpr (QUAD) {
      const int k = 2 * r + (p & 1);
      if (p < 2) return k <= h ? k : -1;
      return k >= 1 && k < h ? n - k : -1;
    } else {
      if (periodic) return p == 0 ? (2 * r <= n ? r : -1) : (r >= 1 && 2 * r < n ? n - r : -1);
      return 2 * r + p < n ? 2 * r + p : -1;
    }
  };
  // The parts of row j from its points: x_j and x_{R-j}; QUAD: x_j, x_{n-j},
  // x_{h-j}, x_{h+j} (points that coincide come as zeros)
  auto fold = [&](int j, const T (&x)[NP], T (&f)[NP]) {
    if constexpr (QUAD) {
      const bool mid = 2 * j == h;
      const T e0 = x[0] + x[1], o0 = j == 0 ? (T)0 : x[0] - x[1], e1 = x[2] + x[3], o1 = j == 0 ? (T)0 : x[2] - x[3];
      f[0] = e0 + e1;
      f[1] = mid ? (T)0 : e0 - e1;
      f[2] = mid ? (T)0 : o0 - o1;
      f[3] = o0 + o1;
    } else {
      f[0] = x[0] + x[1];
      f[1] = self(j) ? (T)0 : x[0] - x[1];
    }
  };
  // whether point q of a row's NP points is one of its own, and its index
  auto own = [&](int j, int q) -> bool {
    if constexpr (QUAD) return q == 0 || (q == 1 ? j > 0 : 2 * j != h && (q == 2 || j > 0));
    else return q == 0 || !self(j);
  };
  auto point = [&](int j, int q) -> int {
    if constexpr (QUAD) return q == 0 ? j : (q == 1 ? n - j : (q == 2 ? h - j : h + j));
    else return q == 0 ? j : R - j;
  };
  // the value at point q of row j from the parts of the inverse
  auto unfold = [&](const T (&f)[NP], int q) -> T {
    if constexpr (QUAD) {
      const T a = q < 2 ? f[0] + f[1] : f[0] - f[1], b = q < 2 ? f[2] + f[3] : f[3] - f[2];
      return q & 1 ? a - b : a + b;
    } else {
      return q ? f[0] - f[1] : f[0] + f[1];
    }
  };

  // ---- load, folded
  // x pass: lines are rows (j, k), their points dealt to the threads in order;
  // q / KP by its reciprocal, exact for q < 16 KP <= 4096
  const unsigned rkp = (1u << 22) / KP + 1;
  __shared__ long lrow[AXIS == 0 ? NL : 1][4];
  __shared__ long lbase[AXIS == 0 ? NL : 1];
  __shared__ double lwt[IO == IO_FIELD_DC ? NL : 1];
  double dc_s = 0, dc_w = 0;
  if constexpr (AXIS == 0) {
    if (t < NL) {
      const int r = bx * NL + t;
      const bool ok = r < n1 * n2;
      const int rj = ok ? r % n1 : 0, rk = ok ? r / n1 : 0;
      lbase[t] = ok ? bp0 * rj + bplane * rk : -1;
      if constexpr (IO == IO_FIELD || IO == IO_FIELD_DC || IO == IO_PACK) {
        const int j = rj + g.olo[1], k = rk + g.olo[2];
        if constexpr (MODE == 0) {
          lrow[t][0] = ok ? io.L.idx(g.olo[0], j, k) : -1;
        } else {
          // the rows the line is written to: owner row, periodic images
          const int N1 = g.N[1], N2 = g.N[2];
          int js[2] = {j, -1}, ks[2] = {k, -1};
          if (g.periodic[1]) js[1] = j == 1 ? N1 - 1 : (j == N1 - 2 ? 0 : -1);
          if (g.periodic[2]) ks[1] = k == 1 ? N2 - 1 : (k == N2 - 2 ? 0 : -1);
          for (int q = 0; q < 4; q++)
            lrow[t][q] = ok && js[q & 1] >= 0 && ks[q >> 1] >= 0 ? io.L.idx(0, js[q & 1], ks[q >> 1]) : -1;
        }
      }
      if constexpr (IO == IO_FIELD_DC) lwt[t] = ok ? owner_weight(g, 1, rj) * owner_weight(g, 2, rk) : 0.0;
      if constexpr (IO == IO_DEFECT) {
        lrow[t][0] = bp0 * nb(g, 1, rj, -1) + bplane * rk;
        lrow[t][1] = bp0 * nb(g, 1, rj, 1) + bplane * rk;
        lrow[t][2] = bp0 * rj + bplane * nb(g, 2, rk, -1);
        lrow[t][3] = bp0 * rj + bplane * nb(g, 2, rk, 1);
      }
    }
    __syncthreads();
  }
  if constexpr (AXIS == 0 && MODE == 0) {
    const double rmean = IO == IO_DEFECT ? io.bmean->s1 / io.bmean->s2 : 0.0;
    const double ihx2 = 1.0 / (g.h[0] * g.h[0]), ihy2 = 1.0 / (g.h[1] * g.h[1]), ihz2 = 1.0 / (g.h[2] * g.h[2]);
    // the value of point m of line l (a line outside the grid reads row 0
    // and is dropped by its caller); mine: the caller is the point's only one
    auto value = [&](int l, int m, bool mine) -> T {
      const long b = lbase[l];
      if constexpr (IO == IO_PLAIN) {
        return B[(b >= 0 ? b : 0) + m];
      } else if constexpr (IO == IO_PACK) {
        return ((const T*)io.P)[(b >= 0 ? lrow[l][0] : 0) + m];
      } else if constexpr (IO == IO_DEFECT) {
        // r = (b - mean) - L phi in FP64 with the 7-point operator
        const float* F = io.phi32;
        const long row = b >= 0 ? b : 0;
        const long o = row + m;
        const double c = F[o];
        const double lx = ((double)F[row + nb(g, 0, m, -1)] - 2 * c + (double)F[row + nb(g, 0, m, 1)]) * ihx2;
        const double ly = ((double)F[lrow[l][0] + m] - 2 * c + (double)F[lrow[l][1] + m]) * ihy2;
        const double lz = ((double)F[lrow[l][2] + m] - 2 * c + (double)F[lrow[l][3] + m]) * ihz2;
        return (T)((io.b64[o] - rmean) - (lx + ly + lz));
      } else {
        // div(u) / dt
        const TV *u = (const TV*)io.u, *v = (const TV*)io.v, *w = (const TV*)io.w;
        const long o = b >= 0 ? lrow[l][0] + m : 0;
        const double du_dx = ((double)u[o + 1] - (double)u[o]) * g.one_over_h[0];
        const double dv_dy = ((double)v[o + io.L.PX] - (double)v[o]) * g.one_over_h[1];
        const double dw_dz = ((double)w[o + io.L.plane] - (double)w[o]) * g.one_over_h[2];
        const double bv = (du_dx + dv_dy + dw_dz) / io.dt;
        if constexpr (IO == IO_FIELD_DC) {
          if (b >= 0 && mine) {
            io.b64[b + m] = bv;
            const double wgt = owner_weight(g, 0, m) * lwt[l];
            dc_s += wgt * bv;
            dc_w += wgt;
          }
        }
        return (T)bv;
      }
    };
    for (int q = t; q < NL * KP; q += nthr) {
      const int l = (q * rkp) >> 22, j = q - l * KP;
      const bool ok = lbase[l] >= 0;
      T f[NP] = {};
      if (j < H) {
        T x[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
          const bool mine = own(j, p);
          const T v = value(l, mine ? point(j, p) : j, mine);
          x[p] = mine ? v : (T)0;
        }
        fold(j, x, f);
      }
#pragma unroll
      for (int p = 0; p < NP; p++) Eo[p * half + at(j, l)] = ok ? f[p] : (T)0;
    }
  } else if constexpr (AXIS == 0) {
    for (int q = t; q < NL * KP; q += nthr) {
      const int l = (q * rkp) >> 22, r = q - l * KP;
      const long b = lbase[l];
      T f[NP];
#pragma unroll
      for (int p = 0; p < NP; p++) {
        const int s = slot(p, r);
        f[p] = B[b >= 0 && s >= 0 ? b + s : 0];
      }
#pragma unroll
      for (int p = 0; p < NP; p++) Eo[p * half + at(r, l)] = b >= 0 && slot(p, r) >= 0 ? f[p] : (T)0;
    }
  } else {
    const int l = t & (NL - 1), step = nthr / NL;
    const int i = bx * NL + l;
    const bool ok = i < n0;
    const T* src = B + (ok ? (AXIS == 1 ? i + bplane * by : i + bp0 * by) : 0);
    // U rows in flight per thread, from always-valid addresses
    constexpr int U = 4;
    for (int q = t / NL; q < KP; q += U * step) {
      T a[U][NP];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int r = q + u * step, j = r < H ? r : 0;
#pragma unroll
        for (int p = 0; p < NP; p++) {
          const int s = MODE == 1 ? max(slot(p, r), 0) : (own(j, p) ? point(j, p) : j);
          a[u][p] = src[s * ms];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int r = q + u * step;
        if (r >= KP) break;
        T f[NP];
        if (MODE == 1) {
#pragma unroll
          for (int p = 0; p < NP; p++) f[p] = ok && slot(p, r) >= 0 ? a[u][p] : (T)0;
        } else {
          const bool in = ok && r < H;
          T x[NP];
#pragma unroll
          for (int p = 0; p < NP; p++) x[p] = in && own(r, p) ? a[u][p] : (T)0;
          fold(r, x, f);
        }
#pragma unroll
        for (int p = 0; p < NP; p++) Eo[p * half + at(r, l)] = f[p];
      }
    }
  }
  __syncthreads();

  // ---- products: acc[part][chain].  Two parts: two chains each, FP64 one
  // per K step of a fragment, FP32 (kBlocked) every eight terms summed from
  // zero and added to alternating totals, so that the longest chain of
  // roundings is 8 + H/16 terms: the solve's error on a line of 120-283 nodes
  // is then that of the mixed-radix transform (2e-7; 3e-7 with the FP64
  // scheme).  Four parts: their rows are half as long, one chain each.
  constexpr int NC = QUAD ? 1 : 2;
  Acc acc[NP][NC];
#pragma unroll
  for (int p = 0; p < NP; p++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[p][c] = Acc{0, 0, 0, 0};
  auto multiply = [&](const T* Md) {
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int c = 0; c < NC; c++) acc[p][c] = Acc{0, 0, 0, 0};
    const Frag* fr = (const Frag*)Md + (long)wave * KS * 64 + lane;
    const long part = (long)P.MT * KS * 64;
    Frag next[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) next[p] = fr[p * part];
    auto step = [&](int s, int par) {
      Frag cur[NP];
      const int s1 = s + 1 < KS ? s + 1 : s;  // next fragments requested before this step's products
#pragma unroll
      for (int p = 0; p < NP; p++) {
        cur[p] = next[p];
        next[p] = fr[p * part + s1 * 64];
      }
      T ln[NP][2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int o = at(8 * s + 4 * h + (lane >> 4), lane & 15);
#pragma unroll
        for (int p = 0; p < NP; p++) ln[p][h] = Eo[p * half + o];
      }
      auto mul = [&](T f, T x, Acc c) { return AXIS == 0 ? Op::mma(x, f, c) : Op::mma(f, x, c); };
      if constexpr (Op::kBlocked) {
        const Acc z = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < NP; p++)
          acc[p][QUAD ? 0 : par] += mul(cur[p][1], ln[p][1], mul(cur[p][0], ln[p][0], z));
      } else {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int p = 0; p < NP; p++) acc[p][QUAD ? 0 : h] = mul(cur[p][h], ln[p][h], acc[p][QUAD ? 0 : h]);
      }
    };
    for (int s = 0; s < KS; s += 2) {
      step(s, 0);
      if (s + 1 < KS) step(s + 1, 1);
    }
    if constexpr (NC == 2)
#pragma unroll
      for (int p = 0; p < NP; p++) acc[p][0] += acc[p][NC - 1];
  };
  const long msize = (long)NP * P.MT * KS * 128;  // one direction's matrices
  // the x passes may have waves without a row tile: they load and store only
  if (AXIS != 0 || wave < P.MT) multiply(M + (MODE == 1 ? msize : 0));

  if constexpr (MODE == 2) {
    // scale every mode by 1/((lx+ly+lz) * norm), constant mode -> 0, and
    // hand the coefficients to the inverse products
    __syncthreads();
    const int l = lane & 15, i = bx * NL + l;
    const double lxy = sc.lam[0][i < n0 ? i : 0] + sc.lam[1][by];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int k = 16 * wave + Op::row(r, lane);
      if (k >= KP) continue;
#pragma unroll
      for (int p = 0; p < NP; p++) {
        const int sl = slot(p, k);
        T x = 0;
        if (sl >= 0) {
          const double s =
              p == 0 && i == 0 && by == 0 && sl == 0 ? 0.0 : (1.0 / (lxy + sc.lam[2][sl])) * sc.inv_norm;
          x = acc[p][0][r] * (T)s;
        }
        Eo[p * half + at(k, l)] = x;
      }
    }
    __syncthreads();
    multiply(M + msize);
  }

  // ---- store
  if constexpr (AXIS != 0) {
    const int i = bx * NL + (lane & 15);
    if (i < n0) {
      T* dst = B + (AXIS == 1 ? i + bplane * by : i + bp0 * by);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = 16 * wave + Op::row(r, lane);
        T f[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) f[p] = acc[p][0][r];
#pragma unroll
        for (int p = 0; p < NP; p++) {
          if (MODE == 0) {
            const int sl = slot(p, k);
            if (sl >= 0) dst[sl * ms] = f[p];
          } else if (k < H && own(k, p)) {
            dst[point(k, p) * ms] = unfold(f, p);
          }
        }
      }
    }
  } else {
    // lines back to LDS, so that whole rows are stored
    const int pl = NP * px;
    __syncthreads();
    const int k = 16 * wave + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      T* x = Eo + Op::row(r, lane) * pl;
      T f[NP];
#pragma unroll
      for (int p = 0; p < NP; p++) f[p] = acc[p][0][r];
#pragma unroll
      for (int p = 0; p < NP; p++) {
        if (MODE == 0) {
          const int sl = slot(p, k);
          if (sl >= 0) x[sl] = f[p];
        } else if (k < H && own(k, p)) {
          x[point(k, p)] = unfold(f, p);
        }
      }
    }
    __syncthreads();
    // a group of 2^lg lanes stores one line
    const int lg = n <= 32 ? 4 : (n <= 64 ? 5 : 6);
    const int m0 = t & ((1 << lg) - 1);
    for (int l = t >> lg; l < NL; l += nthr >> lg) {
      const long b = lbase[l];
      if (b < 0) continue;
      const T* x = Eo + l * pl;
      if constexpr (MODE == 1 && (IO == IO_FIELD || IO == IO_FIELD_DC)) {
        TV* F = (TV*)io.P;
        const int N0 = g.N[0];
        for (int m = m0; m < n; m += 1 << lg) {
          const int i = m + g.olo[0];
          const int i2 = g.periodic[0] ? (i == 1 ? N0 - 1 : (i == N0 - 2 ? 0 : -1)) : -1;
          TV val = (TV)x[m];
          if constexpr (IO == IO_FIELD_DC) {
            // phi = phi_0 + delta in FP64, stored in the field's precision
            val = (TV)((double)x[m] + (double)io.add32[b + m]);
            const double wgt = owner_weight(g, 0, m) * lwt[l];
            dc_s += wgt * (double)val;
            dc_w += wgt;
          }
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const long rb = lrow[l][q];
            if (rb >= 0) {
              F[rb + i] = val;
              if (i2 >= 0) F[rb + i2] = val;
            }
          }
        }
      } else {
        for (int m = m0; m < n; m += 1 << lg) B[b + m] = x[m];
      }
    }
  }
  if constexpr (IO == IO_FIELD_DC) {
    // the workgroup's (W.x, W.1) into its slot of io.partial
    for (int off = 32; off > 0; off >>= 1) {
      dc_s += __shfl_down(dc_s, off, 64);
      dc_w += __shfl_down(dc_w, off, 64);
    }
    __shared__ double red[2][16];
    if (lane == 0) {
      red[0][wave] = dc_s;
      red[1][wave] = dc_w;
    }
    __syncthreads();
    if (t == 0) {
      Red3 s{0, 0, 0};
      for (int q = 0; q < W; q++) {
        s.s1 += red[0][q];
        s.s2 += red[1][q];
      }
      io.partial[bx + gridDim.x * by] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// Periodic lines of even length from which four parts pay: half the products,
// but half the row tiles too, and shorter ones leave the matrix cores waiting
// for loads either way.  Two -> four parts (divergence / unpack / y / z pass,
// us): FP64 78^3 points 9.8 / 9.2 / 8.0 / 11.7 -> 10.6 / 9.9 / 8.8 / 14.0, 102^3
// 15.0 / 12.9 / 11.5 / 18.3 -> 15.5 / 11.8 / 11.5 / 18.9, 122^3 20.1 / 16.1 /
// 15.8 / 24.7 -> 18.8 / 14.3 / 14.1 / 21.9, 180^3 49.0 / 44.0 / 41.8 / 77.4 ->
// 47.2 / 32.9 / 30.5 / 51.0, 302^3 336 / 248 / 215 / 409 -> 273 / 175 / 136 /
// 324; FP32 102^3 11.7 / 10.8 / 9.3 / 14.5 -> 12.1 / 10.6 / 9.4 / 15.0, 122^3
// 14.6 / 13.2 / 11.5 / 19.0 -> 13.9 / 11.7 / 10.7 / 17.2, 302^3 203 / 165 / 144
// / 290 -> 157 / 102 / 89 / 179.
constexpr int kQuadMin = 112;

bool dense_plan(int n, bool periodic, DensePlan* P) {
  P->n = n;
  P->periodic = periodic;
  P->quad = periodic && n % 2 == 0 && n >= kQuadMin;
  P->R = periodic ? n : n - 1;
  P->H = (P->quad ? n / 2 : P->R) / 2 + 1;
  P->MT = (P->H + 15) / 16;
  P->KS = (P->H + 7) / 8;
  // one wave per row tile, at most 16 waves in two parts (longer lines in four
  // parts have not been measured)
  return n >= 2 && P->R / 2 + 1 <= 256;
}

static size_t matrix_elems(const DensePlan& P) { return (size_t)P.MT * P.KS * 128; }
static int parts(const DensePlan& P) { return P.quad ? 4 : 2; }

size_t dense_table_elems(const DensePlan& P) { return 2 * parts(P) * matrix_elems(P); }

// The matrices, forward then inverse, one per part (even, odd; QUAD: of even
// and odd k), each as MT x KS fragments of 64 lanes x 2 elements: element h of
// lane q of fragment (t, s) is M[16 t + q % 16][8 s + 4 h + q / 16], zero
// outside.
void dense_table(const DensePlan& P, double* out64, float* out32) {
  const int n = P.n, R = P.R, np = parts(P);
  const long mod = P.periodic ? n : 2L * R;  // angles are 2 pi m / mod
  std::vector<long double> c(mod), s(mod);
  for (long m = 0; m < mod; m++) {
    const long double ang = 2.0L * 3.141592653589793238462643383279502884L * (long double)m / (long double)mod;
    c[m] = cosl(ang);
    s[m] = sinl(ang);
  }
  // exact zeros where the angle is a multiple of a quarter turn
  for (long m = 0; m < mod; m++) {
    if (4 * m == mod || 4 * m == 3 * mod) c[m] = 0;
    if (m == 0 || 2 * m == mod) s[m] = 0;
  }
  const size_t msize = matrix_elems(P);
  // element (row, col) of matrix mat
  auto put = [&](int mat, int row, int col, long double v) {
    const size_t lane = (row & 15) + 16 * (col & 3);
    const size_t e = mat * msize + (((size_t)(row >> 4) * P.KS + (col >> 3)) * 64 + lane) * 2 + ((col >> 2) & 1);
    out64[e] = (double)v;
    if (out32) out32[e] = (float)v;
  };
  for (size_t e = 0; e < 2 * np * msize; e++) out64[e] = 0;
  if (out32)
    for (size_t e = 0; e < 2 * np * msize; e++) out32[e] = 0;
  for (int r = 0; r < P.H; r++)  // spectral row
    for (int part = 0; part < np; part++) {
      const bool sine = P.periodic && part >= np / 2;
      const long k = P.quad ? 2L * r + (part & 1) : (P.periodic ? r : 2L * r + part);
      if (P.periodic ? (sine ? k < 1 || 2 * k >= n : 2 * k > n) : k >= n) continue;
      const bool edge = P.periodic ? k == 0 || 2 * k == n : k == 0 || k == R;  // weight 1 in the inverse sum
      long a = 0;                                                             // j * k modulo the table
      for (int j = 0; j < P.H; j++) {
        const long double f = sine ? -s[a] : c[a];
        put(part, r, j, !P.periodic && j > 0 ? 2 * f : f);
        put(np + part, j, r, edge ? f : 2 * f);
        a += k;
        if (a >= mod) a -= mod;
      }
    }
}

namespace dense {

size_t lds_bytes(const DensePlan& P, int axis, size_t esize) {
  const size_t kp = 8 * (size_t)P.KS;
  return parts(P) * esize * NL * (axis == 0 ? kp + (esize == 8 ? Mm<double>::kPadX : Mm<float>::kPadX) : kp);
}

}  // namespace dense

template <typename T, int AXIS, int MODE, int IO, typename TV>
static void launch_dense_pass(const DGrid& g, const DensePlan& P, const SpectralScale& sc, T* B, long bp0, long bplane,
                            const FusedIO& io, hipStream_t st) {
  const T* M = sizeof(T) == 8 ? (const T*)P.M64 : (const T*)P.M32;
  constexpr int nl = dense::NL;
  const size_t lds = dense::lds_bytes(P, AXIS, sizeof(T));
  const dim3 grd = AXIS == 0
                       ? dim3((unsigned)(((long)g.npts[1] * g.npts[2] + nl - 1) / nl), 1, 1)
                       : dim3((unsigned)((g.npts[0] + nl - 1) / nl), AXIS == 1 ? g.npts[2] : g.npts[1], 1);
  auto* kernel = P.quad ? k_dense<T, AXIS, MODE, IO, TV, true> : k_dense<T, AXIS, MODE, IO, TV, false>;
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  // One wave per row tile; on x more, which load and store lines only.  There
  // a thread's loads wait for one another, point after point, so the pass
  // lasts as long as one thread has points.  A power of two keeps the waves
  // even over the 16 lines of the store; few workgroups get a thread per point
  // of their lines, as long as the device then holds them all at once (4096
  // waves).  Divergence / unpack pass, one wave per row tile -> this rule and
  // the points spread evenly over the threads (us): FP64 31^3 8.4 / 8.2 -> 6.3
  // / 6.2, 65^3 11.9 / 11.9 -> 10.5 / 8.5, 96^3 15.8 / 13.2 -> 12.9 / 10.9,
  // 151^3 42.7 / 31.2 -> 32.6 / 25.9, 181^3 61.6 / 45.0 -> 50.3 / 42.4, 301^3
  // 351 / 256 -> 333 / 242; FP32 151^3 31.7 / 24.6 -> 24.6 / 20.5, 301^3 246 /
  // 172 -> 210 / 159.
  int waves = P.MT;
  if (AXIS == 0) {
    while (waves & (waves - 1)) waves++;
    waves = std::max(waves, std::min({16, 2 * P.KS, 4096 / (int)grd.x}));
  }
  kernel<<<grd, 64 * waves, lds, st>>>(g, P, M, sc, B, bp0, bplane, io);
}

template <typename T>
void launch_dense(const DGrid& g, int axis, int mode, const DensePlan& P, const SpectralScale& sc, T* B, long bp0,
                  long bplane, const FusedIO* io, hipStream_t st) {
  using namespace dense;
  const FusedIO none{};
  if (axis == 1) {
    if (mode == 0) launch_dense_pass<T, 1, 0, IO_PLAIN, T>(g, P, sc, B, bp0, bplane, none, st);
    else launch_dense_pass<T, 1, 1, IO_PLAIN, T>(g, P, sc, B, bp0, bplane, none, st);
  } else if (axis == 2) {
    launch_dense_pass<T, 2, 2, IO_PLAIN, T>(g, P, sc, B, bp0, bplane, none, st);
  } else if (!io) {
    if (mode == 0) launch_dense_pass<T, 0, 0, IO_PLAIN, T>(g, P, sc, B, bp0, bplane, none, st);
    else launch_dense_pass<T, 0, 1, IO_PLAIN, T>(g, P, sc, B, bp0, bplane, none, st);
  } else if (io->pack && mode == 0) {
    launch_dense_pass<T, 0, 0, IO_PACK, T>(g, P, sc, B, bp0, bplane, *io, st);
  } else if (sizeof(T) == 4 && io->res) {
    if constexpr (sizeof(T) == 4) launch_dense_pass<T, 0, 0, IO_DEFECT, T>(g, P, sc, B, bp0, bplane, *io, st);
  } else if (sizeof(T) == 4 && io->dc) {
    if constexpr (sizeof(T) == 4) {
      if (mode == 0) launch_dense_pass<T, 0, 0, IO_FIELD_DC, T>(g, P, sc, B, bp0, bplane, *io, st);
      else launch_dense_pass<T, 0, 1, IO_FIELD_DC, T>(g, P, sc, B, bp0, bplane, *io, st);
    }
  } else if (sizeof(T) == 8 && io->fields_fp32) {
    if constexpr (sizeof(T) == 8) {
      if (mode == 0) launch_dense_pass<T, 0, 0, IO_FIELD, float>(g, P, sc, B, bp0, bplane, *io, st);
      else launch_dense_pass<T, 0, 1, IO_FIELD, float>(g, P, sc, B, bp0, bplane, *io, st);
    }
  } else {
    if (mode == 0) launch_dense_pass<T, 0, 0, IO_FIELD, T>(g, P, sc, B, bp0, bplane, *io, st);
    else launch_dense_pass<T, 0, 1, IO_FIELD, T>(g, P, sc, B, bp0, bplane, *io, st);
  }
}

int dense_x_blocks(const DGrid& g) { return (int)(((long)g.npts[1] * g.npts[2] + dense::NL - 1) / dense::NL); }

template void launch_dense<double>(const DGrid&, int, int, const DensePlan&, const SpectralScale&, double*, long, long,
                                   const FusedIO*, hipStream_t);
template void launch_dense<float>(const DGrid&, int, int, const DensePlan&, const SpectralScale&, float*, long, long,
                                  const FusedIO*, hipStream_t);

}  // namespace mif
