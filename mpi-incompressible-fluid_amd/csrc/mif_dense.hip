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
// V_MFMA_*_16X16X4 tiles: 16 lines by 16 coefficients, K = 4.
//
// Slot order, scaling, the fused divergence, unpack and defect passes are
// those of mif_fft_pow2.hip.
//
// Measured against the mixed-radix kernel (x / y / z pass, us): 128^3 nodes
// between walls, FP64 406 / 407 / 806 -> 17 / 16 / 26; 201^3, FP64 150 / 164 /
// 294 -> 65 / 59 / 111, FP32 115 / 132 / 234 -> 42 / 41 / 77; 256^3, FP64 629 /
// 645 / 1220 -> 116 / 109 / 208; 480 x 480 x 199 points, periodic, FP64 661 /
// 675 / 13572 -> 531 / 516 / 538.  It was faster at every length measured
// from 20 to 481, smooth or not, so every length that one workgroup's 16
// waves can hold takes it (dense_plan); longer ones stay with mif_fft.hip.
// At 256 nodes the products take 4.3 GFLOP per pass (about 55 us at the FP64
// rate) and the memory 60 us: the two phases of a workgroup overlap only
// through the other three workgroups of its CU.
//
// Work split: a workgroup owns 16 lines; each wave owns one of the
// H / 16 row tiles (H = R/2 + 1) of both matrices, for all lines (on x there
// may be waves beyond those, launch_dense_pass).  The
// folded lines (e and o) sit in LDS, the matrices are read fragment by
// fragment from global memory (they are shared by all workgroups and stay in
// L2; a fragment is one 16-byte load per lane in FP64).
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
template <typename T, int AXIS, int MODE, int IO, typename TV>
__global__ void __launch_bounds__(1024) k_dense(DGrid g, DensePlan P, const T* __restrict__ M, SpectralScale sc,
                                               T* __restrict__ B, long bp0, long bplane, FusedIO io) {
  using namespace dense;
  using Op = Mm<T>;
  using Acc = typename Op::acc;
  using Frag = typename Op::frag;
  extern __shared__ __align__(16) unsigned char smem[];
  const int H = P.H, KS = P.KS, KP = 8 * P.KS, n = P.n, R = P.R;
  const bool periodic = P.periodic;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nthr = blockDim.x, W = nthr >> 6;
  const int n0 = g.npts[0], n1 = g.npts[1], n2 = g.npts[2];
  // e and o: [row][line] on the strided axes, [line][row] on x
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
  // spectral slots of row r of the even and odd parts (-1: none)
  auto slot_e = [&](int r) -> int {
    const int s = periodic ? r : 2 * r;
    return (periodic ? 2 * r <= n : s < n) ? s : -1;
  };
  auto slot_o = [&](int r) -> int {
    if (periodic) return r >= 1 && 2 * r < n ? n - r : -1;
    return 2 * r + 1 < n ? 2 * r + 1 : -1;
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
    // and is dropped by its caller)
    auto value = [&](int l, int m) -> T {
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
          if (b >= 0) {
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
      T e = 0, o = 0;
      if (j < H) {
        const T a = value(l, j);
        if (self(j)) {
          e = ok ? a : (T)0;
        } else {
          const T b = value(l, R - j);
          e = ok ? a + b : (T)0;
          o = ok ? a - b : (T)0;
        }
      }
      Eo[at(j, l)] = e;
      Eo[half + at(j, l)] = o;
    }
  } else if constexpr (AXIS == 0) {
    for (int q = t; q < NL * KP; q += nthr) {
      const int l = (q * rkp) >> 22, r = q - l * KP;
      const long b = lbase[l];
      const int se = slot_e(r), so = slot_o(r);
      const T e = B[b >= 0 && se >= 0 ? b + se : 0], o = B[b >= 0 && so >= 0 ? b + so : 0];
      Eo[at(r, l)] = b >= 0 && se >= 0 ? e : (T)0;
      Eo[half + at(r, l)] = b >= 0 && so >= 0 ? o : (T)0;
    }
  } else {
    const int l = t & (NL - 1), step = nthr / NL;
    const int i = bx * NL + l;
    const bool ok = i < n0;
    const T* src = B + (ok ? (AXIS == 1 ? i + bplane * by : i + bp0 * by) : 0);
    // U rows in flight per thread, from always-valid addresses
    constexpr int U = 4;
    for (int q = t / NL; q < KP; q += U * step) {
      T a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int r = q + u * step;
        int s1, s2;
        if (MODE == 1) {
          s1 = slot_e(r);
          s2 = slot_o(r);
          s1 = s1 < 0 ? 0 : s1;
          s2 = s2 < 0 ? 0 : s2;
        } else {
          s1 = r < H ? r : 0;
          s2 = self(s1) ? s1 : R - s1;
        }
        a[u] = src[s1 * ms];
        b[u] = src[s2 * ms];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int r = q + u * step;
        if (r >= KP) break;
        T e, o;
        if (MODE == 1) {
          e = ok && slot_e(r) >= 0 ? a[u] : (T)0;
          o = ok && slot_o(r) >= 0 ? b[u] : (T)0;
        } else {
          const bool in = ok && r < H;
          e = in ? (self(r) ? a[u] : a[u] + b[u]) : (T)0;
          o = in && !self(r) ? a[u] - b[u] : (T)0;
        }
        Eo[at(r, l)] = e;
        Eo[half + at(r, l)] = o;
      }
    }
  }
  __syncthreads();

  // ---- products: acc[.][.][0] even part, [1] odd part, each in two chains.
  // FP64: one per K step of a fragment.  FP32 (kBlocked): every eight terms
  // are summed from zero and added to alternating totals, so that the longest
  // chain of roundings is 8 + H/16 terms: the solve's error on a line of
  // 120-283 nodes is then that of the mixed-radix transform (2e-7; 3e-7 with
  // the FP64 scheme)
  Acc acc[2][2];
#pragma unroll
  for (int c = 0; c < 4; c++) acc[c >> 1][c & 1] = Acc{0, 0, 0, 0};
  auto multiply = [&](const T* Me) {
    const T* Mo = Me + (long)P.MT * KS * 128;
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c >> 1][c & 1] = Acc{0, 0, 0, 0};
    const Frag* fe = (const Frag*)Me + (long)wave * KS * 64 + lane;
    const Frag* fo = (const Frag*)Mo + (long)wave * KS * 64 + lane;
    Frag ne = fe[0], no = fo[0];
    auto step = [&](int s, int par) {
      const Frag ce = ne, co = no;
      const int s1 = s + 1 < KS ? s + 1 : s;  // next fragments requested before this step's products
      ne = fe[s1 * 64];
      no = fo[s1 * 64];
      T le[2], lo[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int o = at(8 * s + 4 * h + (lane >> 4), lane & 15);
        le[h] = Eo[o];
        lo[h] = Eo[half + o];
      }
      auto mul = [&](T f, T x, Acc c) { return AXIS == 0 ? Op::mma(x, f, c) : Op::mma(f, x, c); };
      if constexpr (Op::kBlocked) {
        const Acc z = {0, 0, 0, 0};
        acc[0][par] += mul(ce[1], le[1], mul(ce[0], le[0], z));
        acc[1][par] += mul(co[1], lo[1], mul(co[0], lo[0], z));
      } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          acc[0][h] = mul(ce[h], le[h], acc[0][h]);
          acc[1][h] = mul(co[h], lo[h], acc[1][h]);
        }
      }
    };
    for (int s = 0; s < KS; s += 2) {
      step(s, 0);
      if (s + 1 < KS) step(s + 1, 1);
    }
    acc[0][0] += acc[0][1];
    acc[1][0] += acc[1][1];
  };
  const long msize = 2L * P.MT * KS * 128;  // one direction's two matrices
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
      const int se = slot_e(k), so = slot_o(k);
      T e = 0, o = 0;
      if (se >= 0) {
        const double s = i == 0 && by == 0 && se == 0 ? 0.0 : (1.0 / (lxy + sc.lam[2][se])) * sc.inv_norm;
        e = acc[0][0][r] * (T)s;
      }
      if (so >= 0) o = acc[1][0][r] * (T)((1.0 / (lxy + sc.lam[2][so])) * sc.inv_norm);
      Eo[at(k, l)] = e;
      Eo[half + at(k, l)] = o;
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
        const T a = acc[0][0][r], b = acc[1][0][r];
        if (MODE == 0) {
          const int se = slot_e(k), so = slot_o(k);
          if (se >= 0) dst[se * ms] = a;
          if (so >= 0) dst[so * ms] = b;
        } else if (k < H) {
          dst[k * ms] = a + b;
          if (!self(k)) dst[(R - k) * ms] = a - b;
        }
      }
    }
  } else {
    // lines back to LDS, so that whole rows are stored
    const int pl = 2 * px;
    __syncthreads();
    const int k = 16 * wave + (lane & 15);
    const int se = slot_e(k), so = slot_o(k);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      T* x = Eo + Op::row(r, lane) * pl;
      const T a = acc[0][0][r], b = acc[1][0][r];
      if (MODE == 0) {
        if (se >= 0) x[se] = a;
        if (so >= 0) x[so] = b;
      } else if (k < H) {
        x[k] = a + b;
        if (!self(k)) x[R - k] = a - b;
      }
    }
    __syncthreads();
    // a group of 2^lg lanes stores one line
    const int lg = H <= 16 ? 4 : (H <= 32 ? 5 : 6);
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
bool dense_plan(int n, bool periodic, DensePlan* P) {
  P->n = n;
  P->periodic = periodic;
  P->R = periodic ? n : n - 1;
  P->H = P->R / 2 + 1;
  P->MT = (P->H + 15) / 16;
  P->KS = (P->H + 7) / 8;
  // one wave per row tile, at most 16 waves
  return n >= 2 && P->MT <= 16;
}

size_t dense_table_elems(const DensePlan& P) { return 4 * (size_t)P.MT * P.KS * 128; }

// The four matrices (forward even, forward odd, inverse even, inverse odd),
// each as MT x KS fragments of 64 lanes x 2 elements: element h of lane q of
// fragment (t, s) is M[16 t + q % 16][8 s + 4 h + q / 16], zero outside.
void dense_table(const DensePlan& P, double* out64, float* out32) {
  const int n = P.n, R = P.R;
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
  const size_t msize = (size_t)P.MT * P.KS * 128;
  // element (row, col) of matrix mat
  auto put = [&](int mat, int row, int col, long double v) {
    const size_t lane = (row & 15) + 16 * (col & 3);
    const size_t e = mat * msize + (((size_t)(row >> 4) * P.KS + (col >> 3)) * 64 + lane) * 2 + ((col >> 2) & 1);
    out64[e] = (double)v;
    if (out32) out32[e] = (float)v;
  };
  for (size_t e = 0; e < 4 * msize; e++) out64[e] = 0;
  if (out32)
    for (size_t e = 0; e < 4 * msize; e++) out32[e] = 0;
  for (int r = 0; r < P.H; r++)  // spectral row
    for (int odd = 0; odd < 2; odd++) {
      const long k = P.periodic ? r : 2L * r + odd;
      if (P.periodic ? (odd ? r < 1 || 2 * r >= n : 2 * r > n) : k >= n) continue;
      const bool edge = P.periodic ? r == 0 || 2 * r == n : k == 0 || k == R;  // weight 1 in the inverse sum
      long a = 0;                                                             // j * k modulo the table
      for (int j = 0; j < P.H; j++) {
        const long double f = P.periodic && odd ? -s[a] : c[a];
        put(odd, r, j, !P.periodic && j > 0 ? 2 * f : f);
        put(2 + odd, j, r, edge ? f : 2 * f);
        a += k;
        if (a >= mod) a -= mod;
      }
    }
}

namespace dense {

size_t lds_bytes(const DensePlan& P, int axis, size_t esize) {
  const size_t kp = 8 * (size_t)P.KS;
  return 2 * esize * NL * (axis == 0 ? kp + (esize == 8 ? Mm<double>::kPadX : Mm<float>::kPadX) : kp);
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
  auto* kernel = k_dense<T, AXIS, MODE, IO, TV>;
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
