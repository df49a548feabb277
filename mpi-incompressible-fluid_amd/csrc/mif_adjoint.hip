// mif_adjoint.hip -- adjoint of one RK3 + projection step (no counterpart in
// the reference, which has no adjoint).
//
// The forward step (src/Timestep.cpp:97-141) is, per stage: a stencil update
// with the momentum right-hand side N (quadratic in the velocity,
// include/MomentumEquation.h:43-255) and the pressure gradient; the boundary
// map (Dirichlet faces are constants, periodic ghosts copy interior points,
// src/VelocityTensor.cpp:36-233); the divergence, the spectral solve M, the
// unpack with periodic images; p += phi; u -= dt_s grad(phi) on interior
// points.  Each kernel below is the transpose of a run of those linear maps,
// written as a gather (each output point sums the contributions that the
// forward scatters into it), so no atomics are needed and results are
// deterministic.  One adjoint stage is three kernels around the solve:
//   k_adj_rhs   phi_bar = p_bar - dt_s G^T y_bar, then U^T and W^-1: the
//               packed right-hand side of M^T = W M W^-1 (W = trapezoid
//               weights of the owner nodes)
//   (spectral solve)
//   k_adj_zb    z_bar = B^T (y_bar + D^T W psi / dt_s): the adjoint of the
//               stage output before its boundary map; also N_bar, the adjoint
//               of N's output, and per-block sums of z_bar (body force)
//   k_adj_xb    x_bar = z_bar + J_N(X)^T N_bar (the transposed linearised
//               convection plus the diffusion stencil), and p_bar += b G^T z_bar
//               for the stage's pressure-gradient term
// z_bar and N_bar vanish outside the component interiors (the forward
// computes N and writes the stage update only there), which lets k_adj_xb
// read neighbours without interior tests.
#include <algorithm>

#include "mif_kernels.h"

namespace mif {

__device__ inline bool adj_interior(const DGrid& g, int c, int i, int j, int k) {
  int e[3];
  extents(g, c, e);
  return i >= 1 && j >= 1 && k >= 1 && i <= e[0] - 2 && j <= e[1] - 2 && k <= e[2] - 2;
}

__device__ inline bool in_field(const DGrid& g, int s, int i, int j, int k) {
  int e[3];
  extents(g, s, e);
  return i >= 0 && j >= 0 && k >= 0 && i < e[0] && j < e[1] && k < e[2];
}

__device__ inline double trap_weight(const DGrid& g, int a, int i) {
  if (g.periodic[a]) return 1.0;
  return (i == 0 || i == g.npts[a] - 1) ? 0.5 : 1.0;
}

// Points of a periodic axis that hold copies of index P (P itself first):
// 1 -> also s-1, s-2 -> also 0, on an axis of extent s.
__device__ inline int images(const DGrid& g, int a, int P, int s, int out[2]) {
  out[0] = P;
  int n = 1;
  if (g.periodic[a]) {
    if (P == 1) out[n++] = s - 1;
    if (P == s - 2) out[n++] = 0;
  }
  return n;
}

// ---------------------------------------------------------------------------
// k_adj_rhs: for each owner node o of the packed solve,
//   B(o) = sum over the pressure points R holding o (o and its periodic
//          images) of phi_bar(R), divided by W(o),
//   phi_bar(R) = p_bar(R) + dt_s sum_c (y_bar_c(R + e_c) - y_bar_c(R)) / h_c
// with y_bar_c taken on the interior of component c only.
// ---------------------------------------------------------------------------
// A wave takes 64 points of a row at a time, so that the row's tests and
// addresses are uniform and the loads contiguous (128^3 FP64 right-hand side:
// 38.5 -> 32.8 us against one point per thread with its own index division).
struct RowItem {
  int i, j, k;
};
// Item w of rows of n0 points, n1 rows per plane: nx = ceil(n0 / 64) items per row.
__device__ inline RowItem row_item(int w, int nx, int n1) {
  const int row = w / nx, iw = w - row * nx;
  const int k = row / n1;
  return {64 * iw + (int)(threadIdx.x & 63), row - k * n1, k};
}

template <typename T>
__global__ void __launch_bounds__(256) k_adj_rhs(DGrid g, Layout L, const T* __restrict__ P, AdjVec Y, double dts,
                                                 T* __restrict__ B, long bp0, long bplane, int nx, int items) {
  const int w0 = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (w0 >= items) return;
  const RowItem q = row_item(w0, nx, g.npts[1]);
  const int a = q.i, b = q.j, c = q.k;
  if (a >= g.npts[0]) return;
  const int O[3] = {a + g.olo[0], b + g.olo[1], c + g.olo[2]};
  const long off[3] = {1, L.PX, L.plane};
  // R and R + e_c lie inside the padded array for every pressure point R,
  // so all seven loads are issued unconditionally and the interior masks
  // apply to the values
  auto phib = [&](int r0, int r1, int r2) -> double {
    const int R[3] = {r0, r1, r2};
    const long o = L.idx(r0, r1, r2);
    double hi[3], lo[3];
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
      const T* F = (const T*)Y.f[cc];
      hi[cc] = (double)F[o + off[cc]];
      lo[cc] = (double)F[o];
    }
    const double pv = (double)P[o];
    double acc = 0;
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
      int Rp[3] = {r0, r1, r2};
      Rp[cc] += 1;
      double d = 0;
      if (adj_interior(g, cc, Rp[0], Rp[1], Rp[2])) d += hi[cc];
      if (adj_interior(g, cc, R[0], R[1], R[2])) d -= lo[cc];
      acc += d * g.one_over_h[cc];
    }
    return pv + dts * acc;
  };
  double s = phib(O[0], O[1], O[2]);
  int opts[3][2], nopt[3];
  bool single = true;
  for (int ax = 0; ax < 3; ax++) {
    nopt[ax] = images(g, ax, O[ax], g.N[ax], opts[ax]);
    single = single && nopt[ax] == 1;
  }
  if (!single) {
    for (int qa = 0; qa < nopt[0]; qa++)
      for (int qb = 0; qb < nopt[1]; qb++)
        for (int qc = 0; qc < nopt[2]; qc++)
          if (qa + qb + qc > 0) s += phib(opts[0][qa], opts[1][qb], opts[2][qc]);
  }
  // (the weight is a power of two: its reciprocal is exact)
  const double w = trap_weight(g, 0, a) * trap_weight(g, 1, b) * trap_weight(g, 2, c);
  B[a + bp0 * b + bplane * c] = (T)(w == 1.0 ? s : s * (w == 0.5 ? 2.0 : (w == 0.25 ? 4.0 : 8.0)));
}

// ---------------------------------------------------------------------------
// k_adj_zb: interior points Q of the three components c,
//   z_bar_c(Q) = sum over the points g holding Q (Q and its periodic ghost
//                copies) of y_bar_c(g) + (Wpsi(g - e_c) - Wpsi(g)) / (dt_s h_c)
//   N_bar_c(Q) = alpha z_bar_c(Q) + beta Zo_c(Q)
// with Wpsi = W * psi on owner nodes (zero elsewhere), and per workgroup the
// partial sums of z_bar_c weighted by fcoef, stored (accumulate = 0) or added
// to the workgroup's slot (accumulate = 1: the later stages of one adjoint
// step, launched with the same grid, so slot b always belongs to workgroup b).
// Waves take 64 points of a row at a time (row_item), all components together,
// so that psi is read once for the three; hd holds 1 / (dt_s h_c).  128^3 FP64:
// 91 -> 62 us against one component and point per thread (10 to 13 words per
// point at about 3 TB/s).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_adj_zb(DGrid g, Layout L, AdjVec Y, const T* __restrict__ Bpsi, long bp0,
                                                long bplane, double hd0, double hd1, double hd2, AdjVec Zb, AdjVec Nb,
                                                AdjVec Zo, double alpha, double beta, double fcoef, int accumulate,
                                                double* __restrict__ partial, int jmax, int nx, int items) {
  const double hd[3] = {hd0, hd1, hd2};
  // W * psi at pressure point P (zero off the owner nodes); the load reads
  // a valid address either way
  auto wpsi = [&](int pi, int pj, int pk) -> double {
    const int q0 = pi - g.olo[0], q1 = pj - g.olo[1], q2 = pk - g.olo[2];
    const bool ok = (unsigned)q0 < (unsigned)g.npts[0] && (unsigned)q1 < (unsigned)g.npts[1] &&
                    (unsigned)q2 < (unsigned)g.npts[2];
    const double v = (double)Bpsi[ok ? q0 + bp0 * q1 + bplane * q2 : 0];
    const double w = trap_weight(g, 0, q0) * trap_weight(g, 1, q1) * trap_weight(g, 2, q2);
    return ok ? w * v : 0.0;
  };
  double part[3] = {0, 0, 0};
  const int nw = gridDim.x * 4;
  for (int it = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); it < items; it += nw) {
    const RowItem r = row_item(it, nx, jmax);
    const int i = r.i + 1, j = r.j + 1, k = r.k + 1;
    const long o = L.idx(min(i, L.PX - 1), j, k);
    const double here = wpsi(i, j, k);
    const double below[3] = {wpsi(i - 1, j, k), wpsi(i, j - 1, k), wpsi(i, j, k - 1)};
    T y[3], zo[3] = {(T)0, (T)0, (T)0};
#pragma unroll
    for (int c = 0; c < 3; c++) y[c] = ((const T*)Y.f[c])[o];
    // the later stage's z_bar enters only with beta != 0 (stage 2): the
    // other stages skip its load (a uniform branch)
    if (beta != 0.0) {
#pragma unroll
      for (int c = 0; c < 3; c++) zo[c] = ((const T*)Zo.f[c])[o];
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      int e[3];
      extents(g, c, e);
      if (i > e[0] - 2 || j > e[1] - 2 || k > e[2] - 2) continue;
      double s = (double)(T)((double)y[c] + (below[c] - here) * hd[c]);
      int opts[3][2], nopt[3];
      const int Q[3] = {i, j, k};
      bool single = true;
      for (int ax = 0; ax < 3; ax++) {
        nopt[ax] = images(g, ax, Q[ax], e[ax], opts[ax]);
        single = single && nopt[ax] == 1;
      }
      if (!single) {
        for (int qa = 0; qa < nopt[0]; qa++)
          for (int qb = 0; qb < nopt[1]; qb++)
            for (int qc = 0; qc < nopt[2]; qc++) {
              if (qa + qb + qc == 0) continue;
              const int g0 = opts[0][qa], g1 = opts[1][qb], g2 = opts[2][qc];
              const double d = (wpsi(g0 - (c == 0), g1 - (c == 1), g2 - (c == 2)) - wpsi(g0, g1, g2)) * hd[c];
              s += (double)(T)((double)((const T*)Y.f[c])[L.idx(g0, g1, g2)] + d);
            }
      }
      const T z = (T)s;
      ((T*)Zb.f[c])[o] = z;
      double nbv = alpha * (double)z;
      if (beta != 0.0) nbv += beta * (double)zo[c];
      ((T*)Nb.f[c])[o] = (T)nbv;
      part[c] += (double)z;
    }
  }
  __shared__ double sh[3][4];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    for (int off = 32; off > 0; off >>= 1) part[c] += __shfl_down(part[c], off, 64);
    if ((threadIdx.x & 63) == 0) sh[c][threadIdx.x >> 6] = part[c];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int c = threadIdx.x;
    const double v = fcoef * (sh[c][0] + sh[c][1] + sh[c][2] + sh[c][3]);
    double* slot = &partial[c * gridDim.x + blockIdx.x];
    *slot = accumulate ? *slot + v : v;
  }
}

// out[c] (= or +=) sum of the nblk partials of component c: one workgroup of
// 1024 threads, each loading its kAdjSumPer values per component at once,
// then a fixed-order wave and workgroup reduction (deterministic).
constexpr int kAdjSumThreads = 1024, kAdjSumPer = 4;
static_assert(kAdjSumThreads * kAdjSumPer >= kAdjMaxBlocks, "k_adj_sum covers every partial");
__global__ void __launch_bounds__(kAdjSumThreads) k_adj_sum(const double* __restrict__ partial, int nblk,
                                                            int accumulate, double* __restrict__ out) {
  double v[3][kAdjSumPer];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int q = 0; q < kAdjSumPer; q++) {
      const int b = threadIdx.x + kAdjSumThreads * q;
      const double x = partial[c * nblk + (b < nblk ? b : 0)];
      v[c][q] = b < nblk ? x : 0.0;
    }
  __shared__ double sh[3][kAdjSumThreads / 64];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    double s = (v[c][0] + v[c][1]) + (v[c][2] + v[c][3]);
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[c][threadIdx.x >> 6] = s;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int c = threadIdx.x;
    double s = 0;
    for (int w = 0; w < kAdjSumThreads / 64; w++) s += sh[c][w];
    out[c] = accumulate ? out[c] + s : s;
  }
}

// ---------------------------------------------------------------------------
// k_adj_xb: for every point Q of the three components,
//   x_bar_c(Q) = z_bar_c(Q) + (J_N(X)^T N_bar)_c(Q)
// and, at pressure points, p_bar(Q) += b sum_c (z_bar_c(Q + e_c) - z_bar_c(Q)) / h_c.
//
// With n = N_bar and (a, b) ranging over the axes, N's component c at P holds
// -x_c D_c x_c - sum_a (S_a^c) D_a x_c with S_a^c the four-point sum of x_a
// around P; its transpose needs, per point P, the products
//   G_c(P)   = n_c x_c
//   H_c^a(P) = n_c S_a^c,    S_a^c = x_a(P+a) + x_a(P) + x_a(P-c+a) + x_a(P-c)
//   F_c^a(P) = n_c (x_c(P+a) - x_c(P-a))
// and then, for component c at Q,
//   x_bar_c = z_bar_c + diffusion(n_c) - n_c (x_c(Q+c) - x_c(Q-c)) / 2h_c
//             + (G_c(Q+c) - G_c(Q-c)) / 2h_c + sum_a (H_c^a(Q+a) - H_c^a(Q-a)) / 8h_a
//             - sum_a (F_a^c(Q) + F_a^c(Q-c) + F_a^c(Q+a) + F_a^c(Q+a-c)) / 8h_c
// so that every product is formed once per point instead of at each of the
// points that gather it (which takes X two points away).
//
// A workgroup's 32 x 16 threads are the points of a tile with a one-point
// halo (30 x 14 outputs) and march along k.  The products of a plane go
// through LDS; everything that couples planes stays in registers of the
// column: the four-point sums' halves, the plane differences and the
// contributions to the planes below and above.  X itself needs one plane in
// LDS at a time, with one more halo point.  N_bar is zero outside the component
// interiors and cells outside the arrays read as zero, so no product needs a
// test.  Two columns read as zero too: (0, N1) and (N0, 0), where the stage
// kernels leave what their threads outside a component's interior hold (in
// padding of u and w, and of v), which is no finite number after a run that
// blew up; the components that have a point there have it on an edge of the
// domain, which no product with a nonzero factor takes.  76 KB of LDS, two workgroups (16 waves) per CU; the arithmetic is FP64
// in both forms.  Bound by the LDS and the plane's two barriers: 128^3 FP64 153 ->
// 99 us against gathering X and N_bar from a three-plane ring of six fields (8
// waves per CU, 31 global taps per point); 14 words per point at 2.4 TB/s.  A
// kernel that spills here is slower than that one (the reloads wait for every
// load in flight): 128 VGPRs hold it only with one address register per load.
// ---------------------------------------------------------------------------
constexpr int AXT = 32, AYT = 16;            // threads: the tile with its halo
constexpr int AOX = AXT - 2, AOY = AYT - 2;  // outputs
constexpr int AHX = AXT + 2, AHY = AYT + 2;  // X plane
constexpr int ARING = 2 * (AHX + AYT);       // X plane points outside the threads' own
enum AdjProduct { PN_U, PN_V, PN_W, PG_V, PH_UV, PH_VU, PH_WU, PH_WV, PF_UY, PF_VX, PF_VZ, PF_WY, kAdjProducts };

template <typename T>
__global__ void __launch_bounds__(AXT * AYT) __attribute__((amdgpu_waves_per_eu(4)))
k_adj_xb(DGrid g, Layout L, AdjVec Xv, AdjVec Nbv, AdjVec Zv, AdjVec Xbv, T* __restrict__ P, double bcoef, int ntx,
         int nty, int ntiles, int kchunk) {
  __shared__ T xs[2][3][AHY][AHX];
  __shared__ double pr[kAdjProducts][AYT][AXT];
  const int tid = threadIdx.x, tx = tid % AXT, ty = tid / AXT;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  const int bx = tile % ntx, by = (tile / ntx) % nty, bz = tile / (ntx * nty);
  const int i = bx * AOX - 1 + tx, j = by * AOY - 1 + ty;
  const int k0 = bz * kchunk, kend = min(k0 + kchunk, g.N[2] + 1);  // output planes k0 .. kend-1
  const T* X[3] = {(const T*)Xv.f[0], (const T*)Xv.f[1], (const T*)Xv.f[2]};
  const T* N[3] = {(const T*)Nbv.f[0], (const T*)Nbv.f[1], (const T*)Nbv.f[2]};
  const T* Z[3] = {(const T*)Zv.f[0], (const T*)Zv.f[1], (const T*)Zv.f[2]};
  // this thread's column, and its point of the X plane's outer ring
  auto inside = [&](int ii, int jj) { return ii >= 0 && jj >= 0 && ii < L.PX && jj < L.SY; };
  auto finite = [&](int ii, int jj) { return !(ii == 0 && jj == g.N[1]) && !(ii == g.N[0] && jj == 0); };
  const bool own = inside(i, j) && finite(i, j);
  // lane offsets are 32-bit and the plane's base is uniform, so that a load
  // takes one address register
  const unsigned oo = inside(i, j) ? i + L.PX * j : 0;
  int rx = 0, ry = 0;
  if (tid < AHX) {
    rx = tid;
  } else if (tid < 2 * AHX) {
    rx = tid - AHX;
    ry = AHY - 1;
  } else if (tid < ARING) {
    rx = (tid - 2 * AHX) < AYT ? 0 : AHX - 1;
    ry = 1 + (tid - 2 * AHX) % AYT;
  }
  const int ri = bx * AOX - 2 + rx, rj = by * AOY - 2 + ry;
  const bool ring = tid < ARING;
  const bool rok = ring && inside(ri, rj) && finite(ri, rj);
  const unsigned ro = rok ? ri + L.PX * rj : 0;

  // planes outside the arrays read plane 0 and count as zero
  auto plane_ok = [&](int k) { return k >= 0 && k < L.SZ; };
  auto plane_at = [&](int k) -> long { return plane_ok(k) ? (long)k * L.plane : 0; };
  // (kept out of the compiler's sight from plane to plane: hoisted out of the
  // loop, the sums of base and offset take a register pair per array)
  auto lane = [](unsigned off) {
    asm volatile("" : "+v"(off));
    return off;
  };
  T px[3], pring[3], pn[3];
  auto fetch_x = [&](int k) {
    const long kp = plane_at(k);
    const unsigned a = lane(oo), b = lane(ro);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T* x = X[c] + kp;
      px[c] = x[a];
      pring[c] = x[b];
    }
  };
  auto fetch_n = [&](int k) {
    const long kp = plane_at(k);
    const unsigned a = lane(oo);
#pragma unroll
    for (int c = 0; c < 3; c++) pn[c] = (N[c] + kp)[a];
  };
  auto commit_x = [&](int k) {
    const bool kin = plane_ok(k);
    T(&pl)[3][AHY][AHX] = xs[k & 1];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      pl[c][ty + 1][tx + 1] = own && kin ? px[c] : (T)0;
      if (ring) pl[c][ry][rx] = rok && kin ? pring[c] : (T)0;
    }
  };

  const double A2 = g.one_over_2h[0], B2 = g.one_over_2h[1], C2 = g.one_over_2h[2];
  const double A8 = g.one_over_8h[0], B8 = g.one_over_8h[1], C8 = g.one_over_8h[2];
  const double Dx = g.one_over_h2Re[0], Dy = g.one_over_h2Re[1], Dz = g.one_over_h2Re[2];
  const double D2 = 2 * (Dx + Dy + Dz);
  const bool out = tx >= 1 && ty >= 1 && tx <= AOX && ty <= AOY && i <= g.N[0] && j <= g.N[1];
  // the column of a pressure point (its neighbours above lie in the arrays)
  const bool pcol = out && i < g.N[0] && j < g.N[1];
  const unsigned oz = pcol ? oo : 0;

  // X, f at this thread's point of plane k, displaced within the plane
  auto xat = [&](int k, int c, int di, int dj) -> double { return (double)xs[k & 1][c][ty + 1 + dj][tx + 1 + di]; };
  // planes k0-2 (what plane k0-1 needs of it), then k0-1 and k0 into LDS
  double su0, sv0, x0[3];  // of the plane below: u(P) + u(P+x), v(P) + v(P+y), X(P)
  fetch_x(k0 - 2);
  commit_x(k0 - 2);
  fetch_x(k0 - 1);
  commit_x(k0 - 1);
  fetch_x(k0);
  fetch_n(k0 - 1);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; c++) x0[c] = xat(k0, c, 0, 0);  // (the slot of plane k0-2)
  su0 = x0[0] + xat(k0, 0, 1, 0);
  sv0 = x0[1] + xat(k0, 1, 0, 1);
  __syncthreads();
  commit_x(k0);

  // acc: the outputs of plane m-1 but for what plane m adds; dn: what plane
  // m-1 adds to plane m
  double acc[3] = {0, 0, 0}, dn[3] = {0, 0, 0};
  for (int m = k0 - 1; m <= kend; m++) {
    __syncthreads();
    double n[3];
#pragma unroll
    for (int c = 0; c < 3; c++) n[c] = own && plane_ok(m) ? (double)pn[c] : 0.0;
    // memory requests in the order their values are waited for: the operands
    // of output plane m-1, then plane m+2 of X and m+1 of N_bar, which stay in
    // flight until the next plane
    const int k = m - 1;
    const bool emit = out && k >= k0;
    const long kp = plane_at(k);
    double z[3], zn[3], pv;
#pragma unroll
    for (int c = 0; c < 3; c++) z[c] = (double)(Z[c] + kp)[lane(oo)];
    const unsigned az = lane(oz);
    zn[1] = (double)(Z[1] + kp)[az + L.PX];
    zn[2] = (double)(Z[2] + plane_at(k + 1))[az];
    pv = (double)(P + kp)[az];
    fetch_x(m + 2);
    fetch_n(m + 1);
    // products of plane m
    const double u = xat(m, 0, 0, 0), v = xat(m, 1, 0, 0), w = xat(m, 2, 0, 0);
    double here[3] = {dn[0] - D2 * n[0], dn[1] - D2 * n[1], dn[2] - D2 * n[2]};
    double fv_x, fw_x, fw_y, fu_y, su, sv, swx, swy;
    {
      const double up = xat(m, 0, 1, 0), ud = xat(m, 0, 0, -1);
      su = u + up;
      here[0] -= A2 * n[0] * (up - xat(m, 0, -1, 0));
      fu_y = n[0] * (xat(m, 0, 0, 1) - ud);
      pr[PH_VU][ty][tx] = n[1] * (su + xat(m, 0, 1, -1) + ud);
    }
    {
      const double vp = xat(m, 1, 0, 1), vl = xat(m, 1, -1, 0);
      sv = v + vp;
      here[1] -= B2 * n[1] * (vp - xat(m, 1, 0, -1));
      fv_x = n[1] * (xat(m, 1, 1, 0) - vl);
      pr[PH_UV][ty][tx] = n[0] * (sv + xat(m, 1, -1, 1) + vl);
    }
    {
      const double wl = xat(m, 2, -1, 0), wd = xat(m, 2, 0, -1);
      swx = w + wl;
      swy = w + wd;
      fw_x = n[2] * (xat(m, 2, 1, 0) - wl);
      fw_y = n[2] * (xat(m, 2, 0, 1) - wd);
    }
    const double gu = n[0] * u, gw = n[2] * w;
#pragma unroll
    for (int c = 0; c < 3; c++) pr[PN_U + c][ty][tx] = n[c];
    pr[PG_V][ty][tx] = n[1] * v;
    pr[PH_WU][ty][tx] = n[2] * (su + su0);
    pr[PH_WV][ty][tx] = n[2] * (sv + sv0);
    pr[PF_UY][ty][tx] = fu_y;
    pr[PF_VX][ty][tx] = fv_x;
    pr[PF_WY][ty][tx] = fw_y;
    double fu_z, fv_z, hu_w, hv_w;
    {
      const double u1 = xat(m + 1, 0, 0, 0), v1 = xat(m + 1, 1, 0, 0), w1 = xat(m + 1, 2, 0, 0);
      hu_w = n[0] * (swx + w1 + xat(m + 1, 2, -1, 0));
      hv_w = n[1] * (swy + w1 + xat(m + 1, 2, 0, -1));
      fu_z = n[0] * (u1 - x0[0]);
      fv_z = n[1] * (v1 - x0[1]);
      here[2] -= C2 * n[2] * (w1 - x0[2]);
    }
    pr[PF_VZ][ty][tx] = fv_z;
    x0[0] = u;
    x0[1] = v;
    x0[2] = w;
    su0 = su;
    sv0 = sv;
    // x neighbours lie in the same wave (a wave is two rows of 32 points)
    const double fw_xl = __shfl_up(fw_x, 1, 64), fu_zr = __shfl_down(fu_z, 1, 64);
    zn[0] = __shfl_down(z[0], 1, 64);
    const double gu_l = __shfl_up(gu, 1, 64), gu_r = __shfl_down(gu, 1, 64);
    __syncthreads();
    if (out) {
      auto at = [&](int f, int di, int dj) -> double { return pr[f][ty + dj][tx + di]; };
      const double t1 = fw_x + fw_xl, t2 = fw_y + at(PF_WY, 0, -1);
      const double t3 = fu_z + fu_zr + fv_z + at(PF_VZ, 0, 1);
      // outputs of plane m-1
      if (emit) {
        const double ub = acc[0] + (C8 * hu_w + Dz * n[0] - A8 * t1) + z[0];
        const double vb = acc[1] + (C8 * hv_w + Dz * n[1] - B8 * t2) + z[1];
        const double wb = acc[2] + (C2 * gw + Dz * n[2]) + z[2];
        if (in_field(g, 0, i, j, k)) ((T*)Xbv.f[0] + kp)[lane(oo)] = (T)ub;
        if (in_field(g, 1, i, j, k)) ((T*)Xbv.f[1] + kp)[lane(oo)] = (T)vb;
        if (in_field(g, 2, i, j, k)) ((T*)Xbv.f[2] + kp)[lane(oo)] = (T)wb;
        if (pcol && k < g.N[2])
          (P + kp)[lane(oz)] = (T)(pv + bcoef * ((zn[0] - z[0]) * g.one_over_h[0] + (zn[1] - z[1]) * g.one_over_h[1] +
                                   (zn[2] - z[2]) * g.one_over_h[2]));
      }
      // plane m from its own products
      auto lap = [&](int f) { return Dx * (at(f, 1, 0) + at(f, -1, 0)) + Dy * (at(f, 0, 1) + at(f, 0, -1)); };
      acc[0] = here[0] + lap(PN_U) + A2 * (gu_r - gu_l) +
               B8 * (at(PH_UV, 0, 1) - at(PH_UV, 0, -1)) -
               A8 * ((fv_x + at(PF_VX, -1, 0) + at(PF_VX, 0, 1) + at(PF_VX, -1, 1)) + t1);
      acc[1] = here[1] + lap(PN_V) + B2 * (at(PG_V, 0, 1) - at(PG_V, 0, -1)) +
               A8 * (at(PH_VU, 1, 0) - at(PH_VU, -1, 0)) -
               B8 * ((fu_y + at(PF_UY, 0, -1) + at(PF_UY, 1, 0) + at(PF_UY, 1, -1)) + t2);
      acc[2] = here[2] + lap(PN_W) + A8 * (at(PH_WU, 1, 0) - at(PH_WU, -1, 0)) +
               B8 * (at(PH_WV, 0, 1) - at(PH_WV, 0, -1)) - C8 * t3;
      dn[0] = Dz * n[0] - C8 * hu_w;
      dn[1] = Dz * n[1] - C8 * hv_w;
      dn[2] = Dz * n[2] - C2 * gw - C8 * t3;
    }
    // plane m+2 takes the slot of plane m, which every thread has read
    commit_x(m + 2);
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <typename T>
void launch_adj_rhs(const DGrid& g, const Layout& L, const T* P, const AdjVec& Y, double dts, T* B, long bp0,
                    long bplane, hipStream_t st) {
  const int nx = (g.npts[0] + 63) / 64, items = nx * g.npts[1] * g.npts[2];
  k_adj_rhs<T><<<(unsigned)((items + 3) / 4), 256, 0, st>>>(g, L, P, Y, dts, B, bp0, bplane, nx, items);
}

// Rows per plane, 64-point items per row and items of k_adj_zb: the union of
// the components' interiors.
struct ZbShape {
  int rows, nx, items;
};
static ZbShape zb_shape(const DGrid& g) {
  int top[3] = {0, 0, 0};
  for (int c = 0; c < 3; c++) {
    int e[3];
    extents(g, c, e);
    for (int ax = 0; ax < 3; ax++) top[ax] = std::max(top[ax], e[ax] - 2);
  }
  const int nx = (top[0] + 63) / 64;
  return {top[1], nx, nx * top[1] * top[2]};
}

int adj_zb_blocks(const DGrid& g) { return std::clamp((zb_shape(g).items + 3) / 4, 1, kAdjMaxBlocks); }

template <typename T>
void launch_adj_zb(const DGrid& g, const Layout& L, const AdjVec& Y, const T* Bpsi, long bp0, long bplane, double dts,
                   const AdjVec& Zb, const AdjVec& Nb, const AdjVec& Zo, double alpha, double beta, double fcoef,
                   int accumulate, double* partial,
                   int nblk, hipStream_t st) {
  const ZbShape sh = zb_shape(g);
  k_adj_zb<T><<<nblk, 256, 0, st>>>(g, L, Y, Bpsi, bp0, bplane, g.one_over_h[0] / dts, g.one_over_h[1] / dts,
                                    g.one_over_h[2] / dts, Zb, Nb, Zo, alpha, beta, fcoef, accumulate, partial,
                                    sh.rows, sh.nx, sh.items);
}

void launch_adj_sum(const double* partial, int nblk, int accumulate, double* out, hipStream_t st) {
  k_adj_sum<<<1, kAdjSumThreads, 0, st>>>(partial, nblk, accumulate, out);
}

template <typename T>
void launch_adj_xb(const DGrid& g, const Layout& L, const AdjVec& X, const AdjVec& Nb, const AdjVec& Zb,
                   const AdjVec& Xb, T* P, double bcoef, hipStream_t st) {
  // tiles over points 0..N per axis
  const int ntx = (g.N[0] + AOX) / AOX, nty = (g.N[1] + AOY) / AOY;
  // planes per workgroup: each chunk repeats two planes of products, and a
  // chunk's planes are a serial chain of about 2.6 us each.  Adjoint step, 2 / 4
  // / 6 / 16 planes: 32^3 317 / 333 / 353 / 433 us, 64^3 419 / 410 / 423 / 498, 96^3
  // 637 / 603 / 592 / 622, 128^3 1115 / 1036 / 1023 / 1009, 256^3 6.27 / 5.60 /
  // 5.41 / 5.15 ms
  const int kchunk = (int)std::clamp((long)ntx * nty * (g.N[2] + 1) / 400, 2L, 16L);
  const int ntiles = ntx * nty * ((g.N[2] + kchunk) / kchunk);
  k_adj_xb<T><<<ntiles, AXT * AYT, 0, st>>>(g, L, X, Nb, Zb, Xb, P, bcoef, ntx, nty, ntiles, kchunk);
}

#define MIF_ADJ_INST(T)                                                                                              \
  template void launch_adj_rhs<T>(const DGrid&, const Layout&, const T*, const AdjVec&, double, T*, long, long,       \
                                  hipStream_t);                                                                      \
  template void launch_adj_zb<T>(const DGrid&, const Layout&, const AdjVec&, const T*, long, long, double,            \
                                 const AdjVec&, const AdjVec&, const AdjVec&, double, double, double, int, double*,   \
                                 int, hipStream_t);                                                                  \
  template void launch_adj_xb<T>(const DGrid&, const Layout&, const AdjVec&, const AdjVec&, const AdjVec&,            \
                                 const AdjVec&, T*, double, hipStream_t);

MIF_ADJ_INST(double)
MIF_ADJ_INST(float)

}  // namespace mif
