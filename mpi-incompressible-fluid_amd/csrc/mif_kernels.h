// mif_kernels.h -- launch interfaces of the HIP kernels (host side).
#pragma once

#include <vector>

#include "mif_device.h"

namespace mif {

// Arguments of the fused three-component RK3 stage kernel of the full step
// (src/Timestep.cpp:10-54).  X is the stencil source, A the pointwise
// operand, O1/O2 the outputs; a1, a2, b are the stage coefficients (stage 3
// passes its a3 in a2).
struct Red3;
struct StageArgs {
  const void* X[3];
  const void* A[3];
  void* O1[3];
  void* O2[3];
  const void* p;
  double a1, a2, b;
  double force[3];  // constant body force added to N (zero in the reference)
  // The previous stage's projection, fused into this stage (kinds 2 and 3):
  // when phi is set, X holds that stage's output before its projection and p
  // the pressure before its increment; the kernel reads them as
  // X - pdts grad(phi) (component interiors) and p + phi - mean (mean from
  // pmean, or 0), and stores the incremented p at its tile's points into pout
  // (not p, which neighbouring threads and workgroups read).
  const void* phi;
  double pdts;
  const Red3* pmean;
  void* pout;
};

// Arguments of the velocity-only stage kernel (src/TimestepVelocity.cpp:20-51).
struct VelStageArgs {
  const void* X[3];
  void* V[3];
  void* R[3];
  void* B[3];
  double t, dt;
  FnDesc forcing;
};

struct Red3 {
  double s1, s2, mx;
};

// One axis as products with the transform's matrices (mif_dense.hip), for
// lengths without a specialised kernel: R is the mirror length (n, or n - 1 on
// a Neumann axis), H = R/2 + 1 the rows of the folded line (quad, a line
// folded twice: n/4 + 1), MT and KS its 16-row and 8-column tiles, M the
// fragment tables (null: no dense pass).
struct DensePlan {
  int n, R, H, MT, KS;
  int periodic, quad;
  const double* M64;
  const float* M32;
};

// One axis of the spectral Poisson solve: complex transform length L (= n on
// a periodic axis, 2(n-1) on a Neumann axis), its radix factorisation and
// the twiddle table W[e] = exp(-2 pi i e / L).
struct FftPlan {
  int n, L, periodic;
  int nst;
  int radix[24];
  int Ns[24];
  const double* W64;
  const float* W32;
  // cell-centred Neumann axis: DCT-II/DCT-III of length n = L, with the
  // half-angle table (cos, sin)(pi k / (2L)), k < L
  int dct2;
  const double* H64;
  const float* H32;
  DensePlan dense;
};

// Scaling applied between the forward and inverse transform of the last
// axis: 1 / ((lx[i] + ly[j] + lz[k]) * norm), zero for the constant mode.
struct SpectralScale {
  const double* lam[3];
  double inv_norm;
};

// Neighbour index along axis a of packed index i (d = -1 or +1): periodic
// wrap, cell-centred reflection of the first/last cell, or the node-centred
// even reflection (the 7-point operator of the packed solve).
__device__ inline long nb(const DGrid& g, int a, int i, int d) {
  const int n = g.npts[a];
  int q = i + d;
  if (g.periodic[a]) {
    q = q < 0 ? q + n : (q >= n ? q - n : q);
  } else if (g.cell[a]) {
    // cell-centred: the ghost mirrors the first/last cell
    if (q < 0) q = 0;
    if (q >= n) q = n - 1;
  } else {
    if (q < 0) q = n > 1 ? 1 : 0;
    if (q >= n) q = n > 1 ? n - 2 : 0;
  }
  return q;
}

// Operands of the x passes fused with the divergence (forward) or with the
// unpack into the pressure field (inverse).
struct FusedIO {
  const void* u;
  const void* v;
  const void* w;
  void* P;
  Layout L;
  double dt;
  // the velocity and pressure fields hold FP32 values while the transform
  // runs in FP64 (the mixed form with FP64 transforms)
  int fields_fp32 = 0;
  // x forward pass of a right-hand side held in the pressure field P: it reads
  // the field's owner points (element type T) in place of its buffer
  int pack = 0;
  // mixed form with one FP64 defect sweep (FP32 transforms): the forward
  // pass also stores the FP64 divergence b (packed layout) and per-workgroup
  // owner-weighted sums (W.b, W.1) into partial; the inverse pass adds the
  // first FP32 solution add32 (packed layout) to the correction in FP64,
  // stores the sum, and leaves (W.phi, W.1) of the stored values in partial
  int dc = 0;
  double* b64 = nullptr;
  const float* add32 = nullptr;
  Red3* partial = nullptr;
  // x forward pass of the defect (res): the pass loads r = (b - mean) - L phi
  // in FP64 (b64, bmean, the first FP32 solution phi32, packed layout) instead
  // of its buffer, and transforms it into its buffer
  int res = 0;
  const float* phi32 = nullptr;
  const Red3* bmean = nullptr;
};

// pout = pin + (phi - mean) on the pressure points a stage kernel with a fused
// projection leaves out (outside the union of the components' interiors).
struct PressureRim {
  const void* pin = nullptr;  // null: no rim
  const void* phi = nullptr;
  void* pout = nullptr;
  const Red3* mean = nullptr;
};
// The extents of the stage kernels' tiles (the union of the components'
// interiors) and the rim's point counts per group.
struct RimShape {
  int imax, jmax, kmax;
  long count[3];
};
struct BCArgs {
  void* F[3];
  FnDesc f;
  double t;
  double tf;        // time_factor (BC_ES, BC_VT)
  int count[3][3];  // threads (opposite shell points) per (component, face pair)
};
// The boundary pass and the pressure rim of a stage, in the stage's own
// launch: the stage kernel stores its boundary-adjacent points at their
// periodic images too, and further workgroups fill the wall faces and the rim.
struct StageShell {
  int on = 0;    // 0: not wanted
  // workgroups of a row: of each axis (0: no wall), whose rows are (side,
  // component), and of the rim, whose rows are its three groups
  int nb[3] = {}, nb_rim = 0;
  int blocks() const { return 6 * (nb[0] + nb[1] + nb[2]) + 3 * nb_rim; }
  BCArgs a{};
  PressureRim rim{};
  RimShape rs{};
};
// The shell of a stage (of the full or the velocity-only step) that writes F,
// whose boundary data are f at time t.
StageShell stage_shell(const DGrid& g, const Layout& L, bool full_step, void* const F[3], const FnDesc& f, double t,
                       const PressureRim& rim);

// A stage, and the shell sh with it where there is a kernel for the two: false
// if not, and a boundary pass has to follow.
template <typename T>
bool launch_stage(int stage, const DGrid& g, const Layout& L, const StageArgs& s, const StageShell& sh,
                  hipStream_t st);
template <typename T>
bool launch_vel_stage(int stage, const DGrid& g, const Layout& L, const VelStageArgs& s, const StageShell& sh,
                      hipStream_t st);
// The axis tables (axis_index) of n indices per axis: es_axis_tables returns
// them with the rows AX_SIN and AX_COS empty, which launch_axis_tables fills on
// the device.
std::vector<double> es_axis_tables(const DGrid& g, int n);
void launch_axis_tables(const DGrid& g, double* tab, int n, hipStream_t st);
template <typename T>
void launch_bc(const DGrid& g, const Layout& L, void* const F[3], const FnDesc& f, double t, hipStream_t st,
               const PressureRim& rim = PressureRim{});
template <typename T>
void launch_periodic(const DGrid& g, const Layout& L, T* F, int stag, hipStream_t st);
template <typename T>
void launch_set(const DGrid& g, const Layout& L, T* F, int stag, int comp, const FnDesc& f, double t, int border,
                hipStream_t st);
template <typename T, typename S>
void launch_div_rhs(const DGrid& g, const Layout& L, const T* u, const T* v, const T* w, S* B, long bp0, long bplane,
                    double dt, const FnDesc& gp, double tg, int nhn, hipStream_t st);
template <typename T, typename S>
void launch_pack(const DGrid& g, const Layout& L, const T* P, S* B, long bp0, long bplane, hipStream_t st);
template <typename T, typename S>
void launch_unpack(const DGrid& g, const Layout& L, const S* B, long bp0, long bplane, T* P, hipStream_t st);
template <typename T>
// p += phi (minus mean->s1 / mean->s2 when mean is not null), velocity -= dts grad phi
void launch_project(const DGrid& g, const Layout& L, T* u, T* v, T* w, T* p, const T* phi, double dts, hipStream_t st,
                    const Red3* mean = nullptr, T* pout = nullptr);
template <typename T>
void launch_pgrad(const DGrid& g, const Layout& L, const T* p, T* u, T* v, T* w, hipStream_t st);
template <typename T>
void launch_from_dense(const Layout& L, const int e[3], const double* src, T* dst, hipStream_t st);
template <typename T>
void launch_to_dense(const Layout& L, const int e[3], const T* src, double* dst, hipStream_t st);
template <typename T>
void launch_copy(long n, const T* src, T* dst, hipStream_t st);
template <typename T>
void launch_dot(const Layout& L, const int e[3], const T* a, const T* b, Red3* partial, int nblocks, Red3* out,
                hipStream_t st);
// out[q] = F(ijk[3q], ijk[3q+1], ijk[3q+2]) for q < n (indices checked by the caller).
template <typename T>
void launch_gather(const Layout& L, const T* F, const int* ijk, long n, double* out, hipStream_t st);
template <typename T>
void launch_add_const(const DGrid& g, const Layout& L, T* P, double c, hipStream_t st);
// Exact-solution tables for the norms and adjust_pressure: node-shaped
// fields (element type of the context) holding the exact values; f[0] null
// selects the closed-form descriptor instead.
struct ExactTables {
  const void* f[3];
};
template <typename T>
void launch_norm_velocity(const DGrid& g, const Layout& L, const T* u, const T* v, const T* w, const FnDesc& f,
                          double t, const ExactTables& tab, Red3* partial, int nblocks, Red3* out, hipStream_t st);
template <typename T>
void launch_norm_pressure(const DGrid& g, const Layout& L, const T* p, const FnDesc& f, double t, int adjust,
                          const ExactTables& tab, Red3* partial, int nblocks, Red3* out, hipStream_t st);

// Spectral solve passes on the packed buffer B (extents npts, row pitch bp0,
// plane pitch bplane).  dir: -1 forward, +1 inverse on axes 0 and 1; axis 2 has
// one pass only, forward, scaling and inverse, whatever dir is.
template <typename T>
void launch_fft_axis(const DGrid& g, int axis, int dir, const FftPlan& plan, const SpectralScale& sc, T* B,
                     long bp0, long bplane, hipStream_t st);
// Specialised transform pass (complex lengths 2^k and 3 * 2^k, see
// fft_fast_len); on axis 0 with io set, the forward pass is fused with the
// divergence (mode 0) and the inverse with the unpack into the pressure field
// (mode 1); axis 2 is mode 2, forward, scaling and inverse.  Returns false when
// the length has no specialised kernel.
bool fft_fast_len(int L);
template <typename T>
bool launch_fft_pow2(const DGrid& g, int axis, int mode, const FftPlan& plan, const SpectralScale& sc, T* B, long bp0,
                     long bplane, const FusedIO* io, hipStream_t st);
// The passes as matrix products (mif_dense.hip): axis 0 with mode 0 / 1 (io
// as in launch_fft_pow2), axis 1 with mode 0 / 1, axis 2 is mode 2.
// dense_plan fills the tile counts (false: the line is too long).
bool dense_plan(int n, bool periodic, DensePlan* P);
// The fragment tables of a plan: dense_table_elems elements, in FP64 and (out32
// not null) FP32.
size_t dense_table_elems(const DensePlan& P);
void dense_table(const DensePlan& P, double* out64, float* out32);
template <typename T>
void launch_dense(const DGrid& g, int axis, int mode, const DensePlan& P, const SpectralScale& sc, T* B, long bp0,
                  long bplane, const FusedIO* io, hipStream_t st);
int dense_x_blocks(const DGrid& g);
// Whether the axis-0 pass of a plan has a form fused with the divergence and
// the unpack, and that pass (mode 0 forward, 1 inverse).
bool fused_x_pass(const FftPlan& plan);
template <typename T>
void launch_fused_x(const DGrid& g, int mode, const FftPlan& plan, const SpectralScale& sc, T* B, long bp0, long bplane,
                    const FusedIO& io, hipStream_t st);
bool dense_x_short(const DGrid& g, const FftPlan& plan, bool fp64);
// Workgroups of the specialised x pass of a plan (0 without one), and of the
// fused x pass that runs: the number of partial sums FusedIO::dc leaves.
int pow2_x_blocks(const DGrid& g, const FftPlan& plan, bool fp64);
int fused_x_blocks(const DGrid& g, const FftPlan& plan, bool fp64);
// DCT-II (forward) or DCT-III (inverse) pass of a cell-centred Neumann y
// axis; false when the length (64, 128, 256, 512 or 1024) has no kernel.
template <typename T>
bool launch_dct2_y_any(const DGrid& g, const FftPlan& plan, int inverse, T* B, long bp0, long bplane, hipStream_t st);

// Three component arrays of one velocity-shaped quantity.
struct AdjVec {
  void* f[3];
};

// Adjoint of one step (mif_adjoint.hip).
// Packed right-hand side of the transposed solve from p_bar and y_bar.
template <typename T>
void launch_adj_rhs(const DGrid& g, const Layout& L, const T* P, const AdjVec& Y, double dts, T* B, long bp0,
                    long bplane, hipStream_t st);
// z_bar and N_bar = alpha z_bar + beta Zo of a stage, plus nblk partial sums
// of z_bar per component (partial holds 3 * nblk doubles).
template <typename T>
void launch_adj_zb(const DGrid& g, const Layout& L, const AdjVec& Y, const T* Bpsi, long bp0, long bplane, double dts,
                   const AdjVec& Zb, const AdjVec& Nb, const AdjVec& Zo, double alpha, double beta, double fcoef,
                   int accumulate, double* partial, int nblk, hipStream_t st);
// Workgroups of k_adj_zb (64 points per wave up to this many, grid-stride
// beyond), and the number of partials per component k_adj_sum reduces.
constexpr int kAdjMaxBlocks = 4096;
int adj_zb_blocks(const DGrid& g);
// out[c] = (accumulate: out[c] +) the sum of the nblk <= kAdjMaxBlocks
// partials of component c.
void launch_adj_sum(const double* partial, int nblk, int accumulate, double* out, hipStream_t st);
// x_bar = z_bar + J_N(X)^T N_bar; p_bar += bcoef * G^T z_bar.
template <typename T>
void launch_adj_xb(const DGrid& g, const Layout& L, const AdjVec& X, const AdjVec& Nb, const AdjVec& Zb,
                   const AdjVec& Xb, T* P, double bcoef, hipStream_t st);

// Mixed form: FP64 right-hand side projection and defect correction
// (mif_mixed.hip).
void launch_project_rhs(const DGrid& g, double* B64, float* B32, long bp0, long bplane, Red3* partial, int nblocks,
                        Red3* total, hipStream_t st);
void launch_to64(const DGrid& g, const float* B32, double* P, long bp0, long bplane, hipStream_t st);
void launch_remove_mean(const DGrid& g, double* P, long bp0, long bplane, Red3* partial, int nblocks, Red3* total,
                        hipStream_t st);
void launch_residual(const DGrid& g, const double* b, const double* P, float* B32, long bp0, long bplane,
                     hipStream_t st);
void launch_accumulate(const DGrid& g, double* P, const float* B32, long bp0, long bplane, hipStream_t st);
// One-sweep defect correction with FP32 transforms: the sum of n partial
// (W.x, W.1) pairs into total; a node field minus the mean total holds.
void launch_reduce_partials(const Red3* partial, int n, Red3* total, hipStream_t st);
void launch_sub_mean_field(const DGrid& g, const Layout& L, float* F, const Red3* total, hipStream_t st);

// Streaming-ceiling probe (mif_probe.hip): nr arrays read and nw arrays
// written, n4 16-byte elements each.
constexpr int kStreamMax = 8;
struct StreamArgs {
  const float4* in[kStreamMax];
  float4* out[kStreamMax];
};
void launch_stream(const StreamArgs& a, int nr, int nw, long n4, int blocks, hipStream_t st);

}  // namespace mif
