// mif_device.h -- device-side data model shared by the HIP kernels.
//
// Every field of one context lives in the same padded x-fastest layout:
// element (i,j,k) of any staggering is at i + PX*(j + SY*k), where PX is the
// largest x extent rounded up to 64 bytes and SY the largest y extent.  The
// logical extents of each staggering are those of the reference tensors
// (src/StaggeredTensor.cpp:5-9, src/Constants.cpp:80-85 at one rank); the
// padding is never read as data.  A common layout lets a stencil thread
// address u, v, w and p at one offset.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "../../include/mif_types.h"

namespace mif {

// Single-rank domain constants (src/Constants.cpp:58-120 at Py = Pz = 1).
struct DGrid {
  int N[3];        // Nx, Ny, Nz: node extents incl. periodic ghosts
  int Ng[3];       // global node counts
  int base[3];     // base_i/j/k
  int periodic[3];
  int npts[3];     // Poisson unknowns per axis
  int olo[3];      // first owner index per axis (1 on periodic axes)
  int cell[3];     // 1: cell-centred Neumann axis (stand-alone Poisson solves)
  double h[3], min[3];
  double one_over_2h[3], one_over_8h[3], one_over_h2Re[3], h_over_2[3], one_over_h[3];
  double Re, dt;
};

struct Layout {
  int PX, SY, SZ;  // padded pitch, rows per plane, planes
  long plane;      // PX * SY
  long elems;      // PX * SY * SZ
  int lead;        // elements between the (aligned) allocation start and element 0
  int nt;          // nonzero: the streaming kernels store their outputs non-temporally
  __host__ __device__ inline long idx(int i, int j, int k) const {
    return (long)i + (long)PX * ((long)j + (long)SY * (long)k);
  }
};

// Extents of a field with staggering s (0 = x, 1 = y, 2 = z, 3 = none).
__host__ __device__ inline void extents(const DGrid& g, int s, int e[3]) {
  e[0] = g.N[0];
  e[1] = g.N[1];
  e[2] = g.N[2];
  if (s == 0) e[0] = g.periodic[0] ? g.N[0] : g.N[0] + 1;
  if (s == 1) e[1] = g.N[1] + 1;
  if (s == 2) e[2] = g.N[2] + 1;
}

// ---------------------------------------------------------------------------
// Analytic functions (device closed forms of the reference's generated
// callbacks; see include/mif_types.h for the list).
// ---------------------------------------------------------------------------
// kind kFnFaceTable: boundary data evaluated on the host, for callbacks that
// have no closed form here.  tab holds, for each component q (of a velocity;
// only q = 0 for the Neumann data of a node field) and each face
// f = z-, z+, y-, y+, x-, x+, a plane of values over the field's extents
// along the two other axes, lower axis fastest (face_plane_index), starting
// at tab + toff[q][f]; faces of periodic axes have none.  fn_eval never
// reads it; the boundary and Neumann-data kernels look values up instead.
constexpr int kFnFaceTable = 1000;

struct FnDesc {
  int kind, base;
  double Re, c[3], t0, t1;
  const double* tab;
  long toff[3][6];
  // the context's axis tables (AxisTab), for the closed forms that separate
  // into functions of one coordinate
  const double* axis;
  int an;
};

// Functions of one coordinate tabulated per axis a at its unstaggered (sh = 0)
// and staggered (sh = 1, shifted by -h/2) indices i < n, in FP64: entry i of
// the row at axis_index.  EXP_A, SIN_A, COS_A take (pi/4) x and SIN_D, COS_D
// (pi/2) x, the Ethier-Steinman arguments; row fn + kAxisLow holds what
// rounding such an entry left out.
enum AxisFn { AX_SIN, AX_COS, AX_EXP_A, AX_SIN_A, AX_COS_A, AX_SIN_D, AX_COS_D, kAxisFns };
constexpr int kAxisLow = kAxisFns - AX_EXP_A, kAxisRows = kAxisFns + kAxisLow;
__host__ __device__ inline long axis_index(int a, int sh, int fn, int n) { return ((fn * 3 + a) * 2 + sh) * (long)n; }
inline long axis_elems(int n) { return axis_index(0, 0, kAxisRows, n); }

// Index of point (i, j, k) in the plane of face f (0,1 = z-,z+; 2,3 =
// y-,y+; 4,5 = x-,x+) of a field with extents e.
__host__ __device__ inline long face_plane_index(int face, const int e[3], int i, int j, int k) {
  const int axis = 2 - (face >> 1);
  if (axis == 2) return (long)i + (long)e[0] * j;
  if (axis == 1) return (long)i + (long)e[0] * k;
  return (long)j + (long)e[1] * k;
}

__host__ inline FnDesc make_fn(const mif_function* f) {
  FnDesc d{};
  if (f) {
    d.kind = f->kind;
    d.base = f->base;
    d.Re = f->Re;
    d.c[0] = f->c[0];
    d.c[1] = f->c[1];
    d.c[2] = f->c[2];
    d.t0 = f->t0;
    d.t1 = f->t1;
  }
  return d;
}

#define MIF_PI 3.14159265358979323846

// Ethier-Steinman u (generators/manufsol.py:36-44); v, w by cyclic argument
// permutation.
__device__ inline double es_u(double t, double x, double y, double z, double Re) {
  const double a = MIF_PI / 4, d = MIF_PI / 2;
  return -a * (exp(a * x) * sin(a * y + d * z) + exp(a * z) * cos(a * x + d * y)) * exp(-d * d * t / Re);
}

// Ethier-Steinman p (generators/manufsol.py:55-68).
__device__ inline double es_p(double t, double x, double y, double z, double Re) {
  const double a = MIF_PI / 4, d = MIF_PI / 2;
  const double s = exp(2 * a * x) + exp(2 * a * y) + exp(2 * a * z) +
                   2 * sin(a * x + d * y) * cos(a * z + d * x) * exp(a * (y + z)) +
                   2 * sin(a * y + d * z) * cos(a * x + d * y) * exp(a * (z + x)) +
                   2 * sin(a * z + d * x) * cos(a * y + d * z) * exp(a * (x + y));
  return -a * a / 2 * s * exp(-2 * d * d * t / Re);
}

// d p / d x of the Ethier-Steinman pressure (term-by-term derivative).
__device__ inline double es_dpdx(double t, double x, double y, double z, double Re) {
  const double a = MIF_PI / 4, d = MIF_PI / 2;
  const double S1 = sin(a * x + d * y), C1 = cos(a * z + d * x);
  const double S2 = sin(a * y + d * z), C2 = cos(a * x + d * y);
  const double S3 = sin(a * z + d * x), C3 = cos(a * y + d * z);
  const double s = 2 * a * exp(2 * a * x) + 2 * exp(a * (y + z)) * (a * C2 * C1 - d * S1 * S3) +
                   2 * a * exp(a * (z + x)) * S2 * (C2 - S1) + 2 * exp(a * (x + y)) * C3 * (d * C1 + a * S3);
  return -a * a / 2 * s * exp(-2 * d * d * t / Re);
}

// Forcing of the velocity-only manufactured field: f = u_t + (u.grad)u -
// lap(u)/Re of MIF_FN_VT_VELOCITY (generators/manufsol_velocity.py:40-50),
// simplified, from the sines and cosines of the coordinates and the time.
__host__ __device__ inline double vt_forcing(int c, double sx, double cx, double sy, double cy, double sz, double cz,
                                             double st, double ct, double Re) {
  if (c == 0) return sx * cx * st * st * (2 - 2 * sy * sy - sz * sz) + sx * sz * cy * (ct + 3 * st / Re);
  if (c == 1) return sy * cy * st * st * (2 - 2 * sx * sx - sz * sz) + sy * sz * cx * (ct + 3 * st / Re);
  return sz * cz * st * st * (2 * sx * sx + 2 * sy * sy - 4) + cx * cy * cz * (2 * ct + 6 * st / Re);
}

// Kept out of line: the closed forms are large and only the boundary,
// forcing and set-up kernels evaluate them.  Of a descriptor it takes Re: a
// reference would have every thread copy the kernel's argument to scratch
// first (240 to 336 bytes: a 128^3 FP64 field set to zero 118 -> 17 us, to the
// Ethier-Steinman u 120 -> 30, 257^3 boundary pass of the PT field 52 -> 41,
// velocity-only step at 128^3 with constant forcing 403 -> 196).
__device__ __noinline__ double fn_base(int kind, int c, double t, double x, double y, double z, double Re) {
  switch (kind) {
    case MIF_FN_ZERO:
      return 0.0;
    case MIF_FN_ES_VELOCITY:
      return c == 0 ? es_u(t, x, y, z, Re) : (c == 1 ? es_u(t, y, z, x, Re) : es_u(t, z, x, y, Re));
    case MIF_FN_ES_PRESSURE:
      return es_p(t, x, y, z, Re);
    case MIF_FN_ES_GRAD_P:
      return c == 0 ? es_dpdx(t, x, y, z, Re) : (c == 1 ? es_dpdx(t, y, z, x, Re) : es_dpdx(t, z, x, y, Re));
    case MIF_FN_VT_VELOCITY:
      // generators/manufsol_velocity.py:55-57
      if (c == 0) return sin(x) * cos(y) * sin(z) * sin(t);
      if (c == 1) return cos(x) * sin(y) * sin(z) * sin(t);
      return 2 * cos(x) * cos(y) * cos(z) * sin(t);
    case MIF_FN_VT_FORCING:
      return vt_forcing(c, sin(x), cos(x), sin(y), cos(y), sin(z), cos(z), sin(t), cos(t), Re);
    case MIF_FN_PT_VELOCITY:
    case MIF_FN_PT_GRAD_P:
      // generators/manufsol_pressure.py:36-38 (grad p equals the velocity)
      if (c == 0) return -sin(x) * cos(y) * cos(z) * t;
      if (c == 1) return -cos(x) * sin(y) * cos(z) * t;
      return -cos(x) * cos(y) * sin(z) * t;
    case MIF_FN_PT_PRESSURE:
      return cos(x) * cos(y) * cos(z) * t;
    case MIF_FN_LID_1:
    case MIF_FN_LID_2: {
      // include/TestCaseBoundaries.h:18-56: v = 1 on the lid plane x = 1
      // (test 1) or x = -0.5 (test 2), zero elsewhere.
      const double xl = kind == MIF_FN_LID_1 ? 1.0 : -0.5;
      const double eps = 1e-12;
      return (c == 1 && x < xl + eps && x > xl - eps) ? 1.0 : 0.0;
    }
    default:
      return 0.0;
  }
}

__device__ inline double fn_eval(const FnDesc& f, int c, double t, double x, double y, double z) {
  const bool difference = f.kind == MIF_FN_TIME_DIFFERENCE;
  const int kind = difference ? f.base : f.kind;
  if (kind == MIF_FN_CONSTANT) {
    const double k = c == 0 ? f.c[0] : (c == 1 ? f.c[1] : f.c[2]);
    return difference ? k - k : k;
  }
  const double v = fn_base(kind, c, difference ? f.t1 : t, x, y, z, f.Re);
  return difference ? v - fn_base(kind, c, f.t0, x, y, z, f.Re) : v;
}

// Coordinate of index i along axis a for staggering s: min + h*(base+i),
// minus h/2 on the staggered axis (include/StaggeredTensor.h:95-110,
// include/VelocityTensor.h:16-78).  Contraction is off so that the
// coordinates round exactly as the reference computes them.
__host__ __device__ inline double coord(const DGrid& g, int a, int s, int i) {
#pragma clang fp contract(off)
  double x = g.min[a] + g.h[a] * (double)(g.base[a] + i);
  if (a == s) x = x - g.h_over_2[a];
  return x;
}

// Ethier-Steinman field and pressure gradient, and the velocity-only field,
// from the axis tables, without their factor in time (time_factor).  A sine or
// cosine of a sum of two coordinates is expanded by the addition theorem, so
// a value costs table reads and a few products.  s: staggering, c: component.
// The expansion has more roundings than the sine of a rounded sum, so products
// carry their rounding errors into their sums, and the gradient's entries
// their low parts.  Root mean square error against 80-bit arithmetic at
// boundary points of 1 x 1 x 2, 1.5 x 1 x 2 and 2^3 domains of 65 to 257 nodes,
// relative to the field's, point by point / products of rounded entries / as
// here: velocity 1.08-1.20e-16 / 1.12-1.31e-16 / 0.93-1.05e-16, gradient
// 1.51-2.00e-16 / 1.73-2.25e-16 / 1.22-1.40e-16; on 20^3 1.4e-15 / 8.6e-16 /
// 9.7e-17 and 1.6e-15 / 8e-16 / 1.2e-16.
struct AxisEval {
  const double* tab;
  int n, s, idx[3];
  // a value and what its rounding left out
  struct Wide {
    double h, l;
  };
  __device__ inline double operator()(int a, int fn) const {
    const int i = a == 0 ? idx[0] : (a == 1 ? idx[1] : idx[2]);
    return tab[axis_index(a, a == s ? 1 : 0, fn, n) + i];
  }
  __device__ inline Wide wide(int a, int fn) const { return {(*this)(a, fn), (*this)(a, fn + kAxisLow)}; }
  __device__ static inline Wide mul(double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b;
    return {p, __builtin_fma(a, b, -p)};
  }
  __device__ static inline Wide mul(Wide a, Wide b) {
#pragma clang fp contract(off)
    const double p = a.h * b.h;
    return {p, __builtin_fma(a.h, b.h, -p) + (a.h * b.l + a.l * b.h)};
  }
  __device__ static inline double sum(Wide a, Wide b) {
#pragma clang fp contract(off)
    const double s = a.h + b.h, t = s - a.h;
    return s + (((a.h - (s - t)) + (b.h - t)) + (a.l + b.l));
  }
  __device__ static inline Wide minus(Wide a) { return {-a.h, -a.l}; }
  // sin and cos of (pi/4) x_a + (pi/2) x_b
  __device__ inline double sin_ad(int a, int b) const {
    return sum(mul((*this)(a, AX_SIN_A), (*this)(b, AX_COS_D)), mul((*this)(a, AX_COS_A), (*this)(b, AX_SIN_D)));
  }
  __device__ inline double cos_ad(int a, int b) const {
    return sum(mul((*this)(a, AX_COS_A), (*this)(b, AX_COS_D)), minus(mul((*this)(a, AX_SIN_A), (*this)(b, AX_SIN_D))));
  }
  __device__ inline double wide_sin_ad(int a, int b) const {
    return sum(mul(wide(a, AX_SIN_A), wide(b, AX_COS_D)), mul(wide(a, AX_COS_A), wide(b, AX_SIN_D)));
  }
  __device__ inline double wide_cos_ad(int a, int b) const {
    return sum(mul(wide(a, AX_COS_A), wide(b, AX_COS_D)), minus(mul(wide(a, AX_SIN_A), wide(b, AX_SIN_D))));
  }
  __device__ inline double wide_exp(int a, int b) const {
    const Wide p = mul(wide(a, AX_EXP_A), wide(b, AX_EXP_A));
    return p.h + p.l;
  }
  // es_u, es_dpdx with (x, y, z) = axes (p, q, r)
  __device__ inline double es_velocity(int p, int q, int r) const {
    return -(MIF_PI / 4) * sum(mul((*this)(p, AX_EXP_A), sin_ad(q, r)), mul((*this)(r, AX_EXP_A), cos_ad(p, q)));
  }
  // the gradient's three components share what they take of two axes each
  // (S[a], C[a], E[a]: of a and the axis after it)
  struct GradParts {
    double S[3], C[3], E[3];
  };
  __device__ inline GradParts es_grad_parts() const {
    GradParts t;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int b = (a + 1) % 3;
      t.S[a] = wide_sin_ad(a, b);
      t.C[a] = wide_cos_ad(a, b);
      t.E[a] = wide_exp(a, b);
    }
    return t;
  }
  __device__ inline double es_grad_p(const GradParts& t, int p, int q, int r) const {
#pragma clang fp contract(off)
    const double a = MIF_PI / 4;  // and d = 2 a
    const double v = wide_exp(p, p) + t.E[r] * (t.S[q] * (t.C[p] - t.S[p])) +
                     t.E[q] * __builtin_fma(-2 * t.S[p], t.S[r], t.C[p] * t.C[r]) +
                     t.E[p] * (t.C[q] * __builtin_fma(2.0, t.C[r], t.S[r]));
    return -(a * a * a) * v;
  }
  __device__ inline double vt_velocity(int c) const {
#pragma clang fp contract(off)
    if (c == 0) return (*this)(0, AX_SIN) * (*this)(1, AX_COS) * (*this)(2, AX_SIN);
    if (c == 1) return (*this)(0, AX_COS) * (*this)(1, AX_SIN) * (*this)(2, AX_SIN);
    return 2 * (*this)(0, AX_COS) * (*this)(1, AX_COS) * (*this)(2, AX_COS);
  }
};

// The factor in time of those forms (their only dependence on it).
__host__ inline double time_factor(int kind, double t, double Re) {
  const double d = MIF_PI / 2;
  if (kind == MIF_FN_ES_VELOCITY) return std::exp(-d * d * t / Re);
  if (kind == MIF_FN_ES_GRAD_P) return std::exp(-2 * d * d * t / Re);
  return std::sin(t);  // MIF_FN_VT_VELOCITY
}
// The factor of the Ethier-Steinman gradient's difference between two times,
// without the cancellation of two nearly equal exponentials.
__host__ inline double grad_p_factor_difference(double t1, double t0, double Re) {
  const double d = MIF_PI / 2;
  return std::exp(-2 * d * d * t0 / Re) * std::expm1(-2 * d * d * (t1 - t0) / Re);
}

__device__ inline double eval_at(const DGrid& g, const FnDesc& f, int s, int c, double t, int i, int j, int k) {
  return fn_eval(f, c, t, coord(g, 0, s, i), coord(g, 1, s, j), coord(g, 2, s, k));
}

// Weight of owner index i along axis a in the left null vector of the 1-D
// operator the solve inverts: uniform on periodic and cell-centred axes,
// trapezoid (1/2 at the two end nodes) on node Neumann axes.
__device__ inline double owner_weight(const DGrid& g, int a, int i) {
  if (g.periodic[a] || g.cell[a]) return 1.0;
  return (i == 0 || i == g.npts[a] - 1) ? 0.5 : 1.0;
}

// Workgroups of a launch are dispatched round-robin over the 8 XCDs of the
// device, each with its own L2.  Mapping the dispatch index b of n
// workgroups to this tile index gives every XCD one contiguous range of
// tiles, so tiles that share halo lines run on the same L2.  A bijection on
// [0, n).
__device__ inline int xcd_tile(int b, int n) {
  constexpr int NXCD = 8;
  const int per = n / NXCD, rem = n % NXCD, x = b % NXCD;
  return x * per + (x < rem ? x : rem) + b / NXCD;
}

}  // namespace mif
