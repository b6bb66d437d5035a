// k_plane.h -- complex helpers and the plane tables shared by the kernels that
// factor and solve the per-kz plane systems.
#pragma once

#include <hip/hip_runtime.h>

#include "hz_internal.h"

namespace hz {
namespace {

template <typename T> struct Cx;
template <> struct Cx<float> { typedef float2 t; };
template <> struct Cx<double> { typedef double2 t; };

template <typename C> __device__ __forceinline__ C mk(double x, double y) { C r; r.x = x; r.y = y; return r; }
template <typename C> __device__ __forceinline__ C cmul(C a, C b) {
  C r; r.x = a.x * b.x - a.y * b.y; r.y = a.x * b.y + a.y * b.x; return r;
}
template <typename C> __device__ __forceinline__ C cfma(C a, C b, C c) {  // a*b + c
  C r; r.x = a.x * b.x - a.y * b.y + c.x; r.y = a.x * b.y + a.y * b.x + c.y; return r;
}
template <typename C> __device__ __forceinline__ C cinv(C a) {
  // 1/a with scaling to avoid overflow in |a|^2
  double ax = a.x, ay = a.y;
  double s = fmax(fabs(ax), fabs(ay));
  C r;
  if (s == 0.0) { r.x = ax / 0.0; r.y = 0; return r; }
  double bx = ax / s, by = ay / s;
  double d = s * (bx * bx + by * by);
  r.x = bx / d; r.y = -by / d;
  return r;
}


typedef float hz_v4f __attribute__((ext_vector_type(4)));
typedef double hz_v4d __attribute__((ext_vector_type(4)));

}  // namespace

// Coefficient tables of the plane systems (device pointers).
struct PlaneTabs {
  const double2* cmx;
  const double2* cpx;
  const double2* cdx;
  const double2* cdy;
  const double2* kappa;
  const double* lamz;
  const double2* sig;
};

// The factor chains of k_factor (k_blocktri.hip: mode, m, jbeg and jend as
// there) with every block inverted in registers; false where nx is too wide for
// that in precision prec, and nothing is launched.
bool launch_factor_reg(hz_problem* p, int prec, const PlaneTabs& tb, int blocks, int* st, int mode, int m, void* G,
                       void* Gb, int jbeg, int jend, hipStream_t s);


// Twisted plane solves (k_tri.hip): whether a width has them, the bytes of the
// packed blocks, the packing of the factor chains (G, Gb) into Gtw, and the
// solve of nrhs vectors (wide: complex64 adjoint with the sums in FP64, to
// TRI_WIDE_MAX columns).
constexpr int TRI_WIDE_MAX = 144;
bool tri_available(int nx);
size_t tri_bytes(const hz_problem* p, size_t elem);
void pack_tri(hz_problem* p, int prec, hipStream_t s);
void solve_tri(hz_problem* p, int prec, int nrhs, void* x, bool adjoint, bool wide, hipStream_t s);

// Groups of 8 complex64 right-hand sides on the one-directional factors
// (k_rows.hip): whether a problem has them, and the solve of nrhs vectors.
bool rows_available(const hz_problem* p);
void solve_rows(hz_problem* p, int nrhs, void* x, bool adjoint, hipStream_t s);
// The same on the dense twisted blocks (G below tw_m, Gb from there on), to 208
// columns; wide as for solve_tri.
void solve_rows_twisted(hz_problem* p, int nrhs, void* x, bool adjoint, bool wide, hipStream_t s);

}  // namespace hz
