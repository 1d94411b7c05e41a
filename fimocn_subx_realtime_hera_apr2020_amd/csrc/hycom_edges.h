// The edge interpolation's expressions (hycom_edgvar.F90), shared by the
// kernels that form edge values (hycom_edgvar.hip) and by momtum, which uses
// them without storing them (hycom_momtum.hip).
#pragma once
#include "hycom_internal.h"

namespace fimhip {
namespace hyc {

// the edges before and after edge e of a cell with np edges
__device__ __forceinline__ int e_prev(int e, int np) { return e == 0 ? np - 1 : e - 1; }
__device__ __forceinline__ int e_next(int e, int np) { return e == np - 1 ? 0 : e + 1; }
// a register array's entry at edge e's previous and next edge: with e a
// constant of an unrolled loop, every index is a constant and only the
// wrap-around selects on np (a run-time index would put the array in scratch)
__device__ __forceinline__ double at_prev(const double (&a)[NPP], int e, int np) {
  return e == 0 ? (np == 6 ? a[5] : a[4]) : a[e == 0 ? 0 : e - 1];
}
__device__ __forceinline__ double at_next(const double (&a)[NPP], int e, int np) {
  return e < 4 ? a[e < 4 ? e + 1 : 0] : (e == 4 ? (np == 5 ? a[0] : a[5]) : a[0]);
}
// the extent to which a sidewall is present (hycom_edgvar.F90:479-493; its
// fourth argument is not used)
// (clamped to 0..1: the division is left out where the clamp decides)
__device__ __forceinline__ double blokf(double dp, double plo, double pbx) {
  const double n = plo - pbx, d = hmax(H_EPSIL, dp);
  double b = n <= 0. ? 0. : 1.;
  if (!(n <= 0. || n >= d)) b = n / d;
  return b;
}

// The neighbours' Montgomery potential and specific volume with the sidewall
// blend (hycom_edgvar.F90:367-410): a neighbour's value gives way to the
// cell's own as the layer lies below the neighbour's bottom, and a land
// neighbour's is the cell's own
__device__ __forceinline__ void sidewall(int ci, double di, double pik1, const double (&PB)[NPP], double mi,
                                         const double (&M)[NPP], double svi, const double (&SV)[NPP],
                                         double (&nm)[NPP], double (&ns)[NPP]) {
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const double blok = ci_open(ci, e) ? blokf(di, pik1, PB[e]) : 1.;
    nm[e] = M[e] * (1. - blok) + mi * blok;
    ns[e] = SV[e] * (1. - blok) + svi * blok;
  }
}

// one velocity pair rotated and interpolated to edge e (uvedge's layer loop)
struct UV {
  double u, v;
};
struct Rot {
  double cs[4], sn[4];
};
__device__ __forceinline__ UV uv_edge(const Rot &rt, bool wi, bool wpx, bool wm1, bool wp1,
                                      double ui, double vi, double ux, double vx, double um1, double vm1, double up1,
                                      double vp1) {
  const double *cs = rt.cs, *sn = rt.sn;
  double u1 = cs[0] * ui + sn[0] * vi;
  double v1 = -sn[0] * ui + cs[0] * vi;
  double u2, v2;
  if (wpx) {
    u2 = cs[1] * ux + sn[1] * vx;
    v2 = -sn[1] * ux + cs[1] * vx;
    if (!wi) {          // the neighbour is ocean and the cell is not
      u1 = u2 * H_SLIP;
      v1 = v2 * H_SLIP;
    }
  } else {
    u2 = u1 * H_SLIP;
    v2 = v1 * H_SLIP;
  }
  const double u3 = wm1 ? cs[2] * um1 + sn[2] * vm1 : 0.;
  const double v3 = wm1 ? -sn[2] * um1 + cs[2] * vm1 : 0.;
  const double u4 = wp1 ? cs[3] * up1 + sn[3] * vp1 : 0.;
  const double v4 = wp1 ? -sn[3] * up1 + cs[3] * vp1 : 0.;
  return UV{(8. * (u1 + u2) + u3 + u4) * H_DIVBY18, (8. * (v1 + v2) + v3 + v4) * H_DIVBY18};
}

// The tables of a cell's edges in LDS: the column's lanes load one or two
// values each (a table value that every lane loads for itself costs the
// column's lanes a load each).
constexpr int VT_CS = 0, VT_SN = 4 * NPP, VT_SVE = 8 * NPP, VT_N = 10 * NPP;
__device__ __forceinline__ Rot rot_of(const double *tab, int e) {
  Rot rt;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    rt.cs[j] = tab[VT_CS + e * 4 + j];
    rt.sn[j] = tab[VT_SN + e * 4 + j];
  }
  return rt;
}

}  // namespace hyc
}  // namespace fimhip
