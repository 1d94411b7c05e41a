// HYCOM's edge interpolation (FIMsrc/fim/horizontal/hycom_edgvar.F90,
// bclin_edgvar with uvedge and blokf) on the GPU, in FP64, with the
// reference's operations in its order.  Kernels, lanes over layers as in the
// continuity kernels:
//   hyc_janjic   (janjic_ocn only) the layer-mean geopotential integrated
//                hydrostatically to each layer's mid pressure in the
//                neighbouring columns, nudged below the silhouette depth, and
//                geop_edg from the six results  (200-265, 437-462).
//   hyc_vnorm    total velocities of both leapfrog levels, rotated into each
//                edge's frame from the cell, its neighbour and the two joint
//                neighbours, and their components normal to the edge
//                (6-124, 273-296; hycom_cnuity.F90:98-106); the interface
//                pressure of the mid-time thickness (the column sum through
//                LDS)
//   hyc_edgint   interface pressure and thickness on the edges: each edge's
//                two sequential chains (down from the shallower bottom, then
//                up, limited by the interpolated thickness) run on one lane
//                over increments the column's lanes put in LDS  (300-418)
// A neighbour's column values are loaded once per lane and shared by the
// three edges that use it (as the edge's cell or as a joint neighbour).
//
// fimhip_ocn_edgvar runs these three: cnuity reads of the edges the normal
// velocities and the thickness, and momtum forms what it needs at the edges
// from the cells again.  An edge array is six times a cell array, and the
// kernels are bound by memory: with the reference's nine edge arrays written
// here and read there G7 x 32 layers took 0.82 ms a step in this file's
// kernels and 0.66 in momtum's, and take 0.31 and 0.53.  The public
// edge arrays are formed when one is asked for (ocn_form_edges), by
//   hyc_uvedge   the edge velocities of one leapfrog level, and the kinetic
//                energy on the edges (411-412)
//   hyc_edgint   in its full form, with the edge pressures, Montgomery
//                potential and specific volume
// from the values the interpolation saw, which momtum and cnuity leave in
// place (HycState's dpe, pbe and p0e, HycEdg's other pair of velocities).
#include <type_traits>

#include "hycom_edges.h"

namespace fimhip {
namespace hyc {
namespace {

#define HG(i, k) ed.geop[(size_t)(i) * (kdm + 1) + (k)]
#define HPR(i, e, k) ed.pr_edg[((size_t)(i) * NPP + (e)) * (kdm + 1) + (k)]

template <int LPC>
__global__ void __launch_bounds__(256) hyc_janjic(HycGrid g, HycState s, HycEdg ed) {
  constexpr int CPB = 256 / LPC;
  __shared__ double sp[CPB][LPC + 1], sg[CPB][LPC + 1], sv[CPB][LPC];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k, cc = c.cc;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  const int np = ci_np(ci);
  const double p_lyr = .5 * (HP(i, kk) + HP(i, kk + 1));
  const double glyr = .5 * (HG(i, kk) + HG(i, kk + 1));
  double silhou = 1.e33;        // the shallowest ocean neighbour's bottom
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const double pb = HP(nb[e], kdm);
    if (ci_open(ci, e)) silhou = hmin(silhou, pb);
  }
  const double plyrk = hmin(p_lyr, silhou);
  double gx[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    gx[e] = glyr;
    if (!ci_open(ci, e)) continue;
    const int ipx = nb[e];
    wave_sync();
    for (int j = k; j <= kdm; j += LPC) {
      sp[cc][j] = HP(ipx, j);
      sg[cc][j] = HG(ipx, j);
    }
    if (live) sv[cc][k] = HC(ed.spcifv, ipx, k);
    else sp[cc][k + 1] = 0.;
    wave_sync();
    if (live) {
      // the first layer whose lower interface is not above plyrk, the last
      // layer if none: eight interfaces are read at a time (one at a time,
      // each waits for LDS: G4 x 48 layers took 40 us, this 17)
      int kx = kdm - 1;
      for (int j0 = 0; j0 < kdm - 1; j0 += CHK) {
        int hit = CHK;
#pragma unroll
        for (int j = CHK - 1; j >= 0; j--) hit = sp[cc][j0 + j + 1] < plyrk ? hit : j;
        if (hit < CHK) {
          kx = j0 + hit < kdm - 1 ? j0 + hit : kdm - 1;
          break;
        }
      }
      if (sp[cc][kx + 1] >= plyrk) gx[e] = sg[cc][kx] - sv[cc][kx] * (plyrk - sp[cc][kx]);
    }
  }
  if (!live) return;
  const double tapr = hmax(0., hmin(1., (p_lyr - silhou) / (100. * H_ONEM)));
#pragma unroll
  for (int e = 0; e < NPP; e++)
    if (e < np) gx[e] = (1. - tapr) * gx[e] + tapr * glyr;
#pragma unroll
  for (int e = 0; e < NPP; e++)
    if (e < np)
      HE(ed.geop_edg, i, e, k) =
          (8. * (glyr + gx[e]) + at_prev(gx, e, np) + at_next(gx, e, np)) * H_DIVBY18;
}

// Bound by memory (four cell arrays gathered, two edge arrays written) as long
// as enough waves are in flight: one level at a time in registers (both: 120
// registers and 235 us at G7 x 32 layers; this 223).
template <int LPC>
__global__ void __launch_bounds__(256, 5) hyc_vnorm(HycGrid g, HycState s, HycEdg ed, int leapm, int leapn) {
  constexpr int CPB = 256 / LPC, NRL = (VT_N + LPC - 1) / LPC, NC = NPP + 1;
  __shared__ double sh[CPB][LPC + 1], tab[CPB][VT_N], trop[CPB][4 * NC];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k, cc = c.cc;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  const int np = ci_np(ci);
  const size_t cz = (size_t)nip * kdm;
  const double *um = ed.uclin + (size_t)(leapm - 1) * cz, *vm = ed.vclin + (size_t)(leapm - 1) * cz;
  const double *un = ed.uclin + (size_t)(leapn - 1) * cz, *vn = ed.vclin + (size_t)(leapn - 1) * cz;
  double rv[NRL];
#pragma unroll
  for (int q = 0; q < NRL; q++) {
    const int j = k + q * LPC;
    rv[q] = j < VT_SN    ? g.cs[(size_t)i * NPP * 4 + j]
            : j < VT_SVE ? g.sn[(size_t)i * NPP * 4 + j - VT_SN]
            : j < VT_N   ? g.sve[(size_t)i * NPP * 2 + j - VT_SVE]
                         : 0.;
  }
  double tv = 0.;
  if (k < 4 * NC) {
    const int x = k % NC == 0 ? i : g.prox[i * NPP + k % NC - 1], lv = k < 2 * NC ? leapm : leapn;
    tv = ((k / NC) % 2 == 0 ? ed.utrop : ed.vtrop)[x * 3 + lv - 1];
  }
  const double p0 = HP(i, 0), d = live ? HC(s.dp + (size_t)(leapm - 1) * cz, i, k) : 0.;
#pragma unroll
  for (int q = 0; q < NRL; q++)
    if (k + q * LPC < VT_N) tab[cc][k + q * LPC] = rv[q];
  if (k < 4 * NC) trop[cc][k] = tv;
  // the interface pressure of the mid-time thickness (273-291)
  const double p = col_pres(sh[cc], d, p0, k, kdm);
  if (live) __builtin_nontemporal_store(p, &HP(i, k + 1));
  if (k == kdm - 1) {
    s.pbe[i] = p;
    s.p0e[i] = p0;
  }
  // total velocities (baroclinic + barotropic; a land neighbour's are not used)
  const auto edges = [&](auto sea) {
    const int cj = sea.value ? CI_SEA : ci, nq = sea.value ? 6 : np;
#pragma unroll
    for (int lv = 0; lv < 2; lv++) {
      const double *tr = trop[cc] + 2 * NC * lv, *u = lv == 0 ? um : un, *v = lv == 0 ? vm : vn;
      double ux[NPP], vx[NPP];
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        ux[e] = HC(u, nb[e], kk) + tr[e + 1];
        vx[e] = HC(v, nb[e], kk) + tr[NC + e + 1];
      }
      const double uo = HC(u, i, kk) + tr[0], vo = HC(v, i, kk) + tr[NC];
      double *out = lv == 0 ? s.vnm : s.vnn;
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        if (e >= nq) break;
        const int em1 = e_prev(e, nq), ep1 = e_next(e, nq);
        const UV r = uv_edge(rot_of(tab[cc], e), true, ci_open(cj, e), ci_open(cj, em1), ci_open(cj, ep1), uo, vo,
                             ux[e], vx[e], at_prev(ux, e, nq), at_prev(vx, e, nq), at_next(ux, e, nq),
                             at_next(vx, e, nq));
        const double vnorm = tab[cc][VT_SVE + e * 2 + 1] * r.u - tab[cc][VT_SVE + e * 2] * r.v;
        if (live) __builtin_nontemporal_store(vnorm, &HE(out, i, e, k));
        __builtin_amdgcn_sched_barrier(0);      // an edge's tables at a time in registers
      }
    }
  };
  if (__all(ci == CI_SEA)) edges(std::true_type());
  else edges(std::false_type());
}

// the public edge velocities of leapfrog level 'slot' from the velocities uc,
// vc; with dpm, the interfaces of that thickness from the top one, p0[i * p0s],
// into pres (whose top interface stays) and, with pbe, its bottom
template <int LPC>
__global__ void __launch_bounds__(256) hyc_uvedge(HycGrid g, HycEdg ed, const double *uc, const double *vc, int slot,
                                                  double *ue, double *ve, const double *dpm, const double *p0,
                                                  int p0s, double *pres, double *pbe, double *uvsq) {
  __shared__ double sh[256 / LPC][LPC + 1];
  __shared__ double tab[256 / LPC][VT_SVE];     // the cell's cs then sn, (4,6) each
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  const int np = ci_np(ci);
  const bool wi = ci_wet(ci);
  constexpr int NRL = (VT_SVE + LPC - 1) / LPC;
  double rv[NRL];
#pragma unroll
  for (int q = 0; q < NRL; q++) {
    const int j = k + q * LPC;
    rv[q] = j < VT_SN ? g.cs[(size_t)i * NPP * 4 + j] : j < VT_SVE ? g.sn[(size_t)i * NPP * 4 + j - VT_SN] : 0.;
  }
  const double uo = HC(uc, i, kk) + ed.utrop[i * 3 + slot - 1];
  const double vo = HC(vc, i, kk) + ed.vtrop[i * 3 + slot - 1];
  double ux[NPP], vx[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int x = nb[e];
    const bool wx = ci_open(ci, e);
    const double a = HC(uc, x, kk) + ed.utrop[x * 3 + slot - 1], b = HC(vc, x, kk) + ed.vtrop[x * 3 + slot - 1];
    ux[e] = wx ? a : H_LAND;
    vx[e] = wx ? b : H_LAND;
  }
  if (dpm && wi) {
    const double p = col_pres(sh[c.cc], live ? HC(dpm, i, k) : 0., p0[(size_t)i * p0s], k, kdm);
    if (live) pres[(size_t)i * (kdm + 1) + k + 1] = p;
    if (pbe && k == kdm - 1) pbe[i] = p;
  }
#pragma unroll
  for (int q = 0; q < NRL; q++)
    if (k + q * LPC < VT_SVE) tab[c.cc][k + q * LPC] = rv[q];
  wave_sync();
  const double ui = wi ? uo : H_LAND;
  const double vi = wi ? vo : H_LAND;
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    UV r{0., 0.};
    if (e < np) {
      const int em1 = e_prev(e, np), ep1 = e_next(e, np);
      r = uv_edge(rot_of(tab[c.cc], e), wi, ci_open(ci, e), ci_open(ci, em1), ci_open(ci, ep1), ui, vi, ux[e], vx[e],
                  at_prev(ux, e, np), at_prev(vx, e, np), at_next(ux, e, np), at_next(vx, e, np));
    }
    if (live) {
      __builtin_nontemporal_store(r.u, &HE(ue, i, e, k));
      __builtin_nontemporal_store(r.v, &HE(ve, i, e, k));
      // the kinetic energy on the edges, from the values just stored (0 on
      // land and in a pentagon's sixth slot)
      if (uvsq) __builtin_nontemporal_store(wi && e < np ? .5 * (r.u * r.u + r.v * r.v) : 0., &HE(uvsq, i, e, k));
    }
  }
}

// FULL: all the public arrays, land included, with the interfaces in pres;
// otherwise the thickness on the ocean's edges alone
template <int LPC, bool FULL>
__global__ void __launch_bounds__(256) hyc_edgint(HycGrid g, HycState s, HycEdg ed, const double *dpm,
                                                  const double *pres) {
  constexpr int CPB = 256 / LPC;
  __shared__ double sh_h[CPB][NPP][LPC + 1], sh_t[CPB][NPP][LPC + 1];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  const int i = c.ok ? c.i : 0, k = c.k, cc = c.cc;
  const bool live = c.ok && k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  const bool wet = c.ok && ci_wet(ci);
  int nb[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (FULL && c.ok && !wet) {
#pragma unroll
    for (int e = 0; e < NPP; e++) {
      if (live) {
        __builtin_nontemporal_store(0., &HE(s.dpm_edg, i, e, k));
        __builtin_nontemporal_store(0., &HE(ed.mont_edg, i, e, k));
        __builtin_nontemporal_store(0., &HE(ed.spcv_edg, i, e, k));
      }
      for (int j = k; j <= kdm; j += LPC) __builtin_nontemporal_store(0., &HPR(i, e, j));
    }
  }
  const int np = ci_np(ci);
  double di = 0.;
  if (wet) {
    di = HC(dpm, i, kk);
    double D[NPP];
#pragma unroll
    for (int e = 0; e < NPP; e++) D[e] = HC(dpm, nb[e], kk);
    // lane e: edge e's lowest interface, the shallower of the two bottoms (0
    // beside land)
    if (k < NPP) sh_h[cc][k][kdm] = ci_open(ci, k) ? hmin(s.pbe[i], s.pbe[g.prox[i * NPP + k]]) : 0.;
    // the increments of each edge's two interface chains; a land neighbour is
    // replaced by the cell itself (300-330)
#pragma unroll
    for (int e = 0; e < NPP; e++) {
      double h = 0., t = 0.;
      if (e < np) {
        const int em1 = e_prev(e, np), ep1 = e_next(e, np);
        const double dx = ci_open(ci, e) ? D[e] : di;
        const double dm1 = ci_open(ci, em1) ? at_prev(D, e, np) : di;
        const double dp1 = ci_open(ci, ep1) ? at_next(D, e, np) : di;
        h = .5 * hmin(hmin(H_TENM, di), dx);
        t = (8. * (di + dx) + dm1 + dp1) * H_DIVBY18;
      }
      if (live) {
        sh_h[cc][e][k] = h;
        sh_t[cc][e][k] = t;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < CPB * NPP) {
    // a lane per edge of the block's columns: its interface pressures down
    // from the lowest, then up, each interface no deeper than the one above
    // plus the interpolated thickness; they replace the increments.  Eight
    // increments are read ahead of the eight interfaces that replace them.
    // (The chains of a wavefront's own columns by that wavefront make four
    // times the LDS instructions, which bound the kernel: 125 us at G7 x 32
    // layers, this 92.  A land column's rows are never read.)
    double *hrow = sh_h[threadIdx.x / NPP][threadIdx.x % NPP];
    const double *trow = sh_t[threadIdx.x / NPP][threadIdx.x % NPP];
    double pr = hrow[kdm];
    int j = kdm - 1;
    for (; j >= CHK; j -= CHK) {
      double h[CHK];
#pragma unroll
      for (int q = 0; q < CHK; q++) h[q] = hrow[j - q];
#pragma unroll
      for (int q = 0; q < CHK; q++) hrow[j - q] = pr = pr - h[q];
    }
    for (; j >= 1; j--) hrow[j] = pr = pr - hrow[j];
    hrow[0] = 0.;
    double prk = 0.;
    j = 0;
    for (; j + CHK <= kdm - 1; j += CHK) {
      double h[CHK], t[CHK];
#pragma unroll
      for (int q = 0; q < CHK; q++) {
        h[q] = hrow[j + 1 + q];
        t[q] = trow[j + q];
      }
#pragma unroll
      for (int q = 0; q < CHK; q++) hrow[j + 1 + q] = prk = hmin(h[q], prk + t[q]);
    }
    for (; j < kdm - 1; j++) hrow[j + 1] = prk = hmin(hrow[j + 1], prk + trow[j]);
  }
  __syncthreads();
  if (!wet) return;
  if (!FULL) {
#pragma unroll
    for (int e = 0; e < NPP; e++)
      if (e < np && live)
        __builtin_nontemporal_store(hmax(0., sh_h[cc][e][k + 1] - sh_h[cc][e][k]), &HE(s.dpm_edg, i, e, k));
    return;
  }
  const double pik1 = pres[(size_t)i * (kdm + 1) + kk + 1];
  const double mi = HC(ed.montg, i, kk), svi = HC(ed.spcifv, i, kk);
  double PB[NPP], M[NPP], SV[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    PB[e] = s.pbe[nb[e]];
    M[e] = HC(ed.montg, nb[e], kk);
    SV[e] = HC(ed.spcifv, nb[e], kk);
  }
  double nm[NPP], ns[NPP];
  sidewall(ci, di, pik1, PB, mi, M, svi, SV, nm, ns);
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    if (e >= np) {
      if (live) {
        __builtin_nontemporal_store(0., &HE(s.dpm_edg, i, e, k));
        __builtin_nontemporal_store(0., &HE(ed.mont_edg, i, e, k));
        __builtin_nontemporal_store(0., &HE(ed.spcv_edg, i, e, k));
      }
      for (int j = k; j <= kdm; j += LPC) __builtin_nontemporal_store(0., &HPR(i, e, j));
      continue;
    }
    const double *hrow = sh_h[cc][e];
    for (int j = k; j <= kdm; j += LPC) __builtin_nontemporal_store(hrow[j], &HPR(i, e, j));
    if (live) {
      __builtin_nontemporal_store(hmax(0., hrow[k + 1] - hrow[k]), &HE(s.dpm_edg, i, e, k));
      __builtin_nontemporal_store((8. * (mi + nm[e]) + at_prev(nm, e, np) + at_next(nm, e, np)) * H_DIVBY18,
                                  &HE(ed.mont_edg, i, e, k));
      __builtin_nontemporal_store((8. * (svi + ns[e]) + at_prev(ns, e, np) + at_next(ns, e, np)) * H_DIVBY18,
                                  &HE(ed.spcv_edg, i, e, k));
    }
  }
}

}  // namespace
}  // namespace hyc
}  // namespace fimhip

using namespace fimhip;
using namespace fimhip::hyc;

template <int LPC>
static void edg_kernels(fimhip_ocn *o, int leapm, int leapn) {
  const HycGrid &g = o->g;
  const HycState &s = o->s;
  const HycEdg &ed = o->ed;
  hipStream_t st = o->stream;
  const dim3 grid(ocn_blocks(o, LPC)), blk(256);
  const double *dpm = s.dp + (size_t)(leapm - 1) * o->nip * o->kdm;
  KT_LAUNCH("hyc_vnorm", st, hyc_vnorm<LPC><<<grid, blk, 0, st>>>(g, s, ed, leapm, leapn));
  KT_LAUNCH("hyc_edgint", st, (hyc_edgint<LPC, false><<<grid, blk, 0, st>>>(g, s, ed, dpm, nullptr)));
}

// the public edge arrays of the instance's current values (now), or of those
// that the last hyc_vnorm saw
template <int LPC>
static void form_kernels(fimhip_ocn *o, int leapm, int leapn, bool now) {
  const HycGrid &g = o->g;
  const HycState &s = o->s;
  HycEdg ed = o->ed;
  ed.uclin = ed.uclin_e; ed.vclin = ed.vclin_e;
  ed.utrop = ed.utrop_e; ed.vtrop = ed.vtrop_e; ed.montg = ed.montg_e; ed.spcifv = ed.spcifv_e;
  hipStream_t st = o->stream;
  const dim3 grid(ocn_blocks(o, LPC)), blk(256);
  const size_t cz = (size_t)o->nip * o->kdm, om = (leapm - 1) * cz, on = (leapn - 1) * cz;
  const double *dpm = !now && o->e_dp_old ? s.dpe : s.dp + om;
  double *pres = now ? s.pres : o->pres_f;
  KT_LAUNCH("hyc_uvedge", st, hyc_uvedge<LPC><<<grid, blk, 0, st>>>(g, ed, ed.uclin + om, ed.vclin + om, leapm, s.um, s.vm,
                                                                    dpm, now ? s.pres : s.p0e, now ? o->kdm + 1 : 1,
                                                                    pres, now ? s.pbe : nullptr, ed.uvsq_edg));
  KT_LAUNCH("hyc_uvedge", st, hyc_uvedge<LPC><<<grid, blk, 0, st>>>(g, ed, ed.uclin + on, ed.vclin + on, leapn, s.un, s.vn,
                                                                    nullptr, nullptr, 0, nullptr, nullptr, nullptr));
  KT_LAUNCH("hyc_edgint_full", st, (hyc_edgint<LPC, true><<<grid, blk, 0, st>>>(g, s, ed, dpm, pres)));
}

template <int LPC>
static void janjic_kernel(fimhip_ocn *o) {
  const dim3 grid(ocn_blocks(o, LPC)), blk(256);
  KT_LAUNCH("hyc_janjic", o->stream, hyc_janjic<LPC><<<grid, blk, 0, o->stream>>>(o->g, o->s, o->ed));
}

// bclin_edgvar on the device-resident arrays (hycom_edgvar.F90:128-478); full:
// with the public edge arrays at once, for a caller that takes them all
static int edg_launch(fimhip_ocn *o, int leapm, int leapn, bool full) {
  if (leapm < 1 || leapm > 2 || leapn < 1 || leapn > 2 || leapm == leapn) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  if (full) {
    const int r = ocn_need_edges(o);
    if (r) return r;
  }
  HycEdg &ed = o->ed;
  ed.uclin_e = ed.uclin; ed.vclin_e = ed.vclin; ed.utrop_e = ed.utrop; ed.vtrop_e = ed.vtrop;
  ed.montg_e = ed.montg; ed.spcifv_e = ed.spcifv;
  const bool l32 = o->kdm <= 32;
  g_ktimer = o->kt;
  if (o->janjic) l32 ? janjic_kernel<32>(o) : janjic_kernel<64>(o);
  if (full) l32 ? form_kernels<32>(o, leapm, leapn, true) : form_kernels<64>(o, leapm, leapn, true);
  else l32 ? edg_kernels<32>(o, leapm, leapn) : edg_kernels<64>(o, leapm, leapn);
  g_ktimer = nullptr;
  o->edges_due = !full;
  o->e_leapm = leapm;
  o->e_leapn = leapn;
  o->e_dp_old = o->e_uv_old = false;
  HIPCHK(hipGetLastError());
  return FIMHIP_OK;
}

int ocn_form_edges(fimhip_ocn *o) {
  if (!o->edges_due) return FIMHIP_OK;
  const int r = ocn_need_edges(o);
  if (r) return r;
  g_ktimer = o->kt;
  if (o->kdm <= 32) form_kernels<32>(o, o->e_leapm, o->e_leapn, false);
  else form_kernels<64>(o, o->e_leapm, o->e_leapn, false);
  g_ktimer = nullptr;
  o->edges_due = false;
  HIPCHK(hipGetLastError());
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_set_janjic(fimhip_ocn *o, int on) {
  if (!o) return FIMHIP_EINVAL;
  o->janjic = on != 0;
  return FIMHIP_OK;
}

// asynchronous on the instance's stream: the continuity step, a download or a
// profile report that follows waits for it
extern "C" int fimhip_ocn_edgvar(fimhip_ocn *o, int leapm, int leapn) {
  if (!o) return FIMHIP_EINVAL;
  return edg_launch(o, leapm, leapn, false);
}

extern "C" int fimhip_ocn_edgvar_r8(fimhip_ocn *o, int nstep, int leapm, int leapn, const double *uclin,
                                   const double *vclin, const double *utrop, const double *vtrop, const double *dp,
                                   double *pres, const double *geop, const double *montg, const double *spcifv,
                                   double *um_edg, double *vm_edg, double *un_edg, double *vn_edg, double *dp_edg,
                                   double *pr_edg, double *geop_edg, double *mont_edg, double *uvsq_edg,
                                   double *spcv_edg) {
  (void)nstep;      // the reference uses it for diagnostics only
  if (!o || !uclin || !vclin || !utrop || !vtrop || !dp || !pres || !geop || !montg || !spcifv || !um_edg ||
      !vm_edg || !un_edg || !vn_edg || !dp_edg || !pr_edg || !geop_edg || !mont_edg || !uvsq_edg || !spcv_edg)
    return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  // inputs, and the one output bclin_edgvar leaves partly untouched (geop_edg
  // outside the ocean, and entirely without janjic_ocn)
  const double *in[] = {uclin, vclin, utrop, vtrop, dp, pres, geop, montg, spcifv, geop_edg};
  const int fi[] = {FIMHIP_OCN_UCLIN, FIMHIP_OCN_VCLIN, FIMHIP_OCN_UTROP, FIMHIP_OCN_VTROP, FIMHIP_OCN_DP,
                    FIMHIP_OCN_PRES, FIMHIP_OCN_GEOP, FIMHIP_OCN_MONTG, FIMHIP_OCN_SPCIFV, FIMHIP_OCN_GEOP_EDG};
  const int nin = o->janjic ? 10 : 9;
  int r = 0;
  for (int j = 0; j < nin; j++)
    if ((r = ocn_put(o, fi[j], in[j]))) return r;
  if ((r = edg_launch(o, leapm, leapn, true))) return r;
  double *outp[] = {pres, um_edg, vm_edg, un_edg, vn_edg, dp_edg, pr_edg, mont_edg, uvsq_edg, spcv_edg, geop_edg};
  const int fo[] = {FIMHIP_OCN_PRES, FIMHIP_OCN_UM_EDG, FIMHIP_OCN_VM_EDG, FIMHIP_OCN_UN_EDG, FIMHIP_OCN_VN_EDG,
                    FIMHIP_OCN_DPM_EDG, FIMHIP_OCN_PR_EDG, FIMHIP_OCN_MONT_EDG, FIMHIP_OCN_UVSQ_EDG,
                    FIMHIP_OCN_SPCV_EDG, FIMHIP_OCN_GEOP_EDG};
  const int nout = o->janjic ? 11 : 10;
  for (int j = 0; j < nout; j++)
    if ((r = ocn_get(o, fo[j], outp[j]))) return r;
  HIPCHK(hipStreamSynchronize(o->stream));
  return FIMHIP_OK;
}
