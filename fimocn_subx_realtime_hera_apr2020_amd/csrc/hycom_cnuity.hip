// The HYCOM ocean's continuity equation (FIMsrc/fim/horizontal/hycom_cnuity.F90,
// subroutine cnuity) on the GPU, in FP64, for a grid whose cells are ocean
// or land (wet).
//
// Each column runs on LPC lanes of a wavefront (LPC = 32 for up to 32
// layers, two columns per wavefront; 64 otherwise), lane k holding layer k.
// Every operation is the reference's, in its order: the sums over a cell's
// edges run in edge order per lane, and the two sums the reference forms
// along the column (interface pressure pres(k+1) = pres(k) + dp(k), and the
// clipped part of each edge's flux) are exact sequential chains over values
// the column's lanes exchange through LDS (a column never leaves its
// wavefront, so the exchange needs no workgroup barrier).  The neighbour
// values of all six edges are loaded unconditionally (every neighbour index
// is a valid cell) and the land/sea mask selects afterwards, so each lane has
// all its gathers in flight at once; a per-cell word packs the edge count,
// the cell's own mask and the mask of its six neighbours.  Blocks are ordered
// so that each XCD works on a contiguous eighth of the cells and neighbour
// rows are found in its L2.  A kernel boundary stands wherever a stage reads
// a neighbour's value that the previous stage writes:
//   hyc_normal   the edges' normal velocities from uploaded edge velocities
//                (fimhip_ocn_edgvar leaves them formed)
//   hyc_flux     low/high-order edge fluxes (98-159), low-order thickness and
//                the in/outflow sums of the antidiffusive fluxes (169-265)
//   hyc_limits   local bounds and limiter ratios              (269-300)
//   hyc_clip     thickness after the limited antidiffusive fluxes, the
//                clipped parts' column sums                    (315-393)
//   hyc_recover  the clipped flux as a barotropic correction and its
//                thickness update; dp from pres               (434-548)
//   hyc_del2p    the biharmonic del2p from the neighbours     (553-603)
//   hyc_bolus    the ratio of each layer to its interface-slope bolus outflow
//                (biharmonic form only)                       (605-683)
//   hyc_bclip    clipped bolus fluxes and update              (685-776)
//   hyc_final    the edge mass flux of all stages, the mass-flux average, the
//                leapfrog time smoothing, the bottom pressure (778-954)
// All of these are bound by memory, and an edge array (six values per cell
// and layer) is six times a cell array, so only three are kept between the
// kernels: the low-order flux, the antidiffusive flux and, at the end, the
// mass flux.  The mass flux of the stages in between is not updated in
// memory: hyc_final forms the limited flux and both barotropic corrections
// again from cell values, and the bolus flux is formed by each kernel that
// reads it.  (With every stage's flux in memory, and the fluxes' sums in a
// kernel of their own, G7 x 32 layers took 1.46 ms a step in these kernels;
// this takes 1.24.)
// A stage's thickness has an array of its own where the next stage reads it
// at the neighbours.
// The duplicate-flux check (chkdup) compares each pair of edge fluxes once
// and sets a flag; the global mass and its drift correction (glob2d) are
// summed on the host in cell order, as the reference does serially.
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "hycom_internal.h"

namespace fimhip {
namespace hyc {
namespace {


// the normal velocities of the ocean's edges from the edge velocities (98-106)
template <int LPC>
__global__ void __launch_bounds__(256) hyc_normal(HycGrid g, HycState s) {
  const int kdm = g.kdm;
  const Col<LPC> c = hcol<LPC>(g.nip);
  if (!c.ok || c.k >= kdm) return;
  const int i = c.i, k = c.k;
  if (!ci_wet(g.cinfo[i])) return;
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    HE(s.vnm, i, e, k) = HSVE(i, e, 1) * HE(s.um, i, e, k) - HSVE(i, e, 0) * HE(s.vm, i, e, k);
    HE(s.vnn, i, e, k) = HSVE(i, e, 1) * HE(s.un, i, e, k) - HSVE(i, e, 0) * HE(s.vn, i, e, k);
  }
}

// the edge fluxes, every cell its own six (the expression of either side of
// an edge is the other's with the roles exchanged), and their sums.  Bound by
// memory: three edge arrays read at the cell and its neighbours' matching
// edges, two written; forming each pair once, by the cell of lower index,
// would read less from the caches and not from HBM, and would need the sums
// in a second pass over both fluxes.
template <int LPC>
__global__ void __launch_bounds__(256) hyc_flux(HycGrid g, HycState s, int leapm, int leapn, double dtleap) {
  __shared__ double scf[256 / LPC][NPP];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int ix[NPP], ex[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    ix[e] = g.prox[i * NPP + e];
    ex[e] = g.proxs[i * NPP + e];
  }
  if (!ci_wet(ci)) {      // (no work array is read on land)
    if (live)
#pragma unroll
      for (int e = 0; e < NPP; e++) __builtin_nontemporal_store(H_LAND, &HE(s.massflx, i, e, k));
    return;
  }
  const double *dpm = s.dp + (size_t)(leapm - 1) * nip * kdm, *dpn = s.dp + (size_t)(leapn - 1) * nip * kdm;
  const int np = ci_np(ci);
  const double mi = HC(dpm, i, kk), d = HC(dpn, i, kk);
  // lane e: the sum of both sides' time step over the length scale of edge e
  if (k < NPP) {
    const int x = g.prox[i * NPP + k] * NPP + g.proxs[i * NPP + k], a = i * NPP + k;
    scf[c.cc][k] = g.rsideln[a] * dtleap * g.rprox_ln[a] + g.rsideln[x] * dtleap * g.rprox_ln[x];
  }
  wave_sync();
  double flx = 0., fp = H_EPSIL, fm = -H_EPSIL;
  // two edges at a time: the six would hold 62 values in flight, and 12
  // waves a compute unit are too few for the loads' latency
  constexpr int HF = 2;
#pragma unroll
  for (int e0 = 0; e0 < NPP; e0 += HF) {
    double va[HF], vb[HF], na[HF], nb[HF], da[HF], db[HF], mx[HF], nx[HF];
#pragma unroll
    for (int h = 0; h < HF; h++) {
      const int e = e0 + h;
      va[h] = HE(s.vnm, i, e, kk);
      vb[h] = HE(s.vnm, ix[e], ex[e], kk);
      da[h] = HE(s.dpm_edg, i, e, kk);
      db[h] = HE(s.dpm_edg, ix[e], ex[e], kk);
      mx[h] = HC(dpm, ix[e], kk);
      na[h] = HE(s.vnn, i, e, kk);
      nb[h] = HE(s.vnn, ix[e], ex[e], kk);
      nx[h] = HC(dpn, ix[e], kk);
    }
#pragma unroll
    for (int h = 0; h < HF; h++) {
      const int e = e0 + h;
      const bool open = ci_open(ci, e);
      const double outgom = .5 * (va[h] - vb[h]);
      const double q = hmin(fabs(outgom) * .5 * scf[c.cc][e], 1.);
      const double dpedg = .5 * (da[h] + db[h]);
      double hi = dpedg * (1. - q) + (outgom >= 0. ? mi : mx[h]) * q;
      hi = hi * outgom;
      const double outgon = .5 * (na[h] - nb[h]);
      const double lo = outgon * (outgon >= 0. ? d : nx[h]);
      const double anti = hi - lo;
      // an edge to land carries no flux; a pentagon's sixth slot is land-valued
      if (live) {
        __builtin_nontemporal_store(open ? lo : e < np ? 0. : H_LAND, &HE(s.massflx, i, e, k));
        if (open) __builtin_nontemporal_store(anti, &HE(s.antiflx, i, e, k));
      }
      if (open) {
        flx = flx + lo;
        if (anti >= 0.) fp = fp + anti;
        else fm = fm + anti;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!live) return;
  double lo = d - flx * g.rarea[i] * dtleap;
  if (lo < 0. && lo + H_ONECM > 0.) lo = 0.;
  __builtin_nontemporal_store(lo, &HC(s.dp_lo, i, k));
  __builtin_nontemporal_store(fp, &HC(s.flxplus, i, k));
  __builtin_nontemporal_store(fm, &HC(s.flxmnus, i, k));
}

template <int LPC>
__global__ void __launch_bounds__(256) hyc_limits(HycGrid g, HycState s, int leapn, double dtleap) {
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok || c.k >= kdm) return;
  const int i = c.i, k = c.k;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  const double *dpn = s.dp + (size_t)(leapn - 1) * nip * kdm;
  const double lo = HC(s.dp_lo, i, k), dn = HC(dpn, i, k);
  double dpmax = hmax(lo, dn), dpmin = hmin(lo, dn);
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int ix = nb[e];
    const double a = HC(s.dp_lo, ix, k), b = HC(dpn, ix, k);
    const double nmax = hmax(hmax(dpmax, a), b), nmin = hmin(hmin(dpmin, a), b);
    const bool open = ci_open(ci, e);
    dpmax = open ? nmax : dpmax;
    dpmin = open ? nmin : dpmin;
  }
  dpmin = hmax(0., dpmin);
  __builtin_nontemporal_store((lo - dpmin) * g.area[i] / (dtleap * HC(s.flxplus, i, k)), &HC(s.rmnus, i, k));
  __builtin_nontemporal_store((lo - dpmax) * g.area[i] / (dtleap * HC(s.flxmnus, i, k)), &HC(s.rplus, i, k));
}

// the limiter of an edge's antidiffusive flux a towards a neighbour with the
// ratios rpx, rmx (315-336)
__device__ __forceinline__ double anti_clip(double a, double rpi, double rmi, double rpx, double rmx) {
  return a >= 0. ? hmin(hmin(1., rmi), rpx) : hmin(hmin(1., rpi), rmx);
}
// the barotropic flux that returns an edge's clipped sum cl (434-453): upstream,
// by the layer's share of the column; that of the bolus fluxes (778-795) forms
// its product in another order
__device__ __forceinline__ double baro_flux(double cl, double di, double rpi, double dx, double rpx) {
  return cl > 0. ? cl * (di * rpi) : (cl < 0. ? cl * (dx * rpx) : 0.);
}
__device__ __forceinline__ double baro_flux_b(double cl, double di, double rpi, double dx, double rpx) {
  return cl > 0. ? cl * di * rpi : (cl < 0. ? cl * dx * rpx : 0.);
}

template <int LPC>
__global__ void __launch_bounds__(256) hyc_clip(HycGrid g, HycState s, double dtleap) {
  __shared__ double sh[256 / LPC][NPP][LPC + 1];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) {
    if (k < NPP) s.clippd[i * NPP + k] = 0.;
    return;
  }
  const double rmi = HC(s.rmnus, i, kk), rpi = HC(s.rplus, i, kk);
  double part[NPP], flx = 0.;
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int ix = nb[e];
    const double a = HE(s.antiflx, i, e, kk);
    const double clip = anti_clip(a, rpi, rmi, HC(s.rplus, ix, kk), HC(s.rmnus, ix, kk));
    const bool open = ci_open(ci, e);
    part[e] = open && live ? a * (1. - clip) : 0.;
    flx = open ? flx + a * clip : flx;
  }
  const double cl = col_sums6<LPC>(sh[c.cc], part, k, kdm);
  if (k < NPP) s.clippd[i * NPP + k] = cl;
  double d = 0.;
  if (live) {
    d = HC(s.dp_lo, i, k) - flx * g.rarea[i] * dtleap;
    if (d < 0. && d + H_ONECM > 0.) d = 0.;
    __builtin_nontemporal_store(d, &HC(s.dpc, i, k));
  }
  const double p = col_pres(sh[c.cc][0], d, HP(i, 0), k, kdm);
  if (k == kdm - 1) s.rpbot[i] = 1. / p;
}

// the clipped fluxes back as an upstream barotropic correction and its
// thickness update (434-491); with interface smoothing, dp again from the
// interface pressures (508-548)
template <int LPC>
__global__ void __launch_bounds__(256) hyc_recover(HycGrid g, HycState s, double dtleap, int smooth) {
  __shared__ double sh[256 / LPC][LPC + 1];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  const double dci = HC(s.dpc, i, kk), rpi = s.rpbot[i];
  double flx = 0.;
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int ix = nb[e];
    const double q = baro_flux(s.clippd[i * NPP + e], dci, rpi, HC(s.dpc, ix, kk), s.rpbot[ix]);
    flx = ci_open(ci, e) ? flx + q : flx;
  }
  double d = 0.;
  if (live) {
    d = dci - flx * g.rarea[i] * dtleap;
    if (d < 0. && d + H_ONECM > 0.) d = 0.;
  }
  const double p0 = HP(i, 0);
  const double p = col_pres(sh[c.cc], d, p0, k, kdm);
  const double pa = __shfl_up(p, 1, LPC);
  const double pk = k > 0 ? pa : p0;         // the interface above layer k
  if (!live) return;
  __builtin_nontemporal_store(p, &HP(i, k + 1));
  __builtin_nontemporal_store(smooth ? p - pk : d, &HC(s.dpr, i, k));
}

template <int LPC>
__global__ void __launch_bounds__(256) hyc_del2p(HycGrid g, HycState s, double biharm) {
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok || c.k >= kdm || c.k < 1) return;
  const int i = c.i, k = c.k;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  double sum = 0.;
  const double pi = HP(i, k), pbi = HP(i, kdm);
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int ix = nb[e];
    const double px = HP(ix, k), pbx = HP(ix, kdm);
    double deltap;
    if (pbx < pi) deltap = pbx - px;
    else if (pbi < px) deltap = pi - pbi;
    else deltap = pi - px;
    sum = ci_open(ci, e) ? sum + deltap : sum;
  }
  const int ncount = __builtin_popcount((ci >> 4) & 63);
  __builtin_nontemporal_store(biharm * sum / (double)ncount + (1. - biharm) * pi, &HC(s.del2p, i, k));
}

// The bolus fluxes of a cell's six edges at lane k's layer (605-646): the
// flux of each interface between two layers, limited to what either side
// holds below it, and the layer's as the difference of its two interfaces'.
// del2p is the interface pressure itself unless the form is biharmonic.
// ed: a few LDS words per edge, filled here by lane e of the column with what
// the neighbour's column has one of (each lane loading them for itself costs
// the column a load per edge and value)
template <int LPC>
__device__ __forceinline__ void bolus_fluxes(const HycGrid &g, const HycState &s, int i, int ci, const int (&nb)[NPP],
                                             int k, double dtleap, double thkdff, double biharm,
                                             double (*ed)[NPP], double (&f)[NPP]) {
  const int kdm = g.kdm;
  const int kk = k < kdm ? k : 0;
  double pxk[NPP], dx[NPP];
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    pxk[e] = HP(nb[e], kk);
    dx[e] = biharm > 0. ? HC(s.del2p, nb[e], kk) : 0.;
  }
  if (k < NPP) {
    const int x = g.prox[i * NPP + k];
    ed[0][k] = HP(x, kdm);
    ed[1][k] = g.area[x];
    ed[2][k] = (double)ci_np(g.cinfo[x]);
    ed[3][k] = g.sideln[i * NPP + k];
  }
  const double pik = HP(i, kk), pbi = HP(i, kdm);
  const double di = biharm > 0. ? HC(s.del2p, i, kk) : pik;
  const double flxmn = -((pbi - pik) * g.area[i] / (double)ci_np(ci));
  wave_sync();
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    // the limited flux of interface k (between layers k-1 and k), lanes 1..kdm-1
    const double q = dtleap * thkdff * (di - (biharm > 0. ? dx[e] : pxk[e])) * ed[3][e];
    const double flxmx = (ed[0][e] - pxk[e]) * ed[1][e] / ed[2][e];
    const double b = k >= 1 && k < kdm ? hmin(flxmx * .999, hmax(flxmn * .999, q)) : 0.;
    // layer k's flux: interface k+1's minus interface k's (0 above the top),
    // the bottom layer minus interface kdm-1's
    const double bn = __shfl_down(b, 1, LPC);
    f[e] = ci_open(ci, e) ? (k < kdm - 1 ? bn - b : -b) : 0.;
  }
}

// the ratio of each layer's mass to its bolus outflow (664-683)
template <int LPC>
__global__ void __launch_bounds__(256) hyc_bolus(HycGrid g, HycState s, double dtleap, double thkdff, double biharm) {
  __shared__ double sed[256 / LPC][4][NPP];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  const double dr = HC(s.dpr, i, k < kdm ? k : 0);
  double f[NPP], fp = H_EPSIL;
  bolus_fluxes<LPC>(g, s, i, ci, nb, k, dtleap, thkdff, biharm, sed[c.cc], f);
#pragma unroll
  for (int e = 0; e < NPP; e++)
    if (e < ci_np(ci)) fp = fp + hmax(0., f[e]);
  if (k < kdm) __builtin_nontemporal_store(dr * g.area[i] / fp, &HC(s.brat, i, k));
}

template <int LPC>
__global__ void __launch_bounds__(256) hyc_bclip(HycGrid g, HycState s, double dtleap, double thkdff, double biharm,
                                                 double masscor) {
  __shared__ double sh[256 / LPC][NPP][LPC + 1], sed[256 / LPC][4][NPP];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) {
    if (biharm > 0. && k < NPP) s.clippb[i * NPP + k] = 0.;
    return;
  }
  const int np = ci_np(ci);
  const double p0 = HP(i, 0), dr = HC(s.dpr, i, kk);
  double f[NPP], part[NPP], flx = 0.;
  bolus_fluxes<LPC>(g, s, i, ci, nb, k, dtleap, thkdff, biharm, sed[c.cc], f);
  const double rmi = HC(s.brat, i, kk);
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    double b = f[e], pt = 0.;
    if (biharm > 0.) {
      const double clip = b > 0. ? hmin(1., rmi) : hmin(1., HC(s.brat, nb[e], kk));
      const bool doit = ci_open(ci, e) && b != 0.;
      pt = doit ? b * (1. - clip) : 0.;
      b = doit ? b * clip : b;
    }
    part[e] = live ? pt : 0.;
    if (e < np) flx = flx + b;
  }
  if (biharm > 0.) {
    const double cl = col_sums6<LPC>(sh[c.cc], part, k, kdm);
    if (k < NPP) s.clippb[i * NPP + k] = cl;
  }
  double d = 0.;
  if (live) {
    d = dr - flx * g.rarea[i];
    if (d < 0. && d + H_ONECM > 0.) d = 0.;
    d = d * (1. + masscor);
    __builtin_nontemporal_store(d, &HC(s.dptmp, i, k));
  }
  // (the interfaces themselves are read at the neighbours by this kernel:
  // hyc_final stores the new ones)
  const double p = col_pres(sh[c.cc][0], d, p0, k, kdm);
  if (k == kdm - 1) s.rpbotb[i] = 1. / p;
}

// The mass flux of all stages, from the low-order and antidiffusive fluxes and
// the stages' cell values, and the last thickness.  Bound by memory: three
// edge arrays read and two written.
template <int LPC>
__global__ void __launch_bounds__(256, 4) hyc_final(HycGrid g, HycState s, int leapm, int leapn, double dtleap,
                                                 int smooth, double biharm) {
  __shared__ double sh[256 / LPC][LPC + 1], sed[256 / LPC][4][NPP];
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok) return;
  const int i = c.i, k = c.k;
  const bool live = k < kdm;
  const int kk = live ? k : 0;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) {
    if (k == 0) s.aux[i] = 0.;
    return;
  }
  double *dpm = s.dp + (size_t)(leapm - 1) * nip * kdm, *dpn = s.dp + (size_t)(leapn - 1) * nip * kdm;
  const int np = ci_np(ci);
  const double p0 = HP(i, 0);
  const double rmi = HC(s.rmnus, i, kk), rpi = HC(s.rplus, i, kk);
  const double dci = HC(s.dpc, i, kk), rbi = s.rpbot[i];
  // lane e: what edge e's two columns have one of
  double (*ed)[NPP] = sed[c.cc];
  if (k < NPP) {
    const int x = g.prox[i * NPP + k];
    ed[0][k] = s.clippd[i * NPP + k];
    ed[1][k] = s.rpbot[x];
    ed[2][k] = s.clippb[i * NPP + k];
    ed[3][k] = s.rpbotb[x];
  }
  wave_sync();
  double mf[NPP];
  constexpr int HF = 3;      // three edges at a time in registers, for more waves in flight
#pragma unroll
  for (int e0 = 0; e0 < NPP; e0 += HF) {
    double af[HF], rpx[HF], rmx[HF], dcx[HF];
#pragma unroll
    for (int h = 0; h < HF; h++) {
      const int e = e0 + h;
      mf[e] = HE(s.massflx, i, e, kk);
      af[h] = HE(s.antiflx, i, e, kk);
      rpx[h] = HC(s.rplus, nb[e], kk);
      rmx[h] = HC(s.rmnus, nb[e], kk);
      dcx[h] = HC(s.dpc, nb[e], kk);
    }
#pragma unroll
    for (int h = 0; h < HF; h++) {
      const int e = e0 + h;
      const double clip = anti_clip(af[h], rpi, rmi, rpx[h], rmx[h]);
      const double q = baro_flux(ed[0][e], dci, rbi, dcx[h], ed[1][e]);
      mf[e] = ci_open(ci, e) ? mf[e] + af[h] * clip + q : mf[e];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  double dn = HC(smooth ? s.dptmp : s.dpr, i, kk), av[NPP];
  const double dold = HC(dpn, i, kk), dm = HC(dpm, i, kk);
#pragma unroll
  for (int e = 0; e < NPP; e++) av[e] = smooth ? HE(s.mssfx_avg, i, e, kk) : 0.;
  if (smooth && biharm > 0.) {
    const double dtinv = 1. / dtleap;
    const double dti = dn, rci = s.rpbotb[i];
    double flx = 0.;
#pragma unroll
    for (int e = 0; e < NPP; e++) {
      const int ix = nb[e];
      const double q = baro_flux_b(ed[2][e], dti, rci, HC(s.dptmp, ix, kk), ed[3][e]);
      if (e < np) {
        flx = flx + q;
        mf[e] = mf[e] + q * dtinv;
      }
    }
    dn = dn - flx * g.rarea[i];
  }
  double pb = 0.;
  if (smooth) {
    pb = col_pres(sh[c.cc], live ? dn : 0., p0, k, kdm);
    if (live) __builtin_nontemporal_store(pb, &HP(i, k + 1));
  } else if (k == kdm - 1) {
    pb = HP(i, kdm);
  }
  if (!live) return;
#pragma unroll
  for (int e = 0; e < NPP; e++)
    if (e < np) {
      __builtin_nontemporal_store(mf[e], &HE(s.massflx, i, e, k));
      if (smooth) __builtin_nontemporal_store(av[e] + mf[e], &HE(s.mssfx_avg, i, e, k));
    }
  __builtin_nontemporal_store(dn, &HC(dpn, i, k));
  __builtin_nontemporal_store(dm, &HC(s.dpe, i, k));
  __builtin_nontemporal_store(H_ASSLDP * (dold + dn) + (1. - H_ASSLDP - H_ASSLDP) * dm, &HC(dpm, i, k));
  if (k == kdm - 1) s.aux[i] = pb;
}

// duplicate edge fluxes must be equal and opposite bit for bit (chkdup); the
// cell of lower index checks each pair
template <int LPC>
__global__ void __launch_bounds__(256) hyc_check(HycGrid g, HycState s) {
  const int kdm = g.kdm, nip = g.nip;
  const Col<LPC> c = hcol<LPC>(nip);
  if (!c.ok || c.k >= kdm) return;
  const int i = c.i, k = c.k;
  const int ci = g.cinfo[i];
  int nb[NPP];      // neighbours, loaded before the mask is tested
#pragma unroll
  for (int e = 0; e < NPP; e++) nb[e] = g.prox[i * NPP + e];
  if (!ci_wet(ci)) return;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < NPP; e++) {
    const int ix = nb[e], ex = g.proxs[i * NPP + e];
    if (!ci_open(ci, e) || ix < i) continue;
    const double a = HE(s.massflx, i, e, k), b = HE(s.massflx, ix, ex, k);
    bad = bad || (a + b != 0. && a - b != 0.);
  }
  if (bad) atomicOr(s.flag, 1);
}

}  // namespace
}  // namespace hyc
}  // namespace fimhip

using namespace fimhip;
using namespace fimhip::hyc;

static int ocn_launch(fimhip_ocn *o, int nstep, int leapm, int leapn);

extern "C" int fimhip_ocn_create(const fimhip_grid_desc *gd, const double *rprox_ln, int kdm, const int *wet,
                                 double dtleap, double thkdff, double biharm, int device, fimhip_ocn **out) {
  if (!gd || !rprox_ln || !wet || !out || kdm < 2 || kdm > 64 || gd->nip < 12 || !gd->nprox || !gd->prox ||
      !gd->proxs || !gd->sidevec_e || !gd->sideln || !gd->area || !gd->cs || !gd->sn || !gd->sidevec_c ||
      !gd->lat || !(dtleap > 0.))
    return FIMHIP_EINVAL;
  *out = nullptr;
  int ndev = 0;
  HIPCHK(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) return FIMHIP_ENODEV;
  HIPCHK(hipSetDevice(device));
  fimhip_ocn *o = new fimhip_ocn();
  o->device = device;
  o->nip = gd->nip;
  o->kdm = kdm;
  o->dtleap = dtleap;
  o->thkdff = thkdff;
  o->biharm = biharm;
  if (hipStreamCreate(&o->stream) != hipSuccess) { delete o; return FIMHIP_EHIP; }
  o->arena.stream = o->stream;
  const int nip = gd->nip;
  std::vector<int> prox(nip * NPP), proxs(nip * NPP), nprox(nip);
  std::vector<double> rarea(nip), rsideln(nip * NPP, 0.), sve(nip * NPP * 2), sideln(nip * NPP), rpl(nip * NPP);
  o->wet.assign(wet, wet + nip);
  o->area.assign(gd->area, gd->area + nip);
  for (int i = 0; i < nip; i++) {
    const int np = gd->nprox[i];
    if (np < 5 || np > 6) { fimhip_ocn_destroy(o); return FIMHIP_EINVAL; }
    nprox[i] = np;
    // the reference tests wet > 0 in some places and wet == 0 in others
    if (wet[i] < 0) { fimhip_ocn_destroy(o); return FIMHIP_EINVAL; }
    o->wet[i] = wet[i] > 0 ? 1 : 0;
    rarea[i] = 1. / gd->area[i];
    for (int e = 0; e < NPP; e++) {
      const int ee = e < np ? e : np - 1;            // a pentagon's slot 6 repeats slot 5
      const int x = gd->prox[i * NPP + ee] - 1, xs = gd->proxs[i * NPP + ee] - 1;
      if (x < 0 || x >= nip || xs < 0 || xs >= NPP) { fimhip_ocn_destroy(o); return FIMHIP_EINVAL; }
      prox[i * NPP + e] = x;
      proxs[i * NPP + e] = xs;
      sideln[i * NPP + e] = gd->sideln[i * NPP + e];
      rpl[i * NPP + e] = rprox_ln[i * NPP + e];
      if (e < np) rsideln[i * NPP + e] = 1. / gd->sideln[i * NPP + e];
      sve[(i * NPP + e) * 2] = gd->sidevec_e[(i * NPP + e) * 2];
      sve[(i * NPP + e) * 2 + 1] = gd->sidevec_e[(i * NPP + e) * 2 + 1];
    }
  }
  // every edge's twin must point back (each pair of edge fluxes is formed once)
  for (int i = 0; i < nip; i++)
    for (int e = 0; e < nprox[i]; e++) {
      const int x = prox[i * NPP + e], xs = proxs[i * NPP + e];
      if (xs >= nprox[x] || prox[x * NPP + xs] != i) { fimhip_ocn_destroy(o); return FIMHIP_EINVAL; }
    }
  // the packed per-cell word: edge count, own mask, mask of each edge's neighbour
  std::vector<int> cinfo(nip);
  for (int i = 0; i < nip; i++) {
    int w = nprox[i] | (o->wet[i] << 3);
    for (int e = 0; e < nprox[i]; e++)
      if (o->wet[prox[i * NPP + e]]) w |= 1 << (4 + e);
    cinfo[i] = w;
  }
  int r = 0;
  HycGrid &g = o->g;
  g.nip = nip;
  g.kdm = kdm;
  int *pp, *ps, *pc;
  double *pa, *pr, *pv, *psl, *prs, *prl, *pcs, *psn;
  const std::vector<double> csv(gd->cs, gd->cs + (size_t)nip * NPP * 4), snv(gd->sn, gd->sn + (size_t)nip * NPP * 4);
  const std::vector<double> svcv(gd->sidevec_c, gd->sidevec_c + (size_t)nip * NPP * 2);
  // the momentum equation's cell values, with the C library's sin and sqrt as
  // the reference forms them (dyn_init.F90:753, hycom_init.F90:327)
  std::vector<double> corv(nip), meshv(nip);
  for (int i = 0; i < nip; i++) {
    corv[i] = 1.4584e-4 * sin(gd->lat[i]);
    meshv[i] = sqrt(gd->area[i]);
  }
  double *pvc, *pco, *pms;
  if ((r = o->arena.upload(&pp, prox)) || (r = o->arena.upload(&ps, proxs)) || (r = o->arena.upload(&pc, cinfo)) ||
      (r = o->arena.upload(&pa, o->area)) || (r = o->arena.upload(&pr, rarea)) || (r = o->arena.upload(&pv, sve)) ||
      (r = o->arena.upload(&psl, sideln)) || (r = o->arena.upload(&prs, rsideln)) ||
      (r = o->arena.upload(&prl, rpl)) || (r = o->arena.upload(&pcs, csv)) || (r = o->arena.upload(&psn, snv)) ||
      (r = o->arena.upload(&pvc, svcv)) || (r = o->arena.upload(&pco, corv)) || (r = o->arena.upload(&pms, meshv))) {
    fimhip_ocn_destroy(o);
    return r;
  }
  g.prox = pp; g.proxs = ps; g.cinfo = pc;
  g.area = pa; g.rarea = pr; g.sve = pv; g.sideln = psl; g.rsideln = prs; g.rprox_ln = prl;
  g.cs = pcs; g.sn = psn;
  o->mo.svc = pvc; o->mo.corio = pco; o->mo.meshsz = pms;
  o->mo.veldff = 0.1;              // fimnamelist.F90:254
  o->mo.smagcf = 0.3;              // fimnamelist.F90:253
  const size_t cz = (size_t)nip * kdm, ez = cz * NPP;
  HycState &s = o->s;
  const Arena::Arr arrs[] = {
      {&s.dpm_edg, ez}, {&s.dp, 2 * cz}, {&s.pres, (size_t)nip * (kdm + 1)},
      {&s.massflx, ez}, {&s.mssfx_avg, ez},
      // the edge interpolation's inputs and outputs (the others: ocn_need_edges)
      {&o->ed.uclin, 2 * cz}, {&o->ed.vclin, 2 * cz}, {&o->ed.uclin_alt, 2 * cz}, {&o->ed.vclin_alt, 2 * cz},
      {&o->ed.utrop, (size_t)nip * 3}, {&o->ed.vtrop, (size_t)nip * 3},
      {&o->ed.geop, (size_t)nip * (kdm + 1)}, {&o->ed.montg, cz}, {&o->ed.spcifv, cz},
      {&o->ed.geop_edg, ez},
      // the momentum equation's forcing
      {&o->mo.taux, (size_t)nip}, {&o->mo.tauy, (size_t)nip}, {&o->mo.ustarb, (size_t)nip},
      // the tracers and density the transport and the grid generator share
      {&o->tr.temp, cz}, {&o->tr.saln, cz}, {&o->hy.dens, cz}};
  const Arena::Arr work[] = {
      {&s.vnm, ez}, {&s.vnn, ez}, {&s.antiflx, ez}, {&s.dp_lo, cz}, {&s.dpc, cz}, {&s.dpr, cz}, {&s.flxplus, cz},
      {&s.flxmnus, cz}, {&s.rplus, cz}, {&s.rmnus, cz}, {&s.del2p, cz}, {&s.dptmp, cz}, {&s.brat, cz}, {&s.dpe, cz},
      {&o->mo.d4u, cz}, {&o->mo.d4v, cz}, {&o->mo.gradx, cz}, {&o->mo.grady, cz}, {&o->mo.relvor, cz},
      {&o->mo.visc, cz}, {&o->pres_f, (size_t)nip * (kdm + 1)}, {&s.clippd, (size_t)nip * NPP},
      {&s.clippb, (size_t)nip * NPP}, {&s.rpbot, (size_t)nip}, {&s.rpbotb, (size_t)nip}, {&s.aux, (size_t)nip},
      {&s.pbe, (size_t)nip}, {&s.p0e, (size_t)nip}, {&o->mo.drag, (size_t)nip}, {&o->mo.dpbot, (size_t)nip}};
  if ((r = o->arena.alloc_all(work))) { fimhip_ocn_destroy(o); return r; }
  for (auto &a : arrs)
    if ((r = o->arena.alloc(a.p, a.n))) { fimhip_ocn_destroy(o); return r; }
  if ((r = o->arena.alloc(&s.flag, 1))) { fimhip_ocn_destroy(o); return r; }
  if (hipStreamSynchronize(o->stream) != hipSuccess) { fimhip_ocn_destroy(o); return FIMHIP_EHIP; }
  *out = o;
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_destroy(fimhip_ocn *o) {
  if (!o) return FIMHIP_EINVAL;
  (void)hipSetDevice(o->device);
  if (o->stream) (void)hipStreamSynchronize(o->stream);
  o->arena.release();
  delete o->kt;
  if (o->stream) (void)hipStreamDestroy(o->stream);
  delete o;
  return FIMHIP_OK;
}

double *ocn_field(fimhip_ocn *o, int f, size_t *n) {
  const size_t cz = (size_t)o->nip * o->kdm, ez = cz * NPP;
  HycState &s = o->s;
  switch (f) {
    case FIMHIP_OCN_DP: *n = 2 * cz; return s.dp;
    case FIMHIP_OCN_PRES: *n = (size_t)o->nip * (o->kdm + 1); return s.pres;
    case FIMHIP_OCN_UM_EDG: *n = ez; return s.um;
    case FIMHIP_OCN_VM_EDG: *n = ez; return s.vm;
    case FIMHIP_OCN_UN_EDG: *n = ez; return s.un;
    case FIMHIP_OCN_VN_EDG: *n = ez; return s.vn;
    case FIMHIP_OCN_DPM_EDG: *n = ez; return s.dpm_edg;
    case FIMHIP_OCN_MASSFLX: *n = ez; return s.massflx;
    case FIMHIP_OCN_MSSFX_AVG: *n = ez; return s.mssfx_avg;
    case FIMHIP_OCN_UCLIN: *n = 2 * cz; return o->ed.uclin;
    case FIMHIP_OCN_VCLIN: *n = 2 * cz; return o->ed.vclin;
    case FIMHIP_OCN_UTROP: *n = (size_t)o->nip * 3; return o->ed.utrop;
    case FIMHIP_OCN_VTROP: *n = (size_t)o->nip * 3; return o->ed.vtrop;
    case FIMHIP_OCN_GEOP: *n = (size_t)o->nip * (o->kdm + 1); return o->ed.geop;
    case FIMHIP_OCN_MONTG: *n = cz; return o->ed.montg;
    case FIMHIP_OCN_SPCIFV: *n = cz; return o->ed.spcifv;
    case FIMHIP_OCN_PR_EDG: *n = (size_t)o->nip * NPP * (o->kdm + 1); return o->ed.pr_edg;
    case FIMHIP_OCN_GEOP_EDG: *n = ez; return o->ed.geop_edg;
    case FIMHIP_OCN_MONT_EDG: *n = ez; return o->ed.mont_edg;
    case FIMHIP_OCN_UVSQ_EDG: *n = ez; return o->ed.uvsq_edg;
    case FIMHIP_OCN_SPCV_EDG: *n = ez; return o->ed.spcv_edg;
    case FIMHIP_OCN_TAUX: *n = (size_t)o->nip; return o->mo.taux;
    case FIMHIP_OCN_TAUY: *n = (size_t)o->nip; return o->mo.tauy;
    case FIMHIP_OCN_USTARB: *n = (size_t)o->nip; return o->mo.ustarb;
    case FIMHIP_OCN_CUMUFLX: *n = ez; return o->tr.cumuflx;
    case FIMHIP_OCN_DPINIT: *n = cz; return o->tr.dpinit;
    case FIMHIP_OCN_DPFINL: *n = cz; return o->tr.dpfinl;
    case FIMHIP_OCN_TEMP: *n = cz; return o->tr.temp;
    case FIMHIP_OCN_SALN: *n = cz; return o->tr.saln;
    case FIMHIP_OCN_PASSV: *n = o->tr.numtr * cz; return o->tr.numtr > 0 ? o->tr.passv : nullptr;
    case FIMHIP_OCN_DENS: *n = cz; return o->hy.dens;
  }
  return nullptr;
}

// waits for every asynchronous call queued on the instance
extern "C" int fimhip_ocn_sync(fimhip_ocn *o) {
  if (!o) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  HIPCHK(hipStreamSynchronize(o->stream));
  return FIMHIP_OK;
}

extern "C" long long fimhip_ocn_field_size(const fimhip_ocn *o, int f) {
  if (!o) return FIMHIP_EINVAL;
  size_t n = 0;
  (void)ocn_field(const_cast<fimhip_ocn *>(o), f, &n);
  return n ? (long long)n : FIMHIP_EINVAL;
}

int ocn_need_edges(fimhip_ocn *o) {
  const size_t ez = (size_t)o->nip * o->kdm * NPP;
  const Arena::Arr arrs[] = {{&o->s.um, ez}, {&o->s.vm, ez}, {&o->s.un, ez}, {&o->s.vn, ez},
                             {&o->ed.pr_edg, (size_t)o->nip * NPP * (o->kdm + 1)}, {&o->ed.mont_edg, ez},
                             {&o->ed.uvsq_edg, ez}, {&o->ed.spcv_edg, ez}};
  for (auto &a : arrs) {
    const int r = *a.p ? FIMHIP_OK : o->arena.alloc(a.p, a.n);
    if (r) return r;
  }
  return FIMHIP_OK;
}

// an edge array that fimhip_ocn_edgvar leaves to be formed
static bool lazy_edge(int f) {
  return f == FIMHIP_OCN_UM_EDG || f == FIMHIP_OCN_VM_EDG || f == FIMHIP_OCN_UN_EDG || f == FIMHIP_OCN_VN_EDG ||
         f == FIMHIP_OCN_DPM_EDG || f == FIMHIP_OCN_PR_EDG || f == FIMHIP_OCN_MONT_EDG ||
         f == FIMHIP_OCN_UVSQ_EDG || f == FIMHIP_OCN_SPCV_EDG;
}

// An input that the due edge arrays are formed from is about to be replaced:
// the new values go to its other buffer.  (Forming the arrays, 54 cell arrays of
// which a host that uploads its inputs every step reads none, took 3.0 ms at G8
// x 32 layers beside a step of 8.0.)
static int keep_seen(fimhip_ocn *o, double *&cur, double *&alt, const double *seen, size_t n) {
  if (cur != seen) return FIMHIP_OK;
  if (!alt && o->arena.alloc(&alt, n) != FIMHIP_OK) {
    alt = nullptr;
    (void)hipGetLastError();
    return ocn_form_edges(o);
  }
  std::swap(cur, alt);
  return FIMHIP_OK;
}
static int before_put(fimhip_ocn *o, int f, size_t n) {
  if (!o->edges_due) return FIMHIP_OK;
  if (lazy_edge(f)) return ocn_form_edges(o);
  HycEdg &ed = o->ed;
  switch (f) {
    case FIMHIP_OCN_UTROP: return keep_seen(o, ed.utrop, ed.utrop_alt, ed.utrop_e, n);
    case FIMHIP_OCN_VTROP: return keep_seen(o, ed.vtrop, ed.vtrop_alt, ed.vtrop_e, n);
    case FIMHIP_OCN_MONTG: return keep_seen(o, ed.montg, ed.montg_alt, ed.montg_e, n);
    case FIMHIP_OCN_SPCIFV: return keep_seen(o, ed.spcifv, ed.spcifv_alt, ed.spcifv_e, n);
    case FIMHIP_OCN_UCLIN: return keep_seen(o, ed.uclin, ed.uclin_alt, ed.uclin_e, n);
    case FIMHIP_OCN_VCLIN: return keep_seen(o, ed.vclin, ed.vclin_alt, ed.vclin_e, n);
    case FIMHIP_OCN_DP:
      if (!o->e_dp_old) {
        HIPCHK(hipMemcpyAsync(o->s.dpe, o->s.dp + (size_t)(o->e_leapm - 1) * (n / 2), n / 2 * sizeof(double),
                              hipMemcpyDeviceToDevice, o->stream));
        o->e_dp_old = true;
      }
  }
  return FIMHIP_OK;
}

int ocn_put(fimhip_ocn *o, int f, const double *h) {
  size_t n = 0;
  int r = lazy_edge(f) ? ocn_need_edges(o) : FIMHIP_OK;
  if (r) return r;
  if (!ocn_field(o, f, &n)) return FIMHIP_EINVAL;
  if ((r = before_put(o, f, n))) return r;
  HIPCHK(hipMemcpyAsync(ocn_field(o, f, &n), h, n * sizeof(double), hipMemcpyHostToDevice, o->stream));
  if (f == FIMHIP_OCN_UCLIN || f == FIMHIP_OCN_VCLIN) o->alt_stale = true;
  return FIMHIP_OK;
}

int ocn_get(fimhip_ocn *o, int f, double *h) {
  size_t n = 0;
  if (lazy_edge(f)) {
    int r = ocn_need_edges(o);
    if (r || (r = ocn_form_edges(o))) return r;
  }
  const double *d = ocn_field(o, f, &n);
  if (!d) return FIMHIP_EINVAL;
  HIPCHK(hipMemcpyAsync(h, d, n * sizeof(double), hipMemcpyDeviceToHost, o->stream));
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_upload(fimhip_ocn *o, int f, const double *h) {
  if (!o || !h) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  const int r = ocn_put(o, f, h);
  if (r) return r;
  HIPCHK(hipStreamSynchronize(o->stream));
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_download(fimhip_ocn *o, int f, double *h) {
  if (!o || !h) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  const int r = ocn_get(o, f, h);
  if (r) return r;
  HIPCHK(hipStreamSynchronize(o->stream));
  return FIMHIP_OK;
}

template <int LPC>
static void ocn_kernels(fimhip_ocn *o, int leapm, int leapn) {
  const HycGrid &g = o->g;
  const HycState &s = o->s;
  hipStream_t st = o->stream;
  const dim3 grid(ocn_blocks(o, LPC)), blk(256);     // a multiple of 8 blocks: see hcol
  const double dt = o->dtleap;
  const int smooth = o->thkdff != 0.;
  if (!o->edges_due) KT_LAUNCH("hyc_normal", st, hyc_normal<LPC><<<grid, blk, 0, st>>>(g, s));
  KT_LAUNCH("hyc_flux", st, hyc_flux<LPC><<<grid, blk, 0, st>>>(g, s, leapm, leapn, dt));
  KT_LAUNCH("hyc_limits", st, hyc_limits<LPC><<<grid, blk, 0, st>>>(g, s, leapn, dt));
  KT_LAUNCH("hyc_clip", st, hyc_clip<LPC><<<grid, blk, 0, st>>>(g, s, dt));
  KT_LAUNCH("hyc_recover", st, hyc_recover<LPC><<<grid, blk, 0, st>>>(g, s, dt, smooth));
  if (smooth) {
    if (o->biharm > 0.) {
      KT_LAUNCH("hyc_del2p", st, hyc_del2p<LPC><<<grid, blk, 0, st>>>(g, s, o->biharm));
      KT_LAUNCH("hyc_bolus", st, hyc_bolus<LPC><<<grid, blk, 0, st>>>(g, s, dt, o->thkdff, o->biharm));
    }
    KT_LAUNCH("hyc_bclip", st, hyc_bclip<LPC><<<grid, blk, 0, st>>>(g, s, dt, o->thkdff, o->biharm, o->masscor));
  }
  KT_LAUNCH("hyc_final", st, hyc_final<LPC><<<grid, blk, 0, st>>>(g, s, leapm, leapn, dt, smooth, o->biharm));
  KT_LAUNCH("hyc_check", st, hyc_check<LPC><<<grid, blk, 0, st>>>(g, s));
}

// one call of cnuity on the device-resident arrays (hycom_cnuity.F90:21-361)
static int ocn_launch(fimhip_ocn *o, int nstep, int leapm, int leapn) {
  if (nstep < 1 || leapm < 1 || leapm > 2 || leapn < 1 || leapn > 2 || leapm == leapn) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  // the step keeps the thickness at level leapm for the due edge arrays: a
  // second step, or another level, is a step on the arrays themselves
  if (o->e_dp_old || leapm != o->e_leapm) {
    const int r = ocn_form_edges(o);
    if (r) return r;
  }
  if (!o->edges_due) {
    const int r = ocn_need_edges(o);
    if (r) return r;
  }
  HIPCHK(hipMemsetAsync(o->s.flag, 0, sizeof(int), o->stream));
  g_ktimer = o->kt;
  if (o->kdm <= 32) ocn_kernels<32>(o, leapm, leapn);
  else ocn_kernels<64>(o, leapm, leapn);
  o->e_dp_old = true;
  g_ktimer = nullptr;
  HIPCHK(hipGetLastError());
  // the drift correction of the total mass, at the first step and every 10
  // days (977-998): glob2d sums bottom pressure times area over the ocean in
  // cell order
  const double day = (double)nstep * .5 * o->dtleap / 86400.;
  int flag = 0;
  HIPCHK(hipMemcpyAsync(&flag, o->s.flag, sizeof(int), hipMemcpyDeviceToHost, o->stream));
  if (nstep == 1 || fmod(day + .0001, 10.) < .0002) {
    std::vector<double> pb(o->nip);
    HIPCHK(hipMemcpyAsync(pb.data(), o->s.aux, pb.size() * sizeof(double), hipMemcpyDeviceToHost, o->stream));
    HIPCHK(hipStreamSynchronize(o->stream));
    double tot = 0.;
    for (int i = 0; i < o->nip; i++)
      if (o->wet[i]) tot = tot + pb[i] * o->area[i];
    o->totmass = tot / H_GRVITY;
    if (nstep == 1) o->massglb0 = o->totmass;
    o->masscor = o->dtleap * (o->massglb0 - o->totmass) / (o->massglb0 * 10. * 86400.);
  } else {
    HIPCHK(hipStreamSynchronize(o->stream));
  }
  // the reference stops the program here (chkdup, hycom_cnuity.F90:1030-1075)
  return flag ? FIMHIP_EDUP : FIMHIP_OK;
}

extern "C" int fimhip_ocn_cnuity(fimhip_ocn *o, int nstep, int leapm, int leapn) {
  if (!o) return FIMHIP_EINVAL;
  return ocn_launch(o, nstep, leapm, leapn);
}

extern "C" int fimhip_ocn_cnuity_r8(fimhip_ocn *o, int nstep, int leapm, int leapn, const double *um_edg,
                                   const double *vm_edg, const double *un_edg, const double *vn_edg,
                                   const double *dpm_edg, double *dp, double *pres, double *massflx,
                                   double *mssfx_avg) {
  if (!o || !um_edg || !vm_edg || !un_edg || !vn_edg || !dpm_edg || !dp || !pres || !massflx || !mssfx_avg)
    return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  const double *in[] = {um_edg, vm_edg, un_edg, vn_edg, dpm_edg, dp, pres, massflx, mssfx_avg};
  const int fi[] = {FIMHIP_OCN_UM_EDG, FIMHIP_OCN_VM_EDG, FIMHIP_OCN_UN_EDG, FIMHIP_OCN_VN_EDG, FIMHIP_OCN_DPM_EDG,
                    FIMHIP_OCN_DP, FIMHIP_OCN_PRES, FIMHIP_OCN_MASSFLX, FIMHIP_OCN_MSSFX_AVG};
  int r = 0;
  for (int j = 0; j < 9; j++)
    if ((r = ocn_put(o, fi[j], in[j]))) return r;
  r = ocn_launch(o, nstep, leapm, leapn);
  if (r && r != FIMHIP_EDUP) return r;
  double *outp[] = {dp, pres, massflx, mssfx_avg};
  const int fo[] = {FIMHIP_OCN_DP, FIMHIP_OCN_PRES, FIMHIP_OCN_MASSFLX, FIMHIP_OCN_MSSFX_AVG};
  for (int j = 0; j < 4; j++) {
    const int e = ocn_get(o, fo[j], outp[j]);
    if (e) return e;
  }
  HIPCHK(hipStreamSynchronize(o->stream));
  return r;
}

extern "C" int fimhip_ocn_set_dtleap(fimhip_ocn *o, double dtleap) {
  if (!o || !(dtleap > 0.)) return FIMHIP_EINVAL;
  o->dtleap = dtleap;
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_mass(const fimhip_ocn *o, double *totmass, double *massglb0, double *masscor) {
  if (!o || !totmass || !massglb0 || !masscor) return FIMHIP_EINVAL;
  *totmass = o->totmass;
  *massglb0 = o->massglb0;
  *masscor = o->masscor;
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_set_mass(fimhip_ocn *o, double totmass, double massglb0, double masscor) {
  if (!o) return FIMHIP_EINVAL;
  o->totmass = totmass;
  o->massglb0 = massglb0;
  o->masscor = masscor;
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_profile(fimhip_ocn *o, int on) {
  if (!o) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  HIPCHK(hipStreamSynchronize(o->stream));
  delete o->kt;
  o->kt = on ? new KTimer() : nullptr;
  return FIMHIP_OK;
}

// "name count total_ms" lines of the kernels timed since profiling began
extern "C" int fimhip_ocn_profile_report(fimhip_ocn *o, char *buf, int len) {
  if (!o || !buf || len < 1) return FIMHIP_EINVAL;
  buf[0] = 0;
  if (!o->kt) return FIMHIP_OK;
  HIPCHK(hipSetDevice(o->device));
  const int r = o->kt->flush(o->stream);
  if (r) return r;
  std::string out;
  char line[256];
  for (auto &kv : o->kt->acc) {
    snprintf(line, sizeof line, "%s %ld %.6f\n", kv.first.c_str(), kv.second.second, kv.second.first);
    out += line;
  }
  if ((int)out.size() >= len) return FIMHIP_EINVAL;
  memcpy(buf, out.c_str(), out.size() + 1);
  return FIMHIP_OK;
}
