// HYCOM's momentum equation (FIMsrc/fim/horizontal/hycom_momtum.F90, momtum,
// with hycom_dissip.F90's del4prep and dissip) on the GPU, in FP64, with the
// reference's operations in its order.  Two kernels on the column layout of
// the other ocean kernels (lanes over layers), with the boundary where
// dissip reads del4prep's values at the neighbours:
//   hyc_mom_pgf   interface pressure of the new level, the near-bottom
//                 velocity, bottom drag and friction velocity; the pressure
//                 force around the cell's edges (Bernoulli function and p grad
//                 alpha on the mid-time interfaces, or the janjic_ocn
//                 geopotential)  (104-183); vorticity, deformation and
//                 Smagorinsky viscosity from the edge velocities (211-260);
//                 del4prep: minus the mean of the neighbours' velocities
//                 rotated into the cell's frame, walls by the slip condition
//                 (hycom_dissip.F90:9-110); the bottom of dissip's own
//                 pressure column (hycom_dissip.F90:150-159)
//   hyc_mom_upd   dissip: thickness-weighted momentum fluxes through the edges
//                 with the sidewall blend, summed into a tendency
//                 (hycom_dissip.F90:113-272); Coriolis force, wind stress and
//                 bottom drag; the leapfrog update; the downward mixing into
//                 thin bottom layers (a recurrence down the column, on one
//                 lane per velocity component over LDS); the time smoothing
//                 (262-389)
// (All but del4prep in one kernel would save eight cell arrays of traffic and
// holds 180 registers: 650 us at G7 x 32 layers with del4prep beside it,
// these two 527.)
// The sums along a column (the interface pressures, the near-bottom
// velocity) are sequential chains through LDS as in the continuity kernels.
// modesplit is .false. in the reference (hycom_control.F90:5): the
// barotropic forcing (ubforc, vbforc) is not formed.
#include <type_traits>
#include <utility>

#include "div_by.h"
#include "hycom_edges.h"

namespace fimhip {
namespace hyc {
namespace {

constexpr double H_GRV = 9.80665;                 // module_constants grvity
constexpr double H_ONEMM = 0.001 * H_ONEM;
constexpr double H_TENCM = 0.1 * H_ONEM;
constexpr double H_DRCOEF = 3.e-3;                // hycom_constants.F90:44
constexpr double H_ASSLUV = .25;                  // hycom_constants.F90:48
constexpr double H_THSHLD = 1.e-11;               // hycom_dissip.F90:145
constexpr double H_THKTOP = 50. * H_ONEM, H_THKBOT = 10. * H_ONEM, H_CBAR = .5;   // hycom_momtum.F90:87-91

// The chains of the momentum equation's column, one lane each: the interfaces
// below the lane's layer of the new thickness (from p0 and, for dissip, from
// 0), of the mid-time thickness after the time smoothing, and of the one
// before it, which the edge interpolation saw.
struct MomPres {
  double pn, pz, pm, pe;
};
template <int LPC>
__device__ __forceinline__ MomPres mom_pres(double (*buf)[LPC + 1], double dn, double dm, double de, double p0,
                                            double p0e, int k, int kdm) {
  buf[0][k] = dn;
  buf[1][k] = dn;
  buf[2][k] = dm;
  buf[3][k] = de;
  wave_sync();
  if (k < 4) row_chain(buf[k], k == 1 ? 0. : k == 3 ? p0e : p0, kdm);
  wave_sync();
  const MomPres r{buf[0][k], buf[1][k], buf[2][k], buf[3][k]};
  wave_sync();
  return r;
}
// the sums over the column's layers of u and of v, in layer order from 0, on
// every lane
template <int LPC>
__device__ __forceinline__ UV col_total2(double (*buf)[LPC + 1], double u, double v, int k, int kdm) {
  buf[0][k] = u;
  buf[1][k] = v;
  wave_sync();
  if (k < 2) buf[2][k] = row_sum(buf[k], kdm);
  wave_sync();
  const UV r{buf[2][0], buf[2][1]};
  wave_sync();
  return r;
}
// EDGES: the edge values are the public arrays' (an uploaded state);
// otherwise they are formed here from the cells, from the values
// fimhip_ocn_edgvar saw (dpe the mid-time thickness, the arrays named _e; the
// velocities have not changed since), which costs less than storing and reading five edge arrays.
// Bound by memory (six cell arrays gathered at the neighbours) and, nearly as
// much, by the FP64 expressions of the edges: cells away from the coast run
// them without the coast's selections.
template <int LPC, bool EDGES>
__global__ void __launch_bounds__(256, 4) hyc_mom_pgf(HycGrid g, HycState s, HycEdg ed, HycMom m, const double *dpe,
                                                   int leapm, int leapn, int janjic) {
  constexpr int CPB = 256 / LPC;
  constexpr int T_SVC = VT_N, NT = VT_N + 2 * NPP, NRL = (NT + LPC - 1) / LPC, NC = NPP + 1;
  __shared__ double tabs[CPB][NT], sh[CPB][4][LPC + 1], trop[CPB][2 * NC], sbot[CPB][NPP];
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
  const size_t cz = (size_t)nip * kdm, om = (leapm - 1) * cz, on = (leapn - 1) * cz;
  const double *tab = tabs[cc];
  // the tables and the per-cell values of the neighbours, a few per lane
  double rv[NRL];
#pragma unroll
  for (int q = 0; q < NRL; q++) {
    const int j = k + q * LPC;
    rv[q] = j < VT_SN    ? g.cs[(size_t)i * NPP * 4 + j]
            : j < VT_SVE ? g.sn[(size_t)i * NPP * 4 + j - VT_SN]
            : j < VT_N   ? g.sve[(size_t)i * NPP * 2 + j - VT_SVE]
            : j < NT     ? m.svc[(size_t)i * NPP * 2 + j - T_SVC]
                         : 0.;
  }
  double tv = 0., bv = 0.;
  if (!EDGES && k < 2 * NC) tv = (k < NC ? ed.utrop_e : ed.vtrop_e)[(k % NC == 0 ? i : g.prox[i * NPP + k % NC - 1]) * 3 + leapm - 1];
  if (!EDGES && k < NPP) bv = s.pbe[g.prox[i * NPP + k]];
  const double di = live ? HC(s.dp + on, i, k) : 0., dm = live ? HC(s.dp + om, i, k) : 0.;
  const double de = !EDGES && live ? HC(dpe, i, k) : 0.;
  const double p0 = HP(i, 0), p0e = EDGES ? 0. : s.p0e[i];
  const double uold = HC(ed.uclin + on, i, kk), vold = HC(ed.vclin + on, i, kk);
  const double utn = uold + ed.utrop[i * 3 + leapn - 1], vtn = vold + ed.vtrop[i * 3 + leapn - 1];
#pragma unroll
  for (int q = 0; q < NRL; q++)
    if (k + q * LPC < NT) tabs[cc][k + q * LPC] = rv[q];
  if (!EDGES && k < 2 * NC) trop[cc][k] = tv;
  if (!EDGES && k < NPP) sbot[cc][k] = bv;
  // the new level's interfaces: pn1 below the layer, pn0 above, pb the bottom
  // (every shuffle is taken by all the column's lanes: a lane that skips one
  // gives no value to the lane that reads it)
  const MomPres pr = mom_pres<LPC>(sh[cc], di, dm, de, p0, p0e, k, kdm);
  const double pn1 = pr.pn;
  const double pn1_up = __shfl_up(pn1, 1, LPC);
  const double pn0 = k > 0 ? pn1_up : p0;
  const double pb = __shfl(pn1, kdm - 1, LPC);
  if (k == kdm - 1) m.dpbot[i] = pr.pz;
  // the near-bottom velocity (thkbot above the bottom) and the drag
  const double q = hmin(H_THKBOT, pb);
  const double wgt = hmin(pn1, pb - q) - hmin(pn0, pb - q);
  const UV bot = col_total2<LPC>(sh[cc], live ? utn * wgt : 0., live ? vtn * wgt : 0., k, kdm);
  if (k == 0) {
    const double botvel = sqrt(bot.u * bot.u + bot.v * bot.v) / H_THKBOT;
    m.drag[i] = hmin(H_DRCOEF * (botvel + H_CBAR) * H_ONEM / H_THKBOT, 1. / m.batrop);
    m.ustarb[i] = sqrt(H_DRCOEF) * botvel;
  }
  // the interfaces of the pressure force are the mid-time ones (recomputed at
  // every edge in the reference, to the same values), the new level's with
  // janjic_ocn
  const double pk1 = janjic ? pn1 : pr.pm;
  const double pk1_up = __shfl_up(pk1, 1, LPC);
  const double pk0 = k > 0 ? pk1_up : p0;
  if (!live) return;
  __builtin_nontemporal_store(pk1, &HP(i, k + 1));
  const double ra = g.rarea[i];
  const auto edges = [&](auto sea) {
    const int cj = sea.value ? CI_SEA : ci, nq = sea.value ? 6 : np;
    // del4prep
    {
      double ux[NPP], vx[NPP], avgu = 0., avgv = 0.;
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        ux[e] = HC(ed.uclin + on, nb[e], k);
        vx[e] = HC(ed.vclin + on, nb[e], k);
      }
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        if (e >= nq) break;
        double ungbor, vngbor;
        if (ci_open(cj, e)) {
          const double c0 = tab[VT_CS + e * 4], s0 = tab[VT_SN + e * 4];
          const double c1 = tab[VT_CS + e * 4 + 1], s1 = tab[VT_SN + e * 4 + 1];
          const double uedge = c1 * ux[e] + s1 * vx[e];
          const double vedge = -s1 * ux[e] + c1 * vx[e];
          ungbor = c0 * uedge - s0 * vedge;
          vngbor = s0 * uedge + c0 * vedge;
        } else {
          ungbor = H_SLIP * uold;
          vngbor = H_SLIP * vold;
        }
        avgu = avgu + ungbor;
        avgv = avgv + vngbor;
      }
      const double factor = 1. / nq;
      __builtin_nontemporal_store(uold - avgu * factor, &HC(m.d4u, i, k));
      __builtin_nontemporal_store(vold - avgv * factor, &HC(m.d4v, i, k));
    }
    __builtin_amdgcn_sched_barrier(0);      // one section's values at a time in registers
    // the velocities and the kinetic energy on the edges, the velocity
    // derivatives from the tangential velocity along them
    double uvsq[NPP], dudx = 0., dudy = 0., dvdx = 0., dvdy = 0.;
    {
      double ux[NPP], vx[NPP], ui = 0., vi = 0.;
      if (!EDGES) {
        ui = HC(ed.uclin + om, i, k) + trop[cc][0];
        vi = HC(ed.vclin + om, i, k) + trop[cc][NC];
#pragma unroll
        for (int e = 0; e < NPP; e++) {      // (a land neighbour's are not used)
          ux[e] = HC(ed.uclin + om, nb[e], k) + trop[cc][e + 1];
          vx[e] = HC(ed.vclin + om, nb[e], k) + trop[cc][NC + e + 1];
        }
      }
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        uvsq[e] = 0.;
        if (e >= nq) break;
        double ue, ve;
        if (EDGES) {
          ue = HE(s.um, i, e, k);
          ve = HE(s.vm, i, e, k);
          uvsq[e] = HE(ed.uvsq_edg, i, e, k);
        } else {
          const int em1 = e_prev(e, nq), ep1 = e_next(e, nq);
          const UV r = uv_edge(rot_of(tab, e), true, ci_open(cj, e), ci_open(cj, em1), ci_open(cj, ep1), ui, vi,
                               ux[e], vx[e], at_prev(ux, e, nq), at_prev(vx, e, nq), at_next(ux, e, nq),
                               at_next(vx, e, nq));
          ue = r.u;
          ve = r.v;
          uvsq[e] = .5 * (r.u * r.u + r.v * r.v);
        }
        const double s0 = tab[VT_SVE + e * 2], s1 = tab[VT_SVE + e * 2 + 1];
        dudx = dudx + s1 * ue;
        dudy = dudy - s0 * ue;
        dvdx = dvdx + s1 * ve;
        dvdy = dvdy - s0 * ve;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    dudx = dudx * ra;
    dudy = dudy * ra;
    dvdx = dvdx * ra;
    dvdy = dvdy * ra;
    const double da = dudx - dvdy, db = dudy + dvdx;
    const double deform = sqrt(da * da + db * db);
    const double smag = deform * m.meshsz[i] * m.smagcf;
    __builtin_nontemporal_store(dvdx - dudy, &HC(m.relvor, i, k));
    __builtin_nontemporal_store(hmax(m.veldff, smag), &HC(m.visc, i, k));
    __builtin_amdgcn_sched_barrier(0);
    // the pressure force around the edges
    double pgfx = 0., pgfy = 0.;
    if (janjic) {
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        if (e >= nq) break;
        const double t = HE(ed.geop_edg, i, e, k) + uvsq[e];
        pgfx = pgfx - t * tab[T_SVC + e * 2 + 1];
        pgfy = pgfy + t * tab[T_SVC + e * 2];
      }
    } else {
      double mo[NPP], sp[NPP];
      if (EDGES) {
#pragma unroll
        for (int e = 0; e < NPP; e++) {
          mo[e] = HE(ed.mont_edg, i, e, k);
          sp[e] = HE(ed.spcv_edg, i, e, k);
        }
      } else {
        double PB[NPP], M[NPP], SV[NPP], nm[NPP], ns[NPP];
        const double mi = HC(ed.montg_e, i, k), svi = HC(ed.spcifv_e, i, k);
#pragma unroll
        for (int e = 0; e < NPP; e++) {
          PB[e] = sbot[cc][e];
          M[e] = HC(ed.montg_e, nb[e], k);
          SV[e] = HC(ed.spcifv_e, nb[e], k);
        }
        sidewall(cj, de, pr.pe, PB, mi, M, svi, SV, nm, ns);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < NPP; e++) {
          mo[e] = (8. * (mi + nm[e]) + at_prev(nm, e, nq) + at_next(nm, e, nq)) * H_DIVBY18;
          sp[e] = (8. * (svi + ns[e]) + at_prev(ns, e, nq) + at_next(ns, e, nq)) * H_DIVBY18;
        }
      }
#pragma unroll
      for (int e = 0; e < NPP; e++) {
        if (e >= nq) break;
        const double t = mo[e] + uvsq[e];
        const double c0 = tab[T_SVC + e * 2], c1 = tab[T_SVC + e * 2 + 1];
        pgfx = pgfx - t * c1;
        pgfy = pgfy + t * c0;
        pgfx = pgfx + .5 * (pk0 + pk1) * sp[e] * c1;
        pgfy = pgfy - .5 * (pk0 + pk1) * sp[e] * c0;
      }
    }
    __builtin_nontemporal_store(pgfx * ra, &HC(m.gradx, i, k));
    __builtin_nontemporal_store(pgfy * ra, &HC(m.grady, i, k));
  };
  if (__all(ci == CI_SEA)) edges(std::true_type());
  else edges(std::false_type());
}

// The new velocities go to the other pair of arrays, and the two are swapped:
// what the edge interpolation saw stays in place.  Bound by memory (three
// cell arrays gathered, nine read at the cell, four written).
template <int LPC>
__global__ void __launch_bounds__(256) hyc_mom_upd(HycGrid g, HycState s, HycEdg ed, HycMom m, int leapm, int leapn,
                                                   double dtleap) {
  constexpr int CPB = 256 / LPC;
  constexpr int T_SL = 4 * NPP, NT = T_SL + 2 * NPP, NRL = (NT + LPC - 1) / LPC;
  __shared__ double tabs[CPB][NT], sx[CPB][5][LPC + 1];
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
  const size_t cz = (size_t)nip * kdm, om = (leapm - 1) * cz, on = (leapn - 1) * cz;
  const double *dpn = s.dp + on, *tab = tabs[cc];
  // by edge: cs, sn of the cell and of the neighbour; the lengths; the
  // neighbours' bottoms
  double rv[NRL];
#pragma unroll
  for (int q = 0; q < NRL; q++) {
    const int j = k + q * LPC;
    rv[q] = j < T_SL         ? (j & 1 ? g.sn : g.cs)[((size_t)i * NPP + (j >> 2)) * 4 + ((j >> 1) & 1)]
            : j < T_SL + NPP ? g.sideln[(size_t)i * NPP + j - T_SL]
            : j < NT         ? m.dpbot[g.prox[i * NPP + j - T_SL - NPP]]
                             : 0.;
  }
  const double di = HC(dpn, i, kk), ui = HC(m.d4u, i, kk), vi = HC(m.d4v, i, kk);
  const double ra = g.rarea[i];
#pragma unroll
  for (int q = 0; q < NRL; q++)
    if (k + q * LPC < NT) tabs[cc][k + q * LPC] = rv[q];
  // dissip's own column, from 0
  const double pz = col_pres(sx[cc][0], live ? di : 0., 0., k, kdm);
  double du = 0., dv = 0.;
  const auto edges = [&](auto sea) {
    const int cj = sea.value ? CI_SEA : ci, nq = sea.value ? 6 : np;
    const double factor = ra / hmax(di, H_THSHLD);
    double ux[NPP], vx[NPP], dx[NPP];
#pragma unroll
    for (int e = 0; e < NPP; e++) {
      ux[e] = HC(m.d4u, nb[e], kk);
      vx[e] = HC(m.d4v, nb[e], kk);
      dx[e] = HC(dpn, nb[e], kk);
    }
#pragma unroll
    for (int e = 0; e < NPP; e++) {
      if (e >= nq) break;
      const double c0 = tab[e * 4], s0 = tab[e * 4 + 1];
      const double urot = c0 * ui + s0 * vi;
      const double vrot = -s0 * ui + c0 * vi;
      double ungbor, vngbor;
      if (ci_open(cj, e)) {
        const double c1 = tab[e * 4 + 2], s1 = tab[e * 4 + 3];
        ungbor = c1 * ux[e] + s1 * vx[e];
        vngbor = -s1 * ux[e] + c1 * vx[e];
        const double blokd = blokf(di, pz, tab[T_SL + NPP + e]);
        ungbor = (1. - blokd) * ungbor + blokd * urot * H_SLIP;
        vngbor = (1. - blokd) * vngbor + blokd * vrot * H_SLIP;
      } else {
        ungbor = urot * H_SLIP;
        vngbor = vrot * H_SLIP;
      }
      const double a = hmax(di, H_THSHLD), b = hmax(dx[e], H_THSHLD);
      const double hh = a * b / (a + b);
      const double sl = tab[T_SL + e];
      const double ufx = (ungbor - urot) * sl * 2. * hh;
      const double vfx = (vngbor - vrot) * sl * 2. * hh;
      const double uflux = c0 * ufx - s0 * vfx;
      const double vflux = s0 * ufx + c0 * vfx;
      du = du + uflux * factor;
      dv = dv + vflux * factor;
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (__all(ci == CI_SEA)) edges(std::true_type());
  else edges(std::false_type());
  const double pk = HP(i, kk), pk1 = HP(i, kk + 1), pb = HP(i, kdm), drag = m.drag[i];
  const double um = HC(ed.uclin + om, i, kk), vm = HC(ed.vclin + om, i, kk);
  const double uold = HC(ed.uclin + on, i, kk), vold = HC(ed.vclin + on, i, kk);
  const double relvor = HC(m.relvor, i, kk), visc = HC(m.visc, i, kk);
  const double gradx = HC(m.gradx, i, kk), grady = HC(m.grady, i, kk);
  const double cor = m.corio[i];
  const double uzeta = um * (relvor + cor) + ed.utrop[i * 3 + leapm - 1] * relvor;
  const double vzeta = vm * (relvor + cor) + ed.vtrop[i * 3 + leapm - 1] * relvor;
  const double thn = hmax(di, H_ONEMM);
  double ustres = m.taux[i] * H_GRV / H_THKTOP * (hmin(pk1 + H_ONEMM, H_THKTOP) - hmin(pk, H_THKTOP)) / thn;
  double vstres = m.tauy[i] * H_GRV / H_THKTOP * (hmin(pk1 + H_ONEMM, H_THKTOP) - hmin(pk, H_THKTOP)) / thn;
  const double q = (hmax(pb - H_THKBOT, pk1) - hmax(pb - H_THKBOT, hmin(pk1 - H_ONEMM, pk))) / thn;
  const double utn = uold + ed.utrop[i * 3 + leapn - 1], vtn = vold + ed.vtrop[i * 3 + leapn - 1];
  ustres = ustres - drag * utn * q;
  vstres = vstres - drag * vtn * q;
  const double un = uold + dtleap * (gradx + vzeta + du * visc + ustres);
  const double vn = vold + dtleap * (grady - uzeta + dv * visc + vstres);
  // downward momentum mixing into thin bottom layers: each layer below the
  // first takes (slab - q) of the final value of the layer above
  const double slab = hmax(H_TENCM, pk1 - pb + H_TENM);
  const double qq = hmin(di, slab);
  sx[cc][0][k] = un;
  sx[cc][1][k] = vn;
  sx[cc][2][k] = qq;
  sx[cc][3][k] = slab;
  sx[cc][4][k] = div_rcp(slab);
  wave_sync();
  if (k < 2) {
    double *x = sx[cc][k];
    const double *sq = sx[cc][2], *ssl = sx[cc][3], *srs = sx[cc][4];
    double prev = x[0];
    int j = 1;
    constexpr int CH = 4;
    for (; j + CH <= kdm; j += CH) {
      double xv[CH], sv[CH], qv[CH], rs[CH];
#pragma unroll
      for (int t = 0; t < CH; t++) {
        xv[t] = x[j + t];
        qv[t] = sq[j + t];
        sv[t] = ssl[j + t];
        rs[t] = srs[j + t];
      }
#pragma unroll
      for (int t = 0; t < CH; t++)
        x[j + t] = prev = div_by(xv[t] * qv[t] + prev * (sv[t] - qv[t]), sv[t], rs[t]);
    }
    for (; j < kdm; j++) x[j] = prev = div_by(x[j] * sq[j] + prev * (ssl[j] - sq[j]), ssl[j], srs[j]);
  }
  wave_sync();
  if (!live) return;
  const double uf = sx[cc][0][k], vf = sx[cc][1][k];
  __builtin_nontemporal_store(uf, &HC(ed.uclin_alt + on, i, k));
  __builtin_nontemporal_store(vf, &HC(ed.vclin_alt + on, i, k));
  __builtin_nontemporal_store(H_ASSLUV * (uold + uf) + (1. - H_ASSLUV - H_ASSLUV) * um, &HC(ed.uclin_alt + om, i, k));
  __builtin_nontemporal_store(H_ASSLUV * (vold + vf) + (1. - H_ASSLUV - H_ASSLUV) * vm, &HC(ed.vclin_alt + om, i, k));
}

}  // namespace
}  // namespace hyc
}  // namespace fimhip

using namespace fimhip;
using namespace fimhip::hyc;

template <int LPC>
static void mom_kernels(fimhip_ocn *o, int leapm, int leapn) {
  const HycGrid &g = o->g;
  const HycState &s = o->s;
  const HycEdg &ed = o->ed;
  const HycMom &m = o->mo;
  hipStream_t st = o->stream;
  const dim3 grid(ocn_blocks(o, LPC)), blk(256);
  const int janjic = o->janjic ? 1 : 0;
  const double *dpe = o->e_dp_old ? s.dpe : s.dp + (size_t)(leapm - 1) * o->nip * o->kdm;
  if (o->edges_due)
    KT_LAUNCH("hyc_mom_pgf", st,
              (hyc_mom_pgf<LPC, false><<<grid, blk, 0, st>>>(g, s, ed, m, dpe, leapm, leapn, janjic)));
  else
    KT_LAUNCH("hyc_mom_pgf_edg", st,
              (hyc_mom_pgf<LPC, true><<<grid, blk, 0, st>>>(g, s, ed, m, nullptr, leapm, leapn, janjic)));
  KT_LAUNCH("hyc_mom_upd", st, hyc_mom_upd<LPC><<<grid, blk, 0, st>>>(g, s, ed, m, leapm, leapn, o->dtleap));
}

// momtum on the device-resident arrays (hycom_momtum.F90:16-389)
static int mom_launch(fimhip_ocn *o, int leapm, int leapn) {
  if (leapm < 1 || leapm > 2 || leapn < 1 || leapn > 2 || leapm == leapn) return FIMHIP_EINVAL;
  if (!(o->mo.batrop > 0.)) return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  HycEdg &ed = o->ed;
  // a second momtum since the edge interpolation, one at other levels, or one
  // on other velocities, is one on the arrays themselves
  if (o->e_uv_old || leapm != o->e_leapm || ed.uclin != ed.uclin_e || ed.vclin != ed.vclin_e) {
    const int r = ocn_form_edges(o);
    if (r) return r;
  }
  if (!o->edges_due) {
    const int r = ocn_need_edges(o);
    if (r) return r;
  }
  if (o->alt_stale) {       // land keeps its velocities: the other pair needs them too
    const size_t n = 2 * (size_t)o->nip * o->kdm * sizeof(double);
    HIPCHK(hipMemcpyAsync(ed.uclin_alt, ed.uclin, n, hipMemcpyDeviceToDevice, o->stream));
    HIPCHK(hipMemcpyAsync(ed.vclin_alt, ed.vclin, n, hipMemcpyDeviceToDevice, o->stream));
    o->alt_stale = false;
  }
  g_ktimer = o->kt;
  if (o->kdm <= 32) mom_kernels<32>(o, leapm, leapn);
  else mom_kernels<64>(o, leapm, leapn);
  g_ktimer = nullptr;
  std::swap(ed.uclin, ed.uclin_alt);
  std::swap(ed.vclin, ed.vclin_alt);
  o->e_uv_old = true;
  HIPCHK(hipGetLastError());
  return FIMHIP_OK;
}

extern "C" int fimhip_ocn_set_momtum(fimhip_ocn *o, double batrop, double veldff, double smagcf) {
  if (!o || !(batrop > 0.)) return FIMHIP_EINVAL;
  o->mo.batrop = batrop;
  o->mo.veldff = veldff;
  o->mo.smagcf = smagcf;
  return FIMHIP_OK;
}

// asynchronous on the instance's stream, like fimhip_ocn_edgvar
extern "C" int fimhip_ocn_momtum(fimhip_ocn *o, int leapm, int leapn) {
  if (!o) return FIMHIP_EINVAL;
  return mom_launch(o, leapm, leapn);
}

extern "C" int fimhip_ocn_momtum_r8(fimhip_ocn *o, int nstep, int leapm, int leapn, const double *utrop,
                                   const double *vtrop, double *uclin, double *vclin, const double *um_edg,
                                   const double *vm_edg, const double *geop_edg, const double *mont_edg,
                                   const double *uvsq_edg, const double *spcv_edg, const double *taux,
                                   const double *tauy, double *ubforc, double *vbforc, const double *dp,
                                   double *pres, double *ustarb) {
  (void)nstep;
  (void)ubforc;     // formed only under modesplit, which the reference has off
  (void)vbforc;
  if (!o || !utrop || !vtrop || !uclin || !vclin || !um_edg || !vm_edg || !geop_edg || !mont_edg || !uvsq_edg ||
      !spcv_edg || !taux || !tauy || !dp || !pres || !ustarb)
    return FIMHIP_EINVAL;
  HIPCHK(hipSetDevice(o->device));
  const double *in[] = {utrop, vtrop, uclin, vclin, um_edg, vm_edg, geop_edg, mont_edg, uvsq_edg, spcv_edg,
                        taux, tauy, dp, pres, ustarb};
  const int fi[] = {FIMHIP_OCN_UTROP, FIMHIP_OCN_VTROP, FIMHIP_OCN_UCLIN, FIMHIP_OCN_VCLIN, FIMHIP_OCN_UM_EDG,
                    FIMHIP_OCN_VM_EDG, FIMHIP_OCN_GEOP_EDG, FIMHIP_OCN_MONT_EDG, FIMHIP_OCN_UVSQ_EDG,
                    FIMHIP_OCN_SPCV_EDG, FIMHIP_OCN_TAUX, FIMHIP_OCN_TAUY, FIMHIP_OCN_DP, FIMHIP_OCN_PRES,
                    FIMHIP_OCN_USTARB};
  int r = 0;
  for (int j = 0; j < 15; j++)
    if ((r = ocn_put(o, fi[j], in[j]))) return r;
  if ((r = mom_launch(o, leapm, leapn))) return r;
  double *outp[] = {uclin, vclin, pres, ustarb};
  const int fo[] = {FIMHIP_OCN_UCLIN, FIMHIP_OCN_VCLIN, FIMHIP_OCN_PRES, FIMHIP_OCN_USTARB};
  for (int j = 0; j < 4; j++)
    if ((r = ocn_get(o, fo[j], outp[j]))) return r;
  HIPCHK(hipStreamSynchronize(o->stream));
  return FIMHIP_OK;
}
