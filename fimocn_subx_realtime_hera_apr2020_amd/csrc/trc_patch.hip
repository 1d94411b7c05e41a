// trcadv1 of the device-resident FP64 step over patches of cells
// (trcadv_compute.F90:19-150 with the reconstructions of edgvar3.F90:65-132).
//
// A block takes one patch of cells for one tracer, lane = level: it stages the
// tracer of the patch and of two neighbour rings in LDS, and each wavefront
// then takes core cells in turn: both cells' reconstructions of the six edges
// (the neighbours' from their own stencils in LDS), the high- and low-order
// fluxes, the antidiffusive fluxes and their in- and outflow sums, the
// low-order tendency and the bounded low-order tracer.  Every operation is the
// reference's, in its order, so the results keep their bits.
//
// What bounds it: HBM traffic.  With the reconstructions stored by edgvar3 and
// read back with the neighbours' the two kernels moved 816 B per cell-level
// for 4 tracers, this one and the thickness's reconstruction 560 B and the
// halo, at 4 TB/s.  G7 x 64: trcadv1 and edgvar3 1.35 + 0.64 -> 1.31 + 0.17 ms;
// G6 x 50 x 5 tracers: 0.57 -> 0.45 ms; G5: 0.12 ms both ways; G3: 24 -> 19 us.  The coefficients and indexes of a cell come as one row by
// vector loads, a cell ahead, handed out by v_readlane (as scalar loads each
// batch waits for the scalar cache); the cell's other inputs are loaded before
// the reconstructions, whose arithmetic covers their latency.  All tracers of
// a patch run in turn on one XCD, whose L2 then holds the patch's rows and
// mass fluxes.
#include <algorithm>

#include "ens_internal.h"
#include "host_common.h"

namespace fimhip {

#define C2(a, ipn, k) (a)[(size_t)(ipn) * nvl + (k)]
#define E3(a, ipn, e, k) (a)[((size_t)(ipn) * NPP + (e)) * nvl + (k)]
#define TAB(a, t, s, ipn, k) (a)[(((size_t)(t) * 3 + (s)) * nip + (ipn)) * nvl + (k)]

namespace {

constexpr int NW = 8;                // wavefronts per block
// words of a cell's row: own coefficients, the neighbours' of the shared
// edges (36 doubles each), the LDS byte offsets of the neighbours' stencil
// cells (36 of 16 bits) and of the neighbours (6 of 16 bits), and the
// neighbours' edge slots, cell * 6 + slot (6)
constexpr int R_OWN = 0, R_NBR = 72, R_ST = 144, R_NB = 162, R_EX = 165, ROW = 171, ROWP = 192;

__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ int lnb(const int4 &en, int e) {
  return e < 4 ? (en.y >> (8 * e)) & 0xff : (en.z >> (8 * (e - 4))) & 0xff;
}
__device__ __forceinline__ int enp(const int4 &en) { return (en.z >> 16) & 0xff; }

// word 64 i + lane in the i-th.  Every lane stays active from the load of a
// row to its last word (lanes above the column compute on level 0's values and
// store nothing): a copy of a row's register that the compiler makes while some
// lanes are off would lose their words.
struct Row { int a, b, c; };
__device__ __forceinline__ int row_i(const Row &r, int w) {
  return __builtin_amdgcn_readlane(w < 64 ? r.a : w < 128 ? r.b : r.c, w & 63);
}
__device__ __forceinline__ double row_d(const Row &r, int w) {
  const unsigned lo = (unsigned)row_i(r, w), hi = (unsigned)row_i(r, w + 1);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ int row_h(const Row &r, int w0, int i) {   // i-th 16-bit field from word w0
  const int p = row_i(r, w0 + (i >> 1));
  return i & 1 ? (p >> 16) & 0xffff : p & 0xffff;
}
__device__ __forceinline__ double lds_at(const double *a, int byte_off, int k) {
  return *(const double *)((const char *)a + byte_off + 8 * k);
}

__global__ void __launch_bounds__(256) k_patch_rows(DevGrid g, EnsTiles ts, int *rows) {
  const int p = blockIdx.x, n0 = ts.cnt[p].x;
  const int4 *ent = ts.ent + ts.off[p];
  for (int q = threadIdx.x; q < n0; q += blockDim.x) {
    const int4 en = ent[q];
    int *row = rows + (size_t)en.x * ROWP;
    for (int e = 0; e < NPP; e++) {
      const int l = lnb(en, e), xs = (en.w >> (4 * e)) & 0xf;
      const int4 ex = ent[l];
      const int x = ex.x, nx = enp(ex);
      row[R_EX + e] = x * NPP + xs;
      ((unsigned short *)(row + R_NB))[e] = (unsigned short)(512 * l);
      for (int j = 0; j < NPP; j++) {
        const long long a = __double_as_longlong(g.hfcoef[((size_t)en.x * NPP + e) * NPP + j]);
        const long long b = __double_as_longlong(j < nx ? g.hfcoef[((size_t)x * NPP + xs) * NPP + j] : 0.);
        row[R_OWN + 2 * (e * NPP + j)] = (int)a;
        row[R_OWN + 2 * (e * NPP + j) + 1] = (int)(a >> 32);
        row[R_NBR + 2 * (e * NPP + j)] = (int)b;
        row[R_NBR + 2 * (e * NPP + j) + 1] = (int)(b >> 32);
        ((unsigned short *)(row + R_ST))[e * NPP + j] = (unsigned short)(512 * (j < nx ? lnb(ex, j) : l));
      }
    }
  }
}

// One core cell: its row is here, its stencil's tracer in LDS; lane: of the
// wavefront, k: its level, or 0 above the column (live).  A pentagon
// neighbour's sixth stencil value is the neighbour's own (difference 0) with
// coefficient 0, and PENT keeps it out of the sum.
template <int NP, bool THETA>
__device__ __forceinline__ void flux_col(const DevGrid &g, const DevState &s, const AB &ab, int t, int cell, int i, int lane,
                                         int k, bool live, double rar, int pent, const Row &row, const double *Str) {
  const int nip = g.nip, nvl = g.nvl;
  const int nf = ab.nf - 1, of = ab.of - 1, vof = ab.vof - 1;
  const size_t csz = (size_t)nip * nvl;
  const double *mf = s.massfx + (size_t)nf * csz * NPP;
  // every global load of the cell first
  double m[NP], mx_[NP];
#pragma unroll
  for (int e = 0; e < NP; e++) {
    m[e] = E3(mf, cell, e, k);
    mx_[e] = mf[(size_t)row_i(row, R_EX + e) * nvl + k];
  }
  const double dpc = dmax(1.e-11, C2(s.dp, cell, k));
  const double td = C2(s.trdp + t * csz, cell, k), tlof = TAB(s.trl_tdcy, t, of, cell, k);
  const double tlov = TAB(s.trl_tdcy, t, vof, cell, k);
  const double ti = Str[i * 64 + lane];
  double v[NP], te[NP];
#pragma unroll
  for (int e = 0; e < NP; e++) v[e] = lds_at(Str, row_h(row, R_NB, e), lane);
  if (THETA) {
#pragma unroll
    for (int e = 0; e < NP; e++) te[e] = (2. * (ti + v[e]) + v[(e + NP - 1) % NP] + v[(e + 1) % NP]) * (1. / 6.);
  } else {
#pragma unroll
    for (int e = 0; e < NP; e++) {
      double own = ti, oth = v[e];
#pragma unroll
      for (int j = 0; j < NP; j++) own = own + (v[j] - ti) * row_d(row, R_OWN + 2 * (e * NPP + j));
#pragma unroll
      for (int j = 0; j < NPP; j++) {
        const double q = (lds_at(Str, row_h(row, R_ST, e * NPP + j), lane) - v[e]) * row_d(row, R_NBR + 2 * (e * NPP + j));
        if (j < NPP - 1 || !((pent >> e) & 1)) oth = oth + q;
      }
      te[e] = 0.5 * (own + oth);
      // formed here, not in the branch of the live lanes below, to which the
      // compiler would move the arithmetic and keep all the row's words
      asm volatile("" : "+v"(te[e]));
    }
  }
  double af[NP], acc = 0., sp = 0., sm = 0., mx = ti, mn = ti;
#pragma unroll
  for (int e = 0; e < NP; e++) {
    const double flx_hi = m[e] * te[e];
    const double fl = 0.5 * ((m[e] + fabs(m[e])) * ti - (mx_[e] + fabs(mx_[e])) * v[e]);
    const double a = flx_hi - fl;
    af[e] = a;
    sp = sp - dmin(0., a);
    sm = sm + dmax(0., a);
    acc = acc + fl;
    mx = dmax(mx, v[e]);
    mn = dmin(mn, v[e]);
  }
  if (!live) return;
#pragma unroll
  for (int e = 0; e < NP; e++) __builtin_nontemporal_store(af[e], &E3(s.antiflx + t * csz * NPP, cell, e, k));
  const double tlo = -acc * rar;
  __builtin_nontemporal_store(tlo, &TAB(s.trl_tdcy, t, nf, cell, k));
  const double trcdp_lo = td + ab.ab1 * tlo + ab.ab2 * tlof + ab.ab3 * tlov;
  mx = dmax(0., mx);
  mn = dmax(0., mn);
  C2(s.trcr_lo + t * csz, cell, k) = dmax(mn, dmin(mx, trcdp_lo / dpc));
  __builtin_nontemporal_store(sp, &C2(s.tr_rp + t * csz, cell, k));
  __builtin_nontemporal_store(sm, &C2(s.tr_rm + t * csz, cell, k));
}

template <bool THETA>
__device__ __forceinline__ void flux_cells(const DevGrid &g, const DevState &s, const EnsTiles &ts, const AB &ab, int t,
                                           const int4 &ev, double rarl, int w, int n0, int lane,
                                           const double *Str) {
  const int jl = (n0 - 1 - w) / NW;
  auto load_row = [&](int j) {
    const int *r = ts.core_row + (size_t)__builtin_amdgcn_readlane(ev.x, min(j, jl)) * ROWP + lane;
    return Row{r[0], r[64], r[128]};
  };
  const bool live = lane < g.nvl;
  const int k = live ? lane : 0;
  Row row = load_row(0);
  for (int i = w, j = 0; i < n0; i += NW, j++) {
    const Row nrow = load_row(j + 1);
    const int cell = __builtin_amdgcn_readlane(ev.x, j), z = __builtin_amdgcn_readlane(ev.z, j);
    const long long b = __double_as_longlong(rarl);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, j), hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), j);
    const double rar = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    if (((z >> 16) & 0xff) == 6) flux_col<6, THETA>(g, s, ab, t, cell, i, lane, k, live, rar, (z >> 24) & 0x3f, row, Str);
    else flux_col<5, THETA>(g, s, ab, t, cell, i, lane, k, live, rar, (z >> 24) & 0x3f, row, Str);
    row = nrow;
  }
}

__global__ void __launch_bounds__(64 * NW) k_p_trcadv1(DevGrid g, DevState s, EnsTiles ts, AB ab) {
  extern __shared__ double Str[];      // the tracer of rings 0-2
  const int nvl = g.nvl, ntra = g.ntra;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.y), k = threadIdx.x;
  // each XCD takes a contiguous eighth of the patches, every tracer of a patch in turn
  const int q = blockIdx.x >> 3, per = (ts.npatch + 7) >> 3;
  const int p = (blockIdx.x & 7) * per + q / ntra, t = q % ntra;
  if (p >= ts.npatch) return;          // the whole block: before the barrier
  const int *cn = (const int *)(ts.cnt + p);
  const int n0 = ldc(cn, 0), n2 = ldc(cn, 2), off = ldc(ts.off, p);
  const int4 ev = ts.ent[off + min(w + k * NW, n2 - 1)];   // lane j: the wavefront's j-th tile cell
  const int kc = k < nvl ? k : 0;
  const double *tr = s.tr + (size_t)t * g.nip * nvl + kc;
  constexpr int J0 = (TRC64_LIMITS.lo + NW - 1) / NW;
  double v[J0];
#pragma unroll
  for (int j = 0; j < J0; j++)
    if (w + j * NW < n2) v[j] = tr[(size_t)__builtin_amdgcn_readlane(ev.x, j) * nvl];
#pragma unroll
  for (int j = 0; j < J0; j++)
    if (w + j * NW < n2) Str[(w + j * NW) * 64 + k] = v[j];
  const double rarl = g.rarea[ev.x];
  __syncthreads();
  if (w >= n0) return;
  if (t == 0) flux_cells<true>(g, s, ts, ab, t, ev, rarl, w, n0, k, Str);
  else flux_cells<false>(g, s, ts, ab, t, ev, rarl, w, n0, k, Str);
}

}  // namespace

void patch_pentagons(const HostGrid &h, TileHost &t) {
  for (size_t p = 0; p < t.cnt.size(); p++)
    for (int i = 0; i < t.cnt[p][0]; i++) {
      auto &en = t.ent[t.off[p] + i];
      for (int e = 0; e < NPP; e++)
        if (h.nprox[h.prox[(size_t)en[0] * NPP + e]] != NPP) en[2] |= 1 << (24 + e);
    }
}

int patch_tables(Arena &a, const HostGrid &h, const DevGrid &g, int core, EnsTiles &ts) {
  TileHost t;
  int r = ens_build_tiles(h, g.nip, {2, std::min(core, TRC64_LIMITS.core), TRC64_LIMITS.r, TRC64_LIMITS.lo, TRC64_LIMITS.tile}, t);
  if (r) return r;
  patch_pentagons(h, t);
  if ((r = ens_upload_tiles(a, t, ts))) return r;
  ts.lo_max = 0;
  for (auto &c : t.cnt) ts.lo_max = std::max(ts.lo_max, c[2]);
  int *rows = nullptr;
  if ((r = a.alloc(&rows, (size_t)g.nip * ROWP))) return r;
  k_patch_rows<<<ts.npatch, 256, 0, a.stream>>>(g, ts, rows);
  if (hipGetLastError() != hipSuccess) return FIMHIP_EHIP;
  ts.core_row = rows;
  return 0;
}

void launch_patch_trcadv1(const DevGrid &g, const DevState &s, const EnsTiles &ts, const AB &ab, hipStream_t st) {
  const size_t sh = (size_t)ts.lo_max * 64 * sizeof(double);
  k_p_trcadv1<<<(ts.npatch + 7) / 8 * 8 * g.ntra, dim3(64, NW), sh, st>>>(g, s, ts, ab);
}

}  // namespace fimhip
