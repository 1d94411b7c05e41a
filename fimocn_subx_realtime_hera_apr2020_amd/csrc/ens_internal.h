// The batched mixed-precision form: several members (ensemble members or
// other instances on the same grid) advanced by the same kernels.
//
// Precision split (per field):
//   FP32  winds, tracers, tracer mass, their Adams-Bashforth histories, the
//         edge values (of the edge wind only its normal component is stored;
//         momtum forms the full edge winds itself), the FCT work arrays and
//         the mass fluxes;
//   FP64  layer thickness and its AB history (mass conservation), interface
//         pressure and Exner function, Montgomery potential (also on the
//         edges, formed where momtum needs it) and geopotential (the
//         pressure-gradient force), and all of hybgen.
// Each edge's mass flux is taken from one side (the lower cell index) and
// negated on the other, so the FP32 fluxes cancel exactly in the global sum.
//
// Layout: the plain form's layout with the cell index replaced by the column
// index col = member * nip + cell (ncol = members * nip):
//   cell (nvl, ncol)   level (nvl+1, ncol)   edge (nvl, 6, ncol)
//   tracer (nvl, ncol, ntra)   AB (nvl, ncol, 3)   tracer AB (nvl, ncol, 3, ntra)
// (the tracers' edge values are formed where they are used); the mass flux
// keeps only the current slot.
#pragma once
#include <array>
#include <vector>

#include "fimhip_internal.h"

namespace fimhip {

struct HostGrid;
struct Arena;

// Patches of cells with their neighbour rings, of three kernels: the fused
// tracer FCT (three rings) and trcadv12 (two; both fct_tiles.hip) of the batched
// form, and the FP64 step's trcadv1 (two; trc_patch.hip).  Per patch the
// cumulative ends n0..n3 of its core and rings in its list of tile cells (with
// two rings n3 is n2), and per tile cell an entry of four ints: the cell index;
// the local indices in the tile of its neighbours 0-3 (8 bits each); of
// neighbours 4-5 and its edge count (8 bits each); the neighbours' indices of
// the shared edges, proxs (4 bits each).  The local indices are set for all but
// the last ring (0 there).  In the FP64 tables bits 24-29 of a core cell's third
// int mark the edges whose neighbour is a pentagon.  core_row: per core cell
// what the two-ring kernels hand out lane by lane, CORE_ROW words a cell in
// trcadv12's format (k_core_rows), ROWP in the FP64 trcadv1's (k_patch_rows).
// words of trcadv12's core rows and where their parts begin (k_core_rows in
// fct_tiles.hip)
constexpr int CR_NBR = 36, CR_ST = 72, CR_NB = 90, CORE_ROW = 96;
struct EnsTiles {
  int npatch;
  const int *off;      // (npatch + 1) first tile cell of each patch
  const int4 *cnt;     // (npatch) n0, n1, n2, n3
  const int4 *ent;
  const int *core_row; // not the fused FCT's
  int r_max, lo_max;   // most cells of a patch in rings 0-1 and 0-2
};

// FP32 copies of the grid metrics (the reference stores them in FP32).
struct EnsGrid {
  DevGrid d;                 // FP64 metrics and the neighbour tables
  const float *cs, *sn, *svc, *sve, *sideln, *hfcoef;
  const float *area, *rarea, *corio, *grndspd, *dfflen;
  EnsTiles tiles;            // the patch partition of the fused tracer FCT
  EnsTiles ptiles;           // and that of trcadv12, with its core rows
};

struct EnsState {
  int members, ncol;
  float *us, *vs, *u2, *v2;
  int keep_trdp;                     // the tracer mass trcadv3 forms is read again (transport-only steps; otherwise hystat writes it)
  float *tr_alt, *trdp_alt;          // the other buffer of tr / trdp (the fused FCT writes it)
  double *dp, *pr, *ex, *ph, *mp, *sdot, *exsmo, *psrf, *ptdcy, *thbuf;
  float *tr, *trdp;
  float *u_tdcy, *v_tdcy, *dpl_tdcy;
  double *dp_tdcy;
  float *trc_tdcy, *trl_tdcy;
  float *massfx, *ws, *relvor;
  float *vn_edg, *dp_edg;             // vn_edg: normal edge wind
  float *pgx, *pgy;                   // the edge-pressure line integrals of cnuity5 (per cell-level)
  float *th0;                                  // theta at the start of the step
  float *antifx, *delp_lo, *r_plus, *r_mnus;
  float *antiflx, *trmax, *trmin, *tr_rp, *tr_rm;
  StepCtl *ctl;
  // Land/sea mask per column (0 = land), or null (every column wet).  An edge
  // carries mass and tracer flux only if both of its cells are wet (as the
  // ocean's continuity gates its fluxes, hycom_cnuity.F90:100-125); a land
  // column keeps its thickness, winds and tracers, and the Laplacian
  // momentum diffusion through a land edge is zero.
  const unsigned char *wet;
};
// wet(column) of a mask that may be null
__device__ __forceinline__ bool col_wet(const unsigned char *wet, int col) { return !wet || ldc(wet, col) != 0; }

// Launch shapes ("tiles"): columns per 256-lane-or-smaller block and whether
// the block index is remapped so that each XCD works on a contiguous range of
// cells (neighbour columns then share that XCD's L2).
constexpr int ENS_NTILES = 8;                       // cols {1,2,4,8} x swizzle {0,1}
inline int tile_cols(int t) { return 1 << (t & 3); }
inline bool tile_swz(int t) { return (t >> 2) & 1; }

// The numbers are part of the interface (fimhip_ens_set_tile).  trcadv12 has the
// number of the trcadv1 it took the place of; trcadv2's is kept, without a
// kernel, so that the numbers after it stay.
enum EnsKernel {
  EK_EDGVAR1 = 0, EK_EDGVAR3, EK_CNUITY12, EK_CNUITY3, EK_CNUITY45, EK_TRCADV12, EK_TRCADV2_NONE, EK_TRCADV3,
  EK_MOMTUM, EK_HYSTAT, EK_MASSADV1, EK_MASSADV2, EK_TRCFCT, EK_NKERNELS
};
extern const char *const ens_kernel_names[EK_NKERNELS];

// Class-B transport of the batched form: the tracers (nvl, ncol, ntrb) FP32,
// the ring of the last three steps' mass fluxes (nvl, 6, ncol, 3) and their
// AB-weighted time integral (nvl, 6, ncol) FP32, the thickness at the start of
// the integration and the vertical mass flux (nvl, ncol) FP64, and per class-B
// tracer the fct3d work fields (FP32; uan on the edges).
struct EnsClassB {
  int ntrb, dtratio;
  float *trb, *ring, *cumufx;
  double *dpinit, *w;
  float *fld, *vfx, *fmx, *fmn, *fld1, *flp, *fln, *uan;
};
void ens_launch_class_b_init(const EnsGrid &g, const EnsState &s, const EnsClassB &b, hipStream_t st);
void ens_launch_class_b_step(const EnsGrid &g, const EnsState &s, const EnsClassB &b, bool move, hipStream_t st);

// Sizes of the fused tracer FCT's patches (its LDS tile).
constexpr int FCT_CORE_MAX = 64;               // core cells of a patch
constexpr int FCT_R_MAX = 112;                 // cells in rings 0-1
constexpr int FCT_LO_MAX = 160;                // cells in rings 0-2
constexpr int FCT_TILE_MAX = 208;              // cells in rings 0-3
struct TileHost {
  std::vector<int> off;
  std::vector<std::array<int, 4>> cnt, ent;
};
struct TileLimits { int rings, core, r, lo, tile; };  // rings; most cells in the core, rings 0-1, 0-2, 0-3
constexpr TileLimits TRC_LIMITS = {2, 48, 84, 124, 124};   // trcadv12's patches: three blocks per CU
constexpr TileLimits TRC64_LIMITS = {2, 44, 80, 120, 120}; // the FP64 step's trcadv1
constexpr TileLimits FCT_LIMITS = {3, FCT_CORE_MAX, FCT_R_MAX, FCT_LO_MAX, FCT_TILE_MAX};
int ens_build_tiles(const HostGrid &h, int nip, const TileLimits &lim, TileHost &out);
int ens_upload_tiles(Arena &a, const TileHost &t, EnsTiles &d);
// marks in t's core cells the edges whose neighbour is a pentagon
void patch_pentagons(const HostGrid &h, TileHost &t);
// the FP64 step's patches of at most 'core' cells and their rows (trc_patch.hip)
int patch_tables(Arena &a, const HostGrid &h, const DevGrid &g, int core, EnsTiles &ts);
void launch_patch_trcadv1(const DevGrid &g, const DevState &s, const EnsTiles &ts, const AB &ab, hipStream_t st);
int ens_make_core(Arena &a, const TileHost &t, EnsGrid &g);   // g.ptiles' core rows
// the fused tracer FCT: reads s.tr / s.trdp, writes s.tr_alt / s.trdp_alt
void ens_launch_trcadv12(int tile, const EnsGrid &g, const EnsState &s, hipStream_t st);
void ens_launch_trc_fct(int tile, const EnsGrid &g, const EnsState &s, hipStream_t st);

void ens_launch_abstart(const EnsState &s, double dt, hipStream_t st);
void ens_launch(int kernel, int tile, const EnsGrid &g, const EnsState &s, hipStream_t st);
void ens_launch_pres_from_exner(const EnsGrid &g, const EnsState &s, hipStream_t st);
void ens_launch_trdp(const EnsGrid &g, const EnsState &s, hipStream_t st);
void ens_launch_hystat_init(const EnsGrid &g, const EnsState &s, hipStream_t st);
void ens_launch_convert_member(const EnsGrid &g, const EnsState &s, int member, const DevState &src,
                               hipStream_t st);
// count fields of n values: FP32 ones 'stride' apart to consecutive FP64 ones, and back
void ens_launch_widen(const float *src, double *dst, size_t n, size_t stride, int count, hipStream_t st);
void ens_launch_narrow(const double *src, float *dst, size_t n, size_t stride, int count, hipStream_t st);
void ens_launch_globsum(const EnsGrid &g, const EnsState &s, double *part64, float *part32, int nblocks,
                        hipStream_t st);

}  // namespace fimhip
