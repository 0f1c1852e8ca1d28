// Device-side layer view and kernel launchers of the COMCOT step.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace gc {

struct GaugeDev;

// What one step kernel needs of a layer.  Planes are column-major NX*NY
// float (index (J-1)*NX + I-1), time level 1 (in) and 2 (out) bound per
// launch from the layer's current parity.
struct DevLayer {
  int nx, ny;
  int is_root;     // outermost layer: loop ranges of ID==1 and the OPEN ring
  int modscm;      // 0: modified-scheme (SCM) term on
  int linchk;      // 1: convection terms on
  int fric;        // 1: Manning friction on (FRIC_SWITCH != 1)
  float rx, ry, grx, gry, dt;
  float kfric;     // (0.5*DT*GRAV)*FM*FM, the Fortran's CONST*FM*FM
  const float *h;
  const float *coef;   // per-row table (comcot_consts.h), spherical only
  const float *rowc;   // row-major copy of the coefficients (comcot_consts.h, kRowCoef floats a row)
  const float *r24;    // optional R2|R4 planes (drop-in fallback), else null
  const float *z1, *m1, *n1;
  float *z2, *m2, *n2;
  float *dzp;          // DZ(:,:,2) plane, kept for nonlinear parents, else null
  // wet-only max and first arrival, fused into the step when zmax != null
  float *zmax;
  int *arrival;
  int *ctl;            // root-step counters: read ctl[ctl_in], write ctl[1-ctl_in]
  int ctl_in, advance; // advance: this launch writes the next counter
  float arr_thr;
  float kf26;          // drag_scaled(kfric) (fastdiv.h)
  // MAX_AMP's maximum (GPUOutput.cu:46-53: no wet test, NaN replaces),
  // fused into the step of the outermost layer when != null
  float *zraw;
  // SPONGE_LAYER's coefficients COEFX per column I and COEFY per row J
  // (boundaries.f90:206-246), applied after the momentum pass when != null
  const float *sponge_cx, *sponge_cy;
  // 1: the single-layer step kernels (launch_step, launch_step2) write the
  // new level-2 planes Z2, M2, N2 of interior tiles with nontemporal
  // stores.  For a layer whose one step moves more bytes than the chip's
  // last-level cache holds, the next step finds none of them in a cache
  // anyway, and streaming them keeps the depth and maximum planes there;
  // for a layer small enough to stay in L2, streaming spares each kernel
  // end the write-back of the whole new level.  The batch kernels always
  // store through the caches.
  int stream_out;
  // bytes of the layer's block, which starts with h and holds every plane
  // above; 0 when they do not fit in one buffer descriptor (4 GB)
  unsigned block_bytes;
  // A nested layer's boundary fluxes of the next sub-step (one slot of
  // DevNest::edge) or null: a fused step then writes them, under JNQ's wet
  // test, where it otherwise writes 0, and the next sub-step needs no JNQ.
  const float *edge;
  // Host side, a nested layer's fused step only: the view of its linear root
  // whose momentum + next continuity (kMomentMass) launch_step runs beside the
  // step, in the same launch where that is faster.
  const DevLayer *beside;
  // ngauge > 0, the fused step of an outermost layer without nested ones: the
  // launch also samples these gauges of the step before, from z1, into
  // gauge_ring (launch_gauges' layout)
  const GaugeDev *gauges;
  float *gauge_ring;
  int ngauge, gauge_cap;
};
// Slot layout: M of rows 1..NY at column 1 and at column NX, then N of
// columns 1..NX at row 1 and at row NY.
constexpr size_t edge_floats(int nx, int ny) { return 2 * ((size_t)nx + ny); }

// kMomentMass: the momentum half of root step k of a linear outermost
// layer with nested layers, with the continuity (+ open boundary) of step
// k+1 in the same launch.  Nothing runs between the two in the root step
// order: momentum(k) reads Z(k) (after JNZ) and the level-1 fluxes and
// writes M(k), N(k) to level 2; continuity(k+1) reads Z(k), M(k), N(k)
// and writes Z(k+1) into the buffer that held Z(k-1), which linear
// momentum does not read.  The view's z1 is Z(k), its z2 that buffer.
enum StepMode { kFused = 0, kMassOnly = 1, kMomentOnly = 2, kMomentMass = 3 };

// One pass over all tiles of a layer (tile shape chosen by variant).
hipError_t launch_step(const DevLayer &L, int mode, bool nl, bool sph, int variant,
                       hipStream_t st);
int num_tile_variants();
void tile_variant_shape(int v, int *tx, int *ty);
bool tile_variant_is_tile(int v);  // the tiles come first, marching strips after them
// What a fused step of this view runs at variant `variant`: tiles of tx x ty, or
// marching strips of -tx columns in segments of ty rows.
void fused_form(const DevLayer &L, bool nl, bool sph, int variant, int *tx, int *ty);

// Two root steps of a linear outermost layer without children in one
// launch (temporal blocking); shape 0..6 = tiles of 64x8, 32x16, 64x16 with
// 256 threads, 64x16 with 512 and 1024, 32x16 with 512, 64x32 with 1024.
// Reads level 1, writes level 2 (two steps later); with zmax set, the
// wet maximum and arrival take both steps and the counter advances by 2.
hipError_t launch_step2(const DevLayer &L, bool sph, int shape, hipStream_t st);
constexpr int kStep2Shapes = 7;
// tile of two-step shape `shape`
void step2_shape(int shape, int *tx, int *ty);

// Root steps of a spherical linear outermost layer without children in the
// marching kernels (march.hip): 2 or 4 per launch, level 1 in, level 2 out,
// bookkeeping as launch_step2.  march_applies says whether a layer's view can
// take them (row-major coefficients, no R2/R4 planes, no MAX_AMP maximum or
// sponge, planes within 4 GB).
constexpr int kMarchSteps = 4;
inline bool march_applies(const DevLayer &L) {
  return L.is_root && L.rowc && !L.r24 && !L.zraw && !L.sponge_cx && L.block_bytes != 0;
}
hipError_t launch_march_linear(const DevLayer &L, int steps, hipStream_t st);
// kMomentMass of a spherical root in the marching form
hipError_t launch_march_moment_mass(const DevLayer &L, hipStream_t st);

// One fused step of a nonlinear layer with friction and convection in the
// marching kernels (march_nl.hip), in segments of seg rows; march_nl_seg
// gives the segments that suit a layer, 0 where the LDS tiles are faster.
inline bool march_nl_applies(const DevLayer &L, bool sph) {
  return (!sph || L.rowc) && L.modscm == 1 && L.linchk == 1 && L.fric && !L.r24 && !L.zraw &&
         !L.sponge_cx && L.block_bytes != 0;
}
int march_nl_seg(int nx, int ny);
hipError_t launch_march_nl(const DevLayer &L, bool sph, int seg, hipStream_t st);
// Whether tile variant v is a form of its own on this view: marching strips
// that a layer cannot take are variant 0 again.
inline bool tile_variant_takes(int v, const DevLayer &L, bool nl, bool sph) {
  return tile_variant_is_tile(v) || (nl && march_nl_applies(L, sph));
}

// Reference-semantics maximum (no wet test) plus the wet max/arrival.
hipError_t launch_max(const DevLayer &L, float *zmax_raw, hipStream_t st);

// Output planes of one layer for the reference's file writers, in one pass:
// oz = elevation with DATA_PRT's dry-land mask and tide (output.f90:781-793),
// om/on = copies of the fluxes, ozmax = MAX_AMP's masked maximum
// (output.f90:918-931).  Any output may be null.
struct OutPack {
  const float *z, *h, *m, *n, *zraw;
  float *oz, *om, *on, *ozmax;
  float tide;
  long long count;
};
hipError_t launch_out_pack(const OutPack &p, hipStream_t st);

// One fault plane of the Okada (1985) source as DEFORM_OKADA evaluates it
// (deform.f90:74-191), in FP64: constants of the fault and, for spherical
// layers, the stereographic projection split into per-row and per-column
// factors (deform.f90:494-588 depends on the latitude and the longitude
// separately until the final combination).
struct FaultDev {
  int nx, ny, sph;
  double sin_t, cos_t, halfl, w, hh, del_x, del_y, sn, cs, ds, dd;
  double two_rk0, sxi0, cxi0;  // spherical: 2 R K0, sin/cos of XI0
  const double *row;           // spherical: {sin XI, cos XI} per row J
  const double *col;           // spherical: {sin, cos}(LM - LM0) per column I
  double dx, dy, xl, yl;       // Cartesian: spacing, projected grid origin
};
// deform = vertical seafloor displacement of every cell of the layer
hipError_t launch_okada(const FaultDev &f, float *deform, hipStream_t st);
// CELL_INTERP (all_grids.f90:859-934): a nested layer's deformation from its
// parent's, in REAL; corners are the child's IS, IE, JS, JE in the parent
hipError_t launch_cell_interp(const float *parent, int pnx, float *child, int cnx, int cny,
                              const int *corners, int rel_size, hipStream_t st);
// Z1 += D and H -= D (deform.f90:55-64, UPDATE_BATH initialization.f90:
// 2410-2460); zraw != null also restarts MAX_AMP's maximum at the new Z1
hipError_t launch_apply_deform(float *z1, float *h, const float *deform, float *zraw, size_t n,
                               hipStream_t st);

// Nesting: child boundary fluxes for sub-step t (1 = JNQ, >1 = NEWQ)
struct DevNest {
  // parent
  int pnx, pny, p_sph, p_nl, p_r24;
  const float *ph, *pz2, *pm1, *pn1, *pcoef, *pr24;
  float pgrx, pgry;
  float *xflux, *yflux;  // parent cache (NX,2), (NY,2)
  // child
  int cnx, cny, rel_size, rel_time;
  int is, ie, js, je;    // footprint in the parent, 1-based
  const float *ch, *cz1, *cz2;
  float *cm1, *cn1;      // child level-1 fluxes, boundary written
  float *pz2_out;        // parent level-2 Z, footprint written by JNZ
  // the interface fluxes of the next `ahead` sub-steps, before the wet test,
  // go to ahead slots of edge (see DevLayer::edge)
  int ahead;
  float *edge;
  // launch_jnz, next_t > 0: JNQ/NEWQ of sub-step next_t (after UPDATE, so on
  // the child's level 2, whose fluxes are cm2, cn2) in the same launch
  int next_t;
  float *cm2, *cn2;
};
hipError_t launch_jnq(const DevNest &N, int t, hipStream_t st);
hipError_t launch_jnz(const DevNest &N, hipStream_t st);

// SC_OPTION = 1 coupling of a Cartesian child to its spherical parent
// (all_grids.f90:996-1425): boundary fluxes bilinear in the parent's fluxes
// at the positions POS/CXY that SUBGRID_MATCHING's reverse UTM projection
// gives every child cell, and the parent's elevation averaged from the wet
// child cells that fall in each parent cell.
struct DevSc {
  // parent (spherical)
  int pnx, pny, p_nl, p_modscm, p_r24;
  const float *ph, *pz2, *pm1, *pn1, *pcoef, *pr24;
  float *pm2, *pn2;    // parent level-2 fluxes: NEWQ_SC's band forecasts
  float *pz2_out;      // parent level-2 elevation, averaged by JNZ_SC
  // child (Cartesian)
  int cnx, cny, rel_time;
  float half;          // REAL(REL_SIZE**2)/2
  const int *pos;      // POS(NX,NY,2), component-major
  const float *cxy;    // CXY(NX,NY,4), component-major
  const float *ch, *cz_now, *cz2;  // H, newest Z (Fortran level 2 after UPDATE), level-2 buffer
  float *cm1, *cn1;    // child level-1 fluxes, boundary written
  const int *steps_done;  // root steps completed: the child's first sub-step ever sees Z2 = 0
  int band[4][4];      // M bands (left, right edge), N bands (top, bottom): IS, IE, JS, JE
  int corners[4];      // the POS extent
  const int *jnz_off, *jnz_idx;  // per parent cell of the extent: its child cells in Fortran order
};
hipError_t launch_sc_edges(const DevSc &S, int t, hipStream_t st);
hipError_t launch_sc_jnz(const DevSc &S, hipStream_t st);
// CELL_INTERP_SC (all_grids.f90:938-992): a child's deformation from its parent's
hipError_t launch_sc_cell_interp(const float *parent, int pnx, int pny, float *child, int cnx,
                                 int cny, const int *pos, const float *cxy, hipStream_t st);

// ---- batch engine: one persistent launch over the tiles of many layers
struct BatchDesc {
  DevLayer L;
  int tiles_x, ntiles;
};
struct alignas(8) BatchItem {
  int slot, tile;  // descriptor index, tile index within that layer
};
struct BatchLaunch {
  const BatchDesc *descs;
  const BatchItem *items;
  const int *qstart;  // 9 entries: items of XCD queue q are [qstart[q], qstart[q+1])
  int *heads;         // 8 queue heads, zero before the launch
  int nitems;
  int dry;            // 1: the layers' views carry no maximum planes
};
// Fused launches take tile shape `shape` (batch_shape): 0-2 the persistent
// form and 3-5 the grid form of 64 x 8, 32 x 16 and 64 x 16 tiles, and for
// nonlinear layers 6 = grid form of 32 x 8 tiles (one cell per thread), 7 and
// 8 = marching strips, four waves of 8 or 14 rows to an item.  Continuity and
// momentum halves of nested parents use 64 x 8.  prepare: only look up
// the kernel's resident-workgroup count (do it before a graph capture).
int batch_num_shapes();
void batch_shape(int k, int *tx, int *ty);
constexpr int kBatchGridShape = 3, kBatchForcedShapes = 6, kBatchSmallShape = 6, kBatchMarchShape = 7;
inline bool batch_shape_takes(int shape, const DevLayer &L, bool nl, bool sph) {
  return shape < kBatchSmallShape || (nl && (shape < kBatchMarchShape || march_nl_applies(L, sph)));
}
// The shape of a fused launch that nobody tuned: marching strips where the
// layers together give their SIMDs enough rows (the lines of march_nl_seg),
// one cell per thread below, 64 x 8 tiles for linear layers.
inline int batch_rule_shape(const DevLayer *layers, int n, bool nl) {
  if (!nl) return kBatchGridShape;
  long long rows = 0;
  for (int k = 0; k < n; ++k) rows += (long long)((layers[k].nx + 59) / 60) * layers[k].ny / 1024;
  return rows < 16 ? kBatchSmallShape : (rows < 36 ? kBatchMarchShape : kBatchMarchShape + 1);
}
hipError_t launch_batch(const BatchLaunch &B, int mode, bool nl, bool sph, int shape,
                        hipStream_t st, bool prepare = false);
// Two root steps of single-layer linear layers, one workgroup per item;
// items tile each layer with step2_shape(shape) tiles.
hipError_t launch_batch2(const BatchLaunch &B, bool sph, int shape, hipStream_t st);
// Two-step shape 6 of the batch is the marching form for spherical layers
// (and a tile of the same size for Cartesian ones); kStep2TileShape suits any.
constexpr int kStep2March = 6, kStep2TileShape = 4;
inline bool step2_shape_takes(int shape, const DevLayer &L, bool sph) {
  return shape != kStep2March || !sph || march_applies(L);
}
// The marching forms of launch_batch and launch_batch2.
hipError_t launch_batch_march_nl(const BatchLaunch &B, bool sph, int seg, hipStream_t st);
hipError_t launch_batch_march2(const BatchLaunch &B, hipStream_t st);
// JNQ/NEWQ and JNZ of several nests in one launch: nest n owns blocks
// [start[n], start[n+1]) of 128 threads; *_block_count gives each one's share.
int jnq_block_count(const DevNest &N);
int jnz_block_count(const DevNest &N);
hipError_t launch_jnq_multi(const DevNest *nests, const int *start, int nnest, int nblocks,
                            int t, hipStream_t st);
hipError_t launch_jnz_multi(const DevNest *nests, const int *start, int nnest, int nblocks,
                            hipStream_t st);
hipError_t launch_fill_i32(int *p, int n, int v, hipStream_t st);
// ---- gauges: bilinear samples of the elevation after each root step
struct GaugeDev {
  int lid, ki, kj, nx;   // layer, 1-based lower-left stencil cell, layer width
  float cx, cy, tide;    // GET_TS weights and tide-level offset
  int pad;
};
struct ZNow {
  const float *z[20];    // current elevation plane of each layer id (index = id)
};
// Sample n gauges into ring[g * cap + (step - 1) % cap], step = *step_now
// (the root steps completed), with GET_TS's arithmetic (output.f90:1085-1094).
hipError_t launch_gauges(const GaugeDev *g, int n, const ZNow &z, const int *step_now,
                         float *ring, int cap, hipStream_t st);

// Streaming copy of bytes (a multiple of 16) from src to dst.
hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t st);
// Self-check of the short divisions and square root (fastdiv.h) against
// the IEEE operations: out[6g..6g+5] = lane g's mismatches of div12 and
// sqrt_inrange (over its slice of all floats) and of div_inrange (over
// per_lane random in-range pairs), then its first mismatching x, pair
// (a << 32 | b) and square-root argument; 256*blocks lanes.
// powf_manning(x[q], 2.3333333f) -> pw[q] and expf_det(x[q]) -> ex[q], q < n.
hipError_t launch_detmath_eval(const float *x, long long n, float *pw, float *ex,
                               hipStream_t st);
hipError_t launch_division_check(unsigned long long seed, int per_lane, unsigned long long *out,
                                 int blocks, hipStream_t st);
// The same of its refined reciprocal: out[3g..3g+2] = lane g's divisors tested,
// mismatches and the bits of its first one; 256*blocks lanes.
hipError_t launch_reciprocal_check(unsigned long long *out, int blocks, hipStream_t st);

}  // namespace gc
