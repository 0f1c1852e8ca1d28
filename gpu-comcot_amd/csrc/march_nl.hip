// Register-marching step of nonlinear layers: one time step, every plane
// read and written once.
//
// A wavefront holds a strip of 64 columns (60 written) and marches along J.
// Row r enters the continuity pass, then the flux-point quantities of row r
// (X) and r - 1 (Y), the X momentum of row r - 1 and the Y momentum of row
// r - 2, all from rows held in registers; neighbouring columns come from the
// neighbouring lanes.  There is no LDS traffic but the pow/exp tables, and
// no barrier in the loop.  A strip's halo rows skip the momentum passes: they
// are two thirds of a row's instructions (4096x3072 118.3 us per step with
// them, 115.5 without; 1201x901 Cartesian 20.2 and 18.3).
//
// The nonlinear step is bound by VALU issue (the fused tile takes 560
// instructions per cell).  Marching shares what the tile form computes
// again in every cell that reads it: the advection quotients P*P/D, P*Q/D of
// a flux point serve the point itself and its four neighbours (a tile
// divides anew for each, eight divisions a cell instead of four), the flux
// depths, averaged fluxes and wet tests likewise; tests of neighbouring
// cells are shifts of lane masks in scalar registers; and staging, halo
// recomputation and per-cell index arithmetic go.
//
// Values are those of the tile kernels bit for bit: the same operations on
// the same operands (CONMASS_S mass.f90:227-277 / CONMASS :162-224, OPEN
// boundaries.f90:22-202, CONMOME_S moment.f90:783-1384 / CONMOME :280-780).
// Where a Fortran case takes A - B, B - A, A or -A of two quotients, the
// form here is +-(A - B) with B = 0 in the one-sided cases; the two differ
// in the sign of a zero term only, which the EPS test on the flux clears.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "comcot_consts.h"
#include "detmath.h"
#include "fastdiv.h"
#include "kernels.h"
#include "march.h"

namespace gc {

namespace {

typedef unsigned long long Mask;
#define GC_BALLOT(c) __builtin_amdgcn_ballot_w64(c)

// What the momentum of a flux point between cell a and cell b (b = I + 1 or
// J + 1) reads.
struct Face {
  float p, cross;        // own flux, averaged flux across
  float ha, hb, za, zb;  // depth and new elevation of the two cells
  float dza, dzb;        // their total depths (Cartesian shoreline case)
  float d1;              // a quarter of their sum, DP/DQ(.,.,1) where >= GX
  Mask wa, wb;           // DZ > GX of the two cells
};

// The wet/dry cases of CONMOME(_S) (moment.f90:396-425, 892-921): depth DD
// for the pressure term, DF for friction, and the lanes that move at all.
// Where both cells are wet DD is twice d1, above GX, and H(a) > ELMAX leaves
// the depth at the point above ELMAX too; the one-sided cases are only
// evaluated in waves that hold a wet cell beside a dry one.
template <bool SPH>
__device__ __forceinline__ Mask face_depths(const Face &f, float &DD, float &DF) {
  Mask act = f.wa & f.wb;
  DD = f.d1 + f.d1;
  DF = fmaxf(f.d1, 1.0e-3f);
  if (f.wa ^ f.wb) {
    const Mask out = f.wa & ~f.wb & GC_BALLOT(f.hb + f.za > kGx);
    const Mask in = ~f.wa & f.wb & GC_BALLOT(f.ha + f.zb > kGx);
    const float hface = f.ha > kGx ? 0.5f * (f.ha + f.hb) : 0.0f;
    const float part = SPH ? hface + 0.5f * (f.za + f.zb) : 0.5f * (lanes(out) ? f.dza : f.dzb);
    const Mask one = (out | in) & ~GC_BALLOT(hface <= kElmax) & ~GC_BALLOT(part < kGx);
    DD = lanes(one) ? part : DD;
    DF = lanes(one) ? fmaxf(part, 1.0e-3f) : DF;
    act |= one;
  }
  return act & ~GC_BALLOT(f.ha <= kElmax);
}

__device__ __forceinline__ float friction(const DevLayer &L, const Face &f, float DF,
                                          const gcdet::Tables &tab) {
  return div_inrange(L.kfric * sqrt_inrange(f.p * f.p + f.cross * f.cross),
                     gcdet::powf_manning(DF, kManExp, tab));
}

// One upwind term fac * (+-(a - b)): b is the quotient of the upwind
// neighbour, 0 where that one is dry (gone), neg the lanes flowing backwards.
__device__ __forceinline__ float upwind(float fac, float a, float fwd, float back, Mask gone, Mask neg) {
  float b = lanes(neg) ? fwd : back;
  b = lanes(gone) ? 0.0f : b;
  const float t = a - b;
  return fac * (lanes(neg) ? -t : t);
}

// EPS and V_LIMIT (moment.f90:565-572, 1054-1060), 0 in the lanes that do
// not move (V_LIMIT * DD is above EPS, so the order of the two is free)
__device__ __forceinline__ float limited(float x, float DD, Mask act) {
  const float lim = kVLimit * DD;
  const float y = fabsf(x) > lim ? copysignf(lim, x) : x;
  return lanes(act & ~GC_BALLOT(fabsf(x) < kEps)) ? y : 0.0f;
}

// One step of strip S (layers with friction and convection, FRIC_SWITCH = 0
// and LAYGOV other than 9).  COL: the strip's cells or halo lie within
// SPAN + 2 columns of the grid's edge (loads are clamped, OPEN, the ghost
// column and the ranges of the Fortran loops apply); ROW: the same for rows;
// otherwise all of that compiles away.
template <bool SPH, bool COL, bool ROW, bool MX, bool ST>
__device__ __forceinline__ void march_nl(const DevLayer &L, const Strip S, int step,
                                         const gcdet::Tables &tab) {
  // halo columns and rows; rows in flight, and unrolled (the rings of three
  // rows then rotate without moves)
  constexpr int HW = 2, D = COL || ROW ? 2 : 3;
  const int nx = L.nx, ny = L.ny, lane = threadIdx.x & (kWave - 1);
  const int i = S.c0 - HW + lane;
  const int ic = COL ? min(max(i, 1), nx) : i;
  const bool own = lane >= HW && lane < kWave - HW && (!COL || i <= nx);
  const int vld = (ic - 1) * 4, vst = own ? vld : kNoStore;
  const bool root = L.is_root;
  // column masks: the ring's or ghost column I = 1, column NX, the columns
  // where the momentum ranges and the convection terms hold
  const Mask col1 = COL ? GC_BALLOT(i == 1) : 0, coln = COL ? GC_BALLOT(i == nx) : 0;
  const Mask colx = COL ? GC_BALLOT(i >= (root ? 1 : 2) && i <= nx - 1) : ~0ull;
  const Mask coly = COL ? GC_BALLOT(i >= (root ? 1 : 2) && i <= (root ? nx - 1 : nx)) : ~0ull;
  const Mask conv_col = COL ? GC_BALLOT(i > kSpan && i < nx - kSpan) : ~0ull;
  const Mask ghost = COL ? GC_BALLOT(i < 2) : 0;
  const int ra = S.j0 - HW, rb = S.j1 + HW;
  const Block B = block_of(L);
  const unsigned pitch = (unsigned)nx * 4u;
  const unsigned oz1 = plane_off(L, L.z1), om1 = plane_off(L, L.m1), on1 = plane_off(L, L.n1),
                 oz2 = plane_off(L, L.z2), om2 = plane_off(L, L.m2), on2 = plane_off(L, L.n2),
                 omax = plane_off(L, L.zmax), oarr = plane_off(L, L.arrival);
  const float zt = breaking_floor(L.dt);
  // a nested layer's boundary fluxes of the next sub-step: M of the side
  // columns comes row by row, N of rows 1 and NY once.  Lanes without one, and
  // every lane where there are none, read past the table: 0.
  const bool has_edge = (COL || ROW) && L.edge;
  const Block E = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(L.edge), 0, has_edge ? (int)(edge_floats(nx, ny) * sizeof(float)) : 0, 0x00027000);
  const Mask edge_col = has_edge ? col1 | coln : 0;
  auto edge_n = [&](int row_off) {
    return get(E, has_edge && i >= 1 && i <= nx ? (row_off + i - 1) * 4 : kNoStore, 0);
  };
  const float n_lo = ROW ? edge_n(2 * ny) : 0.0f, n_hi = ROW ? edge_n(2 * ny + nx) : 0.0f;

  float ph[D], pz[D], pm[D], pn[D], pq[D], pe[D];
  auto load = [&](int j, int k) {
    const unsigned b = (unsigned)((ROW ? min(max(j, 1), ny) : min(j, rb)) - 1) * pitch;
    ph[k] = get(B, vld, b);
    pz[k] = get(B, vld, oz1 + b);
    pm[k] = get(B, vld, om1 + b);
    pn[k] = get(B, vld, on1 + b);
    if (MX) pq[k] = get(B, vld, omax + b);
    if (COL) {
      const int je = min(max(j, 1), ny) - 1;
      pe[k] = get(E, lanes(edge_col) ? ((i == 1 ? 0 : ny) + je) * 4 : kNoStore, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < D; ++k) load(ra + k, k);
  // rows r, r - 1, r - 2 at index 0, 1, 2
  float H[3] = {}, M[2] = {}, N[3] = {}, NR[2] = {}, Z[3] = {}, DZ[3] = {}, brk[3] = {1, 1, 1};
  float me[2] = {};
  float d1[2] = {}, xqq[2] = {}, pp[2] = {}, pc[3] = {};              // X points
  float e1[3] = {}, xpp[3] = {}, qq[4] = {}, qc[3] = {};              // Y points
  Mask W[3] = {}, ZD[3] = {};   // DZ > GX, DZ < GX
  Mask slow[3] = {};            // lanes whose breaking factor is not 1
  Mask P1[2] = {}, PX[3] = {};  // X points: depth below GX; that or a dry cell
  Mask Q1[4] = {}, QY[3] = {};  // Y points
  // whether row j is written: halo rows need no momentum
  auto live = [&](int j) { return (unsigned)(j - S.j0) <= (unsigned)(S.j1 - S.j0); };
  Row4 c0 = row_coef(L, ra, 0);

  auto row = [&](int r, int k) __attribute__((always_inline)) {
    const Row4 C = c0;
    Row4 CX, CY;
    if (SPH) {
      c0 = row_coef(L, r + 1, 0);
      CX = row_coef(L, r - 1, 1);
      CY = row_coef(L, r - 2, 2);
    }
    H[0] = ph[k];
    M[0] = pm[k];
    N[0] = pn[k];
    const float z1 = pz[k], zl = MX ? pq[k] : 0.0f;
    if (COL) me[0] = pe[k];
    load(r + D, k);
    const int vz = live(r) ? vst : kNoStore;

    // ---- continuity at row r
    {
      float zz;
      const float mw = west(M[0]);
      if (SPH) {
        NR[0] = N[0] * C[2];
        zz = z1 - C[0] * (M[0] - mw) - C[1] * (NR[0] - NR[1]);
      } else {
        zz = z1 - L.rx * (M[0] - mw) - L.ry * (N[0] - N[1]);
      }
      if (fabsf(zz) < kEps) zz = 0.0f;
      const float dd = zz + H[0];
      Mask up = (SPH ? GC_BALLOT(H[0] >= kElmax) : GC_BALLOT(H[0] > kElmax)) & GC_BALLOT(dd >= kGx);
      DZ[0] = lanes(up) ? dd : 0.0f;
      Z[0] = lanes(up) ? zz : -H[0];
      // H + Z2 of a wet cell is DZ, of a dry one 0
      Mask wet = GC_BALLOT(DZ[0] > kGx);
      W[0] = wet;
      if ((COL || ROW) && root) {  // the radiating ring
        const bool row_end = ROW && (r == 1 || r == ny);
        const Mask ring = row_end ? ~0ull : (col1 | coln);
        if (ring) {
          const bool w1 = lanes(col1), wn = lanes(coln);
          const float u = w1 ? M[0] : mw;
          float a, b;
          bool neg;
          if (row_end) {
            b = r == 1 ? N[0] : N[1];
            const bool corner = w1 | wn;
            a = corner ? u : 0.5f * (M[0] + mw);
            neg = r == 1 ? b > 0.0f : b < 0.0f;
            neg |= corner & (w1 ? u > 0.0f : u < 0.0f);
          } else {
            a = (w1 & !(H[1] > kGx)) ? N[0] : 0.5f * (N[0] + N[1]);
            b = u;
            neg = w1 ? u > 0.0f : u < 0.0f;
          }
          const float zr = radiate(H[0], sqrtf(kGrav * H[0]), a, b, neg);
          Z[0] = lanes(ring) ? zr : Z[0];
          DZ[0] = lanes(ring) ? 0.0f : DZ[0];
          wet = (wet & ~ring) | (ring & GC_BALLOT(H[0] + zr > kGx));
          W[0] &= ~ring;
          up &= ~ring;
        }
      } else if (COL || ROW) {  // ghost row and column
        const Mask g = ROW && r < 2 ? ~0ull : ghost;
        Z[0] = lanes(g) ? 0.0f : Z[0];
        DZ[0] = lanes(g) ? 0.0f : DZ[0];
        wet &= ~g;
        W[0] &= ~g;
        up &= ~g;
      }
      ZD[0] = ~up;
      const unsigned g = (unsigned)(r - 1) * pitch;
      if ((COL || ROW) && !root) {  // UPDATE's copies (all_grids.f90:323-324)
        const float ze = east(Z[0]);
        const float zo = lanes(col1) ? ze : Z[0];
        if (ROW) put<ST>(B, S.j0 == 1 && r == 2 ? vst : kNoStore, oz2, zo);
        put<ST>(B, ROW && r == 1 ? kNoStore : vz, oz2 + g, zo);
      } else {
        put<ST>(B, vz, oz2 + g, Z[0]);
      }
      if (MX) {  // wet maximum and first arrival
        const Mask more = wet & GC_BALLOT(Z[0] > zl);
        put<false>(B, lanes(more) ? vz : kNoStore, omax + g, Z[0]);
        const Mask first = wet & GC_BALLOT(Z[0] >= L.arr_thr) & ~GC_BALLOT(zl >= L.arr_thr);
        put<false>(B, lanes(first) ? vz : kNoStore, oarr + g, __int_as_float(step));
      }
      // WAVE_BREAKING's factor (moment.f90:1272-1384; the tile kernels'
      // breaking_coef states the ranges)
      const float dz = fabsf(Z[0] - z1);
      brk[0] = 1.0f;
      slow[0] = GC_BALLOT(dz > zt * __builtin_amdgcn_sqrtf(DZ[0]));
      if (slow[0]) {
        const float c = sqrt_inrange(kGrav * DZ[0]);
        const float dzdt_f = 0.08f * c, dzdt_i = 0.65f * c;
        const float dzdt = div_by(dz, L.dt, recip_refined(L.dt));
        if (dzdt > dzdt_f)
          brk[0] = gcdet::expf_det(-(1.0f * ((dzdt - dzdt_f) / (dzdt_i - dzdt_f))), tab);
      }
    }
    // ---- flux points X(r): depth, averaged N, advection quotients
    {
      d1[0] = 0.25f * (DZ[0] + east(DZ[0]));
      P1[0] = GC_BALLOT(d1[0] < kGx);
      const float ns = ROW && r == 1 ? N[0] : N[1];
      xqq[0] = 0.25f * (N[0] + east(N[0]) + ns + east(ns));
      const float y = recip_refined(d1[0]);
      pp[0] = div_by(M[0] * M[0], d1[0], y);
      pc[0] = div_by(M[0] * xqq[0], d1[0], y);
      PX[0] = ZD[0] | (ZD[0] >> 1) | P1[0];
    }
    // ---- flux points Y(r - 1)
    {
      e1[1] = 0.25f * (DZ[1] + DZ[0]);
      Q1[1] = GC_BALLOT(e1[1] < kGx);
      const float ms = M[1] + M[0];
      float mw0 = west(M[1]), mw1 = west(M[0]);
      if (COL) {
        mw0 = lanes(col1) ? M[1] : mw0;
        mw1 = lanes(col1) ? M[0] : mw1;
      }
      xpp[1] = 0.25f * (ms + mw0 + mw1);
      const float y = recip_refined(e1[1]);
      qq[1] = div_by(N[1] * N[1], e1[1], y);
      qc[1] = div_by(N[1] * xpp[1], e1[1], y);
      QY[1] = ZD[1] | ZD[0] | Q1[1];
    }
    // ---- X momentum at row j = r - 1
    {
      const int j = r - 1;
      const Face f{M[1], xqq[1], H[1], east(H[1]), Z[1], east(Z[1]), DZ[1], SPH ? 0.0f : east(DZ[1]),
                   d1[1], W[1], W[1] >> 1};
      float DD, DF, X = 0.0f;
      Mask act = live(j) ? face_depths<SPH>(f, DD, DF) : 0;
      if (COL || ROW) act &= !ROW || (root ? j <= ny - 1 : j >= 2) ? colx : 0;
      const float pe = east(pp[1]), pw = west(pp[1]);
      if (act) {
        X = f.p - (SPH ? CX[0] : L.grx) * DD * (f.zb - f.za);
        const Mask drag = SPH ? act & ~GC_BALLOT(drag_vanishes(L.kf26, f.p, f.cross, DF, X)) : ~0ull;
        float FF = 0.0f;
        if (drag) {
          FF = friction(L, f, DF, tab);
          X = X - FF * f.p;
        }
        if (SPH) X = X + CX[1] * f.cross;
        Mask conv = ~P1[1];
        if (COL || ROW) conv &= !ROW || (j > kSpan && j < ny - kSpan) ? conv_col : 0;
        const Mask pn = GC_BALLOT(f.p < 0.0f), qn = GC_BALLOT(f.cross < 0.0f);
        const Mask gx = (pn & ((P1[1] >> 1) | (ZD[1] >> 1))) | (~pn & ((P1[1] << 1) | ZD[1]));
        const Mask gy = (qn & PX[0]) | (~qn & PX[2]);
        float ax = upwind(SPH ? CX[2] : L.rx, pp[1], pe, pw, gx, pn);
        float ay = upwind(SPH ? CX[3] : L.ry, pc[1], pc[0], pc[2], gy, qn);
        if (slow[1]) ax = brk[1] * ax, ay = brk[1] * ay;
        const float adv = X - ax - ay;
        X = lanes(conv) ? adv : X;
        if (drag) X = div_inrange(X, 1.0f + FF);
        X = limited(X, DD, act);
      }
      if (COL) {
        const bool dry = H[1] + (lanes(col1) ? f.zb : Z[1]) <= kGx;
        X = lanes(!ROW || j >= 2 ? edge_col : 0) ? (dry ? 0.0f : me[1]) : X;
      }
      put<ST>(B, live(j) ? vst : kNoStore, om2 + (unsigned)(j - 1) * pitch, X);
    }
    // ---- Y momentum at row j = r - 2
    {
      const int j = r - 2;
      const Face f{N[2], xpp[2], H[2], H[1], Z[2], Z[1], DZ[2], DZ[1], e1[2], W[2], W[1]};
      float DD, DF, Y = 0.0f;
      Mask act = live(j) ? face_depths<SPH>(f, DD, DF) : 0;
      if (COL || ROW) act &= !ROW || (j <= ny - 1 && (root || j >= 2)) ? coly : 0;
      const float qe = east(qc[2]), qw = west(qc[2]);
      if (act) {
        Y = f.p - (SPH ? CY[0] : L.gry) * DD * (f.zb - f.za);
        const Mask drag = SPH ? act & ~GC_BALLOT(drag_vanishes(L.kf26, f.p, f.cross, DF, Y)) : ~0ull;
        float FF = 0.0f;
        if (drag) {
          FF = friction(L, f, DF, tab);
          if (SPH) Y = Y - FF * f.p;
        }
        if (SPH) Y = Y - CY[1] * f.cross;
        Mask conv = ~Q1[2];
        if (COL || ROW) conv &= !ROW || (j > kSpan && j < ny - kSpan) ? conv_col : 0;
        const Mask qn = GC_BALLOT(f.p < 0.0f), pn = GC_BALLOT(f.cross < 0.0f);
        const Mask gy = (qn & (Q1[1] | ZD[1])) | (~qn & (Q1[3] | ZD[2]));
        const Mask gx = (pn & (QY[2] >> 1)) | (~pn & (QY[2] << 1));
        float ay = upwind(SPH ? CY[3] : L.ry, qq[2], qq[1], qq[3], gy, qn);
        float ax = upwind(SPH ? CY[2] : L.rx, qc[2], qe, qw, gx, pn);
        if (slow[2]) ax = brk[2] * ax, ay = brk[2] * ay;
        const float adv = Y - ax - ay;
        Y = lanes(conv) ? adv : Y;
        if (drag) Y = div_inrange(Y, 1.0f + FF);
        Y = limited(Y, DD, act);
      }
      if (ROW && has_edge && (j == 1 || j == ny)) {
        const bool dry = H[2] + (j == 1 ? Z[1] : Z[2]) <= kGx;
        Y = lanes(~col1) ? (dry ? 0.0f : (j == 1 ? n_lo : n_hi)) : Y;
      }
      put<ST>(B, live(j) ? vst : kNoStore, on2 + (unsigned)(j - 1) * pitch, Y);
    }
    // ---- the rows move on
#define GC_SHIFT2(a) a[1] = a[0]
#define GC_SHIFT3(a) a[2] = a[1], a[1] = a[0]
    GC_SHIFT3(H); GC_SHIFT2(M); GC_SHIFT3(N); GC_SHIFT2(NR); GC_SHIFT3(Z); GC_SHIFT3(DZ); GC_SHIFT3(brk);
    if (COL) GC_SHIFT2(me);
    GC_SHIFT2(d1); GC_SHIFT2(xqq); GC_SHIFT2(pp); GC_SHIFT3(pc);
    e1[2] = e1[1]; xpp[2] = xpp[1]; qc[2] = qc[1];
    qq[3] = qq[2]; qq[2] = qq[1];
    GC_SHIFT3(W); GC_SHIFT3(ZD); GC_SHIFT3(slow); GC_SHIFT2(P1); GC_SHIFT3(PX);
    Q1[3] = Q1[2]; Q1[2] = Q1[1]; QY[2] = QY[1];
#undef GC_SHIFT2
#undef GC_SHIFT3
    __builtin_amdgcn_sched_barrier(0);
  };
  // The first loads are waited for here (vmcnt 0), as in march_linear.
  __builtin_amdgcn_s_waitcnt(0x0f70);
  for (int r = ra; r <= rb; r += D)
#pragma unroll
    for (int u = 0; u < D; ++u) row(r + u, u);
}

__device__ __forceinline__ void stage(gcdet::Tables &dst) {
  constexpr int n = sizeof(gcdet::Tables) / sizeof(double);
  const double *src = reinterpret_cast<const double *>(&gcdet::kTab);
  double *d = reinterpret_cast<double *>(&dst);
  for (int k = threadIdx.x; k < n; k += kMarchBlock) d[k] = src[k];
  __syncthreads();
}

constexpr int kNlWidth = kWave - 4;
// rows at either end whose waves need the ROW form
constexpr int kNlEnd = kSpan + 4;

// How the waves of a launch split a layer: strips of 60 columns.  Strip 0
// and the strips from east on reach the side columns (COL); the middle
// strips take end_rows rows at either end (ROW) in pieces of seg_end rows,
// and segments of seg rows between.  A row of the COL and ROW forms costs up
// to twice a middle one, so those waves take shorter segments and come first.
struct NlGrid {
  int nstrip, east, end_rows, seg_end, nend, seg, nseg, seg_side, nseg_side, first_blocks, per_xcd;
};

// The strip of wave w of the first blocks (side strips, then the middle
// strips' ends); false past the last.
__device__ __forceinline__ bool nl_first(const NlGrid &G, int ny, int w, Strip &S) {
  const int nside = 1 + G.nstrip - G.east, mid = G.east - 1;
  if (w < nside * G.nseg_side) {
    const int k = w % nside;
    S.c0 = (k == 0 ? 0 : G.east + k - 1) * kNlWidth + 1;
    S.j0 = (w / nside) * G.seg_side + 1;
    S.j1 = min(S.j0 + G.seg_side - 1, ny);
    return true;
  }
  w -= nside * G.nseg_side;
  if (w >= 2 * G.nend * mid) return false;
  const int k = w / mid, top = k >= G.nend;  // piece k of the lower end, then of the upper
  S.c0 = (1 + w % mid) * kNlWidth + 1;
  S.j0 = (top ? max(ny - G.end_rows, G.end_rows) + (k - G.nend) * G.seg_end : k * G.seg_end) + 1;
  S.j1 = min(S.j0 + G.seg_end - 1, top ? ny : min(G.end_rows, ny));
  return S.j0 <= S.j1;
}

template <bool SPH, bool MX, bool ST>
__global__ void __launch_bounds__(kMarchBlock) k_march_nl(DevLayer L, NlGrid G) {
  constexpr int WB = kMarchBlock / kWave;
  __shared__ gcdet::Tables tab;
  const int g = step_block(L);
  if (g < 0) return;
  stage(tab);
  int step = 0;
  if (MX) {
    step = L.ctl[L.ctl_in] + 1;
    if (L.advance && g == 0 && threadIdx.x == 0) L.ctl[1 - L.ctl_in] = step;
  }
  Strip S;
  if (g < G.first_blocks) {
    const int w = __builtin_amdgcn_readfirstlane(g * WB + (threadIdx.x >> 6));
    if (!nl_first(G, L.ny, w, S)) return;
    if (S.j0 > kNlEnd && S.j1 <= L.ny - kNlEnd)
      march_nl<SPH, true, false, MX, ST>(L, S, step, tab);
    else
      march_nl<SPH, true, true, MX, ST>(L, S, step, tab);
    return;
  }
  const int b = g - G.first_blocks, mid = G.east - 1;
  const int w = __builtin_amdgcn_readfirstlane(((b & 7) * G.per_xcd + (b >> 3)) * WB + (threadIdx.x >> 6));
  if (w >= mid * G.nseg) return;
  S.c0 = (1 + w % mid) * kNlWidth + 1;
  S.j0 = G.end_rows + (w / mid) * G.seg + 1;
  S.j1 = min(S.j0 + G.seg - 1, L.ny - G.end_rows);
  march_nl<SPH, false, false, MX, ST>(L, S, step, tab);
}

template <bool SPH, bool MX, bool ST>
hipError_t launch_nl(const DevLayer &L, int seg, hipStream_t st) {
  constexpr int WB = kMarchBlock / kWave;
  NlGrid G;
  G.nstrip = (L.nx + kNlWidth - 1) / kNlWidth;
  // first strip with an owned column beyond NX - SPAN - 3
  G.east = std::min(std::max((L.nx - kSpan - 3) / kNlWidth, 1), G.nstrip);
  G.seg = seg;
  G.seg_side = L.is_root ? std::max(seg / 2, 4) : seg;  // OPEN runs in the root's
  G.end_rows = std::max(kNlEnd, G.seg_side);
  G.nend = (G.end_rows + G.seg_side - 1) / G.seg_side;
  G.seg_end = (G.end_rows + G.nend - 1) / G.nend;
  G.nseg_side = (L.ny + G.seg_side - 1) / G.seg_side;
  G.nseg = std::max(0, (L.ny - 2 * G.end_rows + seg - 1) / seg);
  const long long first = (long long)(1 + G.nstrip - G.east) * G.nseg_side + 2LL * G.nend * (G.east - 1);
  const long long mid = (long long)(G.east - 1) * G.nseg;
  G.first_blocks = (int)((first + WB - 1) / WB);
  G.per_xcd = (int)((mid + 8 * WB - 1) / (8 * WB));
  const long long blocks = (long long)G.first_blocks + 8LL * G.per_xcd + gauge_blocks(L);
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_march_nl<SPH, MX, ST>), dim3((unsigned)blocks), dim3(kMarchBlock), 0, st, L, G);
  return hipGetLastError();
}

// The batch form: one workgroup per (layer, tile) item of a 60 x 4 SEG tiling,
// a wave per SEG rows.
template <bool SPH, bool MX, int SEG>
__global__ void __launch_bounds__(kMarchBlock)
    k_batch_march_nl(const BatchDesc *__restrict__ descs, const BatchItem *__restrict__ items, int nitems,
                     int per_xcd) {
  __shared__ gcdet::Tables tab;
  const int it = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (it >= nitems) return;
  const BatchItem w = items[it];
  const int slot = __builtin_amdgcn_readfirstlane(w.slot), t = __builtin_amdgcn_readfirstlane(w.tile);
  const DevLayer L = descs[slot].L;
  const int tiles_x = descs[slot].tiles_x;
  stage(tab);
  int step = 0;
  if (MX) {
    step = L.ctl[L.ctl_in] + 1;
    if (L.advance && t == 0 && threadIdx.x == 0) L.ctl[1 - L.ctl_in] = step;
  }
  const int k = t % tiles_x, east = min(max((L.nx - kSpan - 3) / kNlWidth, 1), tiles_x);
  Strip S;
  S.c0 = k * kNlWidth + 1;
  S.j0 = (t / tiles_x) * 4 * SEG + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * SEG + 1;
  S.j1 = min(S.j0 + SEG - 1, L.ny);
  if (S.j0 > S.j1) return;
  const bool rows = S.j0 > kNlEnd && S.j1 <= L.ny - kNlEnd, cols = k > 0 && k < east;
  if (rows && cols) march_nl<SPH, false, false, MX, false>(L, S, step, tab);
  else if (rows) march_nl<SPH, true, false, MX, false>(L, S, step, tab);
  else march_nl<SPH, true, true, MX, false>(L, S, step, tab);
}

}  // namespace

// Rows of strips per SIMD decide: below about 16 a wave has its SIMD to
// itself and the launch lasts as long as one wave's chain of rows (some 1.1
// us each, four of them halo), which the LDS tiles, eight waves per SIMD,
// beat.  Measured, us per step (64x8 tiles, then segments of 8 / 14 / 20 /
// 32 rows):
//   517x391 (3 rows per SIMD)         14.4, 18.6 / 29 / 30 / 42
//   1024x768 (13)                     21.0, 21.7 / 24 / 30 / 42
//   1201x901 Cartesian (18)           24.9, 18.3 / 22.0 / 28 / 37
//   nest 2048x1536 + 1801x1801 (54)   235, 180 / 172 / 186 / 250 per root step
//   4096x3072 (206)                   153, 123 / 118 / 116 / 116
int march_nl_seg(int nx, int ny) {
  const long long rows = (long long)((nx + kNlWidth - 1) / kNlWidth) * ny / 1024;
  return rows < 16 ? 0 : (rows < 36 ? 8 : (rows < 120 ? 14 : 20));
}

hipError_t launch_march_nl(const DevLayer &L, bool sph, int seg, hipStream_t st) {
  if (!march_nl_applies(L, sph) || seg < 1) return hipErrorInvalidValue;
#define GC_NL(A, C) \
  if (sph == A && (L.zmax != nullptr) == C) \
    return L.stream_out ? launch_nl<A, C, true>(L, seg, st) : launch_nl<A, C, false>(L, seg, st);
  GC_NL(true, true) GC_NL(true, false) GC_NL(false, true) GC_NL(false, false)
#undef GC_NL
  return hipErrorInvalidValue;
}

hipError_t launch_batch_march_nl(const BatchLaunch &B, bool sph, int seg, hipStream_t st) {
  if (B.nitems <= 0) return hipSuccess;
  const int per = (B.nitems + 7) / 8;
#define GC_BM(A, C, SEG)                                                                              \
  if (sph == A && (B.dry == 0) == C && seg == SEG) {                                                  \
    hipLaunchKernelGGL((k_batch_march_nl<A, C, SEG>), dim3(8 * per), dim3(kMarchBlock), 0, st, B.descs, \
                       B.items, B.nitems, per);                                                       \
    return hipGetLastError();                                                                         \
  }
  GC_BM(true, true, 8) GC_BM(true, false, 8) GC_BM(false, true, 8) GC_BM(false, false, 8)
  GC_BM(true, true, 14) GC_BM(true, false, 14) GC_BM(false, true, 14) GC_BM(false, false, 14)
#undef GC_BM
  return hipErrorInvalidValue;
}

}  // namespace gc
