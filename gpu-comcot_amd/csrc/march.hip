// Register-marching kernels: several root steps of a linear outermost layer
// in one pass over its planes.
//
// A wavefront owns a strip of 64 columns and marches along J.  Lane l holds
// column c0 - K + l; each iteration loads one row of Z, M, N, H and moves K
// time steps one row further, step s working s rows behind step 1, so every
// intermediate row lives in registers and neighbouring columns are read
// from the neighbouring lane (DPP wave shifts, free as VALU operands).
// There is no LDS and no barrier.  A step makes one column on each side
// invalid, so a strip writes 64 - 2K columns, and a segment of SEG rows
// takes SEG + 2K iterations; the first 2K, unrolled, only run the steps that
// the strip's rows need of them (an eighth of all for SEG = 24, K = 4).
//
// Against the LDS tiles (k_step2) a cell costs about a third of the
// instructions (no staging, no index arithmetic per cell, no halo ring of
// a tile recomputed) and K steps share one read and one write of the
// planes.
//
// Values are those of the single-step kernels bit for bit: the same
// operations on the same operands in the same order (MASS_S
// mass.f90:61-100, OPEN boundaries.f90:22-202, MOMT_S moment.f90:65-149,
// the wet maximum and first arrival step by step).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "comcot_consts.h"
#include "kernels.h"
#include "march_mm.h"

namespace gc {

namespace {

// K linear root steps of strip S.  COL: the strip holds column I = 1 or NX
// or its halo leaves the grid there; ROW: the same for rows.  Loads are
// then clamped to the grid and OPEN and the index limits of the Fortran
// loops apply; otherwise all of that compiles away.  Each row is
// loaded D rows ahead of its use.  MX: the wet maximum and first
// arrival are kept.
template <int K, bool COL, bool ROW, bool MX, bool ST>
__device__ __forceinline__ void march_linear(const DevLayer &L, const Strip S, int step) {
  // Rows in flight.  The row loop is unrolled by D, so a row's registers stay
  // put until its turn: rotating them would wait for loads just issued.
  constexpr int D = COL || ROW ? 2 : 4;
  const int nx = L.nx, ny = L.ny, lane = threadIdx.x & (kWave - 1);
  const int i = S.c0 - K + lane;
  const int ic = COL ? min(max(i, 1), nx) : i;
  const int vld = (ic - 1) * 4;
  const bool own = lane >= K && lane < kWave - K && (!COL || i <= nx);
  const bool west_end = COL && i == 1, east_end = COL && i == nx;
  const int vst = own ? vld : kNoStore;
  const int ra = S.j0 - K, rb = S.j1 + K;
  const Block B = block_of(L);
  const unsigned pitch = (unsigned)nx * 4u;
  const unsigned oz1 = plane_off(L, L.z1), om1 = plane_off(L, L.m1), on1 = plane_off(L, L.n1),
                 oz2 = plane_off(L, L.z2), om2 = plane_off(L, L.m2), on2 = plane_off(L, L.n2),
                 omax = plane_off(L, L.zmax), oarr = plane_off(L, L.arrival);
  auto base = [&](int j) {
    const int jc = ROW ? min(max(j, 1), ny) : j;
    return (unsigned)(jc - 1) * pitch;
  };

  // levels s = 0..K: Z, M at that level's newest row, M, N and N*R6 one row
  // below (level 0's newest row is the row just loaded)
  float Z[K + 1], M[K + 1], Mb[K], Nb[K], NRb[K];
  // per row r, r-1, ...: depth, momentum factors, wet masks, maximum, arrival
  float H[K + 1], R2[K], R4[K + 1], CC[K], zm[K];
  // (zl: the maximum as loaded; below: how many of the steps so far left it
  // under the arrival threshold, so the first arrival is step + below)
  float zl[K];
  int below[K];
  unsigned long long wet[K + 1];  // lane masks of H > GX
  // row coefficients: R1 R11 R6 R3, and F2 F4 R5
  Row4 C[K + 1], E[K + 1];
#pragma unroll
  for (int s = 0; s <= K; ++s) Z[s] = M[s] = H[s] = R4[s] = 0.0f, wet[s] = 0;
#pragma unroll
  for (int s = 0; s < K; ++s) {
    Mb[s] = Nb[s] = NRb[s] = R2[s] = CC[s] = zm[s] = 0.0f;
    zl[s] = 0.0f;
    below[s] = 0;
  }
#pragma unroll
  for (int s = 0; s <= K; ++s) C[s] = row_coef(L, ra, 0), E[s] = row_coef(L, ra, 3);

  float ph[D], pz[D], pm[D], pn[D], pq[D];
  auto load = [&](int j, int k) {
    const unsigned b = base(ROW ? j : min(j, rb));
    ph[k] = get(B, vld, b);
    pz[k] = get(B, vld, oz1 + b);
    pm[k] = get(B, vld, om1 + b);
    pn[k] = get(B, vld, on1 + b);
    if (MX) pq[k] = get(B, vld, omax + b);
  };
#pragma unroll
  for (int k = 0; k < D; ++k) load(ra + k, k);
  Row4 cnext = row_coef(L, ra, 0), enext = row_coef(L, ra, 3);

  // k: the row's load slot; active: the steps that run (the rows that the
  // strip's first rows need of step s + 1 begin 1 + 2 s rows after row ra)
  auto row = [&](int r, int k, int active) __attribute__((always_inline)) {
    // ---- row r enters: shift the per-row values down
#pragma unroll
    for (int s = K; s > 0; --s) {
      H[s] = H[s - 1];
      C[s] = C[s - 1];
      E[s] = E[s - 1];
      R4[s] = R4[s - 1];
      wet[s] = wet[s - 1];
    }
#pragma unroll
    for (int s = K - 1; s > 0; --s) {
      R2[s] = R2[s - 1];
      if (COL) CC[s] = CC[s - 1];
      if (MX) {
        zm[s] = zm[s - 1];
        zl[s] = zl[s - 1];
        below[s] = below[s - 1];
      }
    }
    C[0] = cnext;
    E[0] = enext;
    const float h = ph[k];
    float zc = pz[k], mc = pm[k], nc = pn[k];
    if (MX) {
      zm[0] = zl[0] = pq[k];
      below[0] = 0;
    }
    cnext = row_coef(L, r + 1, 0);
    enext = row_coef(L, r + 1, 3);
    load(r + D, k);
    const float he = east(h);
    H[0] = h;
    wet[0] = __builtin_amdgcn_ballot_w64(h > kGx);
    R2[0] = E[0][0] * (0.5f * (h + he));   // used where both cells are wet: HP > 0
    R4[1] = E[1][1] * (0.5f * (H[1] + h));
    if (COL) CC[0] = sqrtf(kGrav * h);

#pragma unroll
    for (int s = 0; s < K; ++s) {  // step s + 1 at row q
      const int q = r - s;
      if (s >= active) {
        if (s == active) Mb[s] = mc, Nb[s] = nc, NRb[s] = nc * C[s][2];
        continue;
      }
      const float hq = H[s];
      // continuity
      const float nr = nc * C[s][2];
      const float mw = west(mc);
      float zz = zc - C[s][0] * (mc - mw) - C[s][1] * (nr - NRb[s]);
      if (fabsf(zz) < kEps) zz = 0.0f;
      const float t = zz + hq;
      float zn = t <= kEps ? -hq : zz;
      zn = lanes(wet[s]) ? zn : 0.0f;
      bool w = lanes(wet[s] & __builtin_amdgcn_ballot_w64(t > kGx));
      if (ROW && (q == 1 || q == ny)) {
        // bottom and top rows; the corners take their own fluxes
        const float b = q == 1 ? nc : Nb[s];
        const float u = west_end ? mc : mw;
        const bool corner = west_end | east_end;
        const float a = corner ? u : 0.5f * (mc + mw);
        bool neg = q == 1 ? b > 0.0f : b < 0.0f;
        neg |= corner & (west_end ? u > 0.0f : u < 0.0f);
        zn = radiate(hq, sqrtf(kGrav * hq), a, b, neg);
        w = hq + zn > kGx;
      } else if (COL) {
        // left and right columns
        const float u = west_end ? mc : mw;
        const float a = (west_end & !(H[s + 1] > kGx)) ? nc : 0.5f * (nc + Nb[s]);
        const bool neg = west_end ? u > 0.0f : u < 0.0f;
        const bool ring = west_end | east_end;
        const float zr = radiate(hq, CC[s], a, u, neg);
        zn = ring ? zr : zn;
        w = ring ? hq + zr > kGx : w;
      }
      // momentum: M at row q, N at row q - 1
      const float ns = ROW && q == 1 ? nc : Nb[s];
      const float tn = nc + east(nc) + ns + east(ns);
      float mn = mc - R2[s] * (east(zn) - zn) + C[s][3] * tn;
      // M(I) needs I and I + 1 wet; |M| < EPS goes to 0
      mn = lanes(wet[s] & (wet[s] >> 1) & ~__builtin_amdgcn_ballot_w64(fabsf(mn) < kEps)) ? mn : 0.0f;
      if (COL) mn = east_end ? 0.0f : mn;
      const float sum = Mb[s] + mc;
      float sw = west(sum);
      if (COL) sw = west_end ? sum : sw;
      const float tm = sw + Mb[s] + mc;
      float nn = Nb[s] - R4[s + 1] * (zn - Z[s + 1]) - E[s + 1][2] * tm;
      nn = lanes(wet[s + 1] & wet[s] & ~__builtin_amdgcn_ballot_w64(fabsf(nn) < kEps)) ? nn : 0.0f;
      if (ROW && q - 1 == ny) nn = 0.0f;
      if (MX) {  // wet maximum and first arrival of step s + 1 at row q
        zm[s] = (w & (zn > zm[s])) ? zn : zm[s];
        below[s] += zm[s] >= L.arr_thr ? 0 : 1;
      }
      // the level below is done with its rows
      Mb[s] = mc;
      Nb[s] = nc;
      NRb[s] = nr;
      // hand over: the next step works one row behind, on the values this
      // level held before this iteration
      const float zo = Z[s + 1], mo = M[s + 1];
      Z[s + 1] = zn;
      M[s + 1] = mn;
      if (s + 1 < K) {
        zc = zo;
        mc = mo;
        nc = nn;
      } else {
        const unsigned g = (unsigned)(q - 1) * pitch;
        const int vq = q >= S.j0 && q <= S.j1 ? vst : kNoStore;
        const int vn = q - 1 >= S.j0 && q - 1 <= S.j1 ? vst : kNoStore;
        put<ST>(B, vq, oz2 + g, zn);
        put<ST>(B, vq, om2 + g, mn);
        put<ST>(B, vn, on2 + g - pitch, nn);
        if (MX) {
          put<false>(B, zm[s] != zl[s] ? vq : kNoStore, omax + g, zm[s]);
          const bool hit = !(zl[s] >= L.arr_thr) & (below[s] < K);
          put<false>(B, hit ? vq : kNoStore, oarr + g, __int_as_float(step + below[s]));
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Rows beyond rb (the unrolled loop's remainder) load row rb again and
  // store nothing.  The first loads are waited for here (vmcnt 0): otherwise
  // the wait at the loop's head has to serve the entry, where they are the
  // newest operations, and would stop for everything in flight on each turn.
  __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll
  for (int u = 0; u < 2 * K; ++u) row(ra + u, u % D, (u + 1) / 2);
  static_assert(2 * K % D == 0, "the row loop starts at load slot 0");
  for (int r = ra + 2 * K; r <= rb; r += D)
#pragma unroll
    for (int u = 0; u < D; ++u) row(r + u, u, K);
}

// K = 0: march_moment_mass, otherwise K steps of march_linear.
template <int K, bool MX, bool ST>
__global__ void __launch_bounds__(kMarchBlock) k_march_linear(DevLayer L, MarchGrid G) {
  if constexpr (K == 0) {
    march_mm_block<MX, ST>(L, G, blockIdx.x);
  } else {
    int step = 0;
    if (MX) {
      step = L.ctl[L.ctl_in] + 1;
      if (L.advance && blockIdx.x == 0 && threadIdx.x == 0) L.ctl[1 - L.ctl_in] = step + K - 1;
    }
    Strip S;
    if (!march_strip<K>(G, L.ny, blockIdx.x, S)) return;
    if ((int)blockIdx.x < G.side_blocks) march_linear<K, true, true, MX, ST>(L, S, step);
    else if (S.j0 - K >= 2 && S.j1 + K <= L.ny - 1) march_linear<K, false, false, MX, ST>(L, S, step);
    else march_linear<K, false, true, MX, ST>(L, S, step);
  }
}

template <int K, bool MX, bool ST>
hipError_t launch_grid(const DevLayer &L, const MarchGrid &G, long long blocks, hipStream_t st) {
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_march_linear<K, MX, ST>), dim3((unsigned)blocks), dim3(kMarchBlock), 0, st,
                     L, G);
  return hipGetLastError();
}

template <int K>
hipError_t launch_grid(const DevLayer &L, const MarchGrid &G, long long blocks, hipStream_t st) {
  if (L.zmax)
    return L.stream_out ? launch_grid<K, true, true>(L, G, blocks, st)
                        : launch_grid<K, true, false>(L, G, blocks, st);
  return L.stream_out ? launch_grid<K, false, true>(L, G, blocks, st)
                      : launch_grid<K, false, false>(L, G, blocks, st);
}

// The batch form of two root steps: one workgroup per (layer, tile) item of a
// 60 x 32 tiling, a wave per 8 rows.
template <bool MX>
__global__ void __launch_bounds__(kMarchBlock)
    k_batch_march2(const BatchDesc *__restrict__ descs, const BatchItem *__restrict__ items, int nitems,
                   int per_xcd) {
  constexpr int K = 2, W = kWave - 2 * K, SEG = 8;
  const int it = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (it >= nitems) return;
  const BatchItem w = items[it];
  const int slot = __builtin_amdgcn_readfirstlane(w.slot), t = __builtin_amdgcn_readfirstlane(w.tile);
  const DevLayer L = descs[slot].L;
  const int tiles_x = descs[slot].tiles_x;
  int step = 0;
  if (MX) {
    step = L.ctl[L.ctl_in] + 1;
    if (L.advance && t == 0 && threadIdx.x == 0) L.ctl[1 - L.ctl_in] = step + K - 1;
  }
  Strip S;
  S.c0 = (t % tiles_x) * W + 1;
  S.j0 = (t / tiles_x) * 4 * SEG + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * SEG + 1;
  S.j1 = min(S.j0 + SEG - 1, L.ny);
  if (S.j0 > S.j1) return;
  const bool rows = S.j0 - K >= 2 && S.j1 + K <= L.ny - 1;
  const bool cols = S.c0 - K >= 2 && S.c0 - K + kWave - 1 <= L.nx - 1;
  if (cols && rows) march_linear<K, false, false, MX, false>(L, S, step);
  else if (cols) march_linear<K, false, true, MX, false>(L, S, step);
  else march_linear<K, true, true, MX, false>(L, S, step);
}

}  // namespace

// Rows of strips per SIMD decide the split.  With few of them a wave has
// its SIMD to itself, an instruction then takes about 8 cycles instead of 4,
// and a launch lasts as long as one wave's rows: short segments.  Measured,
// us per root step with four steps a launch (two-step tiles before):
//   96x72 (0 rows per SIMD)  side segments of 2 rows 3.04, of 4 3.86 (6.9)
//   517x391 (3)              4 rows, sides 2 3.33; 8, 2 3.96; 8, 4 4.00 (6.9)
//   1024x768 (14)            8, 4 4.48; 4, 2 4.49; 12, 4 5.7 (11.0; best tile 8.5)
//   1500x1200 (31)           12, 4 6.95; 8, 2 7.34; 4, 2 7.74
//   2051x1537 (55)           12, 4 9.84; 20, 8 9.73; 8, 4 10.1; 16, 8 10.5 (28.8)
//   4096x3072 (222)          20, 8 27.5; 16, 8 28.6; 24, 8 28.2; 32, 8 29.7 (99.6)
// Two steps a launch: 3.83, 4.05, 4.90, -, 11.6, 48.  Side strips run OPEN on
// every row (about 1.6 times the time per row).
struct MarchPlan {
  int seg, seg_side;
};
static MarchPlan march_plan(const DevLayer &L) {
  const long long rows = (long long)((L.nx + 55) / 56) * L.ny / 1024;
  if (rows < 10) return {4, 2};
  if (rows < 24) return {8, 4};
  return rows < 120 ? MarchPlan{12, 4} : MarchPlan{20, 8};
}

hipError_t launch_march_linear(const DevLayer &L, int steps, hipStream_t st) {
  if (!march_applies(L)) return hipErrorInvalidValue;
  const MarchPlan p = march_plan(L);
  MarchGrid G;
  if (steps == 2) {
    const long long blocks = march_grid<2>(L, p.seg, p.seg_side, G);
    return launch_grid<2>(L, G, blocks, st);
  }
  if (steps != kMarchSteps) return hipErrorInvalidValue;
  const long long blocks = march_grid<kMarchSteps>(L, p.seg, p.seg_side, G);
  return launch_grid<kMarchSteps>(L, G, blocks, st);
}

hipError_t launch_march_moment_mass(const DevLayer &L, hipStream_t st) {
  if (!march_applies(L)) return hipErrorInvalidValue;
  MarchGrid G;
  const long long blocks = mm_grid<>(L, G);
  return launch_grid<0>(L, G, blocks, st);
}

hipError_t launch_batch_march2(const BatchLaunch &B, hipStream_t st) {
  if (B.nitems <= 0) return hipSuccess;
  const int per = (B.nitems + 7) / 8;
  if (B.dry)
    hipLaunchKernelGGL(k_batch_march2<false>, dim3(8 * per), dim3(kMarchBlock), 0, st, B.descs, B.items,
                       B.nitems, per);
  else
    hipLaunchKernelGGL(k_batch_march2<true>, dim3(8 * per), dim3(kMarchBlock), 0, st, B.descs, B.items,
                       B.nitems, per);
  return hipGetLastError();
}

}  // namespace gc
