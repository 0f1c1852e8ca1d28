// The momentum + next continuity march of a nested linear root, and the split
// of a linear layer into strips (march.hip, and the launches that run a
// root's march beside a child's step).
#pragma once

#include "march.h"

namespace gc {

namespace {

// The momentum half of root step k of a nested linear root and the continuity
// (+ OPEN) of step k + 1 (kMomentMass): row r enters with Z(k) and the level-1
// fluxes, M(k) follows at row r, N(k) at r - 1, Z(k + 1) at r - 1.  One halo
// column and row on each side.
//
// Bound by memory for large layers (32 bytes a cell) and by one wave's chain
// of rows for small ones; the tile form stages five planes in LDS, works out
// the momentum of a halo ring again and passes two barriers.
template <bool COL, bool ROW, bool MX, bool ST>
__device__ __forceinline__ void march_moment_mass(const DevLayer &L, const Strip S, int step) {
  constexpr int D = COL || ROW ? 2 : 4;
  const int nx = L.nx, ny = L.ny, lane = threadIdx.x & (kWave - 1);
  const int i = S.c0 - 1 + lane;
  const int ic = COL ? min(max(i, 1), nx) : i;
  const int vld = (ic - 1) * 4;
  const int vst = lane >= 1 && lane < kWave - 1 && (!COL || i <= nx) ? vld : kNoStore;
  const bool west_end = COL && i == 1, east_end = COL && i == nx;
  const int ra = S.j0 - 1, rb = S.j1 + 1;
  const Block B = block_of(L);
  const unsigned pitch = (unsigned)nx * 4u;
  const unsigned oz1 = plane_off(L, L.z1), om1 = plane_off(L, L.m1), on1 = plane_off(L, L.n1),
                 oz2 = plane_off(L, L.z2), om2 = plane_off(L, L.m2), on2 = plane_off(L, L.n2),
                 omax = plane_off(L, L.zmax), oarr = plane_off(L, L.arrival);
  float ph[D], pz[D], pm[D], pn[D], pq[D];
  auto load = [&](int j, int k) {
    const unsigned b = (unsigned)((ROW ? min(max(j, 1), ny) : min(j, rb)) - 1) * pitch;
    ph[k] = get(B, vld, b);
    pz[k] = get(B, vld, oz1 + b);
    pm[k] = get(B, vld, om1 + b);
    pn[k] = get(B, vld, on1 + b);
    if (MX) pq[k] = get(B, vld, omax + b);
  };
#pragma unroll
  for (int k = 0; k < D; ++k) load(ra + k, k);
  // index 0: row r, 1: row r - 1, 2: row r - 2; m, n: level 1, M, N: new
  float h[3] = {}, z[2] = {}, m[2] = {}, n[2] = {}, M[2] = {}, N[2] = {}, NR[2] = {};
  unsigned long long wet[2] = {};
  Row4 C[2], E[2];
  Row4 cnext = row_coef(L, ra, 0), enext = row_coef(L, ra, 3);
  C[0] = cnext, E[0] = enext;

  auto row = [&](int r, int k) __attribute__((always_inline)) {
    const int q = r - 1;
    h[2] = h[1], h[1] = h[0], z[1] = z[0], m[1] = m[0], n[1] = n[0];
    M[1] = M[0], N[1] = N[0], NR[1] = NR[0], wet[1] = wet[0], C[1] = C[0], E[1] = E[0];
    C[0] = cnext;
    E[0] = enext;
    h[0] = ph[k], z[0] = pz[k], m[0] = pm[k], n[0] = pn[k];
    const float zl = MX ? pq[k] : 0.0f;
    cnext = row_coef(L, r + 1, 0);
    enext = row_coef(L, r + 1, 3);
    load(r + D, k);
    wet[0] = __builtin_amdgcn_ballot_w64(h[0] > kGx);
    const unsigned g = (unsigned)(r - 1) * pitch, gq = g - pitch;
    const int vr = r >= S.j0 && r <= S.j1 ? vst : kNoStore;
    const int vq = q >= S.j0 && q <= S.j1 ? vst : kNoStore;
    if (MX) {  // wet maximum and first arrival of step k
      const unsigned long long w = __builtin_amdgcn_ballot_w64(h[0] + z[0] > kGx);
      put<false>(B, lanes(w & __builtin_amdgcn_ballot_w64(z[0] > zl)) ? vr : kNoStore, omax + g, z[0]);
      const unsigned long long first = w & __builtin_amdgcn_ballot_w64(z[0] >= L.arr_thr) &
                                       ~__builtin_amdgcn_ballot_w64(zl >= L.arr_thr);
      put<false>(B, lanes(first) ? vr : kNoStore, oarr + g, __int_as_float(step));
    }
    // M at row r
    const float ns = ROW && r == 1 ? n[0] : n[1];
    const float tn = n[0] + east(n[0]) + ns + east(ns);
    const float r2 = E[0][0] * (0.5f * (h[0] + east(h[0])));
    float mn = m[0] - r2 * (east(z[0]) - z[0]) + C[0][3] * tn;
    mn = lanes(wet[0] & (wet[0] >> 1) & ~__builtin_amdgcn_ballot_w64(fabsf(mn) < kEps)) ? mn : 0.0f;
    if (COL) mn = east_end ? 0.0f : mn;
    M[0] = mn;
    put<ST>(B, vr, om2 + g, mn);
    // N at row q
    const float sum = m[1] + m[0];
    float sw = west(sum);
    if (COL) sw = west_end ? sum : sw;
    const float tm = sw + m[1] + m[0];
    const float r4 = E[1][1] * (0.5f * (h[1] + h[0]));
    float nn = n[1] - r4 * (z[0] - z[1]) - E[1][2] * tm;
    nn = lanes(wet[1] & wet[0] & ~__builtin_amdgcn_ballot_w64(fabsf(nn) < kEps)) ? nn : 0.0f;
    if (ROW && q == ny) nn = 0.0f;
    N[0] = nn;
    put<ST>(B, vq, on2 + gq, nn);
    // continuity of step k + 1 at row q
    NR[0] = nn * C[1][2];
    const float mw = west(M[1]);
    float zz = z[1] - C[1][0] * (M[1] - mw) - C[1][1] * (NR[0] - NR[1]);
    if (fabsf(zz) < kEps) zz = 0.0f;
    float zn = zz + h[1] <= kEps ? -h[1] : zz;
    zn = lanes(wet[1]) ? zn : 0.0f;
    if (ROW && (q == 1 || q == ny)) {
      const float b = q == 1 ? N[0] : N[1];
      const float u = west_end ? M[1] : mw;
      const bool corner = west_end | east_end;
      const float a = corner ? u : 0.5f * (M[1] + mw);
      bool neg = q == 1 ? b > 0.0f : b < 0.0f;
      neg |= corner & (west_end ? u > 0.0f : u < 0.0f);
      zn = radiate(h[1], sqrtf(kGrav * h[1]), a, b, neg);
    } else if (COL) {
      const float u = west_end ? M[1] : mw;
      const float a = (west_end & !(h[2] > kGx)) ? N[0] : 0.5f * (N[0] + N[1]);
      const bool neg = west_end ? u > 0.0f : u < 0.0f;
      const float zr = radiate(h[1], sqrtf(kGrav * h[1]), a, u, neg);
      zn = (west_end | east_end) ? zr : zn;
    }
    put<ST>(B, vq, oz2 + gq, zn);
    __builtin_amdgcn_sched_barrier(0);
  };
  __builtin_amdgcn_s_waitcnt(0x0f70);  // as in march_linear
  for (int r = ra; r <= rb; r += D)
#pragma unroll
    for (int u = 0; u < D; ++u) row(r + u, u);
}

// How the waves of a launch split a layer: strips of W columns in segments
// of seg rows.  Strip 0 and the strips from east on reach the grid's side
// columns; their waves cost more per row, so they take shorter segments
// (seg_side) and come first in the grid.
struct MarchGrid {
  int nstrip, east, seg, nseg, seg_side, nseg_side, side_blocks, per_xcd;
};

// The split for strips of W = 64 - 2 HW columns in blocks of WB waves; its
// number of blocks.
template <int HW, int WB = kMarchBlock / kWave>
inline long long march_grid(const DevLayer &L, int seg, int seg_side, MarchGrid &G) {
  constexpr int W = kWave - 2 * HW;
  G.nstrip = (L.nx + W - 1) / W;
  // first strip whose last lane lies beyond column NX - 1
  G.east = L.nx - 1 >= W + kWave - HW ? (L.nx - 1 - kWave + HW) / W + 1 : 1;
  G.east = std::min(G.east, G.nstrip);
  G.seg = seg;
  G.nseg = (L.ny + seg - 1) / seg;
  G.seg_side = seg_side;
  G.nseg_side = (L.ny + seg_side - 1) / seg_side;
  const long long side = (long long)(1 + G.nstrip - G.east) * G.nseg_side;
  const long long mid = (long long)(G.east - 1) * G.nseg;
  G.side_blocks = (int)((side + WB - 1) / WB);
  G.per_xcd = (int)((mid + 8 * WB - 1) / (8 * WB));
  return (long long)G.side_blocks + 8LL * G.per_xcd;
}

// The strip of this wave in block b: side blocks first, then blocks in XCD
// order (block b runs on XCD b % 8; each XCD takes one contiguous run of
// waves, so strips that share halo columns meet in one L2).  False: none.
template <int HW, int WB = kMarchBlock / kWave>
__device__ __forceinline__ bool march_strip(const MarchGrid &G, int ny, int b, Strip &S) {
  constexpr int W = kWave - 2 * HW;
  const int wb = threadIdx.x >> 6;
  if (b < G.side_blocks) {
    const int w = __builtin_amdgcn_readfirstlane(b * WB + wb);
    const int nside = 1 + G.nstrip - G.east;
    if (w >= nside * G.nseg_side) return false;
    const int k = w % nside;
    S.c0 = (k == 0 ? 0 : G.east + k - 1) * W + 1;
    S.j0 = (w / nside) * G.seg_side + 1;
    S.j1 = min(S.j0 + G.seg_side - 1, ny);
    return true;
  }
  const int c = b - G.side_blocks, mid = G.east - 1;
  const int w = __builtin_amdgcn_readfirstlane(((c & 7) * G.per_xcd + (c >> 3)) * WB + wb);
  if ((c >> 3) >= G.per_xcd || w >= mid * G.nseg) return false;  // also past the last block
  S.c0 = (1 + w % mid) * W + 1;
  S.j0 = (w / mid) * G.seg + 1;
  S.j1 = min(S.j0 + G.seg - 1, ny);
  return true;
}

// Block b of momentum + next continuity.
template <bool MX, bool ST, int WB = kMarchBlock / kWave>
__device__ __forceinline__ void march_mm_block(const DevLayer &L, const MarchGrid &G, int b) {
  int step = 0;
  if (MX) {
    step = L.ctl[L.ctl_in] + 1;
    if (L.advance && b == 0 && threadIdx.x == 0) L.ctl[1 - L.ctl_in] = step;
  }
  Strip S;
  if (!march_strip<1, WB>(G, L.ny, b, S)) return;
  if (b < G.side_blocks) march_moment_mass<true, true, MX, ST>(L, S, step);
  else if (S.j0 - 1 >= 2 && S.j1 + 1 <= L.ny - 1) march_moment_mass<false, false, MX, ST>(L, S, step);
  else march_moment_mass<false, true, MX, ST>(L, S, step);
}

// Momentum + next continuity: rows are few and cheap, so short segments.
// Measured, us per root step of a nest with a small child (tiles; segments of
// 2 rows, 4, 8, 12, 16, the side strips' of 2 below 1024x768 and 4 above):
//   256x192 (1 row per SIMD)   17.2, 17.9, 18.9, 20.1, 21.3
//   512x384 (3)                17.3, 18.0, 18.9, 20.1, 21.5
//   1024x768 (12)              24.1, 23.4, 23.7, 23.7, 24.6
//   2048x1536 (51)             36.3, 34.9, 31.8, 30.5, 30.6
template <int WB = kMarchBlock / kWave>
inline long long mm_grid(const DevLayer &L, MarchGrid &G) {
  const long long rows = (long long)((L.nx + 61) / 62) * L.ny / 1024;
  return march_grid<1, WB>(L, rows < 8 ? 2 : (rows < 32 ? 4 : 12), rows < 32 ? 2 : 4, G);
}

// A launch that runs a root's momentum + next continuity beside a step of its
// child deals its blocks out to the two in turn, eight at a time (one to each
// XCD), so that both are in flight from the start; the rest of the longer one
// follows.
struct Beside {
  int mine, root;  // blocks of the step, of the root's march: multiples of 8
  unsigned total() const { return (unsigned)(mine + root); }
};
inline Beside beside_split(long long mine, long long root) {
  return {(int)((mine + 7) / 8 * 8), (int)((root + 7) / 8 * 8)};
}
// The block number within the step, or -1 - that within the root's march.
__device__ __forceinline__ int beside_block(const Beside &B, int b) {
  const int g = b >> 3, both = min(B.mine, B.root) >> 3;
  if (g < 2 * both) return g & 1 ? -1 - ((g >> 1) * 8 + (b & 7)) : (g >> 1) * 8 + (b & 7);
  const int rest = b - 8 * both;
  return B.mine > B.root ? rest : -1 - rest;
}

}  // namespace

}  // namespace gc
