// ptq2_rows.h -- the A11 element pass on nine waves per brick, one per quadrature row, for meshes of
// so few bricks that one brick's latency is what a launch takes (multigrid levels).
//
// Wave w loads and stores the node plane z = w of the brick's tile and runs the quadrature row
// (qb, qc) = (w % 3, w / 3) of all 64 elements (lane = element): contraction of the tile along z and y for
// the row, the three points, and the transposed contraction along x, whose 24 values per element (8 per
// component: the x derivative has no m term) go to LDS.  Then wave w takes component w % 3 and node layer
// w / 3 of every element and finishes the transpose along y and z.  The layers 0 and 1 of a brick's
// elements are different nodes and are added to the output tile at once, the layers 2 after a barrier:
// every node's sum has one order.
//
// The row's coefficients are wave-uniform values, not code: nine waves share one row of code, where nine
// unrolled rows would each be fetched cold.  x runs in the modal form of ptq2_comp.h (derivatives times 2, on
// y and z too; the point weights take it out).
//
// What bounds it: a launch's latency; 8 bricks took 8.2 us and 48 bricks 8.0, of which some 5 us are the 1.2k VALU
// instructions of the three waves that share the first SIMD (12.5 and 10.6 us with three waves per brick).  The FP64
// sums over the slabs added 0.4 us (216 bricks 9.2 -> 9.5 us, overlapping blocks of 16x16x12 elements 10.5 -> 10.9).
#pragma once
#include "ptq2_comp.h"

namespace ptq2 {

constexpr int NUM_CUS = 256;  // of an MI355X
constexpr int RWAVES = 9;
static_assert(RWAVES == TN, "one wave per plane of the tile, and per quadrature row");
constexpr int ROWVALS = 24;  // values per element that a row hands over

template <typename T>
struct RowCoef {
  T b[3], d[3];  // nodal values and twice the derivatives
};
constexpr double RX = 0.77459666924148337704;
template <typename T>
__constant__ const RowCoef<T> c_row[3] = {
    {{T(0.5 * (0.6 + RX)), T(0.4), T(0.5 * (0.6 - RX))}, {T(-2.0 * RX - 1.0), T(4.0 * RX), T(-2.0 * RX + 1.0)}},
    {{T(0.0), T(1.0), T(0.0)}, {T(-1.0), T(0.0), T(1.0)}},
    {{T(0.5 * (0.6 - RX)), T(0.4), T(0.5 * (0.6 + RX))}, {T(2.0 * RX - 1.0), T(-4.0 * RX), T(2.0 * RX + 1.0)}}};

// gradients (times 2) of one field at the row's points: g[d][qa]
template <typename T>
__device__ __forceinline__ void row_points(const T *s, int base, int c, const RowCoef<T> &cb, const RowCoef<T> &cc,
                                           T g[3][3]) {
  constexpr T V1 = T(MOD_V1), V2 = T(MOD_V2), D2 = T(MOD_D2);
  T r[3][3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    T tb[3], td[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const T v0 = tv(s, base, c, i, j, 0), v1 = tv(s, base, c, i, j, 1), v2 = tv(s, base, c, i, j, 2);
      tb[j] = fma(cc.b[2], v2, fma(cc.b[1], v1, cc.b[0] * v0));
      td[j] = fma(cc.d[2], v2, fma(cc.d[1], v1, cc.d[0] * v0));
    }
    r[0][i] = fma(cb.b[2], tb[2], fma(cb.b[1], tb[1], cb.b[0] * tb[0]));
    r[1][i] = fma(cb.d[2], tb[2], fma(cb.d[1], tb[1], cb.d[0] * tb[0]));
    r[2][i] = fma(cb.b[2], td[2], fma(cb.b[1], td[1], cb.b[0] * td[0]));
    if (i == 1) row_fence();
  }
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const T m = r[d][1], b = r[d][2] - r[d][0], a = fma(T(-2), r[d][1], r[d][0] + r[d][2]);
    if (d == 0) {
      g[d][0] = fma(-D2, a, b);
      g[d][1] = b;
      g[d][2] = fma(D2, a, b);
    } else {
      const T p = fma(V2, a, m);
      g[d][0] = fma(-V1, b, p);
      g[d][1] = m;
      g[d][2] = fma(V1, b, p);
    }
  }
}
// the row's stresses dv[d][qa] of component c, transposed along x, into the exchange rows of that component
template <typename T>
__device__ __forceinline__ void row_hand_over(const T dv[3][3], T *ex, int lane) {
  constexpr T V1 = T(MOD_V1), V2 = T(MOD_V2), D2 = T(MOD_D2);
  ex[lane] = dv[0][0] + dv[0][2] + dv[0][1];
  ex[BEL + lane] = D2 * (dv[0][2] - dv[0][0]);
#pragma unroll
  for (int d = 1; d < 3; d++) {
    const T s = dv[d][0] + dv[d][2], f = dv[d][2] - dv[d][0];
    ex[(3 * d - 1) * BEL + lane] = s + dv[d][1];
    ex[(3 * d) * BEL + lane] = V1 * f;
    ex[(3 * d + 1) * BEL + lane] = V2 * s;
  }
}
// component c, node layer k of the element from the nine rows' values: Y[i + 3 j].  bk, dk: the layer's value
// and twice its derivative at the slabs' z.  A slab's rows are summed in T and the slabs in FP64, as
// the three-wave kernel's output tile adds them: with everything in FP32 an element's error is 1.16e-7 on random
// fields (three waves 1.04e-7), with FP64 over the slabs 0.93e-7.
template <typename T>
__device__ __forceinline__ void gather_rows(const T *ex, int lane, int c, const double bk[3], const double dk[3],
                                            double Y[9]) {
#pragma unroll
  for (int n = 0; n < 9; n++) Y[n] = 0.0;
#pragma unroll
  for (int qc = 0; qc < 3; qc++) {
    T RB[9], RD[9];
#pragma unroll
    for (int n = 0; n < 9; n++) RB[n] = RD[n] = T(0);
#pragma unroll
    for (int qb = 0; qb < 3; qb++) {
      const T *e = ex + ((qb + 3 * qc) * ROWVALS + 8 * c) * BEL + lane;
      T t[8];
#pragma unroll
      for (int n = 0; n < 8; n++) t[n] = e[n * BEL];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        if (nzB(qb, j)) {
          RB[3 * j + 1] = fma(T(gB(qb, j)), t[0], RB[3 * j + 1]);
          RB[3 * j + 2] = fma(T(gB(qb, j)), t[1], RB[3 * j + 2]);
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
          if (gD(qb, j) != 0.0) RB[3 * j + i] = fma(T(2.0 * gD(qb, j)), t[2 + i], RB[3 * j + i]);
          if (nzB(qb, j)) RD[3 * j + i] = fma(T(gB(qb, j)), t[5 + i], RD[3 * j + i]);
        }
      }
    }
#pragma unroll
    for (int n = 0; n < 9; n++) Y[n] = fma(bk[qc], (double)RB[n], fma(dk[qc], (double)RD[n], Y[n]));
    row_fence();
  }
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const double m = Y[3 * j], b = Y[3 * j + 1], a = Y[3 * j + 2];
    Y[3 * j] = a - b;
    Y[3 * j + 1] = fma(-2.0, a, m);
    Y[3 * j + 2] = a + b;
  }
}

// one plane of the tile: rows y = 2 it + p of plane z, 27 values each
constexpr int PSTEPS = (TN + 1) / 2;
template <typename T>
__device__ __forceinline__ void plane_load(const Box &b, const Tile &t, const T *__restrict__ g, int z, int lane,
                                           T v[PSTEPS]) {
  const RowLane L(lane);
  const int64_t col = 3 * (t.node0 + min(L.ii, t.tnx - 1) + (int64_t)b.NX * b.NY * min(z, t.tnz - 1)) + L.c;
#pragma unroll
  for (int it = 0; it < PSTEPS; it++) v[it] = g[col + 3 * (int64_t)b.NX * min(2 * it + (L.p & 1), t.tny - 1)];
}
// the same with the Dirichlet dofs as zero (BCListInsertLocalZero, src/dmda_bcs.c:581-608)
template <typename T>
__device__ __forceinline__ void plane_load_masked(const Box &b, const Tile &t, const T *__restrict__ g,
                                                  const uint8_t *__restrict__ mask, int z, int lane, T v[PSTEPS]) {
  plane_load(b, t, g, z, lane, v);
  if (!mask) return;
  uint8_t mk[PSTEPS];
  plane_load(b, t, mask, z, lane, mk);
#pragma unroll
  for (int it = 0; it < PSTEPS; it++) v[it] = mk[it] ? T(0) : v[it];
}
// rows and columns outside the box belong to no element: any value will do there
template <typename T>
__device__ __forceinline__ void plane_put(const T v[PSTEPS], T *s, int z, int lane) {
  const RowLane L(lane);
  if (L.p > 1) return;
#pragma unroll
  for (int it = 0; it < PSTEPS; it++)
    if (2 * it + L.p < TN) s[L.lds_col + TRS * (2 * it + L.p) + TPS * z] = v[it];
}
// the owner-writes store (store_tile_own) of one plane
template <typename T>
__device__ __forceinline__ void plane_store(const Box &b, const BrickId &br, const Tile &t, const double *s,
                                            T *__restrict__ g, T *__restrict__ face, bool add_mode, int z, int lane) {
  if (tile_fast(b, t)) {
    store_rows_full<TN>(b, br, t, s, g, face, add_mode, z, lane);
    return;
  }
  const RowLane L(lane);
  if (L.p > 1 || L.ii >= t.tnx || z >= t.tnz) return;
  const bool ownx = L.ii < 2 * BE || br.bx == b.nbx - 1, lasty = br.by == b.nby - 1,
             ownz = z < 2 * BE || br.bz == b.nbz - 1;
  T *fo = face + (int64_t)br.lin * FACEVALS + L.c;
#pragma unroll
  for (int it = 0; it < PSTEPS; it++) {
    const int y = 2 * it + L.p;
    if (y >= t.tny) continue;
    const T val = T(s[L.lds_col + TRS * y + TPS * z]);
    const bool owny = y < 2 * BE || lasty;
    if (ownx && owny && ownz) {
      T *o = g + 3 * (t.node0 + L.ii + (int64_t)b.NX * (y + (int64_t)b.NY * z)) + L.c;
      *o = add_mode ? *o + val : val;
    } else {
      const int slot = !ownx ? z * TN + y : (!owny ? TN * TN + z * TN + L.ii : 2 * TN * TN + y * TN + L.ii);
      fo[3 * slot] = val;
    }
  }
}

// the row's points from the stored factors F = sqrt(w eta / det) adj(J): dv = F^T (M + M^T), M = F g;
// a quarter takes out the two factors 2
__device__ __forceinline__ void row_stress(const float F[27], const float g[3][3][3], float dv[3][3][3]) {
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const float *f = F + 9 * q;
    float M[3][3], S[3][3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int l = 0; l < 3; l++)
        M[k][l] = g[l][0][q] * f[3 * k] + g[l][1][q] * f[3 * k + 1] + g[l][2][q] * f[3 * k + 2];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      S[k][k] = 0.5f * M[k][k];
#pragma unroll
      for (int l = 0; l < k; l++) S[k][l] = S[l][k] = 0.25f * (M[k][l] + M[l][k]);
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int l = 0; l < 3; l++) dv[l][k][q] = S[0][l] * f[k] + S[1][l] * f[3 + k] + S[2][l] * f[6 + k];
    row_fence();
  }
}

// LDS of the FP32 pass: the velocity tile, later the output tile (FP64 sums) in its place, and the rows'
// values.
struct RowsLds32 {
  double Ts[3 * TCS];
  float Ex[RWAVES * ROWVALS * BEL];
};
// The pass from wave w's plane v of the velocity tile to the output tile L.Ts; fs: the lane's factors of row w.
__device__ __forceinline__ void a11_rows32(RowsLds32 &L, const float v[PSTEPS], const float *__restrict__ fs,
                                           bool active, int w, int lane) {
  float *Us = reinterpret_cast<float *>(L.Ts);
  float F[27];
#pragma unroll
  for (int n = 0; n < 27; n++) F[n] = fs[n * BEL];
  plane_put(v, Us, w, lane);
  lds_barrier();
  const int base = lane_base(lane);
  {
    const RowCoef<float> cb = c_row<float>[w % 3], cc = c_row<float>[w / 3];
    float g[3][3][3], dv[3][3][3];  // [component][d][qa]
#pragma unroll
    for (int c = 0; c < 3; c++) {
      row_points(Us, base, c, cb, cc, g[c]);
      row_fence();
    }
    row_stress(F, g, dv);
#pragma unroll
    for (int c = 0; c < 3; c++) row_hand_over(dv[c], L.Ex + (ROWVALS * w + 8 * c) * BEL, lane);
  }
  lds_barrier();  // the velocities are read, the rows' values written
  for (int n = threadIdx.x; n < 3 * TCS; n += RWAVES * BEL) L.Ts[n] = 0.0;
  const int c = w % 3, k = w / 3;
  double Y[9], bk[3], dk[3];
#pragma unroll
  for (int qc = 0; qc < 3; qc++) {
    bk[qc] = c_row<double>[qc].b[k];
    dk[qc] = c_row<double>[qc].d[k];
  }
  gather_rows(L.Ex, lane, c, bk, dk, Y);
  lds_barrier();
  double *o = L.Ts + base + c * TCS + TPS * k;
#pragma unroll
  for (int half = 0; half < 2; half++) {
    if (active && (k == 2) == (half == 1)) {
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) lds_add(o + xo(i) + TRS * j, Y[i + 3 * j]);
    }
    lds_barrier();
  }
}

__device__ __forceinline__ void a11_rows32_brick(const Box &b, const BrickId &br, const float *__restrict__ u,
                                                 const uint8_t *__restrict__ mask, const float *__restrict__ fac,
                                                 float *__restrict__ y, int add_mode, float *__restrict__ facebuf) {
  __shared__ RowsLds32 L;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / BEL), lane = (int)threadIdx.x - BEL * w;
  const Tile t = tile_of(b, br);
  float v[PSTEPS];
  plane_load_masked(b, t, u, mask, w, lane, v);
  // the factor slots of lanes without an element hold something, and nobody takes their outputs
  a11_rows32(L, v, fac + ((int64_t)br.lin * 243 + 27 * w) * BEL + lane, lane_active(t, lane), w, lane);
  plane_store(b, br, t, L.Ts, y, facebuf, add_mode != 0, w, lane);
}

// Overlapping blocks: 4x4x4 elements each, three elements apart, so that every node is complete in
// one block (of the nodes 0 .. 8 along an axis an inner block has 1 .. 7 and owns 1 .. 6).  With 64 / 27 of the work
// there are no face slots, and an apply with its Chebyshev update or its Dirichlet rows is one launch.
__host__ __device__ constexpr int own_blocks(int m) { return m <= BE ? 1 : (m - BE + 2) / 3 + 1; }
struct OwnAxis {
  int e0, lo, hi;  // first element; owned tile nodes lo .. hi
  __device__ __forceinline__ OwnAxis(int k, int m)
      : e0(3 * k), lo(k > 0 ? 1 : 0), hi(3 * k + BE < m ? 6 : 2 * (m - 3 * k)) {}
};
// y = A x with y = x on the mask's dofs (CH: the Chebyshev update of co instead); single-rank boxes
template <bool CH>
__device__ __forceinline__ void a11_rows32_own(const Box &b, int bid, const float *__restrict__ x,
                                               const uint8_t *__restrict__ mask, const float *__restrict__ fac,
                                               float *__restrict__ y, const ChebOut<float> &co) {
  __shared__ RowsLds32 L;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / BEL), lane = (int)threadIdx.x - BEL * w;
  const int nx = own_blocks(b.mx), ny = own_blocks(b.my);
  const OwnAxis ax(bid % nx, b.mx), ay(bid / nx % ny, b.my), az(bid / (nx * ny), b.mz);
  Tile t;
  t.ex0 = ax.e0; t.ey0 = ay.e0; t.ez0 = az.e0;
  t.nex = min(BE, b.mx - t.ex0); t.ney = min(BE, b.my - t.ey0); t.nez = min(BE, b.mz - t.ez0);
  t.tnx = 2 * t.nex + 1; t.tny = 2 * t.ney + 1; t.tnz = 2 * t.nez + 1;
  t.node0 = 2 * (t.ex0 + (int64_t)b.NX * (t.ey0 + (int64_t)b.NY * t.ez0));
  float v[PSTEPS], xv[PSTEPS], bv[PSTEPS], dv[PSTEPS], pv[PSTEPS] = {};
  uint8_t mk[PSTEPS] = {};
  plane_load(b, t, x, w, lane, xv);
  if (mask) plane_load(b, t, mask, w, lane, mk);
  if (CH) {  // the update's operands travel behind the tile
    plane_load(b, t, co.b, w, lane, bv);
    plane_load(b, t, co.dinv, w, lane, dv);
    if (co.pkm1) plane_load(b, t, co.pkm1, w, lane, pv);
  }
#pragma unroll
  for (int it = 0; it < PSTEPS; it++) v[it] = mk[it] ? 0.0f : xv[it];  // BCListInsertLocalZero, src/dmda_bcs.c:581-608
  const LaneElem e = lane_elem(lane);
  const int ex = min(t.ex0 + e.lx, b.mx - 1), ey = min(t.ey0 + e.ly, b.my - 1), ez = min(t.ez0 + e.lz, b.mz - 1);
  const int64_t brick = ex / BE + (int64_t)b.nbx * (ey / BE + (int64_t)b.nby * (ez / BE));
  a11_rows32(L, v, fac + (brick * 243 + 27 * w) * BEL + elem_lane(ex % BE, ey % BE, ez % BE), lane_active(t, lane), w,
             lane);
  const RowLane R(lane);
  if (R.p > 1 || R.ii < ax.lo || R.ii > ax.hi || w < az.lo || w > az.hi) return;
  const int64_t col = 3 * (t.node0 + R.ii + (int64_t)b.NX * b.NY * w) + R.c;
#pragma unroll
  for (int it = 0; it < PSTEPS; it++) {
    const int yy = 2 * it + R.p;
    if (yy < ay.lo || yy > ay.hi) continue;
    const int64_t gi = col + 3 * (int64_t)b.NX * yy;
    const float val = mk[it] ? xv[it] : (float)L.Ts[R.lds_col + TRS * yy + TPS * w];
    if (CH)
      co.out[gi] = cheb_value(co, dv[it], bv[it], val, xv[it], pv[it], co.pkm1 != nullptr);
    else
      y[gi] = val;
  }
}

}  // namespace ptq2
