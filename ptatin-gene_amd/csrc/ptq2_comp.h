// ptq2_comp.h -- the FP64 A11 (and full-block) element pass on four waves per brick.
//
// Four waves share a brick of 4x4x4 elements (lane = element, as everywhere): U wave c (0, 1, 2) owns
// component c of the velocity and of the output, the G wave the geometry.  Per quadrature row (three
// points along x) the U waves contract their components to reference gradients at the three points
// and the G wave the coordinates to adjugate and determinant; the values change hands through LDS;
// U wave q runs the stress of the row's point q for all 64 elements; and the stresses go back to the
// U waves, which run the transposed contractions of their component.  What that buys over one wave
// holding everything:
//   - an element's 27 values of one component are 27 doubles, so a whole element's contraction
//     stays in registers and no partial sum is formed twice;
//   - two workgroups (eight waves) fit a CU where the one-wave form had four waves, each SIMD
//     runs two waves, and one workgroup's loads and stores travel behind the other's arithmetic;
//   - U wave c's outputs touch only component c of the output tile, so the waves never add to the
//     same LDS word and the sum order stays the program order;
//   - a brick's latency falls with the number of waves that share it, which is what small meshes
//     see.
// Four waves because the SIMDs of a CU are filled in turn from the first for every workgroup: three
// waves per brick leave the fourth SIMD idle, six fit once instead of twice.
//
// The 1D contractions work on (m, b, a) = (u1, u2 - u0, u0 - 2 u1 + u2) instead of the nodal
// values: with x = sqrt(3/5), u(+-x) = m + 0.3 a +- (x/2) b, u(0) = m, 2 u'(+-x) = b +- 2 x a and
// 2 u'(0) = b, 5 operations for three values and three derivatives against 14 with the nodal
// tables.  A brick takes 6.4k VALU instructions, the one-wave form with nodal tables 12.9k.  All derivatives
// carry the factor 2; it is taken out in the point weights (w / 8:
// J' = 2 J, adj(J') = 4 adj(J), det J' = 8 det J, and the transposed derivative applies 2 again).
//
// What bounds it: a workgroup's chain of load, nine rows with a barrier each, output and store takes
// 21k cycles alone and 33k beside a second workgroup (a row 1.3k and 1.8k, of which ~0.6k are VALU),
// and two workgroups fit a CU (212 VGPRs, 81 KB of LDS).  128^3 elements: 1020-1110 us per apply by mesh
// (158 us of it the face pass; this pass' loads and stores alone 547 us), 1300-1330 us with the one-wave kernel;
// 8^3 (one brick's latency): 17 us against 39 us; 37x22x45: 36 us against 48 us.
#pragma once
#include "ptq2_device.h"
#include "ptq2_kernels.h"

namespace ptq2 {

constexpr double MOD_V1 = 0.5 * 0.77459666924148337704;  // value at +-x: coefficient of b
constexpr double MOD_V2 = 0.3;                           //               coefficient of a
constexpr double MOD_D2 = 2.0 * 0.77459666924148337704;  // twice the derivative: coefficient of a
constexpr int CWAVES = 4;                                // U 0, 1, 2 and G

// Workgroup barrier for LDS traffic only: global loads and stores in flight need not drain.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// values that are computed here and not later: without it the compiler sinks a row's sums into the
// branch that finally uses them and keeps their operands alive (spilled) until then
template <int N>
__device__ __forceinline__ void pin(double *v) {
#pragma unroll
  for (int n = 0; n < N; n++) asm volatile("" : "+v"(v[n]));
}

// nodal triple -> (m, b, a) in place, stride S
template <int S>
__device__ __forceinline__ void to_modal3(double *v) {
  const double u0 = v[0], u1 = v[S], u2 = v[2 * S];
  v[0] = u1;
  v[S] = u2 - u0;
  v[2 * S] = fma(-2.0, u1, u0 + u2);
}
// the transpose: dual (m, b, a) -> nodal triple in place
template <int S>
__device__ __forceinline__ void from_dual3(double *v) {
  const double m = v[0], b = v[S], a = v[2 * S];
  v[0] = a - b;
  v[S] = fma(-2.0, a, m);
  v[2 * S] = a + b;
}

// The element's 27 values of one tile component into modal form v[i + 3 j + 9 k].
__device__ __forceinline__ void load_modal(const double *s, int base, int c, double v[27]) {
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) v[i + 3 * j + 9 * k] = s[base + c * TCS + xo(i) + j * TRS + k * TPS];
}
__device__ __forceinline__ void modal_layer(double v[9]) {
#pragma unroll
  for (int j = 0; j < 3; j++) to_modal3<1>(v + 3 * j);
#pragma unroll
  for (int i = 0; i < 3; i++) to_modal3<3>(v + i);
}
// nodal -> modal, the z direction's a still missing: layer 2 keeps the nodal u0 (slab 1, which runs
// first, needs m and b alone, and its wait for the first row is shorter by the rest)
__device__ __forceinline__ void modal27(double v[27]) {
#pragma unroll
  for (int n = 0; n < 9; n++) {
    const double u0 = v[n], u1 = v[n + 9], u2 = v[n + 18];
    v[n] = u1;
    v[n + 9] = u2 - u0;
    v[n + 18] = u0;
  }
  modal_layer(v);
  modal_layer(v + 9);
}

// Reference gradients (times 2) of one field at the three points of quadrature row QB of the current
// slab: g[d][qa].  v[0..8] holds the slab's values along z and
// v[9..17] its derivatives, per modal (x, y) coefficient: in slab 1 (z = 0), which runs first, these
// are m and b themselves; fold_slab0 and fold_slab2 turn them into those of the next slab.
// r0: the row's values (no derivative) per modal x coefficient.
template <int QB>
__device__ __forceinline__ void row_grad(const double v[18], double g[3][3], double r0[3]) {
  constexpr double sy = QB == 0 ? -1.0 : 1.0;
  double r1[3], r2[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const double *ZB = v + i, *ZD = v + 9 + i;  // stride 3 in y
    if (QB == 1) {
      r0[i] = ZB[0];
      r1[i] = ZB[3];
      r2[i] = ZD[0];
    } else {
      r0[i] = fma(sy * MOD_V1, ZB[3], fma(MOD_V2, ZB[6], ZB[0]));
      r1[i] = fma(sy * MOD_D2, ZB[6], ZB[3]);
      r2[i] = fma(sy * MOD_V1, ZD[3], fma(MOD_V2, ZD[6], ZD[0]));
    }
  }
  g[0][1] = r0[1];
  g[0][0] = fma(-MOD_D2, r0[2], r0[1]);
  g[0][2] = fma(MOD_D2, r0[2], r0[1]);
  g[1][1] = r1[0];
  const double p1 = fma(MOD_V2, r1[2], r1[0]);
  g[1][0] = fma(-MOD_V1, r1[1], p1);
  g[1][2] = fma(MOD_V1, r1[1], p1);
  g[2][1] = r2[0];
  const double p2 = fma(MOD_V2, r2[2], r2[0]);
  g[2][0] = fma(-MOD_V1, r2[1], p2);
  g[2][2] = fma(MOD_V1, r2[1], p2);
}
template <int QB>
__device__ __forceinline__ void row_grad(const double v[18], double g[3][3]) {
  double r0[3];
  row_grad<QB>(v, g, r0);
}
// slab 1 -> slab 0; a[n] gets the z direction's a, which slab 2 needs (u0: layer 0, nodal along z only; may be a)
__device__ __forceinline__ void fold_slab0(double v[18], const double u0[9], double a[9]) {
#pragma unroll
  for (int n = 0; n < 9; n++) {
    a[n] = fma(2.0, u0[n] - v[n], v[n + 9]);  // u0 - 2 u1 + u2
    v[n] = fma(-MOD_V1, v[n + 9], fma(MOD_V2, a[n], v[n]));
    v[n + 9] = fma(-MOD_D2, a[n], v[n + 9]);
  }
}
// slab 0 -> slab 2
__device__ __forceinline__ void fold_slab2(double v[18], const double a[9]) {
#pragma unroll
  for (int n = 0; n < 9; n++) {
    const double b = fma(MOD_D2, a[n], v[n + 9]);
    v[n] = fma(2.0 * MOD_V1, b, v[n]);
    v[n + 9] = fma(MOD_D2, a[n], b);
  }
}

// acc (+)= c f, the first contribution without a load of the accumulator
template <bool FIRST>
__device__ __forceinline__ void acc_to(double &acc, double c, double f) {
  acc = FIRST ? c * f : fma(c, f, acc);
}
template <bool FIRST>
__device__ __forceinline__ void acc_one(double &acc, double f) {
  acc = FIRST ? f : acc + f;
}

// Transposed x- and y-contraction of one row's stresses dv[d][qa] of the wave's component into
// the slab sums RB (B-weighted in z) and RD (D-weighted), both [i + 3 j] in dual modal form.
// Rows run in the order 0, 2, 1 within a slab; row 0 starts the sums.
template <int QB>
__device__ __forceinline__ void row_dual(const double dv[3][3], double RB[9], double RD[9]) {
  constexpr bool F = QB == 0;
  constexpr double sy = QB == 0 ? -1.0 : 1.0;
  double t0[3], t1[3], t2[3];
  {
    const double s = dv[0][0] + dv[0][2], d = dv[0][2] - dv[0][0];
    t0[0] = 0.0;  // the derivative has no m term
    t0[1] = s + dv[0][1];
    t0[2] = MOD_D2 * d;
  }
  {
    const double s = dv[1][0] + dv[1][2], d = dv[1][2] - dv[1][0];
    t1[0] = s + dv[1][1];
    t1[1] = MOD_V1 * d;
    t1[2] = MOD_V2 * s;
  }
  {
    const double s = dv[2][0] + dv[2][2], d = dv[2][2] - dv[2][0];
    t2[0] = s + dv[2][1];
    t2[1] = MOD_V1 * d;
    t2[2] = MOD_V2 * s;
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    if (QB == 1) {
      if (i > 0) RB[i] += t0[i];
      RB[i + 3] += t1[i];
      RD[i] += t2[i];
    } else {
      // y: values m, +-V1 b, V2 a (t0 into RB, t2 into RD); derivative b, +-D2 a (t1 into RB)
      if (i > 0) {
        acc_one<F>(RB[i], t0[i]);
        acc_one<F>(RB[i + 3], t1[i]);
        RB[i + 3] = fma(sy * MOD_V1, t0[i], RB[i + 3]);
        acc_to<F>(RB[i + 6], sy * MOD_D2, t1[i]);
        RB[i + 6] = fma(MOD_V2, t0[i], RB[i + 6]);
      } else {
        if (F) RB[0] = 0.0;
        acc_one<F>(RB[3], t1[0]);
        acc_to<F>(RB[6], sy * MOD_D2, t1[0]);
      }
      acc_one<F>(RD[i], t2[i]);
      acc_to<F>(RD[i + 3], sy * MOD_V1, t2[i]);
      acc_to<F>(RD[i + 6], MOD_V2, t2[i]);
    }
  }
}
// a finished slab into the element's dual modal output Y[i + 3 j + 9 k]; slab 1 comes first
template <int QC>
__device__ __forceinline__ void slab_dual(const double RB[9], const double RD[9], double Y[27]) {
  constexpr double sz = QC == 0 ? -1.0 : 1.0;
#pragma unroll
  for (int n = 0; n < 9; n++) {
    if (QC == 1) {
      Y[n] = RB[n];
      Y[n + 9] = RD[n];
    } else {
      Y[n] += RB[n];
      Y[n + 9] = fma(sz * MOD_V1, RB[n], Y[n + 9] + RD[n]);
      const double a = QC == 0 ? MOD_V2 * RB[n] : fma(MOD_V2, RB[n], Y[n + 18]);
      Y[n + 18] = fma(sz * MOD_D2, RD[n], a);
    }
  }
}
__device__ __forceinline__ void dual_to_nodal27(double Y[27]) {
#pragma unroll
  for (int n = 0; n < 9; n++) from_dual3<9>(Y + n);
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int i = 0; i < 3; i++) from_dual3<3>(Y + i + 9 * k);
#pragma unroll
  for (int n = 0; n < 9; n++) from_dual3<1>(Y + 3 * n);
}

// LDS of a brick: the two node tiles while they are read, then the exchange buffers, two of each kind
// (a row's buffers are refilled two barriers later), then the output tile over the odd rows' buffers.
//   A: for each point 10 values per lane, adjugate (9) and determinant;
//   G: for each pair (point q, velocity component c != q) the three gradients;
//   S: for each pair (component c, point q != c) the point's three stresses in component c.
// A component's values at the point with its own number stay in its wave's registers.  The full block (BLK):
//   P: for each point the pressure, from the G wave;
//   T: for each point w (det div u + det fp), to the G wave.
template <bool BLK>
struct CompLds {
  static constexpr int NA = 10, SLOT = 3 * BEL;  // doubles
  static constexpr int A = 0, G = A + 3 * NA * BEL, S = G + 6 * SLOT, P = S + 6 * SLOT, T = P + SLOT;
  static constexpr int ROW = BLK ? T + SLOT : P;
  static constexpr int PARK = 2 * ROW;  // the G wave's own: 27 values (block: 9)
  static constexpr int N = 2 * ROW + (BLK ? 9 : 27) * BEL;
  static_assert(2 * 3 * TCS <= 2 * ROW, "the tiles fit the exchange buffers");
  static_assert(3 * TCS <= S, "the output tile fits a row's A and G buffers");
};
// slot of the ordered pair (a, b), a != b
__device__ __forceinline__ constexpr int pair_slot(int a, int b) { return 2 * a + (b < a ? b : b - 1); }
__device__ __forceinline__ void put3(double *slot, int lane, double a, double b, double c) {
  reinterpret_cast<double2 *>(slot)[lane] = make_double2(a, b);
  slot[2 * BEL + lane] = c;
}
__device__ __forceinline__ void get3(const double *slot, int lane, double &a, double &b, double &c) {
  const double2 v = reinterpret_cast<const double2 *>(slot)[lane];
  a = v.x;
  b = v.y;
  c = slot[2 * BEL + lane];
}

// quadrature rows of a brick in the order they run: slabs 1, 0, 2, each with its rows 0, 2, 1
__host__ __device__ constexpr int row_qc(int r) { return r / 3 == 0 ? 1 : (r / 3 == 1 ? 0 : 2); }
__host__ __device__ constexpr int row_qb(int r) { return r % 3 == 0 ? 0 : (r % 3 == 1 ? 2 : 1); }

// slab 0 -> slab 2 from layer 2 (nodal along z only) instead of a: v = m + V2 a - V1 b and d = b - D2 a in slab 0, and
// u2 = m + (b + a) / 2 gives a (1/2 - V2 + (1/2 + V1) D2) = u2 - v - (1/2 + V1) d
__device__ __forceinline__ void fold_slab2_layer(double v[18], const double u2[9]) {
  constexpr double e = 0.5 + MOD_V1, f = 1.0 / (0.5 - MOD_V2 + e * MOD_D2);
#pragma unroll
  for (int n = 0; n < 9; n++) {
    const double a = f * fma(-e, v[n + 9], u2[n] - v[n]);
    const double b = fma(MOD_D2, a, v[n + 9]);
    v[n] = fma(2.0 * MOD_V1, b, v[n]);
    v[n + 9] = fma(MOD_D2, a, b);
  }
}

// values at a row's three points from its modal x coefficients
__device__ __forceinline__ void row_values(const double r[3], double v[3]) {
  const double s = fma(MOD_V2, r[2], r[0]);
  v[0] = fma(-MOD_V1, r[1], s);
  v[1] = r[0];
  v[2] = fma(MOD_V1, r[1], s);
}

// the G wave
template <bool BLK>
struct GWave {
  using L = CompLds<BLK>;
  double x[3][18];  // modal coordinates: values and derivatives along z in the current slab
  // The z direction's third coefficients (layer 0, then a) are needed between the slabs only: they wait
  // in LDS (all 81 coefficients, beside a row's Jacobians, would spill).  The block needs that LDS for
  // the pressure; there the coordinates' layer 0 or 2 is read again one row ahead (xg, t).
  double *park;
  // block: coordinates relative to the pressure basis' centre; park holds the previous row's at its points
  double t[3][9], avg[3], ps[4], Yp[4], r0[3][3];
  const double *xg;    // the lane's element: its first coordinate
  int64_t gy, gz;      // steps to the next node row and plane

  __device__ __forceinline__ void read_layer(int k) {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) t[c][i + 3 * j] = xg[k * gz + j * gy + 3 * i + c];
  }
  // the continuity sums of the row whose points are parked, then park the next row's points
  template <bool PARK_NEXT>
  __device__ __forceinline__ void continuity(const double *row, int lane, bool first) {
    if (!first) {
      double f[3];
#pragma unroll
      for (int q = 0; q < 3; q++) f[q] = row[L::T + q * BEL + lane];
      Yp[0] += f[0] + f[1] + f[2];
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int q = 0; q < 3; q++) Yp[1 + c] = fma(f[q], park[(3 * c + q) * BEL + lane], Yp[1 + c]);
      pin<4>(Yp);
    }
    if (PARK_NEXT) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        double v[3];
        row_values(r0[c], v);
#pragma unroll
        for (int q = 0; q < 3; q++) park[(3 * c + q) * BEL + lane] = v[q];
      }
    }
  }

  // adjugates and determinants of row R's points
  template <int R>
  __device__ __forceinline__ void forward(double *row, int lane) {
    double Jc[3][3][3];  // [component][d][qa]
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (BLK && (R == 3 || R == 6)) {
#pragma unroll
        for (int n = 0; n < 9; n++) t[c][n] -= avg[c];
        modal_layer(t[c]);
        if (R == 3)
          fold_slab0(x[c], t[c], t[c]);
        else
          fold_slab2_layer(x[c], t[c]);
        pin<18>(x[c]);
      } else if (R == 3 || R == 6) {
        double t[9];
#pragma unroll
        for (int n = 0; n < 9; n++) t[n] = park[(9 * c + n) * BEL + lane];
        if (R == 3) {
          modal_layer(t);
          fold_slab0(x[c], t, t);
#pragma unroll
          for (int n = 0; n < 9; n++) park[(9 * c + n) * BEL + lane] = t[n];
        } else {
          fold_slab2(x[c], t);
        }
        pin<18>(x[c]);
      }
      if constexpr (BLK)
        row_grad<row_qb(R)>(x[c], Jc[c], r0[c]);
      else
        row_grad<row_qb(R)>(x[c], Jc[c]);
    }
    if constexpr (BLK) {
      // the pressure is linear in the coordinates relative to the basis' centre
      double rp[3], pv[3];
#pragma unroll
      for (int i = 0; i < 3; i++) rp[i] = fma(ps[3], r0[2][i], fma(ps[2], r0[1][i], ps[1] * r0[0][i]));
      rp[0] += ps[0];
      row_values(rp, pv);
#pragma unroll
      for (int q = 0; q < 3; q++) row[L::P + q * BEL + lane] = pv[q];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      double J[3][3], A[3][3];
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int c = 0; c < 3; c++) J[d][c] = Jc[c][d][q];
      const double det = adjugate(J, A);
      double2 *o = reinterpret_cast<double2 *>(row + L::A + q * L::NA * BEL) + lane;
      o[0] = make_double2(A[0][0], A[0][1]);
      o[BEL] = make_double2(A[0][2], A[1][0]);
      o[2 * BEL] = make_double2(A[1][1], A[1][2]);
      o[3 * BEL] = make_double2(A[2][0], A[2][1]);
      o[4 * BEL] = make_double2(A[2][2], det);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  template <int R>
  __device__ __forceinline__ void rows(double *buf, int lane) {
    lds_barrier();
    if constexpr (BLK) continuity<true>(buf + ((R + 1) & 1) * L::ROW, lane, R == 0);
    if constexpr (R < 8) {
      row_fence();
      forward<R + 1>(buf + ((R + 1) & 1) * L::ROW, lane);
      if (BLK && R == 1) read_layer(0);
      if (BLK && R == 4) read_layer(2);
      row_fence();
      rows<R + 1>(buf, lane);
    }
  }
};

// U wave C: velocity component C, output component C and the stress of point C of every row.
template <int C, bool BLK>
struct UWave {
  using L = CompLds<BLK>;
  double u[27];          // modal velocity component C
  double Y[27];          // dual modal output component C
  double RB[9], RD[9];
  double own[3];         // gradient of component C at the wave's point
  double eta, eta_n;     // viscosity at the wave's point of this row and the next
  const double *ep;      // the brick's viscosities (uniform)
  const double *fe;      // block: the lane's element's continuity source, or null (uniformly)
  double pq;             // block: the pressure at the wave's point

  __device__ __forceinline__ double load_eta(int r, int lane) const {
    return fast_at(ep + (C + 3 * row_qb(r) + 9 * row_qc(r)) * BEL, (uint32_t)lane);
  }

  // gradients of row R; the two foreign points' values go to G
  template <int R>
  __device__ __forceinline__ void forward(double *row, int lane) {
    if (R == 3) {
      modal_layer(u + 18);
      fold_slab0(u, u + 18, u + 18);
    }
    if (R == 6) fold_slab2(u, u + 18);
    if (R == 3 || R == 6) pin<18>(u);
    double G[3][3];
    row_grad<row_qb(R)>(u, G);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      if (q == C) {
#pragma unroll
        for (int d = 0; d < 3; d++) own[d] = G[d][q];
      } else {
        put3(row + L::G + pair_slot(q, C) * L::SLOT, lane, G[0][q], G[1][q], G[2][q]);
      }
    }
  }

  // the operands of point() and backward() from the exchange buffers, all read at once
  double A[3][3], G[3][3], det;  // G[d][component]
  double dv[3][3];               // stresses of the previous row [d][qa]
  __device__ __forceinline__ void read_point(const double *row, int lane) {
    const double2 *a = reinterpret_cast<const double2 *>(row + L::A + C * L::NA * BEL) + lane;
    const double2 a0 = a[0], a1 = a[BEL], a2 = a[2 * BEL], a3 = a[3 * BEL], a4 = a[4 * BEL];
    A[0][0] = a0.x; A[0][1] = a0.y; A[0][2] = a1.x;
    A[1][0] = a1.y; A[1][1] = a2.x; A[1][2] = a2.y;
    A[2][0] = a3.x; A[2][1] = a3.y; A[2][2] = a4.x;
    det = a4.y;
#pragma unroll
    for (int c = 0; c < 3; c++)
      if (c != C) get3(row + L::G + pair_slot(C, c) * L::SLOT, lane, G[0][c], G[1][c], G[2][c]);
    if (BLK) pq = row[L::P + C * BEL + lane];
  }
  __device__ __forceinline__ void read_stress(const double *row, int lane) {
#pragma unroll
    for (int q = 0; q < 3; q++)
      if (q != C) get3(row + L::S + pair_slot(C, q) * L::SLOT, lane, dv[0][q], dv[1][q], dv[2][q]);
  }

  // stress of row R at point C; the foreign components go to S, the own one to mine
  template <int R>
  __device__ __forceinline__ void point(double *row, int lane, double mine[3]) {
    constexpr double w8 = gw1(C) * gw1(row_qb(R)) * gw1(row_qc(R)) * 0.125;
    double dv[3][3];
#pragma unroll
    for (int d = 0; d < 3; d++) G[d][C] = own[d];
    const double s = (w8 * eta) * rcp64(det);
    if constexpr (BLK) {
      const double tr = stress_action_p(A, G, s, w8 * pq, dv);
      // det is 8 times the determinant, the trace 8 times det div u
      row[L::T + C * BEL + lane] = w8 * (fe ? fma(det, fe[C + 3 * row_qb(R) + 9 * row_qc(R)], tr) : tr);
    } else {
      stress_action(A, G, s, dv);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (c == C) {
#pragma unroll
        for (int d = 0; d < 3; d++) mine[d] = dv[d][c];
      } else {
        put3(row + L::S + pair_slot(c, C) * L::SLOT, lane, dv[0][c], dv[1][c], dv[2][c]);
      }
    }
  }

  // the transposed contractions of row R
  template <int R>
  __device__ __forceinline__ void backward(const double mine[3]) {
#pragma unroll
    for (int d = 0; d < 3; d++) dv[d][C] = mine[d];
    row_dual<row_qb(R)>(dv, RB, RD);
    if (R % 3 == 2) {
      slab_dual<row_qc(R)>(RB, RD, Y);
      pin<row_qc(R) == 1 ? 18 : 27>(Y);
    } else {
      pin<9>(RB);
      pin<9>(RD);
    }
  }

  // Between two barriers: the transposes of row R - 1 and the stress of row R (their operands were
  // filled before the first of them) and the forward contraction of row R + 1.
  template <int R>
  __device__ __forceinline__ void rows(double *buf, int lane, const double prev[3]) {
    lds_barrier();
    double mine[3];
    if (R < 8) eta_n = load_eta(R < 8 ? R + 1 : 8, lane);
    if constexpr (R > 0) read_stress(buf + ((R - 1) & 1) * L::ROW, lane);
    read_point(buf + (R & 1) * L::ROW, lane);
    row_fence();
    if constexpr (R > 0) {
      backward<R - 1>(prev);
      row_fence();
    }
    point<R>(buf + (R & 1) * L::ROW, lane, mine);
    row_fence();
    if constexpr (R < 8) {
      forward<R + 1>(buf + ((R + 1) & 1) * L::ROW, lane);
      row_fence();
      eta = eta_n;
      rows<R + 1>(buf, lane, mine);
    } else {
      lds_barrier();
      read_stress(buf, lane);
      backward<8>(mine);
    }
  }
};

// Walk of one wave over its tile rows: wave w takes the row pairs w, w + 4, ..., lanes 0-26 the even
// and lanes 27-53 the odd row of a pair.  From one step to the next the row number grows by 8, so
// (y, z) goes to (8, z) from y = 0 and to (y - 1, z + 1) otherwise; the element offset (OFF: 32 bits
// where the tile's offsets fit) and the LDS offset follow by one of two increments.
constexpr int WALK = (TPAIRS + CWAVES - 1) / CWAVES;
template <typename OFF>
struct RowWalk {
  int y, z, lds;
  OFF e, sy, sz;
  __device__ __forceinline__ RowWalk(const Box &b, int w, int p) {
    const int r = 2 * w + (p == 1);  // below TN
    y = r;
    z = 0;
    sy = 3 * (OFF)b.NX;
    sz = sy * (OFF)b.NY;
    e = sy * (OFF)y;
    lds = TRS * y;
  }
  __device__ __forceinline__ void next() {
    const bool top = y == 0;
    e += top ? (OFF)(TN - 1) * sy : sz - sy;
    lds += top ? (TN - 1) * TRS : TPS - TRS;
    z += top ? 0 : 1;
    y = top ? TN - 1 : y - 1;
  }
};
static_assert(2 * CWAVES == TN - 1, "a step of the walk is one row less than a plane");
struct RowLane {
  int p, ii, c;  // parity (2 = idle lane), node column, component
  int lds_col;   // LDS offset of the column
  __device__ __forceinline__ explicit RowLane(int lane) {
    p = lane < 2 * RLEN ? lane / RLEN : 2;
    const int col = lane - RLEN * (p < 2 ? p : 0);
    ii = p < 2 ? col / 3 : 0;
    c = p < 2 ? col - 3 * ii : 0;
    lds_col = c * TCS + tx(ii);
  }
};

// wave w's share of the brick's resident coordinate tile, straight from memory into LDS in chunks of
// 1 KiB (no register holds it on the way); complete at the wave's next s_waitcnt vmcnt(0)
constexpr int XCHUNKS = (3 * TCS * 8 + 1023) / 1024;
__device__ __forceinline__ void copy_xtile(const double *xt, double *lds, int w, int lane) {
  typedef __attribute__((address_space(3))) char lchar;
  const char *src = (const char *)uniform_ptr(xt);
  lchar *dst = (lchar *)(uintptr_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lchar *)lds);
#pragma unroll
  for (int k = 0; k < (XCHUNKS + CWAVES - 1) / CWAVES; k++) {
    const int o = 1024 * (CWAVES * k + w);
    if (o + 16 * lane < 3 * TCS * 8)
      __builtin_amdgcn_global_load_lds((const void *)(src + o + 16 * lane),
                                       (__attribute__((address_space(3))) void *)(dst + o), 16, 0, 0);
  }
}

// Wave w's share of the velocity tile and, without a resident one, of the coordinate tile.
template <bool HM, typename OFF>
__device__ __forceinline__ void load_tiles4(const Box &b, const BrickId &br, const Tile &t,
                                            const double *__restrict__ g1, double *__restrict__ s1,
                                            const double *__restrict__ g2, const uint8_t *__restrict__ mask2,
                                            double *__restrict__ s2, int w, int lane) {
  const RowLane L(lane);
  const OFF col = 3 * min(L.ii, t.tnx - 1) + L.c;
  const double *b2 = g2 + 3 * t.node0;
  const uint8_t *bm = mask2 + 3 * t.node0;
  double v2[WALK];
  int mk[WALK];
  RowWalk<OFF> r(b, w, L.p);
#pragma unroll
  for (int k = 0; k < WALK; k++) {
    const OFF e = col + (r.y < t.tny && r.z < t.tnz ? r.e : 0);  // rows past a partial tile: a valid address
    v2[k] = fast_at(b2, e);
    mk[k] = HM ? (int)fast_at(bm, e) : 0;
    r.next();
  }
  if (b.xtile) {
    copy_xtile(b.xtile + (int64_t)br.lin * 3 * TCS, s1, w, lane);
  } else {
    const double *b1 = g1 + 3 * t.node0;
    double v1[WALK];
    RowWalk<OFF> q(b, w, L.p);
#pragma unroll
    for (int k = 0; k < WALK; k++) {
      v1[k] = fast_at(b1, col + (q.y < t.tny && q.z < t.tnz ? q.e : 0));
      q.next();
    }
    __builtin_amdgcn_sched_barrier(0);
    RowWalk<OFF> a(b, w, L.p);
#pragma unroll
    for (int k = 0; k < WALK; k++) {
      if (L.p < 2 && a.z < TN) s1[L.lds_col + a.lds] = v1[k];
      a.next();
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  RowWalk<OFF> q(b, w, L.p);
#pragma unroll
  for (int k = 0; k < WALK; k++) {
    if (L.p < 2 && q.z < TN) {
      // rows and columns outside the box belong to no element of the brick: any value will do
      s2[L.lds_col + q.lds] = mk[k] ? 0.0 : v2[k];  // BCListInsertLocalZero, src/dmda_bcs.c:581-608
    }
    q.next();
  }
  __builtin_amdgcn_s_waitcnt(WAIT_VM0);  // the coordinate tile's copies
}

// The owner-writes store of store_tile_own by four waves.  mask: the brick's Dirichlet rows become
// u's (MatMult semantics; the face pass leaves them alone), or null.
template <bool CH, typename OFF>
__device__ __forceinline__ void store_tile4(const Box &b, const BrickId &br, const Tile &t,
                                            const double *__restrict__ s, double *__restrict__ g,
                                            double *__restrict__ face, bool add_mode, int w, int lane,
                                            const ChebOut<double> *co, const uint8_t *__restrict__ mask,
                                            const double *__restrict__ u) {
  asm volatile("" : "+v"(lane));  // see store_tile
  const RowLane L(lane);
  const bool ownx = L.ii < 2 * BE || br.bx == b.nbx - 1;
  const bool lasty = br.by == b.nby - 1, lastz = br.bz == b.nbz - 1;
  double *fo = face + (int64_t)br.lin * FACEVALS + L.c;
  double *gb = g + 3 * t.node0;
  const OFF col = 3 * min(L.ii, t.tnx - 1) + L.c;
  double v[WALK], val[WALK];
  if (add_mode) {
    RowWalk<OFF> r(b, w, L.p);
#pragma unroll
    for (int k = 0; k < WALK; k++) {
      v[k] = fast_at(gb, col + (r.y < t.tny && r.z < t.tnz ? r.e : 0));
      r.next();
    }
  }
  RowWalk<OFF> q(b, w, L.p);
#pragma unroll
  for (int k = 0; k < WALK; k++) {
    val[k] = s[L.lds_col + (q.z < TN ? q.lds : 0)];
    q.next();
  }
  if (mask) {
    const uint8_t *bm = mask + 3 * t.node0;
    const double *bu = u + 3 * t.node0;
    int mk[WALK];
    RowWalk<OFF> m(b, w, L.p);
#pragma unroll
    for (int k = 0; k < WALK; k++) {
      const OFF e = col + (m.y < t.tny && m.z < t.tnz ? m.e : 0);
      mk[k] = (int)fast_at(bm, e);
      v[k] = fast_at(bu, e);
      m.next();
    }
#pragma unroll
    for (int k = 0; k < WALK; k++) val[k] = mk[k] ? v[k] : val[k];
  }
  __builtin_amdgcn_sched_barrier(0);
  RowWalk<OFF> r(b, w, L.p);
#pragma unroll
  for (int k = 0; k < WALK; k++) {
    if (L.p < 2 && L.ii < t.tnx && r.y < t.tny && r.z < t.tnz) {
      const bool owny = r.y < 2 * BE || lasty, ownz = r.z < 2 * BE || lastz;
      if (ownx && owny && ownz) {
        if constexpr (CH) {
          const int64_t gi = 3 * t.node0 + col + r.e;
          const bool lower = (L.ii == 0 && br.bx > 0) || (r.y == 0 && br.by > 0) || (r.z == 0 && br.bz > 0);
          const bool dir = co->mask && co->mask[gi];
          if (dir || !lower)
            co->out[gi] = cheb_update(*co, gi, dir ? co->x[gi] : val[k]);
          else
            g[gi] = val[k];
        } else {
          fast_at(gb, col + r.e) = add_mode ? v[k] + val[k] : val[k];
        }
      } else {
        const int slot = !ownx ? r.z * TN + r.y : (!owny ? TN * TN + r.z * TN + L.ii : 2 * TN * TN + r.y * TN + L.ii);
        fo[3 * slot] = val[k];
      }
    }
    r.next();
  }
}

// Full 9x9x9 tiles (every interior brick): the rows by planes, U wave w the planes z = 3 w .. 3 w + 2
// with the constant steps of load_tile2_fast, a handful of instructions per row pair where the walk
// takes forty.  The G wave copies the resident coordinate tile.
__device__ __forceinline__ void copy_xtile_all(const double *xt, double *lds, int lane) {
  lds_copy_async<3 * TCS * 8>(xt, lds, lane);
}
template <typename R, typename S>
__device__ __forceinline__ void load_third(const Box &b, const Tile &t, const S *__restrict__ g, int w, int lane,
                                           R v[WSTEPS]) {
  const FastLane L = fast_lane(b, lane);
  const S *g0 = g + 3 * (t.node0 + (int64_t)b.NX * b.NY * (WPLANES * w));
#pragma unroll
  for (int it = 0; it < WSTEPS; it++) v[it] = (R)fast_at(g0, fast_eoff<WSTEPS>(b, L, it));
}
template <bool HM>
__device__ __forceinline__ void put_third(const double v[WSTEPS], const int mk[WSTEPS], double *s, int w, int lane) {
  const FastLane L = fast_lane(Box{}, lane);  // the LDS offsets do not depend on the box
  s += TPS * WPLANES * w;
  if (L.p > 1) return;
#pragma unroll
  for (int it = 0; it < WSTEPS; it++)
    if (it < WSTEPS - 1 || L.p == 0)
      s[(fast_wrap(it) ? L.ldsw : L.lds0) + fast_lds_step(it)] = HM && mk[it] ? 0.0 : v[it];
}
__device__ __forceinline__ void load_tiles_full(const Box &b, const BrickId &br, const Tile &t,
                                                const double *__restrict__ g1, double *__restrict__ s1,
                                                const double *__restrict__ g2, const uint8_t *__restrict__ mask2,
                                                double *__restrict__ s2, int w, int lane) {
  if (w < 3) {
    double v2[WSTEPS];
    int mk[WSTEPS] = {};
    load_third(b, t, g2, w, lane, v2);
    if (!b.xtile) {
      double v1[WSTEPS];
      load_third(b, t, g1, w, lane, v1);
      put_third<false>(v1, mk, s1, w, lane);
    }
    // the flag's load travels with the tile's
    if (mask2 && !(b.bdir && !b.bdir[br.lin])) {
      load_third(b, t, mask2, w, lane, mk);
      put_third<true>(v2, mk, s2, w, lane);  // BCListInsertLocalZero, src/dmda_bcs.c:581-608
    } else {
      put_third<false>(v2, mk, s2, w, lane);
    }
  } else if (b.xtile) {
    copy_xtile_all(b.xtile + (int64_t)br.lin * 3 * TCS, s1, lane);
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
  }
}

// The owner-writes store of a full tile: U wave w stores the planes 3 w .. 3 w + 2 up to 7, the G wave the
// plane 8.
__device__ __forceinline__ void store_tile_full(const Box &b, const BrickId &br, const Tile &t,
                                                const double *__restrict__ s, double *__restrict__ g,
                                                double *__restrict__ face, bool add_mode, int w, int lane) {
  asm volatile("" : "+v"(lane));  // see store_tile
  if (w < 2)
    store_rows_full<3 * TN>(b, br, t, s, g, face, add_mode, WPLANES * w, lane);
  else if (w == 2)
    store_rows_full<2 * TN>(b, br, t, s, g, face, add_mode, 2 * WPLANES, lane);
  else
    store_rows_full<TN>(b, br, t, s, g, face, add_mode, 2 * BE, lane);
}

// The full block's other operands: pressure, continuity output and source (may be null)
struct BlockArgs {
  const double *p, *coords;
  double *yp;
  const double *fp;
};

template <bool BLK>
__device__ __forceinline__ void g_wave(double *lds, const Box &b, const Tile &t, const BlockArgs &ba, bool active,
                                       bool add_mode, int lane) {
  using L = CompLds<BLK>;
  GWave<BLK> W;
  const int base = lane_base(lane);
  W.park = lds + L::PARK;
  double x[3][27];
  double inv[3];
  int64_t e = 0;
  if constexpr (BLK) {
    // lanes without an element take another's coordinates; nobody takes their outputs
    const LaneElem le = lane_elem(lane);
    W.gy = 3 * (int64_t)b.NX;
    W.gz = W.gy * b.NY;
    W.xg = ba.coords + 3 * (t.node0 + 2 * min(le.lx, t.nex - 1)) + 2 * min(le.ly, t.ney - 1) * W.gy +
           2 * min(le.lz, t.nez - 1) * W.gz;
    if (active) e = lane_element(b, t, lane);
#pragma unroll
    for (int n = 0; n < 4; n++) {
      W.ps[n] = ba.p[4 * e + n];
      W.Yp[n] = 0.0;
    }
  }
  lds_barrier();  // the tiles are in LDS
#pragma unroll
  for (int c = 0; c < 3; c++) load_modal(lds, base, c, x[c]);
  lds_barrier();  // every wave has read its tile: the LDS becomes the exchange buffers
  if constexpr (BLK) {
    // P3D_ConstructNi_P1GRel_3D (src/element_utils_q2.c:183-224): centre and scale of the basis
    inv[0] = 1.0 / (x[0][14] - x[0][12]);
    inv[1] = 1.0 / (x[1][16] - x[1][10]);
    inv[2] = 1.0 / (x[2][22] - x[2][4]);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      double sum = 0.0;
#pragma unroll
      for (int n = 0; n < 27; n++) sum += x[c][n];
      W.avg[c] = sum * (1.0 / 27.0);
#pragma unroll
      for (int n = 0; n < 27; n++) x[c][n] -= W.avg[c];
      W.ps[1 + c] *= inv[c];
    }
  }
#pragma unroll
  for (int c = 0; c < 3; c++) {
    modal27(x[c]);
#pragma unroll
    for (int n = 0; n < 18; n++) W.x[c][n] = x[c][n];
    if constexpr (!BLK) {
#pragma unroll
      for (int n = 0; n < 9; n++) W.park[(9 * c + n) * BEL + lane] = x[c][18 + n];
    }
  }
  W.template forward<0>(lds, lane);
  row_fence();
  W.template rows<0>(lds, lane);
  // the odd rows' A and G buffers are idle since the last barrier: the output tile, zeroed for the
  // U waves
  constexpr int N2 = 3 * TCS / 2;  // double2's
  int l2 = lane;
  asm volatile("" : "+v"(l2));  // keep the address arithmetic here
  double2 *z = reinterpret_cast<double2 *>(lds + L::ROW) + l2;
  const double2 zero = make_double2(0.0, 0.0);
#pragma unroll
  for (int n = 0; n < N2 / BEL; n++) z[n * BEL] = zero;
  if (l2 < N2 % BEL) z[N2 / BEL * BEL] = zero;
  lds_barrier();
  if constexpr (BLK) {
    W.template continuity<false>(lds, lane, false);
    if (active) {
      double *o = ba.yp + 4 * e;
      const double r[4] = {-W.Yp[0], -W.Yp[1] * inv[0], -W.Yp[2] * inv[1], -W.Yp[3] * inv[2]};
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = add_mode ? o[i] + r[i] : r[i];
    }
  }
  lds_barrier();
}

template <int C, bool BLK>
__device__ __forceinline__ void u_wave(double *lds, const double *__restrict__ ep, const double *fe, bool active,
                                       int lane) {
  using L = CompLds<BLK>;
  UWave<C, BLK> W;
  const int base = lane_base(lane);
  W.ep = ep;
  W.fe = fe;
  W.eta = W.load_eta(0, lane);
  lds_barrier();
  load_modal(lds + 3 * TCS, base, C, W.u);
  lds_barrier();
  modal27(W.u);
  W.template forward<0>(lds, lane);
  row_fence();
  const double none[3] = {0.0, 0.0, 0.0};
  W.template rows<0>(lds, lane, none);
  dual_to_nodal27(W.Y);
  if (active) {
    double *Ys = lds + L::ROW;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) lds_add(&Ys[base + toff(C, i, j, k)], W.Y[i + 3 * j + 9 * k]);
  }
  lds_barrier();
}

template <bool HM>
__device__ __forceinline__ void load_tiles4(const Box &b, const BrickId &br, const Tile &t,
                                            const double *__restrict__ g1, double *__restrict__ s1,
                                            const double *__restrict__ g2, const uint8_t *__restrict__ mask2,
                                            double *__restrict__ s2, int w, int lane) {
  if (b.fast32)
    load_tiles4<HM, uint32_t>(b, br, t, g1, s1, g2, mask2, s2, w, lane);
  else
    load_tiles4<HM, int64_t>(b, br, t, g1, s1, g2, mask2, s2, w, lane);
}

// The brick br of box b.  mode: OUT_SET, OUT_ADD or OUT_BC (set, and y = u on the mask's Dirichlet dofs).
// CH: store with the fused Chebyshev update of co (store_tile_own<true>).
// BLK: the full block [A11 A12; A21 0] of ba's pressure and continuity output.
template <bool CH, bool BLK = false>
__device__ __forceinline__ void a11_fp64_brick(const Box &b, const BrickId &br, const double *__restrict__ coords,
                                               const double *__restrict__ u, const uint8_t *__restrict__ mask,
                                               const double *__restrict__ eta_bm, double *__restrict__ y, int mode,
                                               double *__restrict__ facebuf, const ChebOut<double> &co,
                                               const BlockArgs &ba = BlockArgs{}) {
  using L = CompLds<BLK>;
  __shared__ double2 lds2[L::N / 2];
  double *lds = reinterpret_cast<double *>(lds2);
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / BEL), lane = (int)threadIdx.x - BEL * w;
  const Tile t = tile_of(b, br);
  const bool active = lane_active(t, lane);
  const bool full = tile_fast(b, t);
  if (full)
    load_tiles_full(b, br, t, coords, lds, u, mask, lds + 3 * TCS, w, lane);
  else if (mask)
    load_tiles4<true>(b, br, t, coords, lds, u, mask, lds + 3 * TCS, w, lane);
  else
    load_tiles4<false>(b, br, t, coords, lds, u, mask, lds + 3 * TCS, w, lane);
  const double *ep = eta_bm + (int64_t)br.lin * 27 * BEL;
  const double *fe = BLK && ba.fp ? ba.fp + 27 * (active ? lane_element(b, t, lane) : 0) : nullptr;
  switch (w) {
    case 0: u_wave<0, BLK>(lds, ep, fe, active, lane); break;
    case 1: u_wave<1, BLK>(lds, ep, fe, active, lane); break;
    case 2: u_wave<2, BLK>(lds, ep, fe, active, lane); break;
    default: g_wave<BLK>(lds, b, t, ba, active, mode == OUT_ADD, lane); break;
  }
  const double *Ys = lds + L::ROW;
  const ChebOut<double> *cp = CH ? &co : nullptr;
  if (mask && b.bdir && !b.bdir[br.lin]) mask = nullptr;  // no Dirichlet dof in the tile
  if (!CH && full && !(mode == OUT_BC && mask)) {
    store_tile_full(b, br, t, Ys, y, facebuf, mode == OUT_ADD, w, lane);
    return;
  }
  if (b.fast32)
    store_tile4<CH, uint32_t>(b, br, t, Ys, y, facebuf, mode == OUT_ADD, w, lane, cp, mode == OUT_BC ? mask : nullptr, u);
  else
    store_tile4<CH, int64_t>(b, br, t, Ys, y, facebuf, mode == OUT_ADD, w, lane, cp, mode == OUT_BC ? mask : nullptr, u);
}

}  // namespace ptq2
