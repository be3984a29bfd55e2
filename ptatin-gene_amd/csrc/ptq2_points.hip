// ptq2_points.hip -- material points -> quadrature points on the device.
//
// The Q1 projection of SwarmUpdateGaussPropertiesLocalL2Projection_Q1_MPntPStokes
// (src/material_point_utils.c:905-955, body :663-830): every point adds w * value and w into
// the 27 nodes of its element (w = the Q1 basis at the point for the 8 vertex nodes, 1 for the
// other 19), nodal value = sum / weight sum, and each quadrature point takes the Q1
// interpolation of its element's vertex values clipped to the element's nodal range.
//
// The reference scatters point by point into the nodes (an order the device cannot keep
// without atomics).  Here the points are bucketed by element, every element sums its points in
// index order into its 8 vertices and, once, into its other nodes (which all weigh a point with 1),
// and every node adds the sums of its <= 8 adjacent elements in ascending element order: fixed
// orders, so the result is bitwise reproducible.
//
// Buckets: a point takes the next free slot of its element (an atomic counter), and the element
// orders its few slots by point index afterwards.  That is one pass over the points (27 us for 0.5 million
// points in 63360 elements, bound by the atomics), where a stable sort of the keys takes some fifteen
// launches (160 us).  Clouds that crowd some element beyond the slots (BUCKET_MAX, or twice the average
// plus 16) go through the sort; their sums run in the same order and give the same bits.
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include <cmath>
#include <cstdarg>
#include <cstdio>

#include "ptq2.h"
#include "ptq2_ctx.h"
#include "ptq2_kernels.h"

namespace ptq2 {
namespace {

constexpr int PTB = 256;

inline unsigned grid_of(int64_t n) {
  const int64_t g = (n + PTB - 1) / PTB;
  return (unsigned)(g < 65535 * 64 ? (g > 0 ? g : 1) : 65535 * 64);
}

constexpr int BUCKET_MAX = 128;  // slots per element at most (two lists of 32 elements fit 32 KiB of LDS)
constexpr int SUM_LANES = 8, SUM_ELEMS = PTB / SUM_LANES;
enum : int { PERR_INDEX = 1, PERR_FINITE = 2, PERR_CROWDED = 4 };

// slots per element of np points in ne elements; 0: sort
inline int bucket_slots(int64_t np, int64_t ne) {
  const int64_t c = (2 * (np / ne) + 16 + 7) / 8 * 8;
  return c <= BUCKET_MAX ? (int)c : 0;
}

// element index in range, local coordinates and values finite; with slots, the point into one of its
// element's
__global__ void k_points_bucket(int64_t np, int64_t ne, const double *__restrict__ xi, const int32_t *__restrict__ wil,
                                const double *__restrict__ eta, const double *__restrict__ rho, int cap,
                                int32_t *__restrict__ cnt, int32_t *__restrict__ slot, int *__restrict__ err) {
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < np; p += (int64_t)gridDim.x * blockDim.x) {
    const int32_t e = wil[p];
    int bits = 0;
    if (e < 0 || (int64_t)e >= ne) {
      bits |= PERR_INDEX;
    } else if (slot) {
      const int k = atomicAdd(cnt + e, 1);
      if (k < cap)
        slot[(int64_t)e * cap + k] = (int32_t)p;
      else
        bits |= PERR_CROWDED;
    }
    bool fin = isfinite(xi[3 * p]) && isfinite(xi[3 * p + 1]) && isfinite(xi[3 * p + 2]) && isfinite(eta[p]);
    if (rho) fin = fin && isfinite(rho[p]);
    if (!fin) bits |= PERR_FINITE;
    if (bits) atomicOr(err, bits);
  }
}

__global__ void k_iota(int64_t n, int32_t *__restrict__ v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = (int32_t)i;
}

// first sorted position of every element (keys sorted ascending): off[e] = lower_bound(e)
__global__ void k_bucket_offsets(int64_t np, int64_t ne, const int32_t *__restrict__ keys, int64_t *__restrict__ off) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e <= ne; e += (int64_t)gridDim.x * blockDim.x) {
    int64_t lo = 0, hi = np;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)keys[mid] < e)
        lo = mid + 1;
      else
        hi = mid;
    }
    off[e] = lo;
  }
}

// the elements adjacent to node index I along one axis (m elements) and the node's local
// index in each: even I is a vertex of elements I/2-1 (local 2) and I/2 (local 0), odd I the
// middle node of element (I-1)/2
__device__ __forceinline__ int adjacent(int I, int m, int el[2], int loc[2]) {
  if (I & 1) {
    el[0] = (I - 1) >> 1;
    loc[0] = 1;
    return 1;
  }
  int n = 0;
  if (I / 2 - 1 >= 0) { el[n] = I / 2 - 1; loc[n] = 2; n++; }
  if (I / 2 < m) { el[n] = I / 2; loc[n] = 0; n++; }
  return n;
}

// Q1 basis of the vertex at local node index l (0 or 2) along one axis at coordinate x
__device__ __forceinline__ double q1_1d(int l, double x) { return l == 0 ? 1.0 - x : 1.0 + x; }
// A point's weight a b at a vertex, and its share of the three sums; fused explicitly, so that the element sums and
// the nodes' own have the same bits.
struct VertexWeight {
  double a, b;
  __device__ __forceinline__ VertexWeight(int lx, int ly, int lz, const double *xi)
      : a(0.125 * q1_1d(lx, xi[0]) * q1_1d(ly, xi[1])), b(q1_1d(lz, xi[2])) {}
};
__device__ __forceinline__ void add_point(double a, double b, double v, double r, double &sv, double &sr, double &sw) {
  const double w = a * b;
  sv = fma(w, v, sv);
  sr = fma(w, r, sr);
  sw = fma(a, b, sw);
}

// Sums over an element's points in index order: eight lanes per element, one per vertex, walk the points
// together (a point's values are one broadcast load).  part, arrays of ne values: 3 l + 0..2 the sums of w
// eta, w rho and w of vertex l, 24..26 those of eta, rho and 1.  Bound by the gathers of the points' values
// (a 64-byte line each), 32 points of a workgroup in flight per step.  27 us for 0.5 million points, and 12 us
// for the nodes' sums, where one thread per node walking its elements' points takes 265 us.
// SLOTS: the points are the element's slots in any order; else they are order[off[e] .. off[e + 1]).
template <bool SLOTS>
__global__ __launch_bounds__(PTB) void k_points_sums(int64_t ne, int cap, const int32_t *__restrict__ cnt,
                                                     const int32_t *__restrict__ slot, const int64_t *__restrict__ off,
                                                     const int32_t *__restrict__ order, const double *__restrict__ xi,
                                                     const double *__restrict__ eta, const double *__restrict__ rho,
                                                     double *__restrict__ part) {
  extern __shared__ int32_t lists[];
  const int g = (int)threadIdx.x / SUM_LANES, l = (int)threadIdx.x % SUM_LANES;
  const int64_t e = (int64_t)blockIdx.x * SUM_ELEMS + g;
  const int32_t *list;
  int64_t n = 0;
  if (SLOTS) {
    int32_t *in = lists + g * cap, *out = lists + (SUM_ELEMS + g) * cap;
    const int m = e < ne ? min(cnt[e], cap) : 0;
    for (int k = l; k < m; k += SUM_LANES) in[k] = slot[e * cap + k];
    __syncthreads();
    for (int k = l; k < m; k += SUM_LANES) {
      int r = 0;  // the indices differ: a point's place is the number of smaller ones
      for (int q = 0; q < m; q++) r += in[q] < in[k];
      out[r] = in[k];
    }
    __syncthreads();
    list = out;
    n = m;
  } else {
    if (e < ne) n = off[e + 1] - off[e];
    list = order + (e < ne ? off[e] : 0);
  }
  if (e >= ne) return;
  const int lx = (l & 1) * 2, ly = (l >> 1 & 1) * 2, lz = (l >> 2) * 2;
  double a1 = 0.0, a2 = 0.0, bw = 0.0, c1 = 0.0, c2 = 0.0;
#pragma unroll 4
  for (int64_t k = 0; k < n; k++) {
    const int64_t p = list[k];
    const VertexWeight w(lx, ly, lz, xi + 3 * p);
    const double v = eta[p], r = rho ? rho[p] : 0.0;
    add_point(w.a, w.b, v, r, a1, a2, bw);
    c1 += v;
    c2 += r;
  }
  part[(3 * l + 0) * ne + e] = a1;
  part[(3 * l + 1) * ne + e] = a2;
  part[(3 * l + 2) * ne + e] = bw;
  if (l == 0) {
    part[24 * ne + e] = c1;
    part[25 * ne + e] = c2;
    part[26 * ne + e] = (double)n;
  }
}

// The points of the sort, for nodes that sum them themselves
struct SortedPoints {
  const int64_t *off;
  const int32_t *order;
  const double *xi, *eta, *rho;
};

// One thread per node: add the sums of the adjacent elements (ascending), divide.  WALK: without room for the
// elements' sums every node forms those it needs, in the same order (265 us for 0.5 million points).
template <bool WALK>
__global__ void k_points_to_nodes(Box b, const double *__restrict__ part, SortedPoints sp, double *__restrict__ neta,
                                  double *__restrict__ nrho) {
  const int64_t nn = (int64_t)b.NX * b.NY * b.NZ, ne = (int64_t)b.mx * b.my * b.mz;
  for (int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; n < nn; n += (int64_t)gridDim.x * blockDim.x) {
    const int I = (int)(n % b.NX), J = (int)((n / b.NX) % b.NY), K = (int)(n / ((int64_t)b.NX * b.NY));
    int ex[2], lx[2], ey[2], ly[2], ez[2], lz[2];
    const int nx = adjacent(I, b.mx, ex, lx), ny = adjacent(J, b.my, ey, ly), nz = adjacent(K, b.mz, ez, lz);
    double a1 = 0.0, a2 = 0.0, bw = 0.0;
    for (int c = 0; c < nz; c++)
      for (int bb = 0; bb < ny; bb++)
        for (int a = 0; a < nx; a++) {
          const int64_t e = (int64_t)ex[a] + (int64_t)b.mx * ((int64_t)ey[bb] + (int64_t)b.my * ez[c]);
          const bool vert = lx[a] != 1 && ly[bb] != 1 && lz[c] != 1;
          if (WALK) {
            double e1 = 0.0, e2 = 0.0, ew = 0.0;
            for (int64_t k = sp.off[e]; k < sp.off[e + 1]; k++) {
              const int64_t p = sp.order[k];
              const VertexWeight w(lx[a], ly[bb], lz[c], sp.xi + 3 * p);
              add_point(vert ? w.a : 1.0, vert ? w.b : 1.0, sp.eta[p], nrho ? sp.rho[p] : 0.0, e1, e2, ew);
            }
            a1 += e1;
            a2 += e2;
            bw += ew;
            continue;
          }
          const double *s = part + 3 * (vert ? lx[a] / 2 + ly[bb] + 2 * lz[c] : 8) * ne + e;
          a1 += s[0];
          if (nrho) a2 += s[ne];
          bw += s[2 * ne];
        }
    neta[n] = bw != 0.0 ? a1 / bw : 0.0;
    if (nrho) nrho[n] = bw != 0.0 ? a2 / bw : 0.0;
  }
}

// One thread per element: Q1 interpolation of the vertex values at the 27 Gauss points
// (the constants of QuadratureCreateGauss_3pnt_3D, src/quadrature.c:136-167), clipped to the
// range of the element's 27 nodal values.  out: 27 values.
__device__ __forceinline__ void interp_element(const Box &b, int64_t e, const double *__restrict__ nv, double *out) {
  const int ex = (int)(e % b.mx), ey = (int)((e / b.mx) % b.my), ez = (int)(e / ((int64_t)b.mx * b.my));
  const int64_t n0 = 2 * (int64_t)ex + (int64_t)b.NX * (2 * (int64_t)ey + (int64_t)b.NY * 2 * (int64_t)ez);
  double lo = 1.0e32, hi = -1.0e32, v[8];
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const double a = nv[n0 + i + (int64_t)b.NX * (j + (int64_t)b.NY * k)];
        lo = a < lo ? a : lo;
        hi = a > hi ? a : hi;
        if (i != 1 && j != 1 && k != 1) v[(i >> 1) + 2 * (j >> 1) + 4 * (k >> 1)] = a;
      }
  const double s = 0.774596669241483, g[3] = {-s, 0.0, s};
#pragma unroll
  for (int q = 0; q < 27; q++) {
    const double x = g[q % 3], y = g[(q / 3) % 3], z = g[q / 9];
    double r = 0.0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const double w = 0.125 * ((c & 1) ? 1.0 + x : 1.0 - x) * ((c & 2) ? 1.0 + y : 1.0 - y) *
                       ((c & 4) ? 1.0 + z : 1.0 - z);
      r += w * v[c];
    }
    r = r < lo ? lo : r;
    r = r > hi ? hi : r;
    out[q] = r;
  }
}

// One field (grid.y) of 64 elements per wave; their 27 values each are turned in LDS, so that a store
// covers consecutive addresses: 13 us for two fields of 63360 elements, 22 us with one thread per element
// and its stores 216 bytes apart.  With an error or a crowded element (err) the outputs stay as they are.
__global__ __launch_bounds__(64) void k_nodes_to_qp(Box b, const double *__restrict__ neta,
                                                    const double *__restrict__ nrho, double *__restrict__ eta_qp,
                                                    double *__restrict__ rho_qp, const int *__restrict__ err) {
  __shared__ double sh[64 * 27];
  if (*err) return;
  const int64_t ne = (int64_t)b.mx * b.my * b.mz, e0 = (int64_t)blockIdx.x * 64;
  const int lane = threadIdx.x;
  const int n = 27 * (int)min((int64_t)64, ne - e0);
  if (e0 + lane < ne) interp_element(b, e0 + lane, blockIdx.y ? nrho : neta, sh + 27 * lane);
  __syncthreads();
  double *o = (blockIdx.y ? rho_qp : eta_qp) + 27 * e0;
#pragma unroll
  for (int k = lane; k < 27 * 64; k += 64)
    if (k < n) o[k] = sh[k];
}

int pfail(ptq2_ctx *c, int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  c->last = buf;
  return code;
}

// hipMalloc that has the context's spare memory (and, with work, this workspace) given back before it fails
hipError_t take(ptq2_ctx *c, void **p, size_t bytes, bool work) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory && ptq2_internal_give_back(c, work)) {
    (void)hipGetLastError();
    e = hipMalloc(p, bytes);
  }
  return e;
}

// device scratch of one projection call, freed on every return path
struct Scratch {
  static constexpr int CAP = 16;  // a call takes at most 11 buffers
  ptq2_ctx *c;
  void *p[CAP] = {};
  int n = 0;
  bool work = true;  // the context's workspace is not in use yet
  explicit Scratch(ptq2_ctx *c_) : c(c_) {}
  ~Scratch() { drop(0); }
  void drop(int keep) {
    while (n > keep) (void)hipFree(p[--n]);
  }
  template <typename T>
  hipError_t get(T **out, size_t bytes) {
    void *q = nullptr;
    if (n == CAP) {
      *out = nullptr;
      return hipErrorOutOfMemory;
    }
    const hipError_t e = take(c, &q, bytes ? bytes : 1, work);
    if (e == hipSuccess) p[n++] = q;
    *out = (T *)q;
    return e;
  }
};

inline size_t align(size_t n) { return (n + 255) / 256 * 256; }

// the context's point workspace, at least `bytes` long (contents lost); none above the caller's limit
hipError_t grow(ptq2_ctx *c, size_t bytes, size_t limit) {
  if (c->pwork_bytes >= bytes && c->pwork_bytes <= limit) return hipSuccess;
  if (c->pwork) (void)hipFree(c->pwork);
  c->pwork = nullptr;
  c->pwork_bytes = 0;
  const hipError_t e = bytes <= limit ? take(c, &c->pwork, bytes, false) : hipErrorOutOfMemory;
  if (e == hipSuccess) c->pwork_bytes = bytes;
  else c->pwork = nullptr;
  return e;
}

}  // namespace
}  // namespace ptq2

#define PCHK(call)                                                                                    \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess) {                                                                           \
      (void)hipGetLastError();                                                                        \
      return ptq2::pfail(c, e_ == hipErrorOutOfMemory ? PTQ2_ERR_ALLOC : PTQ2_ERR_DEVICE, "%s: %s", #call, \
                         hipGetErrorString(e_));                                                      \
    }                                                                                                 \
  } while (0)

extern "C" int ptq2_project_points_q1(ptq2_ctx *c, int64_t np, const double *xi, const int32_t *wil,
                                      const double *eta_p, const double *rho_p, double *eta_qp, double *rho_qp,
                                      unsigned flags) {
  return ptq2_internal_project_points(c, np, xi, wil, eta_p, rho_p, eta_qp, rho_qp, flags, SIZE_MAX);
}

extern "C" int ptq2_internal_project_points(ptq2_ctx *c, int64_t np, const double *xi, const int32_t *wil,
                                            const double *eta_p, const double *rho_p, double *eta_qp, double *rho_qp,
                                            unsigned flags, size_t max_work) {
  using namespace ptq2;
  if (!c) return PTQ2_ERR_INVALID_ARG;
  if (!c->mesh_ready) return pfail(c, PTQ2_ERR_NOT_SETUP, "MF operator not setup: no mesh");
  if (flags & ~PTQ2_DEVICE) return pfail(c, PTQ2_ERR_INVALID_ARG, "bad flags");
  if (np < 0 || (np > 0 && (!xi || !wil || !eta_p)) || !eta_qp || (!rho_p != !rho_qp))
    return pfail(c, PTQ2_ERR_INVALID_ARG, "null point arrays or outputs (rho_p and rho_qp go together)");
  if (np >= ((int64_t)1 << 31)) return pfail(c, PTQ2_ERR_SIZE, "more than 2^31 - 1 points");
  const Box &b = c->box;
  if (b.i0 || b.j0 || b.k0 || b.NX != 2 * b.mx + 1 || b.NY != 2 * b.my + 1 || b.NZ != 2 * b.mz + 1)
    return pfail(c, PTQ2_ERR_UNSUPPORTED, "point projection needs a single-rank box (no ghost layer)");
  PCHK(hipSetDevice(c->device));
  const bool dev = flags & PTQ2_DEVICE;
  const int64_t ne = c->nel, nn = c->nnodes;
  hipStream_t s = c->stream;
  Scratch S(c);
  const double *dxi = xi, *deta = eta_p, *drho = rho_p;
  const int32_t *dwil = wil;
  double *deq = eta_qp, *drq = rho_qp;
  if (!dev) {
    double *t;
    int32_t *w;
    PCHK(S.get(&t, sizeof(double) * 3 * (size_t)np));
    PCHK(hipMemcpyAsync(t, xi, sizeof(double) * 3 * (size_t)np, hipMemcpyHostToDevice, s));
    dxi = t;
    PCHK(S.get(&w, sizeof(int32_t) * (size_t)np));
    PCHK(hipMemcpyAsync(w, wil, sizeof(int32_t) * (size_t)np, hipMemcpyHostToDevice, s));
    dwil = w;
    PCHK(S.get(&t, sizeof(double) * (size_t)np));
    PCHK(hipMemcpyAsync(t, eta_p, sizeof(double) * (size_t)np, hipMemcpyHostToDevice, s));
    deta = t;
    if (rho_p) {
      PCHK(S.get(&t, sizeof(double) * (size_t)np));
      PCHK(hipMemcpyAsync(t, rho_p, sizeof(double) * (size_t)np, hipMemcpyHostToDevice, s));
      drho = t;
    }
    PCHK(S.get(&deq, sizeof(double) * 27 * (size_t)ne));
    if (rho_qp) PCHK(S.get(&drq, sizeof(double) * 27 * (size_t)ne));
  }
  // Workspace, kept in the context until its next mesh or its end: counters (with the error word), slots,
  // element sums and nodal values; where that does not fit, the error word and the nodal values alone.
  int cap = bucket_slots(np, ne);
  bool sums = true;
  const size_t bcnt = align(sizeof(int32_t) * (size_t)(ne + 1)), bpart = sizeof(double) * 27 * (size_t)ne,
               bnodes = sizeof(double) * (size_t)nn * (drho ? 2 : 1);
  S.work = false;
  int *err = nullptr;
  int32_t *slot = nullptr;
  double *part = nullptr, *neta = nullptr, *nrho = nullptr;
  const auto work = [&] {
    const size_t head = sums ? bcnt : align(sizeof(int)), bslot = align(sizeof(int32_t) * (size_t)ne * (size_t)cap),
                 bsums = sums ? bpart : 0;
    const hipError_t e = grow(c, head + bslot + bsums + bnodes, max_work);
    if (e != hipSuccess) return e;
    char *w = (char *)c->pwork;
    err = (int *)w;
    slot = cap ? (int32_t *)(w + head) : nullptr;
    part = sums ? (double *)(w + head + bslot) : nullptr;
    neta = (double *)(w + head + bslot + bsums);
    nrho = drho ? neta + nn : nullptr;
    return hipMemsetAsync(err, 0, sums ? bcnt : sizeof(int), s);
  };
  const auto without_sums = [&] {
    (void)hipGetLastError();
    if (c->pwork) (void)hipFree(c->pwork);
    c->pwork = nullptr;
    c->pwork_bytes = 0;
    cap = 0;
    sums = false;
    return work();
  };
  hipError_t we = work();
  if (we == hipErrorOutOfMemory) we = without_sums();
  PCHK(we);
  SortedPoints sp{nullptr, nullptr, dxi, deta, drho};
  const auto finish = [&] {
    hipLaunchKernelGGL((sums ? k_points_to_nodes<false> : k_points_to_nodes<true>), dim3(grid_of(nn)), dim3(PTB), 0, s, b,
                       (const double *)part, sp, neta, nrho);
    hipLaunchKernelGGL(k_nodes_to_qp, dim3((unsigned)((ne + 63) / 64), nrho ? 2 : 1), dim3(64), 0, s, b, (const double *)neta,
                       (const double *)nrho, deq, drq, (const int *)err);
  };
  const dim3 sgrid((unsigned)((ne + SUM_ELEMS - 1) / SUM_ELEMS));
  if (np > 0) {
    hipLaunchKernelGGL(k_points_bucket, dim3(grid_of(np)), dim3(PTB), 0, s, np, ne, dxi, dwil, deta, drho, cap,
                       (int32_t *)err + 1, slot, err);
    PCHK(hipGetLastError());
  }
  if (slot) {
    // before the host has seen the checks: only checked points are in a slot, and an error leaves the outputs alone
    hipLaunchKernelGGL(k_points_sums<true>, sgrid, dim3(PTB), 2 * SUM_ELEMS * cap * sizeof(int32_t), s, ne, cap,
                       (const int32_t *)err + 1, (const int32_t *)slot, (const int64_t *)nullptr, (const int32_t *)nullptr,
                       dxi, deta, drho, part);
    finish();
    PCHK(hipGetLastError());
  }
  int bits = 0;
  PCHK(hipMemcpyAsync(&bits, err, sizeof(int), hipMemcpyDeviceToHost, s));
  PCHK(hipStreamSynchronize(s));
  if (bits & PERR_INDEX) return pfail(c, PTQ2_ERR_INVALID_ARG, "point element index outside [0, %lld)", (long long)ne);
  if (bits & PERR_FINITE) return pfail(c, PTQ2_ERR_NONFINITE, "non-finite point coordinate or value");
  if (!slot || (bits & PERR_CROWDED)) {
    // stable bucketing by element
    const int had = S.n;
    int32_t *keys, *order, *iota;
    int64_t *off;
    void *tmp;
    size_t tmp_bytes = 0;
    int end_bit = 1;
    while (end_bit < 31 && ((int64_t)1 << end_bit) < ne) end_bit++;
    // the keys are validated non-negative: sort them as unsigned on the bits that can be set
    const uint32_t *ukin = reinterpret_cast<const uint32_t *>(dwil);
    const auto buffers = [&] {
      hipError_t e = S.get(&keys, sizeof(int32_t) * (size_t)np);
      if (e == hipSuccess) e = S.get(&order, sizeof(int32_t) * (size_t)np);
      if (e == hipSuccess) e = S.get(&iota, sizeof(int32_t) * (size_t)np);
      if (e == hipSuccess) e = S.get(&off, sizeof(int64_t) * (size_t)(ne + 1));
      if (e == hipSuccess && np > 0) {
        e = hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, ukin, reinterpret_cast<uint32_t *>(keys), iota, order,
                                               (int)np, 0, end_bit, s);
        if (e == hipSuccess) e = S.get(&tmp, tmp_bytes);
      }
      return e;
    };
    hipError_t be = buffers();
    if (be == hipErrorOutOfMemory && sums) {
      S.drop(had);
      be = without_sums();
      if (be == hipSuccess) be = buffers();
    }
    PCHK(be);
    if (np > 0) {
      hipLaunchKernelGGL(k_iota, dim3(grid_of(np)), dim3(PTB), 0, s, np, iota);
      PCHK(hipGetLastError());
      PCHK(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, ukin, reinterpret_cast<uint32_t *>(keys), iota, order,
                                              (int)np, 0, end_bit, s));
    }
    hipLaunchKernelGGL(k_bucket_offsets, dim3(grid_of(ne + 1)), dim3(PTB), 0, s, np, ne, (const int32_t *)keys, off);
    PCHK(hipGetLastError());
    sp.off = off;
    sp.order = order;
    if (sums)
      hipLaunchKernelGGL(k_points_sums<false>, sgrid, dim3(PTB), 0, s, ne, 0, (const int32_t *)nullptr,
                         (const int32_t *)nullptr, (const int64_t *)off, (const int32_t *)order, dxi, deta, drho, part);
    PCHK(hipMemsetAsync(err, 0, sizeof(int), s));
    finish();
    PCHK(hipGetLastError());
  }
  if (!dev) {
    PCHK(hipMemcpyAsync(eta_qp, deq, sizeof(double) * 27 * (size_t)ne, hipMemcpyDeviceToHost, s));
    if (rho_qp) PCHK(hipMemcpyAsync(rho_qp, drq, sizeof(double) * 27 * (size_t)ne, hipMemcpyDeviceToHost, s));
  }
  // host outputs, or scratch that is freed on return: wait for the kernels that read it
  if (S.n) PCHK(hipStreamSynchronize(s));
  c->last.clear();
  return PTQ2_OK;
}
