// ptq2_ctx.h -- the context behind the opaque ptq2_ctx handle (internal).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "ptq2_device.h"

struct ptq2_ctx {
  int device = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  bool mesh_ready = false, eta_ready = false;
  ptq2::Box box{};
  int64_t nnodes = 0, nvel = 0, nel = 0, npres = 0, nbricks = 0;
  double *coords = nullptr;
  uint8_t *mask = nullptr;       // followed by box.bdir and dir_idx
  int64_t *dir_idx = nullptr;
  int64_t ndir = 0;
  int64_t ndir_ghost = 0;  // the last of dir_idx: dofs of ghost nodes that no brick's tile holds
  double *eta_bm = nullptr;
  float *fac32 = nullptr;
  bool fac32_valid = false;
  double *geo64 = nullptr;  // FP64 per-point geometry sqrt(w/det) adj(J) (mesh only)
  bool geo64_valid = false;
  float *facb32 = nullptr;  // FP32 full-block factors (w det / eta scale, pressure basis)
  bool facb32_valid = false;
  bool has_state = false;
  uint64_t state = 0;
  // bumped by every mesh set-up and every viscosity upload: a multigrid hierarchy built on this
  // context records it and refuses to run once it has changed (its captured graph holds the
  // device buffers of that mesh, and its coarse levels were derived from that viscosity)
  uint64_t gen = 0;
  int *err = nullptr;
  // output path of the A11 applies: all bricks in one launch, each storing the nodes it owns
  // and its upper-face values into its slot of facebuf (FACEVALS doubles per brick), then a
  // pass adds the face slots into their owners (ptq2::launch_a11_*).  One launch keeps the
  // memory phases of some bricks overlapped with the arithmetic of others, which 8 coloured
  // launches of a few waves per SIMD do not.
  void *facebuf = nullptr;
  // Slots of A12 and the diagonal, which need none to run (8 coloured launches): apart from facebuf, which an
  // apply on another stream may be using, and handed from call to call by an event.
  void *facebuf2 = nullptr;  // beside eta_bm, or in spare
  hipEvent_t face2_ev = nullptr;
  bool face2_used = false;             // since the mesh set-up
  hipStream_t face2_stream = nullptr;  // of the last use
  // What a large mesh runs faster with but not only with: the slots facebuf2 and the coordinate tiles box.xtile.
  // Given back when an allocation of this context (or of a hierarchy on it) finds no memory.
  void *spare = nullptr;
  size_t spare_bytes = 0;
  bool spare_held = false;  // a graph that a caller captured may hold its addresses
  // u with the Dirichlet values inserted, for the residual (allocated on first use)
  double *ures = nullptr;
  size_t ures_bytes = 0;
  // workspace of the point projection (allocated on first use)
  void *pwork = nullptr;
  size_t pwork_bytes = 0;
  // stream ordering of the batched apply (created on first use)
  hipEvent_t ev = nullptr;
  // staging for host-pointer calls
  void *su = nullptr, *sy = nullptr;
  size_t su_bytes = 0, sy_bytes = 0;
  double *sp = nullptr, *syp = nullptr;
  size_t sp_bytes = 0, syp_bytes = 0;
  std::string last;
};


// (re)build the FP32 geometric factors of the smoother operator if stale; with block,
// also those of the FP32 full block
int ptq2_internal_build_fac32(ptq2_ctx *c, bool block = false);
// Gives spare memory (and, with work, the projection's workspace) back; whether there was any.  Waits for the device.
bool ptq2_internal_give_back(ptq2_ctx *c, bool work = true);
// whether work on s is being captured into a graph
bool ptq2_internal_capturing(hipStream_t s);
// the tile buffer of the uncoloured output path if this mesh uses it (allocated on first
// use), else nullptr; *rc receives an allocation error
void *ptq2_internal_facebuf(ptq2_ctx *c, int *rc);
// ptq2_project_points_q1 with at most max_work bytes of workspace kept in the context (tests of the path that a
// device without room takes)
extern "C" int ptq2_internal_project_points(ptq2_ctx *c, int64_t np, const double *xi, const int32_t *wil,
                                            const double *eta_p, const double *rho_p, double *eta_qp, double *rho_qp,
                                            unsigned flags, size_t max_work);
