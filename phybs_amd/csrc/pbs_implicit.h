// pbs_implicit.h -- backward-Euler step (the reference's GPU implicit path): per-node assembly
// of the global stiffness matrix and right-hand side, and a Jacobi-preconditioned conjugate-
// gradient solve, all on the device.  Kernels in pbs_implicit.hip, host side in pbs_implicit.cpp.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "pbs_cg_plan.h"
#include "pbs_internal.h"

namespace pbs {

// Matrix layout: 3x3 blocks, one block row per node (solver order), stored as SELL-64: rows are
// grouped in slices of 64 (one wavefront), a slice is as wide as its longest row, and slot j of
// the slice's row l sits at (slice_off[s] + j) * 64 + l; block values are spread over 9
// consecutive slot groups so that each of the 9 loads of a wavefront is one contiguous 256-byte
// (FP32) access.  Padding slots have column = the row itself and zero values.
struct IeCtrl {
  double rz, pAp, alpha, beta, bb, rz0;  // bb = b.D^-1.b
  int k, done, converged, indefinite;
};

struct IeDev {
  int n, nslice, maxit, scalar;    // scalar: one value per slot (block = value x identity)
  // vector passes: entries per group (64, or a slice's 192), groups per block, blocks with one more
  int vec_unit, vec_per, vec_rem, vec_blocks;
  double tol2;                     // (relative residual tolerance)^2
  const int *slice_off;            // nslice + 1, in slot groups of 64
  const int *row_len;              // N
  const int *bcol;                 // slots
  const int *diag_slot;            // N: slot index of each row's diagonal block
  void *A;                         // 9 x slots values of the solver's real type
  double *b, *x, *z, *p, *Ap, *dinv;  // 3N, node-major (x, y, z of a node together)
  double *part_rz, *part_pap;      // partial sums per block: r.z; p.Ap (at the start b.D^-1.b)
  IeCtrl *ctrl;                    // 2: written in turn within an iteration, [0] at its end
};

// Constants of one assembly (scales of the system matrix, fixed-node spring, damping).
struct IeAsm {
  float h, alpha, beta;  // time step, mass and stiffness damping coefficients
  int raw;               // 1: store K itself (no scaling, no mass), skip the right-hand side
  int warm;              // 1: start the solve from the current velocities, 0: from zero
  int has_ext;
};

// Sets the split of the vector passes for the launches alone: blocks of at least 1024 entries (the
// resident solver's plan has whole slices per block, at most 4).
void ie_vec_split(IeDev &d);

// The resident CG (k_cg): partition (pbs_cg_plan.h) and exchange buffers.
struct CgDev {
  int nparts, per_part;           // workgroups (0: not used), vector blocks of each
  int shares;                     // shares of a slice that one wave multiplies (1, 2 or 4)
  int local_max;                  // rows and ghosts of a workgroup, at most
  const int *ghost_off, *ghost;   // per workgroup: node ids of the columns it does not own
  const unsigned short *lcol;     // per slot: local column (own rows, then ghosts)
  double *z, *pap, *rz;           // 2 slots each: 3N values; partials per vector block
  long xch_bytes;                 // of the three together (z first)
  int *abort;                     // set by a workgroup that gave up waiting
  int polls, from;                // polls in vain before it does, from exchange `from` on (before: kPolls)
};

template <typename R> struct IeLaunch {
  // max_width: the widest slice (slots per row)
  static void assemble(const DevMesh<R> &m, const TileDev &td, const DevParams &p, const IeDev &d, const IeAsm &a,
                       int max_width, hipStream_t st);
  static void start(const IeDev &d, hipStream_t st);
  // per-tet 12 x 12 stiffness of the solver tets ids[0 .. num) at positions x (node-major), FP32 out
  static void tet_stiffness(const DevMesh<R> &m, const DevParams &p, const float *inst_mu, const float *inst_lam,
                            const R *x, int num, const int *ids, float *out, hipStream_t st);
  // one CG iteration = dir, spmv, res, each a kernel; e0, e1 (optional): events recording the start
  // and end of the kernel's own dispatch
  static void dir(const IeDev &d, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
  static void spmv(const IeDev &d, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
  static void res(const IeDev &d, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
  // the whole loop after `start` as one cooperative launch, which keeps the start vector in d.p; whether
  // the device can hold it
  static hipError_t resident(const IeDev &d, const CgDev &c, hipStream_t st);
  static bool resident_fits(const CgDev &c, int scalar, int device);
  static void finish(const DevMesh<R> &m, const DevParams &p, float h, const IeDev &d, hipStream_t st);
  // projective dynamics: global matrix, momentum term + iterate start, local step, velocity update
  static void pd_matrix(const DevMesh<R> &m, const DevParams &p, float stiffness, const IeDev &d, hipStream_t st);
  static void pd_begin(const DevMesh<R> &m, const DevParams &p, const IeDev &d, double *srhs, int has_ext,
                       hipStream_t st);
  // inc_pos[4 t + corner] = position of (t, corner) in its node's incidence run
  static void pd_local(const DevMesh<R> &m, const DevParams &p, float stiffness, const int *inc_pos, const double *pos,
                       const double *srhs, double *out, hipStream_t st);
  static void pd_finish(const DevMesh<R> &m, const DevParams &p, float damping, const IeDev &d, hipStream_t st);
};

// Captured CG iterations for one matrix.
struct CgGraphs {
  hipGraphExec_t graph = nullptr;
  double key[2] = {0, 0};  // tol2, maxit the graph was built with
};

struct ImplicitState {
  BlockRows rows;                                   // (kept for the stiffness export)
  IeDev dev{};                                      // backward Euler: 3x3 blocks
  IeDev pd{};                                       // projective dynamics: same layout and vectors, scalar values
  double *pd_s = nullptr;                           // projective dynamics: momentum term (3N)
  // The PD matrix depends only on the rest shape, the masses, the stiffness and the time step: it is
  // built once per (stiffness, h) with its own Jacobi diagonal and reused by later steps.
  bool pd_built = false;
  float pd_stiffness = 0.0f;
  double pd_h = 0.0;
  int *pd_inc_pos = nullptr;                        // projective dynamics: incidence slot of each (tet, corner)
  CgGraphs cg_ie, cg_pd;
  CgDev cg{};                                       // resident solver
  bool cg_fits[2] = {false, false};                 // for 3x3 blocks; for scalar values
  std::vector<hipEvent_t> ev;                       // timing events of the timed replays
  std::vector<void *> allocs;
};

void implicit_release(ImplicitState *S);
void implicit_params_changed(ImplicitState *S);

}  // namespace pbs
