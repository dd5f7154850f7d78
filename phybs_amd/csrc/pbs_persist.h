// pbs_persist.h -- the resident descent kernel (pbs_persist.hip): host-side launch interface.
#pragma once
#include <hip/hip_runtime.h>

#include "pbs_internal.h"
#include "pbs_tiles.h"

namespace pbs {

constexpr int kPersistThreads = 512;
constexpr int kPersistSlots = 8;                          // exchange slots, used in turn
constexpr int kPersistTetsPerThread = 4;                  // at most
constexpr int kPersistOwn = kPersistThreads / 64 * 21;    // owned nodes per workgroup: 21 per wave (3 lanes each)
constexpr int kPersistGhosts = 4 * kPersistThreads / 3;   // ghosts per workgroup: 4 components per thread

// Device copy of a PersistPlan and the exchange buffers.
struct PersistDev {
  int nparts, tet_max, local_max, slot_max;
  const PersistPart *parts;
  const int *ghost;
  const uint4 *lp;
  const unsigned short *run;
  const unsigned long long *mask;
  void *xch;      // kPersistSlots slots of 3N values: positions published after a pass (node-major)
  double *part;   // kPersistSlots slots of (energy, |g|^2) per part
  long xch_bytes; // of xch and part together (part follows xch)
  int *abort;     // set by a workgroup that gave up waiting
  int polls, from; // polls in vain before it does, from pass `from` of the launch on (before: kPolls)
};

template <typename R> struct PersistLaunch {
  static size_t lds_bytes(const PersistDev &d);
  // Most workgroups of the kernel for `material` that the device holds at once (0: not launchable).
  static int max_resident(const PersistDev &d, int material, int device);
  // Runs up to max_passes descent passes from the state in m.ring / m.ctrl / m.hd and leaves it there.
  static hipError_t run(const DevMesh<R> &m, const TileDev &td, const DevParams &p, const PersistDev &d, int max_passes,
                        hipStream_t st);
};

}  // namespace pbs
