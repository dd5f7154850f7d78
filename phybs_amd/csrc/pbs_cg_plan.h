// pbs_cg_plan.h -- host-side plan of the implicit steps' linear system (pbs_implicit.h): the block rows
// in SELL-64 form and the resident solver's partition of them.
#pragma once
#include <cstdint>
#include <vector>

#include "pbs_tiles.h"

namespace pbs {

constexpr int kVecBlocks = 512;  // blocks of a vector pass, at most

// Block rows in solver order: a node's columns are the nodes sharing a tet with it, ascending, itself
// included (the block pattern of allocateGlobalStiffnessMatrix, IsotropicMaterial.cpp:554-644).
struct BlockRows {
  int n = 0, nslice = 0, max_width = 0;  // max_width: the widest slice (slots per row)
  long slots = 0;
  std::vector<int> slice_off, row_len, bcol, diag;  // as IeDev holds them
};
void build_block_rows(const TilePlan &P, BlockRows &B);

// The resident CG (k_cg): a workgroup owns one or two of the vector passes' blocks (whole slices, at
// most 4) and their slices' rows; the columns it does not own are its ghosts.
constexpr int kCgThreads = 512;
constexpr int kCgSlices = 4 * kVecBlocks, kCgWidth = 28;  // at most: slices, slots of a slice
// Ghost components (x, y, z of each ghost) that a thread reads, and the ghosts a workgroup may have.
// Workgroups of 8 slices (4 shares per wave) have the most: 10:1 cells up to 1308.  An eighth component
// costs 8 registers, which the kernels of 3x3 blocks (at most 2 shares) would spill.
constexpr int cg_ghost_entries(int shares) { return shares == 4 ? 8 : 7; }
constexpr int cg_ghosts(int shares) { return cg_ghost_entries(shares) * kCgThreads / 3; }

struct CgPlan {
  int vec_blocks = 0, vec_per = 0, vec_rem = 0;  // slices per block, blocks with one more
  int nparts = 0, per_part = 0;    // workgroups, vector blocks of each
  int shares = 0, local_max = 0, ghost_max = 0;  // as CgDev; ghosts of a workgroup, at most
  std::vector<int> ghost_off, ghost;  // per workgroup: its ghosts, ascending
  std::vector<uint16_t> lcol;         // per slot: local column (own rows, then ghosts)
  int first_slice(int b) const { return b * vec_per + (b < vec_rem ? b : vec_rem); }
};
// False where the system has more slices than 256 workgroups of 8 waves hold (131,072 rows), wider rows
// than the registers, or a workgroup more ghosts than its threads read at once.
bool build_cg_plan(const BlockRows &B, CgPlan &c);

}  // namespace pbs
