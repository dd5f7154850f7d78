// pbs_cg_plan.cpp -- host-side plan of the implicit steps' linear system (see pbs_cg_plan.h).
#include "pbs_cg_plan.h"

#include <algorithm>

namespace pbs {

void build_block_rows(const TilePlan &P, BlockRows &B) {
  B = BlockRows();
  const int N = P.nn;
  std::vector<int> row_off(N + 1, 0), cols, tmp, last(N, -1);  // last: the last row that took a column
  cols.reserve((size_t)N * 16);
  for (int n = 0; n < N; ++n) {
    tmp.assign(1, n);
    last[n] = n;
    for (int e = P.inc_off[n]; e < P.inc_off[n + 1]; ++e) {
      const int *q = &P.tets_new[4 * (size_t)(P.inc[e] >> 2)];
      for (int c = 0; c < 4; ++c)
        if (last[q[c]] != n) {
          last[q[c]] = n;
          tmp.push_back(q[c]);
        }
    }
    std::sort(tmp.begin(), tmp.end());
    cols.insert(cols.end(), tmp.begin(), tmp.end());
    row_off[n + 1] = (int)cols.size();
  }
  B.n = N;
  B.nslice = (N + 63) / 64;
  B.slice_off.assign(B.nslice + 1, 0);
  B.row_len.resize(N);
  for (int n = 0; n < N; ++n) B.row_len[n] = row_off[n + 1] - row_off[n];
  for (int sl = 0; sl < B.nslice; ++sl) {
    int w = 0;
    for (int n = 64 * sl; n < std::min(N, 64 * sl + 64); ++n) w = std::max(w, B.row_len[n]);
    B.slice_off[sl + 1] = B.slice_off[sl] + w;
    B.max_width = std::max(B.max_width, w);
  }
  B.slots = 64L * B.slice_off[B.nslice];
  B.bcol.assign(B.slots, 0);
  B.diag.resize(N);
  for (int n = 0; n < N; ++n) {
    const long g0 = B.slice_off[n >> 6], w = B.slice_off[(n >> 6) + 1] - g0;
    const int lane = n & 63;
    for (long j = 0; j < w; ++j) {
      const bool real = j < B.row_len[n];
      const int c = real ? cols[row_off[n] + j] : n;
      B.bcol[(g0 + j) * 64 + lane] = c;
      if (real && c == n) B.diag[n] = (int)((g0 + j) * 64 + lane);
    }
  }
}

bool build_cg_plan(const BlockRows &B, CgPlan &c) {
  c = CgPlan();
  const int N = B.n;
  if (B.nslice == 0 || B.nslice > kCgSlices || B.max_width > kCgWidth) return false;
  c.vec_blocks = std::min(B.nslice, kVecBlocks);
  c.vec_per = B.nslice / c.vec_blocks;
  c.vec_rem = B.nslice % c.vec_blocks;
  c.per_part = c.vec_blocks > 256 ? 2 : 1;
  c.nparts = (c.vec_blocks + c.per_part - 1) / c.per_part;
  c.lcol.assign(B.slots, 0);
  c.ghost_off.assign(1, 0);
  std::vector<int> local(N, -1), seen;
  for (int g = 0; g < c.nparts; ++g) {
    const int s0 = c.first_slice(g * c.per_part), s1 = c.first_slice(std::min((g + 1) * c.per_part, c.vec_blocks));
    const int n0 = 64 * s0, n1 = std::min(N, 64 * s1);
    c.shares = std::max(c.shares, s1 - s0 <= 2 ? 1 : s1 - s0 <= 4 ? 2 : 4);
    seen.clear();
    for (int n = n0; n < n1; ++n) {
      const long at = B.slice_off[n >> 6];
      for (int j = 0; j < B.row_len[n]; ++j) {
        const int m = B.bcol[(at + j) * 64 + (n & 63)];
        if ((m < n0 || m >= n1) && local[m] < 0) {
          local[m] = 0;
          seen.push_back(m);
        }
      }
    }
    c.ghost_max = std::max(c.ghost_max, (int)seen.size());
    std::sort(seen.begin(), seen.end());
    for (size_t k = 0; k < seen.size(); ++k) local[seen[k]] = n1 - n0 + (int)k;
    for (int sl = s0; sl < s1; ++sl)
      for (long at = 64L * B.slice_off[sl]; at < 64L * B.slice_off[sl + 1]; ++at) {
        const int m = B.bcol[at];  // (a row's padding: its own column; past the last row: any of its own)
        c.lcol[at] = m >= n0 && m < n1 ? (uint16_t)(m - n0) : local[m] >= 0 ? (uint16_t)local[m] : 0;
      }
    for (int m : seen) local[m] = -1;
    c.ghost.insert(c.ghost.end(), seen.begin(), seen.end());
    c.ghost_off.push_back((int)c.ghost.size());
    c.local_max = std::max(c.local_max, n1 - n0 + (int)seen.size());
  }
  return c.ghost_max <= cg_ghosts(c.shares);
}

}  // namespace pbs
