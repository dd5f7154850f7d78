// persist_check.cpp -- CPU-only checks of the resident descent loop's partition
// (build_persist_plan, pbs_tiles.cpp), built with g++ from the planner alone, also under
// AddressSanitizer / UndefinedBehaviorSanitizer.
//
// For every plan: the parts own all nodes once; a part's list holds exactly the tets that touch its
// nodes, each tet's energy is counted by one part; every local id and slot lies inside the sizes
// the kernel allocates; ghosts are the other corners; and, with random FP32 corner values, a node's
// sum over its masked run is bitwise the tile pass's (each tile's run summed from zero in order,
// the owner's partial first, then the halo partials in slot order).
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include "pbs_tiles.h"

#define CHECK(c)                                                             \
  do {                                                                       \
    if (!(c)) {                                                              \
      std::fprintf(stderr, "FAIL line %d: %s (%s)\n", __LINE__, #c, g_name); \
      std::exit(1);                                                          \
    }                                                                        \
  } while (0)
static const char *g_name = "";

static void bar(int nx, int ny, int nz, std::vector<float> &rest, std::vector<int> &tets, unsigned seed) {
  std::mt19937 rng(seed);
  std::uniform_real_distribution<float> U(-0.004f, 0.004f);
  for (int k = 0; k <= nz; ++k)
    for (int j = 0; j <= ny; ++j)
      for (int i = 0; i <= nx; ++i)
        for (int v : {i, j, k}) rest.push_back(0.05f * v + U(rng));
  const int s[3] = {1, nx + 1, (nx + 1) * (ny + 1)};
  static const int P[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  for (int k = 0; k < nz; ++k)
    for (int j = 0; j < ny; ++j)
      for (int i = 0; i < nx; ++i)
        for (auto &p : P) {
          const int a = i + s[1] * j + s[2] * k;
          for (int v : {a, a + s[p[0]], a + s[p[0]] + s[p[1]], a + s[0] + s[1] + s[2]}) tets.push_back(v);
        }
}

static void check(const char *name, const std::vector<float> &rest, const std::vector<int> &tets, int tile, int parts,
                  int per) {
  g_name = name;
  const int N = (int)rest.size() / 3, Tn = (int)tets.size() / 4;
  pbs::TilePlan P;
  std::string msg;
  CHECK(pbs::build_tile_plan(N, rest.data(), Tn, tets.data(), tile, P, msg));
  pbs::PersistPlan Q;
  CHECK(pbs::build_persist_plan(P, parts, per, Q));
  CHECK((int)Q.parts.size() >= 1 && (int)Q.parts.size() <= parts);
  std::mt19937 rng(7);
  std::uniform_real_distribution<float> U(-1.0f, 1.0f);
  std::vector<float> val(4 * (size_t)Tn);
  for (auto &v : val) v = U(rng);
  // the tile pass's sums
  std::vector<float> own(N), halo(P.halo_total);
  for (const auto &ti : P.tiles) {
    std::vector<float> rec(4 * (size_t)ti.tet_cnt);
    for (int s = 0; s < ti.tet_cnt; ++s) {
      const uint32_t *w = &P.tet_lp[4 * (size_t)(ti.tet_start + s)];
      const int q[4] = {(int)(w[2] & 0xffff), (int)(w[2] >> 16), (int)(w[3] & 0xffff), (int)(w[3] >> 16)};
      for (int c = 0; c < 4; ++c) rec[q[c]] = val[4 * (size_t)(ti.tet_start + s) + c];
    }
    for (int l = 0; l < ti.own_cnt + ti.halo_cnt; ++l) {
      float a = 0.0f;
      for (int j = P.tile_off[ti.off_start + l]; j < P.tile_off[ti.off_start + l + 1]; ++j) a += rec[j];
      if (l < ti.own_cnt) own[ti.own_start + l] = a;
      else halo[P.halo_slot[ti.halo_off + l - ti.own_cnt]] = a;
    }
  }
  std::vector<int> node_seen(N, 0), counted(Tn, 0);
  int next = 0;
  for (const auto &p : Q.parts) {
    CHECK(p.own_start == next && p.own_cnt >= 0);
    next += p.own_cnt;
    CHECK(p.own_cnt <= Q.own_max && p.ghost_cnt <= Q.ghost_max && p.own_cnt + p.ghost_cnt <= Q.local_max);
    CHECK(p.tet_cnt <= Q.tet_max && p.slots + 64 <= Q.slot_max);
    const int n1 = p.own_start + p.own_cnt;
    std::vector<float> rec(Q.slot_max, 1e30f);
    std::vector<int> touched(Tn, 0), ghost_used(p.ghost_cnt, 0), written(p.slots, 0);
    for (int k = 0; k < p.tet_cnt; ++k) {
      const int t = Q.tet[p.tet_off + k];
      CHECK(t >= 0 && t < Tn && !touched[t]);
      touched[t] = 1;
      const uint32_t *w = &Q.lp[4 * (size_t)(p.tet_off + k)];
      if (w[2] >> 31) ++counted[t];
      const int l[4] = {(int)(w[0] & 0xffff), (int)(w[0] >> 16), (int)(w[1] & 0xffff), (int)(w[1] >> 16)};
      const uint32_t w2 = w[2] & 0x7fffffffu;
      const int q[4] = {(int)(w2 & 0xffff), (int)(w2 >> 16), (int)(w[3] & 0xffff), (int)(w[3] >> 16)};
      for (int c = 0; c < 4; ++c) {
        CHECK(l[c] < p.own_cnt + p.ghost_cnt && q[c] < Q.slot_max);
        const int n = P.tets_new[4 * (size_t)t + c];
        if (l[c] < p.own_cnt) {
          CHECK(n == p.own_start + l[c] && q[c] < p.slots && !written[q[c]]);
          written[q[c]] = 1;
        } else {
          CHECK(n == Q.ghost[p.ghost_off + l[c] - p.own_cnt] && (n < p.own_start || n >= n1) && q[c] >= p.slots);
          ghost_used[l[c] - p.own_cnt] = 1;
        }
        rec[q[c]] = val[4 * (size_t)t + c];
      }
    }
    for (int t = 0; t < Tn; ++t) {
      bool touches = false;
      for (int c = 0; c < 4; ++c) {
        const int n = P.tets_new[4 * (size_t)t + c];
        touches |= n >= p.own_start && n < n1;
      }
      CHECK(touches == (touched[t] != 0));
    }
    for (int u : ghost_used) CHECK(u);
    for (int u : written) CHECK(u);
    CHECK(Q.run[p.run_off] == 0 && Q.run[p.run_off + p.own_cnt] == p.slots);
    for (int i = 0; i < p.own_cnt; ++i) {
      const int n = p.own_start + i, r0 = Q.run[p.run_off + i], len = Q.run[p.run_off + i + 1] - r0;
      CHECK(len >= 0 && len <= 64);
      ++node_seen[n];
      float f = 0.0f, a = 0.0f;
      for (int j = 0; j < len; ++j) {
        a += rec[r0 + j];
        if ((Q.mask[p.run_off + i] >> j) & 1) {
          f += a;
          a = 0.0f;
        }
      }
      CHECK(a == 0.0f);
      float ref = own[n];
      for (int e = P.bnd_off[n]; e < P.bnd_off[n + 1]; ++e) ref += halo[e];
      CHECK(f == ref);
    }
  }
  CHECK(next == N);
  for (int n = 0; n < N; ++n) CHECK(node_seen[n] == 1);
  for (int t = 0; t < Tn; ++t) CHECK(counted[t] == 1);
  std::printf("%s: %zu parts, own %d ghosts %d tets %d slots %d\n", name, Q.parts.size(), Q.own_max, Q.ghost_max, Q.tet_max,
              Q.slot_max);
}

int main() {
  static const int dims[][3] = {{1, 1, 1}, {2, 3, 5}, {4, 4, 16}, {7, 5, 31}, {12, 12, 50}};
  for (auto &d : dims)
    for (int tile : {64, 256})
      for (int parts : {1, 7, 256}) {
        std::vector<float> rest;
        std::vector<int> tets;
        bar(d[0], d[1], d[2], rest, tets, 3);
        // one node no tet touches, and node ids in a random order
        for (float v : {0.3f, 0.2f, 0.1f}) rest.push_back(v);
        const int N = (int)rest.size() / 3;
        std::vector<int> perm(N);
        for (int i = 0; i < N; ++i) perm[i] = i;
        std::mt19937 rng(5);
        for (int i = N - 1; i > 0; --i) std::swap(perm[i], perm[rng() % (i + 1)]);
        std::vector<float> r2(rest.size());
        for (int i = 0; i < N; ++i)
          for (int k = 0; k < 3; ++k) r2[3 * (size_t)perm[i] + k] = rest[3 * (size_t)i + k];
        for (int &v : tets) v = perm[v];
        const std::string name = std::to_string(d[0]) + "x" + std::to_string(d[1]) + "x" + std::to_string(d[2]) + " tile " +
                                 std::to_string(tile) + " parts " + std::to_string(parts);
        if (parts == 1 && N > 5000) continue;  // slots beyond 15 bits: refused, see below
        check(name.c_str(), r2, tets, tile, parts, 32);
      }
  {  // what cannot be held is refused
    std::vector<float> rest;
    std::vector<int> tets;
    bar(12, 12, 50, rest, tets, 3);
    pbs::TilePlan P;
    pbs::PersistPlan Q;
    std::string msg;
    g_name = "refusals";
    CHECK(pbs::build_tile_plan((int)rest.size() / 3, rest.data(), (int)tets.size() / 4, tets.data(), 64, P, msg));
    CHECK(!pbs::build_persist_plan(P, 1, 32, Q));
  }
  std::printf("persist_check: all passed\n");
  return 0;
}
