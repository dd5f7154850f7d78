// cg_plan_check.cpp -- CPU-only checks of the resident CG's partition (build_block_rows, build_cg_plan,
// pbs_cg_plan.cpp), built with g++, also under AddressSanitizer / UndefinedBehaviorSanitizer.
//
// For every plan, what a workgroup of the kernel does with it is replayed: its own rows' entries, and
// those of the ghosts that its threads read (cg_ghost_entries components each), are the ones written
// to the local vector; every column of every own row must then be found there.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include "pbs_cg_plan.h"

#define CHECK(c)                                                             \
  do {                                                                       \
    if (!(c)) {                                                              \
      std::fprintf(stderr, "FAIL line %d: %s (%s)\n", __LINE__, #c, g_name); \
      std::exit(1);                                                          \
    }                                                                        \
  } while (0)
static const char *g_name = "";

// Bar of cells with edges e[0], e[1], e[2].
static void bar(const int *d, const double *e, std::vector<float> &rest, std::vector<int> &tets) {
  for (int k = 0; k <= d[2]; ++k)
    for (int j = 0; j <= d[1]; ++j)
      for (int i = 0; i <= d[0]; ++i)
        for (double v : {i * e[0], j * e[1], k * e[2]}) rest.push_back((float)(0.02 * v));
  const int s[3] = {1, d[0] + 1, (d[0] + 1) * (d[1] + 1)};
  static const int P[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  for (int k = 0; k < d[2]; ++k)
    for (int j = 0; j < d[1]; ++j)
      for (int i = 0; i < d[0]; ++i)
        for (auto &p : P) {
          const int a = i + s[1] * j + s[2] * k;
          for (int v : {a, a + s[p[0]], a + s[p[0]] + s[p[1]], a + s[0] + s[1] + s[2]}) tets.push_back(v);
        }
}

static bool plan(const std::vector<float> &rest, const std::vector<int> &tets, pbs::BlockRows &B, pbs::CgPlan &c) {
  pbs::TilePlan P;
  std::string msg;
  CHECK(pbs::build_tile_plan((int)rest.size() / 3, rest.data(), (int)tets.size() / 4, tets.data(), 64, P, msg));
  pbs::build_block_rows(P, B);
  // the rows: each node's columns ascending, without repeats, itself among them and marked
  for (int n = 0; n < B.n; ++n) {
    const long at = B.slice_off[n >> 6];
    std::vector<int> want{n};
    for (int e = P.inc_off[n]; e < P.inc_off[n + 1]; ++e)
      for (int k = 0; k < 4; ++k) want.push_back(P.tets_new[4 * (size_t)(P.inc[e] >> 2) + k]);
    std::sort(want.begin(), want.end());
    want.erase(std::unique(want.begin(), want.end()), want.end());
    CHECK((int)want.size() == B.row_len[n] && B.row_len[n] <= B.slice_off[(n >> 6) + 1] - at);
    for (int j = 0; j < B.row_len[n]; ++j) CHECK(B.bcol[(at + j) * 64 + (n & 63)] == want[j]);
    CHECK(B.bcol[B.diag[n]] == n);
  }
  return pbs::build_cg_plan(B, c);
}

static void check(const char *name, const std::vector<float> &rest, const std::vector<int> &tets, int at_least) {
  g_name = name;
  pbs::BlockRows B;
  pbs::CgPlan c;
  CHECK(plan(rest, tets, B, c));
  CHECK(c.nparts <= 256 && c.vec_blocks <= pbs::kVecBlocks && c.first_slice(c.vec_blocks) == B.nslice);
  CHECK((int)c.ghost_off.size() == c.nparts + 1);
  int most = 0;
  for (int g = 0; g < c.nparts; ++g) {
    const int s0 = c.first_slice(g * c.per_part), s1 = c.first_slice(std::min((g + 1) * c.per_part, c.vec_blocks));
    const int n0 = 64 * s0, own = std::min(B.n, 64 * s1) - n0, gcnt = c.ghost_off[g + 1] - c.ghost_off[g];
    const int *ghost = c.ghost.data() + c.ghost_off[g];
    CHECK(s1 - s0 <= 2 * c.shares && own + gcnt <= c.local_max);
    most = std::max(most, gcnt);
    // the node whose direction each entry of the local vector holds, as the threads write them
    std::vector<int> holds(3 * (size_t)c.local_max, -1);
    for (int i = 0; i < 3 * own; ++i) holds[i] = 3 * n0 + i;
    for (int tid = 0; tid < pbs::kCgThreads; ++tid)
      for (int u = 0; u < pbs::cg_ghost_entries(c.shares); ++u) {
        const int e = tid + u * pbs::kCgThreads;
        if (e < 3 * gcnt) holds[3 * own + e] = 3 * ghost[e / 3] + e % 3;
      }
    for (int sl = s0; sl < s1; ++sl)
      for (long at = 64L * B.slice_off[sl]; at < 64L * B.slice_off[sl + 1]; ++at) {
        CHECK(c.lcol[at] < own + gcnt);
        if (64 * sl + (int)(at & 63) >= B.n) continue;
        for (int k = 0; k < 3; ++k) CHECK(holds[3 * (size_t)c.lcol[at] + k] == 3 * B.bcol[at] + k);
      }
  }
  CHECK(most == c.ghost_max && most >= at_least);
  std::printf("%s: %d nodes, %d workgroups, %d shares, at most %d ghosts\n", name, B.n, c.nparts, c.shares, most);
}

int main(int argc, char **argv) {
  const bool quick = argc > 1;  // under the sanitizers: the small ones and one large
  // dimensions, cell edges, ghosts that the largest workgroup has at least
  struct Case {
    int d[3];
    double e[3];
    int ghosts;
  };
  static const Case cases[] = {{{1, 1, 1}, {1, 1, 1}, 0},      {{2, 4, 12}, {1, 1, 1}, 1},    {{16, 16, 60}, {1, 1, 10}, 200},
                               {{30, 30, 30}, {1, 1, 16}, 300}, {{60, 60, 33}, {1, 1, 10}, 1195}, {{45, 45, 30}, {1, 1, 16}, 600},
                               {{33, 29, 127}, {1, 1, 1}, 500}, {{50, 50, 49}, {1, 1, 5}, 1195},  {{50, 50, 49}, {1, 1, 20}, 1195},
                               {{100, 100, 11}, {1, 1, 10}, 1195}, {{16, 16, 450}, {1, 1, 0.05}, 1195}, {{180, 180, 3}, {1, 1, 16}, 1195}};
  int n = 0;
  for (auto &k : cases) {
    if (quick && ++n > 5) break;
    std::vector<float> rest;
    std::vector<int> tets;
    bar(k.d, k.e, rest, tets);
    const std::string name = std::to_string(k.d[0]) + "x" + std::to_string(k.d[1]) + "x" + std::to_string(k.d[2]) + " of " +
                             std::to_string(k.e[0]) + " " + std::to_string(k.e[1]) + " " + std::to_string(k.e[2]);
    check(name.c_str(), rest, tets, k.ghosts);
  }
  // what cannot be held is refused: more slices, wider rows, more ghosts (nodes joined at random)
  g_name = "refusals";
  auto refused = [](int nodes, int tn, int hub) {
    std::mt19937 rng(11);
    std::vector<float> rest;
    std::vector<int> tets;
    for (int i = 0; i < 3 * nodes; ++i) rest.push_back((float)(rng() % 10007) * 1e-3f);
    for (int t = 0; t < tn; ++t) {
      int v[4];
      do {
        for (int &x : v) x = (int)(rng() % nodes);
        if (t < hub) v[0] = 0;
      } while (v[0] == v[1] || v[0] == v[2] || v[0] == v[3] || v[1] == v[2] || v[1] == v[3] || v[2] == v[3]);
      tets.insert(tets.end(), v, v + 4);
    }
    pbs::BlockRows B;
    pbs::CgPlan c;
    return !plan(rest, tets, B, c);
  };
  CHECK(refused(64 * pbs::kCgSlices + 1, 4, 0));
  CHECK(!refused(64 * pbs::kCgSlices, 4, 0));
  CHECK(refused(100, 20, 20));
  CHECK(refused(64 * pbs::kCgSlices, 16 * pbs::kCgSlices, 0));
  std::printf("cg_plan_check: all passed\n");
  return 0;
}
