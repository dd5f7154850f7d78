// pbs_tiles.h -- host-side partition of a tet mesh for the tiled descent kernels.
#pragma once
#include <stdint.h>

#include <string>
#include <vector>

namespace pbs {

// Nodes are renumbered in Morton order and tets sorted by their smallest new node id.  Tile b
// owns the nodes [own_start, own_start + own_cnt) and the tets whose smallest node it owns --
// a contiguous tet range [tet_start, tet_start + tet_cnt) -- so every tet is evaluated once.
// Tiles are cut so that each holds at most tile_tets tets, 1024 owned nodes and, unless one
// node's tets alone exceed it, max(64, tile_tets / 2) local nodes.  A tile's tets also reach "halo"
// nodes owned by later tiles; the tile writes one partial force per owned and per halo node,
// and the node pass adds a node's partials in tile order.  Halo partial slots are numbered by
// owner node, so each node's partials are contiguous and the node pass reads them coalesced.
//
// Inside a tile, node i (local id: owned nodes first, then halo nodes) receives the corner
// contributions run [off[i], off[i+1]) of the tile's contribution array, ordered by tet, then
// corner.  Each tet carries its corners' local node ids and the position of each corner in that
// array, so the tet pass writes every corner force straight into its slot and the gather sums
// contiguous runs.
struct TileInfo {
  int own_start, own_cnt;  // owned nodes
  int halo_off, halo_cnt;  // halo node ids: halo[halo_off .. +halo_cnt); partial slots likewise
  int tet_start, tet_cnt;  // owned tets (solver order)
  int off_start;           // run offsets: tile_off[off_start .. off_start + own_cnt + halo_cnt]
  int inst;                // mesh instance (batched solvers; 0 otherwise)
};

struct TilePlan {
  int nn = 0, nt = 0;
  // instances (independent meshes of a batched solver) own contiguous node, tet and tile ranges
  int ninst = 1;
  std::vector<int> inst_node_off, inst_tet_off, inst_tile_off;
  int tile_tets = 0, ntiles = 0;
  std::vector<int> inst_tile_tets;  // per instance: its tile size
  int lcap = 0;                     // max local nodes (owned + halo) over tiles
  int tcap = 0;                     // max tets over tiles
  long halo_total = 0;              // sum of halo counts = number of halo partial slots
  std::vector<int> perm, iperm;     // node: new -> old, old -> new
  std::vector<int> tperm, itperm;   // tet:  new -> old, old -> new
  std::vector<int> tets_new;        // 4 per tet, new order, new node ids
  std::vector<int> inc_off, inc;    // per new node: 4*new_tet + corner, in ascending original tet id
  std::vector<TileInfo> tiles;
  std::vector<int> halo;            // new node ids
  std::vector<uint16_t> tile_off;   // per tile: local node count + 1 run offsets
  std::vector<uint32_t> tet_lp;     // 4 words per tet: local ids (c0 | c1 << 16, c2 | c3 << 16),
                                    // contribution positions (likewise)
  std::vector<int> bnd_off;         // per node: its halo partial slots [bnd_off[n], bnd_off[n+1]), tile order
  std::vector<int> halo_slot;       // per halo entry (tile, halo node): its partial slot
};

// Builds the plan.  rest: 3N AoS; tets: 4T.  tile_tets: max tets per tile (1 .. 16383).
// Returns false (with msg) if a tile exceeds the 16-bit local index limits.
bool build_tile_plan(int nn, const float *rest, int nt, const int *tets, int tile_tets, TilePlan &plan,
                     std::string &msg);
// Batched: ninst meshes, instance i owning nodes [node_off[i], node_off[i+1]) and tets
// [tet_off[i], tet_off[i+1]) of the concatenated arrays (tets hold global node ids inside their
// instance's range).  Each instance is planned on its own with its tile size inst_tile_tets[i];
// the plans are concatenated (plan.tile_tets = the largest of them).
bool build_batch_plan(int ninst, const int *node_off, const int *tet_off, const float *rest, const int *tets,
                      const int *inst_tile_tets, TilePlan &plan, std::string &msg);
// The same with one tile size for every instance.
bool build_batch_plan(int ninst, const int *node_off, const int *tet_off, const float *rest, const int *tets,
                      int tile_tets, TilePlan &plan, std::string &msg);

// Partition for the resident descent kernel (pbs_persist.hip): one workgroup per part, a part owning
// a contiguous node run and evaluating every tet that touches an owned node (tets across parts are
// evaluated by each of them, so that no forces have to be exchanged, only positions).  A part's
// local nodes are its owned nodes, then the other corners of its tets (ghosts, ascending).  An
// owned node's contributions form one run, ordered as the tile pass adds them: its own tile's
// tets, then those of the other tiles in tile order, each tile's in (tet, corner) order; bit j of
// its mask is set where entry j ends one tile's partial sum.
struct PersistPart {
  int own_start, own_cnt;
  int ghost_off, ghost_cnt;  // ghost[ghost_off ..)
  int tet_off, tet_cnt;      // tet[tet_off ..), lp likewise
  int run_off;               // run[run_off .. run_off + own_cnt], mask[run_off ..)
  int slots;                 // contributions of the owned nodes
};
struct PersistPlan {
  std::vector<PersistPart> parts;
  std::vector<int> ghost;       // solver node ids
  std::vector<int> tet;         // solver tet ids
  std::vector<uint32_t> lp;     // 4 words per entry as TilePlan::tet_lp; corners of ghosts get the slots
                                // `slots` + (entry & 63), which nothing reads; bit 31 of the third word:
                                // the part owns the tet's smallest node (it counts the tet's energy)
  std::vector<uint16_t> run;    // per part own_cnt + 1 run offsets
  std::vector<uint64_t> mask;   // per entry of run
  int own_max = 0, local_max = 0, ghost_max = 0, tet_max = 0, slot_max = 0;
};
// Builds the partition of a single mesh into at most max_parts parts of about nodes_per_part nodes
// or more.  Returns false where a node has more than 64 incident tets.
bool build_persist_plan(const TilePlan &P, int max_parts, int nodes_per_part, PersistPlan &Q);

}  // namespace pbs
