// pbs_kernels.hip -- HIP kernels of the descent solver for gfx950 (CDNA4, wave64).
//
// One descent pass = k_tile (each tet once, per tile: force, energy, Hessian diagonal on refresh
// passes, gathered per node in LDS) -> k_node (owned + halo partials, Jacobi step, Chebyshev,
// energy and |g|^2 partials) -> k_control (FP64 reduction in a fixed order and the line-search /
// Chebyshev / buffer-role decisions).  This replaces the reference's computeForceKd /
// updateNodesNextIter / updateChebyshev / thrust::reduce and the host loop of
// CUDAInterface::doDescentOpt (CUDAInterface.cu:482-1007) with no host round trip and no atomics.
// k_tet + k_gather evaluate forces and the Hessian diagonal for the standalone material calls.
//
// Layout: nodes are renumbered in Morton order and tets sorted by their smallest node.  The vectors
// of the descent pass (iterates, inertial target, partial forces, Hessian diagonal) are node-major,
// xyz of a node together, so that a tile's scattered halo nodes cost one access each and not three;
// the state between steps is 3 planes (x | y | z) of nn values; per-tet rest data are 10 planes (Dm^-1
// entries, volume) plus 16 bytes per tet of tile-local ids and contribution slots for the tile
// pass; per-tet force records of the standalone calls are 12 consecutive values.
#include <algorithm>
#include <type_traits>

#include <hip/hip_ext.h>

#include "pbs_pass.h"

namespace pbs {

// ---------------------------------------------------------------------------------------------
// Deterministic block reduction of a double: wave64 shuffle tree, then the waves' sums in order.
// The result is valid in thread 0.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double block_sum(double v, double *lds) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) lds[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
    for (int i = 0; i < nw; ++i) r += lds[i];
  }
  __syncthreads();
  return r;
}

// N block sums at once (one LDS exchange): the same order per value as block_sum; lds holds 16 N.
template <int N> __device__ __forceinline__ void block_sums(double (&v)[N], double *lds) {
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[j] += __shfl_down(v[j], off, 64);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0)
#pragma unroll
    for (int j = 0; j < N; ++j) lds[16 * j + w] = v[j];
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      double r = 0.0;
      for (int i = 0; i < nw; ++i) r += lds[16 * j + i];
      v[j] = r;
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------------------------
// Setup: rest-shape data (compute_DmInv_ANs_Mass, CUDAInterface.cu:273-325; TetMesh.cpp:189-216).
// Contraction is off so that Dm^-1, volumes and masses round exactly as the FP32 reference
// formulas written out without fused multiply-adds.
// ---------------------------------------------------------------------------------------------
#pragma clang fp contract(off)
__global__ void k_setup_tets(DevParams p, const float *__restrict__ rest, const int4 *__restrict__ tets,
                             float *__restrict__ dmi, float *__restrict__ vol, int *__restrict__ flag) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.nt) return;
  const int N = p.nn, T = p.nt;
  const int4 q = tets[t];
  if (q.x < 0 || q.y < 0 || q.z < 0 || q.w < 0 || q.x >= N || q.y >= N || q.z >= N || q.w >= N) {
    atomicOr(flag, 1);
    return;
  }
  const int qn[4] = {q.x, q.y, q.z, q.w};
  float r[4][3];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int k = 0; k < 3; ++k) r[c][k] = rest[k * N + qn[c]];
  float Dmi[9], V;
  const float det = rest_shape(r, Dmi, V);
  if (!(det > 0.0f)) atomicOr(flag, 2);
  vol[t] = V;
#pragma unroll
  for (int i = 0; i < 9; ++i) dmi[(size_t)i * T + t] = Dmi[i];
}

// Lumped mass gathered over the incidence list in ascending tet order (the reference's float
// atomics, CUDAInterface.cu:297-301, sum in an unspecified order); gravity force from the mass
// before constrained nodes get fixed_mass (CUDAInterface.cu:716-719).
__global__ void k_setup_nodes(DevParams p, const int *__restrict__ inc_off, const int *__restrict__ inc,
                              const float *__restrict__ vol, const int *__restrict__ mask, float *__restrict__ mass,
                              float *__restrict__ mnode, float *__restrict__ gforce) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= p.nn) return;
  float m = 0.0f;
  for (int e = inc_off[n]; e < inc_off[n + 1]; ++e) {
    const float w = vol[inc[e] >> 2] / 4.0f * p.density;
    m += w;
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) gforce[(size_t)d * p.nn + n] = p.grav[d] * m;
  mass[n] = mask[n] ? p.fixed_mass : m;
  mnode[n] = mask[n] ? -1.0f : m;
}
#pragma clang fp contract(on)

// ---------------------------------------------------------------------------------------------
// Per-tet pass: forces, energy, optional Hessian diagonal (computeForceKd, CUDAInterface.cu:495-568).
// One thread per tet; node positions are gathered from the 3 planes, rest data read coalesced.
// ---------------------------------------------------------------------------------------------
template <typename R, int MAT>
__global__ void __launch_bounds__(256) k_tet(DevParams p, const Ctrl *__restrict__ ctrl, Ring<R> ring,
                                             const int4 *__restrict__ tets, const float *__restrict__ dmi,
                                             const float *__restrict__ vol, R *__restrict__ frec,
                                             float *__restrict__ hrec, double *__restrict__ etet,
                                             R *__restrict__ tete, int force_hd, TileDev td) {
  __shared__ double lds[16];
  if (ctrl->done) return;
  const int hd = force_hd >= 0 ? force_hd : ctrl->hd_now;
  const R *__restrict__ x = ring.b[ctrl->cur];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int T = p.nt;
  double e = 0.0;
  if (t < T) {
    const int4 q = tets[t];
    R Dmi[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) Dmi[i] = (R)dmi[(size_t)i * T + t];
    const R V = (R)vol[t];
    R Ds[9];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const R x0 = x[3 * (size_t)q.x + k];
      Ds[3 * k + 0] = x[3 * (size_t)q.y + k] - x0;
      Ds[3 * k + 1] = x[3 * (size_t)q.z + k] - x0;
      Ds[3 * k + 2] = x[3 * (size_t)q.w + k] - x0;
    }
    R F[9];
    mul3(Ds, Dmi, F);
    R f12[12], h12[12], en;
    int lo = 0, hi = td.ninst;  // instance of tet t
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (td.inst_tet_off[mid] <= t) lo = mid;
      else hi = mid;
    }
    const R mu = (R)td.inst_mu[lo], lam = (R)td.inst_lam[lo];
    if (hd) {
      if (MAT == 0) neo_tet<R, true>(F, Dmi, V, mu, lam, f12, en, h12);
      else stretch_tet<R, true>(F, Dmi, V, mu, lam, f12, en, h12);
      float *hr = hrec + 12 * (size_t)t;
#pragma unroll
      for (int i = 0; i < 12; ++i) hr[i] = (float)h12[i];
    } else {
      if (MAT == 0) neo_tet<R, false>(F, Dmi, V, mu, lam, f12, en, h12);
      else stretch_tet<R, false>(F, Dmi, V, mu, lam, f12, en, h12);
    }
    R *fr = frec + 12 * (size_t)t;
#pragma unroll
    for (int i = 0; i < 12; ++i) fr[i] = f12[i];
    if (p.clamp == 1) en = en > (R)0 ? en : (R)0;                  // CUDAInterface.cu:549
    else if (p.clamp == 2) en = en > (R)1e-6 ? en : (R)0;          // IsotropicNeohookeanMaterial.cpp:129
    if (tete) tete[t] = en;
    e = (double)en;
  }
  const double s = block_sum(e, lds);
  if (threadIdx.x == 0) etet[blockIdx.x] = s;
}

// The fields of a control block that a descent pass's tile and node kernels read.
struct PassCtl {
  int done, cur, nxt, last, hd_now, check_now, cheb_now;
  float alpha, omega_next;
};
__device__ __forceinline__ PassCtl pass_ctl(const Ctrl *c) {
  return {c->done, c->cur, c->nxt, c->last, c->hd_now, c->check_now, c->cheb_now, c->alpha, c->omega_next};
}

// XCD-aware tile order: workgroups are dispatched round-robin over the 8 XCDs, so block i runs
// on XCD i % 8.  Giving each XCD a contiguous range of tiles keeps neighbouring tiles (which
// share halo nodes and halo tets) in the same 4 MB L2.
__device__ __forceinline__ int xcd_tile(int bid, int nblk) {
  const int per = (nblk + 7) >> 3;
  const int xcd = bid & 7, k = bid >> 3;
  const int full = nblk - 8 * (per - 1);  // XCDs that get `per` tiles (the rest get per - 1)
  const int start = xcd < full ? xcd * per : full * per + (xcd - full) * (per - 1);
  return start + k;
}

// Local node i's run of contributions, and a halo node's partial slot.
struct NodeRun {
  unsigned run;  // first contribution, and the next run's in the high half
  int slot;
};
__device__ __forceinline__ NodeRun node_run(const TileInfo &ti, const TileDev &td, int i) {
  const unsigned short *off = td.tile_off + ti.off_start + i;
  return {(unsigned)off[0] | (unsigned)off[1] << 16, i < ti.own_cnt ? 0 : td.halo_slot[ti.halo_off + (i - ti.own_cnt)]};
}

// Gather of one tile: each thread sums the contribution runs of its local nodes in order and
// writes one partial (xyz) per owned node and per halo node (at its slot); the sums
// are formed in R whatever the contributions' type Q.
template <typename R, typename Q>
__device__ __forceinline__ void tile_gather(int phase, const TileInfo &ti, const TileDev &td, const Q *__restrict__ rec,
                                            NodeRun n0, R *__restrict__ fown, R *__restrict__ hpart,
                                            float *__restrict__ fownh, float *__restrict__ hparth) {
  constexpr int W = ContribWidth<Q>::value;
  const int L = ti.own_cnt + ti.halo_cnt;
  for (int i = threadIdx.x; i < L; i += blockDim.x) {
    const NodeRun n = i == (int)threadIdx.x ? n0 : node_run(ti, td, i);
    const int o0 = n.run & 0xffff, o1 = n.run >> 16;
    const size_t d0 = 3 * (size_t)(i < ti.own_cnt ? ti.own_start + i : n.slot);
    // the run is summed in order; FP32 contributions are read 4 at a time ahead of their additions
    // (slots past the run clamped to its first slot and not added: 4 % of the FP32 tile pass), FP64
    // ones one at a time (4 ahead: 3 % slower)
    constexpr int U = sizeof(Q) == 4 ? 4 : 1;
    if (phase == 0) {
      R a0 = (R)0, a1 = (R)0, a2 = (R)0;
      for (int j = o0; j < o1; j += U) {
        Q t[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const Q *r = rec + W * (j + u < o1 ? j + u : o0);
          t[u][0] = r[0];
          t[u][1] = r[1];
          t[u][2] = r[2];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (j + u < o1) {
            a0 += (R)t[u][0];
            a1 += (R)t[u][1];
            a2 += (R)t[u][2];
          }
      }
      R *o = i < ti.own_cnt ? fown : hpart;
      o[d0] = a0;
      o[d0 + 1] = a1;
      o[d0 + 2] = a2;
    } else {
      float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
      for (int j = o0; j < o1; j += U) {
        Q t[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const Q *r = rec + W * (j + u < o1 ? j + u : o0);
          t[u][0] = r[0];
          t[u][1] = r[1];
          t[u][2] = r[2];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (j + u < o1) {
            a0 += (float)t[u][0];
            a1 += (float)t[u][1];
            a2 += (float)t[u][2];
          }
      }
      float *o = i < ti.own_cnt ? fownh : hparth;
      o[d0] = a0;
      o[d0 + 1] = a1;
      o[d0 + 2] = a2;
    }
  }
}

// Byte offset of the tile pass's rest-position region in LDS (after the positions and the
// contribution slots; 16-byte aligned).
template <typename R> __host__ __device__ inline size_t tile_rest_offset(const TileDev &td) {
  const size_t b = (4 * (size_t)td.lcap + 4 * (size_t)ContribWidth<R>::value * td.tcap) * sizeof(R);
  return (b + 15) & ~(size_t)15;
}

// ---------------------------------------------------------------------------------------------
// Tile pass (per-tet half of computeForceKd, CUDAInterface.cu:495-568): one workgroup per tile
// evaluates each of the tile's tets once -- force, energy on check passes, Hessian diagonal on
// refresh passes -- and writes every corner contribution into its precomputed slot of an LDS
// array in which each local node's contributions form one contiguous run (ordered by tet, then
// corner).  The gather then sums each run in that fixed order (no atomics) and writes one partial
// per owned node (fown) and per halo node (hpart).
//   LDS: positions of local nodes (4 R each), contributions (4 per tet, W values each), rest
//   positions of local nodes (float4 each).
//   HBM per tet: 16 B of local ids / slots.  Dm^-1 and the volume are not streamed from memory
//   (40 B per tet): they are recomputed from the staged rest positions with the setup kernel's
//   own FP32 arithmetic (rest_shape), so they are bitwise the stored values.
// ---------------------------------------------------------------------------------------------
// One tile, all phases: stage the local nodes' positions and rest positions, evaluate the tets
// (phase 0 forces and energies; phase 1, when hd, the stiffness diagonal), gather each phase.
template <typename R, int MAT, bool F32M>
__device__ __forceinline__ void tile_body(const DevParams &p, int chk, const R *__restrict__ x, const TileDev &td,
                                          int b, const TileInfo &ti, int node0, int hdnow, const float4 *__restrict__ rest,
                                          R *__restrict__ fown, R *__restrict__ hpart, float *__restrict__ fownh,
                                          float *__restrict__ hparth, unsigned char *smem, double *lds_red) {
  const int L = ti.own_cnt + ti.halo_cnt, tid = threadIdx.x;
  typedef typename std::conditional<F32M, float, R>::type C;
  R *sx = (R *)smem;
  C *rec = (C *)(sx + 4 * td.lcap);
  float4 *srest = (float4 *)(smem + tile_rest_offset<R>(td));
  const int nthr = blockDim.x;
  // neo-Hookean: tet tid's local ids and slots, loaded before the staging so that they arrive with
  // it.  The FP64 stretch kernel would lose waves to the 4 registers it holds across the staging (6.3 M
  // tets, 208 -> 261 us; FP32 101 -> 98), so the stretch material loads them after the barrier.
  constexpr bool PRE = MAT == 0;
  const uint4 lp0 = PRE && tid < ti.tet_cnt ? td.tet_lp[(size_t)ti.tet_start + tid] : make_uint4(0, 0, 0, 0);
  const C mu = (C)td.inst_mu[ti.inst], lam = (C)td.inst_lam[ti.inst];
  // the gather's descriptors of the thread's first local node, read now and not after the tets (FP32
  // 70.8 -> 69.3 us at 6.3 M tets); the asm below keeps the reads from being moved back there
  NodeRun n0 = {0, 0};
  if (tid < L) n0 = node_run(ti, td, tid);
  auto stage = [&](int i, int g) {
    const R *xg = x + 3 * (size_t)g;
    sx[4 * i] = xg[0];
    sx[4 * i + 1] = xg[1];
    sx[4 * i + 2] = xg[2];
    srest[i] = rest[g];
  };
  // the first lstride local nodes: ids at a fixed stride, padded with valid ones, so that the staging
  // waits for no descriptor (node0 was read together with it)
  if (tid < td.lstride) stage(tid, node0);
  for (int i = td.lstride + tid; i < L; i += nthr)
    stage(i, i < ti.own_cnt ? ti.own_start + i : td.halo[ti.halo_off + i - ti.own_cnt]);
  asm volatile("" ::"v"(n0.run), "v"(n0.slot));
  __syncthreads();
  double e_el = 0.0;
  // the tile's tets and their gather for one phase
  auto run_phase = [&](auto ph) {
    constexpr int phase = decltype(ph)::value;
    for (int s = tid; s < ti.tet_cnt; s += nthr) {
      const uint4 lp = PRE && s == tid ? lp0 : td.tet_lp[(size_t)ti.tet_start + s];
      auto get_r = [&](float (&r)[4][3]) {
        const int lid[4] = {(int)(lp.x & 0xffff), (int)(lp.x >> 16), (int)(lp.y & 0xffff), (int)(lp.y >> 16)};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float4 q = srest[lid[c]];
          r[c][0] = q.x;
          r[c][1] = q.y;
          r[c][2] = q.z;
        }
      };
      auto get_neo = [&]() {
        float r[4][3];
        get_r(r);
        return NeoRest<C>(r, mu);
      };
      tile_tet<R, C, MAT, phase>(lp, get_r, get_neo, sx, rec, mu, lam, chk, p.clamp, e_el);
    }
    __syncthreads();
    tile_gather<R>(phase, ti, td, rec, n0, fown, hpart, fownh, hparth);
  };
  // The two phases as separate code: as one loop over the phase the compiler would share their common
  // arithmetic, which the forces of the one do not need.
  run_phase(std::integral_constant<int, 0>());
  if (hdnow) {
    __syncthreads();  // the Hessian phase reuses the contribution slots
    run_phase(std::integral_constant<int, 1>());
  }
  if (chk) {
    const double se = block_sum(e_el, lds_red);
    if (tid == 0) td.tpart[b] = se;
  }
}

// F32M (FP64 state only): the per-tet arithmetic in FP32 after F (the mixed mode's early passes).
//
// Bound (neo-Hookean): the staging's scattered halo reads and the LDS, busy in 77 % (FP32) and 68 %
// (FP64) of the cycles, half of that with bank conflicts.  The vector units issue in 86 % and 53 %, but
// forces with a third fewer FP32 instructions left the time as it was.  So node data is node-major
// (the three components of a node in one cache line, its rest position one 16-byte read, instead of
// three lines each), the first lstride ids and the thread's contribution run are read with the
// descriptor instead of after it, and the neo-Hookean force takes one 3x3 product (neo_force).  Average
// of a 64-pass step's launches on 6.3 M tets (64x64x256 cells, twisted by 30 degrees), with planes and
// three products -> now: FP32 78 -> 76 us, FP64 133 -> 123; stretch FP32 134 -> 130, FP64 259 -> 257,
// with polar_rotation_fast 101 and 208 (bound by its vector instructions).  The FP64 neo-Hookean kernel is held to 5 waves per SIMD (at most 102 VGPRs, no
// spilling), as many as the LDS of 256-tet tiles allows (30.8 KB: 5 workgroups per CU).  6 waves with
// 224-tet tiles spill (130 us), 4 waves 114 us.
template <typename R, int MAT, bool F32M>
__global__ void __launch_bounds__(256, (sizeof(R) == 8 && MAT == 0 && !F32M) ? 5 : 1)
k_tile(DevParams p, const Ctrl *__restrict__ ctrl, Ring<R> ring, TileDev td, const float4 *__restrict__ rest,
       R *__restrict__ fown, R *__restrict__ hpart, float *__restrict__ fownh, float *__restrict__ hparth) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double lds_red[16];
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  // One instance: its control block is ctrl[0], read together with the tile descriptor rather than
  // after it, so the staging loads wait for one dependent memory access less.  Several: the
  // tile's instance's block, read once the descriptor has arrived.
  PassCtl c = pass_ctl(ctrl);
  const int node0 = (int)threadIdx.x < td.lstride ? td.ids[(size_t)b * td.lstride + threadIdx.x] : 0;
  const TileInfo ti = td.tiles[b];
  // both reads in flight before either is waited for (otherwise the compiler folds the first into
  // the second, which waits for the descriptor)
  asm volatile("" ::"s"(c.done), "s"(c.cur), "s"(c.hd_now), "s"(c.check_now), "s"(ti.inst));
  if (td.ninst != 1) c = pass_ctl(ctrl + ti.inst);
  if (c.done) return;
  // (the buffer's pointer is selected, not indexed: that would be one more dependent memory access)
  const R *x01 = c.cur & 1 ? ring.b[1] : ring.b[0], *x23 = c.cur & 1 ? ring.b[3] : ring.b[2];
  tile_body<R, MAT, F32M>(p, c.check_now, c.cur & 2 ? x23 : x01, td, b, ti, node0, c.hd_now, rest, fown, hpart, fownh,
                          hparth, smem, lds_red);
}

// ---------------------------------------------------------------------------------------------
// Node pass (updateNodesNextIter + updateChebyshev, CUDAInterface.cu:572-623): force = owned
// partial + the node's halo partials in tile order; Jacobi-preconditioned step with Chebyshev.
// g = (x - x~) m/h^2 - f - s (m grav + f_ext), s = 1 (REF_GPU) or 2 (REF_CPU, DescentOptimize.cpp:51-52).
// ---------------------------------------------------------------------------------------------
// GRAD_ONLY: only the |g|^2 partials (the warm start's gradient passes); nothing else is written.
template <typename R, bool GRAD_ONLY>
__global__ void __launch_bounds__(256)
k_node(DevParams p, const Ctrl *__restrict__ ctrl, Ring<R> ring, TileDev td, const R *__restrict__ fown,
       const R *__restrict__ hpart, const float *__restrict__ fownh, const float *__restrict__ hparth,
       float *__restrict__ hd, const float *__restrict__ mnode, const float *__restrict__ ext,
       const R *__restrict__ xt) {
  __shared__ double lds_red[48];
  // One instance: control block ctrl[0], node blocks of 256 from node 0, read without waiting for
  // the block's instance.  Several: the block's instance first.
  PassCtl c = pass_ctl(ctrl);
  asm volatile("" ::"s"(c.done), "s"(c.cur), "s"(c.nxt), "s"(c.last), "s"(c.hd_now), "s"(c.cheb_now), "s"(c.alpha),
               "s"(c.omega_next));  // read now, not folded into the several-instance read below
  int n0 = 256 * (int)blockIdx.x, nend = p.nn;
  if (td.ninst != 1) {
    const int inst = td.blk_inst[blockIdx.x];
    c = pass_ctl(ctrl + inst);
    n0 = td.blk_start[blockIdx.x];
    nend = td.inst_node_off[inst + 1];
  }
  if (c.done) return;
  const int hdnow = c.hd_now, cheb = c.cheb_now;
  const R alpha = (R)c.alpha, om = (R)c.omega_next;
  const R *__restrict__ x = ring.b[c.cur];
  const R *__restrict__ xl = ring.b[c.last];
  R *__restrict__ xn = ring.b[c.nxt];
  const int n = n0 + (int)threadIdx.x;
  const int N = p.nn;
  double en = 0.0, g2 = 0.0, f2 = 0.0;
  if (n < nend) {
    // every load of the node that depends on no other is issued first (the flags are uniform), so
    // the thread waits for memory about twice (these loads, then its halo partials), not once per
    // array
    const int b0 = td.bnd_off[n], b1 = td.bnd_off[n + 1];
    const float m = mnode[n];  // the node's mass, or -1: fixed
    const bool fixed = m < 0.0f;
    R f[3], xc[3], xtv[3], xlv[3];
    float hv[3], ev[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const size_t i = 3 * (size_t)n + d;
      f[d] = fown[i];
      xc[d] = x[i];
      xtv[d] = xt[i];
      xlv[d] = (R)0;
      ev[d] = 0.0f;
      hv[d] = 0.0f;
    }
    if (!GRAD_ONLY && cheb)
#pragma unroll
      for (int d = 0; d < 3; ++d) xlv[d] = xl[3 * (size_t)n + d];
    if (p.has_ext)
#pragma unroll
      for (int d = 0; d < 3; ++d) ev[d] = ext[(size_t)d * N + n];
    if (!GRAD_ONLY)
#pragma unroll
      for (int d = 0; d < 3; ++d) hv[d] = hdnow ? fownh[3 * (size_t)n + d] : hd[3 * (size_t)n + d];
    for (int e = b0; e < b1; ++e) {
      const R *hp = hpart + 3 * (size_t)e;
#pragma unroll
      for (int d = 0; d < 3; ++d) f[d] += hp[d];
    }
    if (!GRAD_ONLY && hdnow) {
      for (int e = b0; e < b1; ++e) {
        const float *hp = hparth + 3 * (size_t)e;
#pragma unroll
        for (int d = 0; d < 3; ++d) hv[d] += hp[d];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) hd[3 * (size_t)n + d] = hv[d];
    }
    if (fixed) {
      if (!GRAD_ONLY)
#pragma unroll
        for (int d = 0; d < 3; ++d) xn[3 * (size_t)n + d] = xc[d];
    } else {
      const R hstep = (R)p.h;
      const R mh2 = (R)m / (hstep * hstep);
      R e = (R)0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const R dd = xc[d] - xtv[d];
        R fe = (R)(p.grav[d] * m);  // = the setup's gravity force (mass before the fixed override)
        if (p.has_ext) fe += (R)ev[d];
        const R gr = dd * mh2 - f[d] - (R)p.ext_scale * fe;
        e += (R)0.5 * dd * dd * mh2 - fe * xc[d];
        g2 += (double)gr * (double)gr;
        f2 += (double)f[d] * (double)f[d];
        if (!GRAD_ONLY) {
          R nx = xc[d] - alpha * gr / ((R)hv[d] + mh2);
          if (cheb) nx = om * (nx - xlv[d]) + xlv[d];
          xn[3 * (size_t)n + d] = nx;
        }
      }
      if (!GRAD_ONLY) en += (double)e;
    }
  }
  if (!GRAD_ONLY && p.f32math) {  // mixed mode: also |f|^2, the scale of the FP32 force rounding
    double v[3] = {en, g2, f2};
    block_sums<3>(v, lds_red);
    if (threadIdx.x == 0) {
      td.npart[2 * blockIdx.x] = v[0];
      td.npart[2 * blockIdx.x + 1] = v[1];
      td.fpart[blockIdx.x] = v[2];
    }
  } else {
    double v[2] = {en, g2};
    block_sums<2>(v, lds_red);
    if (threadIdx.x == 0) {
      td.npart[2 * blockIdx.x] = v[0];
      td.npart[2 * blockIdx.x + 1] = v[1];
    }
  }
}

// acc[k] += v[K i + k] for i = first, first + 1024, ... below end, in that order: the loads of 8
// consecutive terms are issued before their additions (indices past the end are clamped to
// `first`, whose value is then not added), so the thread waits for memory once per 8 terms
// instead of once per term, and the sums are those of the plain loop.
template <int K>
__device__ __forceinline__ void strided_sum(const double *__restrict__ v, int first, int end, double *acc) {
  constexpr int U = 8;
  for (int base = first; base < end; base += U * 1024) {
    double t[U][K];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u * 1024 < end ? base + u * 1024 : first;
#pragma unroll
      for (int k = 0; k < K; ++k) t[u][k] = v[(size_t)K * i + k];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (base + u * 1024 < end)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] += t[u][k];
  }
}

// Control step, one workgroup per instance: FP64 sums in a fixed order of the instance's tile
// energies (check passes) and node-block partials (energy, |g|^2), then the loop control of the
// reference.
__global__ void __launch_bounds__(1024) k_control(DevParams p, Ctrl *__restrict__ ctrl, TileDev td) {
  __shared__ double la[1024], lc[1024], lf[1024];
  const int inst = blockIdx.x;
  ctrl += inst;
  if (ctrl->done) return;
  const int tid = threadIdx.x;
  double a = 0.0, c = 0.0;
  if (ctrl->check_now) strided_sum<1>(td.tpart, td.inst_tile_off[inst] + tid, td.inst_tile_off[inst + 1], &a);
  {
    double ac[2] = {a, c};
    strided_sum<2>(td.npart, td.inst_blk_off[inst] + tid, td.inst_blk_off[inst + 1], ac);
    a = ac[0];
    c = ac[1];
  }
  const bool mix = p.f32math != 0;  // mixed mode: also |f|^2 of this pass, the FP32 force scale
  double f = 0.0;
  if (mix) strided_sum<1>(td.fpart, td.inst_blk_off[inst] + tid, td.inst_blk_off[inst + 1], &f);
  la[tid] = a;
  lc[tid] = c;
  lf[tid] = f;
  __syncthreads();
  // pairwise tree: levels 512 .. 64 through LDS, levels 32 .. 1 inside wavefront 0 by shuffles,
  // which pair lane t with lane t + st exactly as the LDS levels pair slots
  for (int st = 512; st >= 64; st >>= 1) {
    if (tid < st) {
      la[tid] += la[tid + st];
      lc[tid] += lc[tid + st];
      if (mix) lf[tid] += lf[tid + st];
    }
    __syncthreads();
  }
  if (tid < 64) {
    double E = la[tid], g2 = lc[tid], f2 = lf[tid];
#pragma unroll
    for (int st = 32; st > 0; st >>= 1) {
      E += __shfl_down(E, st, 64);
      g2 += __shfl_down(g2, st, 64);
      if (mix) f2 += __shfl_down(f2, st, 64);
    }
    if (tid == 0) {
      Ctrl C = *ctrl;
      if (p.f32math) C.fnorm = sqrt(f2);
      control_apply(p, C, E, g2);
      *ctrl = C;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Step start (initDescentOpt, CUDAInterface.cu:482-493; DescentOptimize.cpp:35-41) and the
// device loop state reset.
// ---------------------------------------------------------------------------------------------
template <typename R>
__global__ void k_step_init(DevParams p, Ctrl *__restrict__ ctrl, int ninst, Ring<R> ring, const R *__restrict__ xpos,
                            const R *__restrict__ v, const R *__restrict__ vl, R *__restrict__ xt) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < p.nn) {
    const R h = (R)p.h;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const size_t i = (size_t)d * p.nn + n;
      const R t = xpos[i] + v[i] * h;
      xt[3 * (size_t)n + d] = t;
      R x0;
      if (p.semantics == 1) x0 = t + (R)(p.init_momentum * p.h) * (v[i] - vl[i]);
      else if (sizeof(R) == 4) x0 = (R)((double)t + (double)p.init_momentum * (double)(v[i] - vl[i]) * (double)p.h);
      else x0 = t + (R)p.init_momentum * (v[i] - vl[i]) * h;
      ring.b[0][3 * (size_t)n + d] = x0;
    }
  }
  if (n < ninst) {  // one control block per instance
    Ctrl C;
    C.k = 0;
    C.budget = p.iterations;
    C.passes = 0;
    C.rollbacks = 0;
    C.converged = 0;
    C.used_learned = 0;
    C.first = 1;
    C.cur = 0;
    C.nxt = 1;
    C.last = 2;
    C.old = 3;
    C.hd_now = 1;
    C.check_now = 1;
    C.kc = 0;
    C.alpha = p.alpha0;
    C.rho = 0.0f;
    C.omega = 1.0f;
    float rho = 0.0f, om = 1.0f;
    cheb_schedule(p, 0, rho, om);
    C.rho_next = rho;
    C.omega_next = om;
    C.cheb_now = om != 1.0f;
    C.ws_beta = 0.0f;
    C.E = 0.0;
    C.E_old = 0.0;
    C.g0 = -1.0;
    C.g = 0.0;
    C.g_plain = 0.0;
    C.g_learned = 0.0;
    C.done = (p.iterations <= 0 || p.alpha0 < p.alpha_min) ? 1 : 0;
    ctrl[n] = C;
  }
}

// Step end: velocities (updateVelocity, CUDAInterface.cu:625-639, or DescentOptimize.cpp:183-185)
// and the new positions.
template <typename R>
__global__ void k_step_final(DevParams p, const Ctrl *__restrict__ ctrl, TileDev td, Ring<R> ring, R *__restrict__ xpos,
                             R *__restrict__ v, R *__restrict__ vl, const R *__restrict__ xt,
                             const int *__restrict__ mask) {
  const int inst = td.blk_inst[blockIdx.x];
  const int n = td.blk_start[blockIdx.x] + (int)threadIdx.x;
  if (n >= td.inst_node_off[inst + 1]) return;
  const R *__restrict__ x = ring.b[ctrl[inst].cur];
  const R h = (R)p.h;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const size_t i = (size_t)d * p.nn + n;
    const R xf = x[3 * (size_t)n + d];
    if (p.semantics == 1) {
      vl[i] = v[i];
      v[i] = (R)p.damping * (xf - xpos[i]) / h;
    } else if (!mask[n]) {
      vl[i] = v[i];
      const R vv = v[i] + (xf - xt[3 * (size_t)n + d]) * ((R)1 / h);
      v[i] = (sizeof(R) == 4) ? (R)((double)vv * (double)p.damping) : vv * (R)p.damping;
    }
    xpos[i] = xf;
  }
}

// Control block for a standalone force / Hessian evaluation on ring buffer `cur` (hd, chk: the
// tile pass's Hessian phase and energy partials).
__global__ void k_standalone_ctrl(Ctrl *ctrl, int cur, int hd, int chk) {
  Ctrl C = {};
  C.cur = cur;
  C.nxt = (cur + 1) & 3;
  C.last = (cur + 2) & 3;
  C.old = (cur + 3) & 3;
  C.hd_now = hd;
  C.check_now = chk;
  C.done = 0;
  *ctrl = C;
}

// Per-node sums of the tile pass's partials, in the node pass's order (owned partial, then the
// halo partials in tile order), written as doubles in the caller's node order (AoS): the elastic
// forces (which = 0) or the Hessian diagonal (which = 1) the descent uses.
template <typename R>
__global__ void k_sum_partials(TileDev td, int N, int which, const R *__restrict__ fown, const R *__restrict__ hpart,
                               const float *__restrict__ fownh, const float *__restrict__ hparth,
                               const int *__restrict__ perm, double *__restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int b0 = td.bnd_off[n], b1 = td.bnd_off[n + 1];
  const size_t o = 3 * (size_t)perm[n];
  if (which == 0) {
    R f[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) f[d] = fown[3 * (size_t)n + d];
    for (int e = b0; e < b1; ++e)
#pragma unroll
      for (int d = 0; d < 3; ++d) f[d] += hpart[3 * (size_t)e + d];
#pragma unroll
    for (int d = 0; d < 3; ++d) out[o + d] = (double)f[d];
  } else {
    float h[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) h[d] = fownh[3 * (size_t)n + d];
    for (int e = b0; e < b1; ++e)
#pragma unroll
      for (int d = 0; d < 3; ++d) h[d] += hparth[3 * (size_t)e + d];
#pragma unroll
    for (int d = 0; d < 3; ++d) out[o + d] = (double)h[d];
  }
}

// Gather of per-tet records into per-node planes (elastic forces or Hessian diagonal).
template <typename T>
__global__ void k_gather(int N, const int *__restrict__ inc_off, const int *__restrict__ inc,
                         const T *__restrict__ rec, T *__restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  T a = 0, b = 0, c = 0;
  for (int e = inc_off[n]; e < inc_off[n + 1]; ++e) {
    const T *r = rec + 3 * (size_t)inc[e];
    a += r[0];
    b += r[1];
    c += r[2];
  }
  out[n] = a;
  out[N + n] = b;
  out[2 * (size_t)N + n] = c;
}

// AoS (caller's node order) <-> planes (solver's node order); perm maps solver -> caller index.
template <typename A, typename B>
__global__ void k_aos_to_planes(const A *__restrict__ aos, B *__restrict__ planes, const int *__restrict__ perm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t o = 3 * (size_t)(perm ? perm[i] : i);
#pragma unroll
  for (int d = 0; d < 3; ++d) planes[(size_t)d * n + i] = (B)aos[o + d];
}

template <typename A, typename B>
__global__ void k_planes_to_aos(const A *__restrict__ planes, B *__restrict__ aos, const int *__restrict__ perm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t o = 3 * (size_t)(perm ? perm[i] : i);
#pragma unroll
  for (int d = 0; d < 3; ++d) aos[o + d] = (B)planes[(size_t)d * n + i];
}

// Records of W values per tet (solver's tet order) -> FP32 in the caller's order: one thread per output
// value, so that the writes are coalesced; a record is read by neighbouring threads.  Bound by the
// copy to the host behind it (48 B per tet over PCIe).  Reordered on the host instead, the records
// of 202 K tets took 1.3 ms more per call (forces and stiffness diagonals together 4.95 -> 2.29 ms).
template <typename R, int W>
__global__ void k_tets_to_caller(const R *__restrict__ rec, float *__restrict__ out, const int *__restrict__ itperm, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long t = i / W;
  out[i] = (float)rec[(size_t)W * itperm[t] + (i - W * t)];
}
// AoS (caller's node order) <-> node-major (solver's node order).
template <typename A, typename B>
__global__ void k_aos_to_nodes(const A *__restrict__ aos, B *__restrict__ nodes, const int *__restrict__ perm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t o = 3 * (size_t)perm[i];
#pragma unroll
  for (int d = 0; d < 3; ++d) nodes[3 * (size_t)i + d] = (B)aos[o + d];
}
template <typename A, typename B>
__global__ void k_nodes_to_aos(const A *__restrict__ nodes, B *__restrict__ aos, const int *__restrict__ perm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t o = 3 * (size_t)perm[i];
#pragma unroll
  for (int d = 0; d < 3; ++d) aos[o + d] = (B)nodes[3 * (size_t)i + d];
}

__global__ void k_fill(float *p, float v, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------------------------
// Launch wrappers
// ---------------------------------------------------------------------------------------------
static inline int nblk(long n, int bs) { return (int)((n + bs - 1) / bs); }

// A launch that, given events, records its own start and end in them.
template <typename F, typename... Args>
static void launch_timed(F kernel, dim3 grid, dim3 block, size_t lds, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                         Args... args) {
  if (e0) hipExtLaunchKernelGGL(kernel, grid, block, (std::uint32_t)lds, st, e0, e1, 0u, args...);
  else hipLaunchKernelGGL(kernel, grid, block, lds, st, args...);
}

template <typename R>
void Launch<R>::setup_tets(const DevMesh<R> &m, const DevParams &p, int bs, hipStream_t st) {
  if (p.nt > 0) hipLaunchKernelGGL(k_setup_tets, dim3(nblk(p.nt, bs)), dim3(bs), 0, st, p, m.rest, m.tets, m.dmi, m.vol, m.flag);
}
template <typename R>
void Launch<R>::setup_nodes(const DevMesh<R> &m, const DevParams &p, int bs, hipStream_t st) {
  hipLaunchKernelGGL(k_setup_nodes, dim3(nblk(p.nn, bs)), dim3(bs), 0, st, p, m.inc_off, m.inc, m.vol, m.mask, m.mass,
                     m.mnode, m.gforce);
}
template <typename R>
void Launch<R>::tet(const DevMesh<R> &m, const TileDev &td, const DevParams &p, int bs, int force_hd, int write_e,
                    hipStream_t st) {
  if (p.nt <= 0) return;
  R *te = write_e ? m.tete : nullptr;
  if (p.material == 0)
    hipLaunchKernelGGL((k_tet<R, 0>), dim3(nblk(p.nt, bs)), dim3(bs), 0, st, p, m.ctrl, m.ring, m.tets, m.dmi, m.vol, m.frec, m.hrec, m.etet, te, force_hd, td);
  else
    hipLaunchKernelGGL((k_tet<R, 1>), dim3(nblk(p.nt, bs)), dim3(bs), 0, st, p, m.ctrl, m.ring, m.tets, m.dmi, m.vol, m.frec, m.hrec, m.etet, te, force_hd, td);
}
template <typename R>
size_t Launch<R>::tile_lds(const TileDev &td) {
  return tile_rest_offset<R>(td) + 16 * (size_t)td.lcap;
}
template <typename R>
void Launch<R>::tile_pass(const DevMesh<R> &m, const TileDev &td, const DevParams &p, hipStream_t st, hipEvent_t e0,
                          hipEvent_t e1) {
  const size_t lds = tile_lds(td);
  const bool f32m = sizeof(R) == 8 && p.f32math;
#define PBS_TILE_LAUNCH(MAT, F32M)                                                                               \
  launch_timed(k_tile<R, MAT, F32M>, dim3(td.ntiles), dim3(td.threads), lds, st, e0, e1, p, m.ctrl, m.ring, td, \
               m.rest4, m.fown, m.hpart, m.fownh, m.hparth)
  if (p.material == 0 && !f32m) PBS_TILE_LAUNCH(0, false);
  else if (p.material == 0) PBS_TILE_LAUNCH(0, true);
  else if (!f32m) PBS_TILE_LAUNCH(1, false);
  else PBS_TILE_LAUNCH(1, true);
#undef PBS_TILE_LAUNCH
}
template <typename R>
void Launch<R>::node_pass(const DevMesh<R> &m, const TileDev &td, const DevParams &p, hipStream_t st, hipEvent_t e0,
                          hipEvent_t e1) {
  launch_timed(k_node<R, false>, dim3(td.nblk), dim3(256), 0, st, e0, e1, p, m.ctrl, m.ring, td, m.fown, m.hpart,
               m.fownh, m.hparth, m.hd, m.mnode, m.ext, m.xt);
}
template <typename R>
void Launch<R>::grad_pass(const DevMesh<R> &m, const TileDev &td, const DevParams &p, hipStream_t st) {
  hipLaunchKernelGGL((k_node<R, true>), dim3(td.nblk), dim3(256), 0, st, p, m.ctrl, m.ring, td, m.fown, m.hpart,
                     m.fownh, m.hparth, m.hd, m.mnode, m.ext, m.xt);
}
template <typename R>
void Launch<R>::control(const DevMesh<R> &m, const TileDev &td, const DevParams &p, hipStream_t st, hipEvent_t e0,
                        hipEvent_t e1) {
  launch_timed(k_control, dim3(td.ninst), dim3(1024), 0, st, e0, e1, p, m.ctrl, td);
}
template <typename R>
void Launch<R>::step_init(const DevMesh<R> &m, const TileDev &td, const DevParams &p, int bs, hipStream_t st) {
  hipLaunchKernelGGL((k_step_init<R>), dim3(nblk(std::max(p.nn, td.ninst), bs)), dim3(bs), 0, st, p, m.ctrl, td.ninst,
                     m.ring, m.xpos, m.v, m.vl, m.xt);
}
template <typename R>
void Launch<R>::step_final(const DevMesh<R> &m, const TileDev &td, const DevParams &p, hipStream_t st) {
  hipLaunchKernelGGL((k_step_final<R>), dim3(td.nblk), dim3(256), 0, st, p, m.ctrl, td, m.ring, m.xpos, m.v, m.vl, m.xt,
                     m.mask);
}
template <typename R>
void Launch<R>::standalone_ctrl(const DevMesh<R> &m, int cur, hipStream_t st, int hd, int chk) {
  hipLaunchKernelGGL(k_standalone_ctrl, dim3(1), dim3(1), 0, st, m.ctrl, cur, hd, chk);
}
template <typename R>
void Launch<R>::sum_partials(const DevMesh<R> &m, const TileDev &td, const DevParams &p, int which, double *out,
                             hipStream_t st) {
  hipLaunchKernelGGL((k_sum_partials<R>), dim3(nblk(p.nn, 256)), dim3(256), 0, st, td, p.nn, which, m.fown, m.hpart,
                     m.fownh, m.hparth, m.perm, out);
}
template <typename R>
void Launch<R>::gather(const DevMesh<R> &m, const DevParams &p, int bs, int which, void *out, hipStream_t st) {
  if (which == 0)
    hipLaunchKernelGGL((k_gather<R>), dim3(nblk(p.nn, bs)), dim3(bs), 0, st, p.nn, m.inc_off, m.inc, m.frec, (R *)out);
  else
    hipLaunchKernelGGL((k_gather<float>), dim3(nblk(p.nn, bs)), dim3(bs), 0, st, p.nn, m.inc_off, m.inc, m.hrec, (float *)out);
}
template <typename R>
void Launch<R>::aos_to_planes(const float *aos, R *planes, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_aos_to_planes<float, R>), dim3(nblk(n, 256)), dim3(256), 0, st, aos, planes, perm, n);
}
template <typename R>
void Launch<R>::planes_to_aos(const R *planes, float *aos, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_planes_to_aos<R, float>), dim3(nblk(n, 256)), dim3(256), 0, st, planes, aos, perm, n);
}
template <typename R>
void Launch<R>::planes_to_aos64(const R *planes, double *aos, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_planes_to_aos<R, double>), dim3(nblk(n, 256)), dim3(256), 0, st, planes, aos, perm, n);
}
template <typename R>
void Launch<R>::aos64_to_planes(const double *aos, R *planes, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_aos_to_planes<double, R>), dim3(nblk(n, 256)), dim3(256), 0, st, aos, planes, perm, n);
}
template <typename T> void tets_to_caller(const T *rec, float *out, int width, const int *itperm, int nt, hipStream_t st) {
  const long n = (long)width * nt;
  if (n <= 0) return;
  const dim3 g((unsigned)((n + 255) / 256)), b(256);
  if (width == 12)
    hipLaunchKernelGGL((k_tets_to_caller<T, 12>), g, b, 0, st, rec, out, itperm, n);
  else
    hipLaunchKernelGGL((k_tets_to_caller<T, 1>), g, b, 0, st, rec, out, itperm, n);
}
template void tets_to_caller<float>(const float *, float *, int, const int *, int, hipStream_t);
template void tets_to_caller<double>(const double *, float *, int, const int *, int, hipStream_t);
template <typename R>
void Launch<R>::aos_to_nodes(const float *aos, R *nodes, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_aos_to_nodes<float, R>), dim3(nblk(n, 256)), dim3(256), 0, st, aos, nodes, perm, n);
}
template <typename R>
void Launch<R>::nodes_to_aos64(const R *nodes, double *aos, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_nodes_to_aos<R, double>), dim3(nblk(n, 256)), dim3(256), 0, st, nodes, aos, perm, n);
}
void aos_to_planes_f(const float *aos, float *planes, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_aos_to_planes<float, float>), dim3(nblk(n, 256)), dim3(256), 0, st, aos, planes, perm, n);
}
void planes_to_aos_f(const float *planes, float *aos, const int *perm, int n, hipStream_t st) {
  hipLaunchKernelGGL((k_planes_to_aos<float, float>), dim3(nblk(n, 256)), dim3(256), 0, st, planes, aos, perm, n);
}

void fill_f(float *p, float v, long n, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(k_fill, dim3(nblk(n, 256)), dim3(256), 0, st, p, v, n);
}

template struct Launch<float>;
template struct Launch<double>;

}  // namespace pbs
