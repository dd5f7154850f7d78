// pbs_persist.hip -- the descent loop of a small mesh as one resident kernel.
//
// Three launches per pass (tile, node, control) take 9 to 15 us whatever the mesh's size, most of it
// launch latency and, every 32 passes, the host's read-back.  Here the whole loop is one cooperative
// launch: a workgroup owns a run of nodes (pbs_tiles.h, PersistPart), keeps its tets' rest shapes in
// registers and its positions in LDS, evaluates every tet that touches an owned node, steps its
// nodes, and exchanges only positions and the pass's two sums with the other workgroups.  Every
// workgroup then takes the loop's decision itself, from the same sums added in the same order.
//
// Values cross the workgroups as pbs_exchange.h says.
//
// Decisions.  Only a check pass can roll back, and only its sums are waited for at once.  On other
// passes the control goes on as if not converged; the sums are read during the next pass, while the
// other waves wait for the ghosts' positions.  If they say converged, that next pass is dropped: its
// step is not taken and the iterate before it is the result, as if the loop had stopped there.
//
// Slots.  There are 8, pass k uses slot k mod 8.  At the end of pass k a workgroup has the sums of
// pass k - 1 of all workgroups.  Each of them published those after it had consumed what pass k - 3
// published (positions in pass k - 3, sums in pass k - 2 at the latest), so the workgroup then clears
// its entries of pass k - 3.  The clearing is waited for (vmcnt) before it publishes its sums of pass
// k + 1.  A reader polls a slot in pass k when it has the sums of pass k - 2, whose owners had
// cleared what pass k - 6 and those before it published: it never meets what pass k - 8 left.
//
// Waiting ends: the launch is cooperative, so all workgroups are resident, and every poll is bounded;
// a workgroup that gives up sets *abort and ends, so do the others (one that has all values of the last
// pass writes its nodes back first), and the host starts the step again on the three launches.
//
// Bound: the chain of one pass, not bytes or arithmetic.  43 K tets, FP64: about 7,400 cycles, of
// which tets 2,000, gather 1,500, node step 700, the exchange of positions across the XCDs 2,500, the
// rest barriers.  The decisions (sums over the workgroups and the control, 4,600 cycles when waited
// for) are off that chain on all but check passes.  Wall time of a step, three launches -> resident:
// 1.5 K tets FP32, 96 passes, 876 -> 276 us; 43 K tets FP64, rel-grad 1e-4, 29.4 -> 7.3 ms.
//
// Iterates are bitwise those of the three launches as long as the loop decides alike (same functions,
// contributions added in the same groups and order).  The energy and |g|^2 are FP64 sums in another
// fixed order, so a decision can differ where one of them is within its last bits of the other side of
// a comparison; from there on alpha, the budget and the iterates do.
#include <algorithm>

#include "pbs_exchange.h"
#include "pbs_pass.h"
#include "pbs_persist.h"

namespace pbs {
namespace {

constexpr int T = kPersistThreads, NW = T / 64;
constexpr int CW = NW - 1;  // the wave that runs the loop's control: the last to have tets or nodes
// Sum over each 8 lanes, the same in all of them.
__device__ __forceinline__ double sum8(double v) {
  auto step = [&](auto ctrl) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, decltype(ctrl)::value, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
    v += __builtin_bit_cast(double, (unsigned long long)(unsigned)hi << 32 | (unsigned)lo);
  };
  step(std::integral_constant<int, 0xb1>());   // lanes 1 0 3 2 of each 4
  step(std::integral_constant<int, 0x4e>());   // lanes 2 3 0 1
  step(std::integral_constant<int, 0x141>());  // lanes 7 .. 0 of each 8
  return v;
}

template <typename R> __host__ __device__ inline size_t rec_offset(const PersistDev &d) {
  // after positions and saved positions (4 R per local node each) and rest positions (float4)
  return 8 * (size_t)d.local_max * sizeof(R) + 16 * (size_t)d.local_max;
}

// Sum of a node's run for one component, as the tile pass and the node pass form it: each tile's
// partial from zero in order, the partials added in order (A: the type of the sums).  Without
// branches: an entry that ends a partial moves it to the sum, others move zero (neither sum is ever
// -0).  What is read past the run (less than 2 U entries, inside the array) goes into a partial that
// nothing takes any more.
template <typename A, typename R>
__device__ __forceinline__ A run_sum(const R *__restrict__ rec, int len, unsigned long long mask) {
  constexpr int W = ContribWidth<R>::value, U = 8;
  A f = (A)0, a = (A)0;
  R t[U];
#pragma unroll
  for (int u = 0; u < U; ++u) t[u] = rec[W * u];
  for (int j = 0; j < len; j += U) {
    R next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) next[u] = rec[W * (j + U + u)];
    const unsigned m = (unsigned)(mask >> j);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool end = (m >> u) & 1;
      a += (A)t[u];
      f += end ? a : (A)0;
      a = end ? (A)0 : a;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) t[u] = next[u];
  }
  return f;
}

// What the control wave tells the others after a pass.
struct Next {
  int done, converged, late, rolled, chk, hd, cheb;  // late: the pass before had converged
  float alpha, omega;
};

template <typename R, int MAT, int K>
__global__ void __launch_bounds__(T)
k_persist(DevParams p, PersistDev d, Ctrl *__restrict__ ctrl, Ring<R> ring, const float4 *__restrict__ rest,
          float *__restrict__ hd, const float *__restrict__ mnode, const float *__restrict__ ext,
          const R *__restrict__ xt, const float *__restrict__ lame, int max_passes) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[2][NW];
  __shared__ Next next;
  __shared__ int gave_up;
  constexpr int W = ContribWidth<R>::value;
  R *sx = (R *)smem, *so = sx + 4 * d.local_max;
  float4 *srest = (float4 *)(so + 4 * d.local_max);
  R *rec = (R *)(smem + rec_offset<R>(d));
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, N = p.nn, G = d.nparts;
  const PersistPart pt = d.parts[blockIdx.x];
  // the control wave keeps the control block in registers
  Ctrl c = *ctrl;
  if (c.done) return;  // the same in every workgroup: nobody writes ctrl before all have published
  if (tid == 0) gave_up = 0;
  // positions of the local nodes: current and rollback iterate
  {
    const R *x = ring.b[c.cur], *xo = ring.b[c.old];
    for (int i = tid; i < 3 * (pt.own_cnt + pt.ghost_cnt); i += T) {
      const int l = i / 3, k = i % 3;
      const int n = l < pt.own_cnt ? pt.own_start + l : d.ghost[pt.ghost_off + l - pt.own_cnt];
      sx[4 * l + k] = x[3 * (size_t)n + k];
      so[4 * l + k] = xo[3 * (size_t)n + k];
      if (k == 0) srest[l] = rest[n];
    }
  }
  __syncthreads();
  const R mu = (R)lame[0], lam = (R)lame[1];
  // this thread's tets: local ids and slots, and what the neo-Hookean forces need of the rest shape
  uint4 lp[K];
  NeoRest<R> neo[K];
  auto get_r = [&](const uint4 &q, float (&r)[4][3]) {
    const int lid[4] = {(int)(q.x & 0xffff), (int)(q.x >> 16), (int)(q.y & 0xffff), (int)(q.y >> 16)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float4 v = srest[lid[c]];
      r[c][0] = v.x;
      r[c][1] = v.y;
      r[c][2] = v.z;
    }
  };
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (pt.tet_cnt == 0) break;
    lp[k] = d.lp[pt.tet_off + min(tid + k * T, pt.tet_cnt - 1)];
    if (MAT == 0) {
      float r[4][3];
      get_r(lp[k], r);
      neo[k] = NeoRest<R>(r, mu);
    }
  }
  // this thread's node component: 21 nodes per wave, 3 lanes each
  const int own = w * 21 + lane / 3, dc = lane % 3;
  const bool mine = lane < 63 && own < pt.own_cnt;
  const int n = pt.own_start + (mine ? own : 0);
  const size_t ni = 3 * (size_t)n + dc;
  const float m = mnode[n];
  const bool fixed = m < 0.0f;
  const R hstep = (R)p.h, mh2 = (R)m / (hstep * hstep), xtv = xt[ni];
  R fe = (R)(p.grav[dc] * m);
  if (p.has_ext) fe += (R)ext[(size_t)dc * N + n];
  R x = ring.b[c.cur][ni], xl = ring.b[c.last][ni], xo = ring.b[c.old][ni];
  float hv = hd[ni];
  const int r0 = mine ? d.run[pt.run_off + own] : 0, len = mine ? d.run[pt.run_off + own + 1] - r0 : 0;
  const unsigned long long mask = mine ? d.mask[pt.run_off + own] : 0ULL;
  // ghost components, entries 3 ghost + component, over the threads of the other waves
  constexpr int GH = (3 * kPersistGhosts + T - 65) / (T - 64);
  int gnode[GH], gl[GH];
#pragma unroll
  for (int u = 0; u < GH; ++u) {
    const int i = tid + u * (T - 64), g = i / 3;
    const bool on = w != CW && g < pt.ghost_cnt;
    gnode[u] = on ? 3 * d.ghost[pt.ghost_off + g] + i % 3 : -1;
    gl[u] = 4 * (pt.own_cnt + g) + i % 3;
  }
  R *xch = (R *)d.xch;
  __syncthreads();
  int chk = c.check_now, hdnow = c.hd_now, cheb = c.cheb_now;
  R alpha = (R)c.alpha, om = (R)c.omega_next;
  // control wave: whether the pass before has its verdict pending, its sums as read at the pass's start,
  // k modulo the refresh and check periods, and the last k of the Chebyshev profile
  bool pending = false;
  unsigned long long be[4], bg[4];
  int khd = c.k % p.hd_refresh, kchk = c.k % p.energy_check, kprof = 0;
  for (int i = 0; i < p.profile_n; ++i) kprof = max(kprof, p.profile_k[i]);
  auto read_sums = [&](int q, bool energy) {
    const double *pp = d.part + (size_t)q * G * 2;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = lane + 64 * u;
      be[u] = energy && i < G ? poll(pp + 2 * i) : 0;
      bg[u] = i < G ? poll(pp + 2 * i + 1) : 0;
    }
  };
  for (int pass = 0; pass < max_passes; ++pass) {
    const int slot = pass & (kPersistSlots - 1);
    const int before = (pass + kPersistSlots - 1) & (kPersistSlots - 1);
    const int polls = pass < d.from ? kPolls : d.polls;
    if (w == CW && pending) read_sums(before, false);
    double e_el = 0.0;
    // forces of this workgroup's tets into the contribution slots; phase 1: the stiffness diagonal
    auto tets_phase = [&](auto ph) {
      constexpr int phase = decltype(ph)::value;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (tid + k * T < pt.tet_cnt) {
          uint4 q = lp[k];
          const int count = q.z >> 31;
          q.z &= 0x7fffffffu;
          tile_tet<R, R, MAT, phase>(q, [&](float (&r)[4][3]) { get_r(q, r); }, [&]() { return neo[k]; }, sx, rec, mu, lam,
                                     chk & count, p.clamp, e_el);
        }
    };
    tets_phase(std::integral_constant<int, 0>());
    __syncthreads();
    const R f = run_sum<R>(rec + W * r0 + dc, len, mask);
    if (hdnow) {
      __syncthreads();
      tets_phase(std::integral_constant<int, 1>());
      __syncthreads();
      hv = run_sum<float>(rec + W * r0 + dc, len, mask);
    }
    // node step (k_node's formulas per component)
    R nx = x;
    double en = 0.0, g2 = 0.0;
    {
      const R dd = x - xtv;
      const R gr = dd * mh2 - f - (R)p.ext_scale * fe;
      if (chk) {
        const R term = (R)0.5 * dd * dd * mh2 - fe * x;
        const R t1 = __shfl_down(term, 1, 64), t2 = __shfl_down(term, 2, 64);
        R e = (R)0;
        e += term;
        e += t1;
        e += t2;
        if (mine && !fixed && dc == 0) en = (double)e;
      }
      if (mine && !fixed) {
        g2 = (double)gr * (double)gr;
        nx = x - alpha * gr / ((R)hv + mh2);
        if (cheb) nx = om * (nx - xl) + xl;
      }
    }
    // clearings of the pass before are complete before this workgroup's sums are published
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (mine) publish(xch + (size_t)slot * 3 * N + 3 * (size_t)n + dc, nx);
    {
      const double ew = chk ? wave_sum(e_el + en) : 0.0, gw = wave_sum(g2);
      if (lane == 0) {
        red[0][w] = ew;
        red[1][w] = gw;
      }
    }
    // own positions; after a check the old iterate is still needed: then they wait for the verdict
    if (!chk && mine) sx[4 * own + dc] = nx;
    __syncthreads();
    typename Bits<R>::type gv[GH];
    if (w == 0 && G > 1 && lane < 16) {  // this workgroup's sums: energy in lanes 0 to 7, |g|^2 in 8 to 15
      const double v = sum8(red[lane >> 3][lane & 7]);
      if ((lane & 7) == 0) publish(d.part + ((size_t)slot * G + blockIdx.x) * 2 + (lane >> 3), v);
    }
    if (w == CW) {  // the loop's decision
      // the sums over all workgroups (G <= 256), read again until all are there
      auto sums = [&](int q, bool energy, double &E, double &g) {
        int spin = 0;
        while (true) {
          bool wait = false;
#pragma unroll
          for (int u = 0; u < 4; ++u) wait = wait || be[u] == Bits<double>::none || bg[u] == Bits<double>::none;
          if (!wait) break;
          if (give_up(spin, polls, d.abort)) {
            gave_up = 1;
            break;
          }
          read_sums(q, energy);
        }
        double pe = 0.0, pg = 0.0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          pe += __builtin_bit_cast(double, be[u]);
          pg += __builtin_bit_cast(double, bg[u]);
        }
        E = wave_sum(pe);
        g = wave_sum(pg);
      };
      bool now = chk || c.k + 1 >= c.budget || pass + 1 == max_passes;
      const int rb0 = c.rollbacks;
      const double tol = p.relgrad_tol * c.g0, far = 1.001 * (tol * tol);
      double E = 0.0, g = 0.0;
      bool late = false;
      if (G == 1) {
#pragma unroll
        for (int i = 0; i < NW; ++i) {
          E += red[0][i];
          g += red[1][i];
        }
        now = now || (p.relgrad_tol > 0.0 && !(g > far));
      }
      if (pending) {  // the pass before: the control went on as if it had not converged
        sums(before, false, E, g);
        if (p.relgrad_tol > 0.0 && !(g > far)) {  // (mostly it is, and the root is not needed)
          c.g = sqrt(g);
          late = c.g <= tol;
        }
        if (late) {
          --c.k;
          c.converged = c.done = 1;
        }
      }
      pending = G > 1 && !late && !now;
      if (!late && !now) {  // as control_apply on a pass that neither checks nor ends the loop
        c.rho = c.rho_next;
        c.omega = c.omega_next;
        ++c.k;
        ++c.passes;
        khd = khd + 1 == p.hd_refresh ? 0 : khd + 1;
        kchk = kchk + 1 == p.energy_check ? 0 : kchk + 1;
        c.hd_now = khd == 0;
        c.check_now = kchk == 0;
        float rho = c.rho, o = c.omega;
        if (c.k - c.kc <= kprof) cheb_schedule(p, c.k - c.kc, rho, o);
        else o = 4.0f / (4.0f - rho * rho * o);
        c.rho_next = rho;
        c.omega_next = o;
        c.cheb_now = o != 1.0f;
      } else if (!late) {
        if (G > 1) {
          read_sums(slot, chk != 0);
          sums(slot, chk != 0, E, g);
        }
        control_apply(p, c, E, g);
        khd = c.k % p.hd_refresh;
        kchk = c.k % p.energy_check;
      }
      if (lane == 0)
        next = {c.done, c.converged, late, c.rollbacks != rb0, c.check_now, c.hd_now, c.cheb_now, c.alpha, c.omega_next};
    } else {  // the ghosts' new positions
      bool wait;
      int spin = 0;
      do {
        wait = false;
#pragma unroll
        for (int u = 0; u < GH; ++u) gv[u] = gnode[u] >= 0 ? poll(xch + (size_t)slot * 3 * N + gnode[u]) : 0;
#pragma unroll
        for (int u = 0; u < GH; ++u) wait = wait || gv[u] == Bits<R>::none;
        if (wait && give_up(spin, polls, d.abort)) {
          gave_up = 1;
          break;
        }
      } while (wait);
      if (!chk) {
#pragma unroll
        for (int u = 0; u < GH; ++u)
          if (gnode[u] >= 0) sx[gl[u]] = __builtin_bit_cast(R, gv[u]);
      }
    }
    __syncthreads();
    if (gave_up) {
      if (tid == 0) __hip_atomic_store(d.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    const Next nt = next;
    // clear what was published three passes ago
    const int was = (pass + kPersistSlots - 3) & (kPersistSlots - 1);
    if (pass >= 3) {
      if (mine) clear(xch + (size_t)was * 3 * N + 3 * (size_t)n + dc);
      if (G > 1 && tid < 2) clear(d.part + ((size_t)was * G + blockIdx.x) * 2 + tid);
    }
    if (nt.converged) {  // the iterate the forces were evaluated at is the result
      if (nt.late) x = xl;
      break;
    }
    if (chk) {
      const int locals = pt.own_cnt + pt.ghost_cnt;
      if (nt.rolled) {  // back to the iterate of the last accepted check
        for (int i = tid; i < 4 * locals; i += T) sx[i] = so[i];
      } else {
        for (int i = tid; i < 4 * locals; i += T) so[i] = sx[i];
        __syncthreads();
        if (mine) sx[4 * own + dc] = nx;
        if (w != CW) {
#pragma unroll
          for (int u = 0; u < GH; ++u)
            if (gnode[u] >= 0) sx[gl[u]] = __builtin_bit_cast(R, gv[u]);
        }
      }
      __syncthreads();
    }
    if (nt.rolled) {
      x = xo;
    } else {
      if (chk) xo = x;
      xl = x;
      x = nx;
    }
    chk = nt.chk;
    hdnow = nt.hd;
    cheb = nt.cheb;
    alpha = (R)nt.alpha;
    om = (R)nt.omega;
    if (nt.done) break;
  }
  // state back in fixed roles
  if (mine) {
    ring.b[0][ni] = x;
    ring.b[1][ni] = xl;
    ring.b[2][ni] = xo;
    hd[ni] = hv;
  }
  if (blockIdx.x == 0 && tid == 64 * CW) {
    c.cur = 0;
    c.last = 1;
    c.old = 2;
    c.nxt = 3;
    *ctrl = c;
  }
}

__global__ void k_persist_fill(uint4 *__restrict__ p, long n, int *__restrict__ abort) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  if (i == 0) *abort = 0;
}

template <typename R> const void *kernel_of(int material, int tet_max) {
  const int k = (tet_max + T - 1) / T;
  if (material == 0)
    return k <= 1 ? (const void *)k_persist<R, 0, 1> : k == 2 ? (const void *)k_persist<R, 0, 2> : (const void *)k_persist<R, 0, 4>;
  return k <= 1 ? (const void *)k_persist<R, 1, 1> : k == 2 ? (const void *)k_persist<R, 1, 2> : (const void *)k_persist<R, 1, 4>;
}

}  // namespace

template <typename R> size_t PersistLaunch<R>::lds_bytes(const PersistDev &d) {
  return rec_offset<R>(d) + (size_t)ContribWidth<R>::value * d.slot_max * sizeof(R);
}
template <typename R> int PersistLaunch<R>::max_resident(const PersistDev &d, int material, int device) {
  int coop = 0, cus = 0, per = 0;
  if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess || !coop) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel_of<R>(material, d.tet_max), T, lds_bytes(d)) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return per > 0 ? cus : 0;  // one per CU: the loop's latency, not its occupancy, is what counts
}
template <typename R>
hipError_t PersistLaunch<R>::run(const DevMesh<R> &m, const TileDev &td, const DevParams &p, const PersistDev &d,
                                 int max_passes, hipStream_t st) {
  const long n16 = d.xch_bytes / 16;
  hipLaunchKernelGGL(k_persist_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st, (uint4 *)d.xch, n16, d.abort);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  DevParams dp = p;
  PersistDev pd = d;
  Ctrl *ctrl = m.ctrl;
  Ring<R> ring = m.ring;
  const float4 *rest = m.rest4;
  const float *mnode = m.mnode, *ext = m.ext, *lame = td.inst_mu;
  float *hd = m.hd;
  const R *xt = m.xt;
  void *args[] = {&dp, &pd, &ctrl, &ring, &rest, &hd, &mnode, &ext, &xt, &lame, &max_passes};
  return hipLaunchCooperativeKernel(kernel_of<R>(p.material, d.tet_max), dim3(d.nparts), dim3(T), args,
                                    (unsigned)lds_bytes(d), st);
}
template struct PersistLaunch<float>;
template struct PersistLaunch<double>;

}  // namespace pbs
