// pbs_persist.hip -- the descent loop of a small mesh as one resident kernel.
//
// Three launches per pass (tile, node, control) take 9 to 15 us whatever the mesh's size, most of it
// launch latency and, every 32 passes, the host's read-back.  Here the whole loop is one cooperative
// launch: a workgroup owns a run of nodes (pbs_tiles.h, PersistPart), keeps its tets' rest shapes in
// registers and its positions in LDS, evaluates every tet that touches an owned node, steps its
// nodes, and exchanges only positions and the pass's two sums with the other workgroups.  Every
// workgroup then takes the loop's decision itself, from the same sums added in the same order.
//
// Exchange.  Values cross workgroups as relaxed atomics at agent scope (8 or 4 bytes each, written
// through to and read from the point where all XCDs see them), and they are their own flags: a slot
// holds all-ones bits until its owner has written it, a reader polls until it does not (a computed
// value with that bit pattern, a NaN, is replaced by another NaN).  There are 4 slots, pass k uses
// slot k mod 4.  An owner clears its entries of slot k - 1 once it has the sums of pass k of all
// workgroups: each of them has then consumed pass k - 1.  The clearing is waited for (vmcnt) before
// the workgroup publishes its sums of pass k + 1, and a reader polls slot k + 3 only after it has
// seen those, so it never meets what was published in pass k - 1.
//
// Waiting ends: the launch is cooperative, so all workgroups are resident, and every poll is bounded;
// a workgroup that gives up sets *abort and ends, so do the others, nothing is written back, and the
// host runs the step through the three launches.
//
// Bound: the chain of one pass (tets, gather, two block sums, one exchange across the XCDs) and not
// bytes or arithmetic.  Wall time of a step, three launches -> resident: 1.5 K tets FP32, 96 passes,
// 875 -> 417 us; 43 K tets FP64, rel-grad 1e-4, 28.0 -> 13.8 ms.
//
// Iterates are bitwise those of the three launches (same functions, contributions added in the same
// groups and order); the energy and |g|^2 are FP64 sums in another fixed order.
#include <algorithm>

#include "pbs_pass.h"
#include "pbs_persist.h"

namespace pbs {
namespace {

constexpr int T = kPersistThreads, NW = T / 64;
constexpr int kSpin = 1 << 20;  // polls before giving up (about a second)

template <typename R> struct Bits;
template <> struct Bits<double> {
  typedef unsigned long long type;
  static constexpr type none = ~0ULL, nan = 0x7ff8000000000000ULL;
};
template <> struct Bits<float> {
  typedef unsigned type;
  static constexpr type none = ~0U, nan = 0x7fc00000U;
};
template <typename R> __device__ __forceinline__ void publish(R *p, R v) {
  typedef typename Bits<R>::type B;
  B b = __builtin_bit_cast(B, v);
  if (b == Bits<R>::none) b = Bits<R>::nan;
  __hip_atomic_store((B *)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename R> __device__ __forceinline__ void clear(R *p) {
  __hip_atomic_store((typename Bits<R>::type *)p, Bits<R>::none, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename R> __device__ __forceinline__ typename Bits<R>::type poll(const R *p) {
  return __hip_atomic_load((const typename Bits<R>::type *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename R> __host__ __device__ inline size_t rec_offset(const PersistDev &d) {
  // after positions and saved positions (4 R per local node each) and rest positions (float4)
  return 8 * (size_t)d.local_max * sizeof(R) + 16 * (size_t)d.local_max;
}

// Sum of a node's run for one component, as the tile pass and the node pass form it: each tile's
// partial from zero in order, the partials added in order (A: the type of the sums).
template <typename A, typename R>
__device__ __forceinline__ A run_sum(const R *__restrict__ rec, int len, unsigned long long mask) {
  constexpr int W = ContribWidth<R>::value, U = 4;
  A f = (A)0, a = (A)0;
  for (int j = 0; j < len; j += U) {
    R t[U];
#pragma unroll
    for (int u = 0; u < U; ++u) t[u] = rec[W * (j + u < len ? j + u : 0)];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (j + u < len) {
        a += (A)t[u];
        if ((mask >> (j + u)) & 1) {
          f += a;
          a = (A)0;
        }
      }
  }
  return f;
}

template <typename R, int MAT, int K>
__global__ void __launch_bounds__(T)
k_persist(DevParams p, PersistDev d, Ctrl *__restrict__ ctrl, Ring<R> ring, const float4 *__restrict__ rest,
          float *__restrict__ hd, const float *__restrict__ mnode, const float *__restrict__ ext,
          const R *__restrict__ xt, const float *__restrict__ lame, int max_passes) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Ctrl C;
  __shared__ double red[2][NW];
  __shared__ int gave_up;
  constexpr int W = ContribWidth<R>::value;
  R *sx = (R *)smem, *so = sx + 4 * d.local_max;
  float4 *srest = (float4 *)(so + 4 * d.local_max);
  R *rec = (R *)(smem + rec_offset<R>(d));
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, N = p.nn, G = d.nparts;
  const PersistPart pt = d.parts[blockIdx.x];
  if (tid == 0) {
    C = *ctrl;
    gave_up = 0;
  }
  __syncthreads();
  if (C.done) return;  // the same in every workgroup: nobody has written ctrl yet
  // positions of the local nodes: current and rollback iterate
  {
    const R *x = ring.b[C.cur], *xo = ring.b[C.old];
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
  R x = ring.b[C.cur][ni], xl = ring.b[C.last][ni], xo = ring.b[C.old][ni];
  float hv = hd[ni];
  const int r0 = mine ? d.run[pt.run_off + own] : 0, len = mine ? d.run[pt.run_off + own + 1] - r0 : 0;
  const unsigned long long mask = mine ? d.mask[pt.run_off + own] : 0ULL;
  // this thread's ghost components: entries 3 ghost + component
  constexpr int GH = 4;
  int gnode[GH], gl[GH];
#pragma unroll
  for (int u = 0; u < GH; ++u) {
    const int i = tid + u * T, g = i / 3;
    const bool on = g < pt.ghost_cnt;
    gnode[u] = on ? 3 * d.ghost[pt.ghost_off + g] + i % 3 : -1;
    gl[u] = 4 * (pt.own_cnt + g) + i % 3;
  }
  R *xch = (R *)d.xch;
  __syncthreads();
  for (int pass = 0; pass < max_passes; ++pass) {
    const int slot = pass & 3;
    const int chk = C.check_now, hdnow = C.hd_now, cheb = C.cheb_now;
    const R alpha = (R)C.alpha, om = (R)C.omega_next;
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
    // clearings of the pass before are complete before this workgroup's sums are published
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
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
      const R term = (R)0.5 * dd * dd * mh2 - fe * x;
      const R t1 = __shfl_down(term, 1, 64), t2 = __shfl_down(term, 2, 64);
      if (mine && !fixed) {
        R e = (R)0;
        e += term;
        e += t1;
        e += t2;
        if (dc == 0) en = (double)e;
        g2 = (double)gr * (double)gr;
        nx = x - alpha * gr / ((R)hv + mh2);
        if (cheb) nx = om * (nx - xl) + xl;
      }
    }
    if (mine) publish(xch + (size_t)slot * 3 * N + 3 * (size_t)n + dc, nx);
    if (G > 1) {
      const double ew = wave_sum(e_el + en), gw = wave_sum(g2);
      if (lane == 0) {
        red[0][w] = ew;
        red[1][w] = gw;
      }
      __syncthreads();
      if (tid < 2) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < NW; ++i) v += red[tid][i];
        publish(d.part + ((size_t)slot * G + blockIdx.x) * 2 + tid, v);
      }
    }
    // the sums of all workgroups and the ghosts' new positions
    double pe = e_el + en, pg = g2;
    typename Bits<R>::type gv[GH];
    {
      unsigned long long be = 0, bg = 0;
      const double *pp = d.part + ((size_t)slot * G + tid) * 2;
      bool wait;
      int spin = 0;
      do {
        wait = false;
        if (G > 1 && tid < G) {
          be = poll(pp);
          bg = poll(pp + 1);
        }
#pragma unroll
        for (int u = 0; u < GH; ++u) gv[u] = gnode[u] >= 0 ? poll(xch + (size_t)slot * 3 * N + gnode[u]) : 0;
        if (G > 1 && tid < G) wait = be == Bits<double>::none || bg == Bits<double>::none;
#pragma unroll
        for (int u = 0; u < GH; ++u) wait = wait || gv[u] == Bits<R>::none;
        if (wait && (++spin >= kSpin || (spin % 1024 == 0 && __hip_atomic_load(d.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))) {
          gave_up = 1;
          break;
        }
      } while (wait);
      if (G > 1) {
        pe = tid < G ? __builtin_bit_cast(double, be) : 0.0;
        pg = tid < G ? __builtin_bit_cast(double, bg) : 0.0;
        __syncthreads();  // red is read
      }
    }
    {
      const double ew = wave_sum(pe), gw = wave_sum(pg);
      if (lane == 0) {
        red[0][w] = ew;
        red[1][w] = gw;
      }
    }
    __syncthreads();
    if (gave_up) {
      if (tid == 0) __hip_atomic_store(d.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    const bool had_check = chk != 0;
    const int rb0 = C.rollbacks;
    __syncthreads();
    if (tid == 0) {
      double E = 0.0, g = 0.0;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        E += red[0][i];
        g += red[1][i];
      }
      Ctrl c = C;
      control_apply(p, c, E, g);
      C = c;
    }
    __syncthreads();
    // clear what the pass before published
    const int was = (pass + 3) & 3;
    if (pass > 0) {
      if (mine) clear(xch + (size_t)was * 3 * N + 3 * (size_t)n + dc);
      if (G > 1 && tid < 2) clear(d.part + ((size_t)was * G + blockIdx.x) * 2 + tid);
    }
    if (C.converged) break;  // the iterate the forces were evaluated at is the result
    const int locals = pt.own_cnt + pt.ghost_cnt;
    if (C.rollbacks != rb0) {  // back to the iterate of the last accepted check
      x = xo;
      for (int i = tid; i < 4 * locals; i += T) sx[i] = so[i];
    } else {
      if (had_check) {
        xo = x;
        for (int i = tid; i < 4 * locals; i += T) so[i] = sx[i];
        __syncthreads();
      }
      xl = x;
      x = nx;
      if (mine) sx[4 * own + dc] = nx;
#pragma unroll
      for (int u = 0; u < GH; ++u)
        if (gnode[u] >= 0) sx[gl[u]] = __builtin_bit_cast(R, gv[u]);
    }
    __syncthreads();
    if (C.done) break;
  }
  // state back in fixed roles
  if (mine) {
    ring.b[0][ni] = x;
    ring.b[1][ni] = xl;
    ring.b[2][ni] = xo;
    hd[ni] = hv;
  }
  if (blockIdx.x == 0 && tid == 0) {
    Ctrl c = C;
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
