// pbs_implicit.hip -- kernels of the backward-Euler step (computeInnerforces,
// computeGlobalStiffnessMatrix and doBackEuler, CUDAInterface.cu:784-884, as driven by
// fvm.cpp:179-183).
//
// The reference scatters 144 float atomics per tet into a CSR matrix (computeGlobalK,
// CUDAInterface.cu:234-271) and solves with a sparse Cholesky factorisation.  Here one thread
// owns one block row (a node): it walks the node's incident tets in a fixed order, evaluates the
// 3x12 stiffness strip of its corner in closed form and accumulates it into its own SELL-64
// slots, so the assembly is deterministic and atomic-free; the solve is a Jacobi-preconditioned
// conjugate gradient in FP64 whose scalars stay on the device.
#include <algorithm>

#include <hip/hip_ext.h>

#include "pbs_device.h"
#include "pbs_exchange.h"
#include "pbs_implicit.h"

namespace pbs {
namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ size_t val_idx(long group, int q, int lane) {
  return ((size_t)group * 9 + q) * 64 + lane;
}

// XCD-contiguous block order: workgroup i runs on XCD i % 8; giving each XCD a contiguous range
// of row blocks keeps a row's neighbours (mostly in the same or the adjacent blocks, in Morton
// order) in that XCD's L2.
__device__ __forceinline__ int xcd_block(int bid, int nblk) {
  const int per = (nblk + 7) >> 3;
  const int xcd = bid & 7, k = bid >> 3;
  const int full = nblk - 8 * (per - 1);
  const int start = xcd < full ? xcd * per : full * per + (xcd - full) * (per - 1);
  return start + k;
}

// Sum of v over the 256 threads of the block in a fixed order (wave tree, then the 4 waves).
__device__ __forceinline__ double block_sum256(double v, double *lds) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) lds[w] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0) t = (lds[0] + lds[1]) + (lds[2] + lds[3]);
  __syncthreads();
  return t;
}

// Sum of nb per-block partials by one block of NT threads in a fixed order, in two halves so that
// other loads can be issued in between: the first takes the thread's first 8 terms v[tid], v[tid +
// NT], ... (indices past the end clamped, not added later), the second adds them, any further ones
// and the block's threads; every thread of the block gets the sum.
template <int NT> struct PartialSum {
  double t[8];
  __device__ __forceinline__ void load(const double *__restrict__ v, int nb, int base = 0) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = base + u * NT + (int)threadIdx.x;
      t[u] = v[i < nb ? i : nb - 1];
    }
  }
  __device__ __forceinline__ double sum(const double *__restrict__ v, int nb, double *lds) {
    double a = 0.0;
    for (int base = 0;;) {
#pragma unroll
      for (int u = 0; u < 8; ++u) a += base + u * NT + (int)threadIdx.x < nb ? t[u] : 0.0;
      base += 8 * NT;
      if (base >= nb) break;
      load(v, nb, base);
    }
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = a;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) r += lds[i];
    return r;
  }
};

// The partials of p.Ap (one per slice) as PartialSum takes them: where the vector passes' blocks are
// whole slices, each block's slices are added first (at most 4 each, 512 blocks).
__device__ __forceinline__ int first_slice(const IeDev &d, int b) { return b * d.vec_per + min(b, d.vec_rem); }
__device__ __forceinline__ void load_pap(const IeDev &d, PartialSum<256> &part) {
  if (d.vec_unit != 192) {
    part.load(d.part_pap, d.nslice);
    return;
  }
  double v[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int b = min(u * 256 + (int)threadIdx.x, d.vec_blocks - 1), s = first_slice(d, b), n = first_slice(d, b + 1) - s;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[u][i] = i < n ? d.part_pap[s + i] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) part.t[u] = ((v[u][0] + v[u][1]) + v[u][2]) + v[u][3];
#pragma unroll
  for (int u = 2; u < 8; ++u) part.t[u] = 0.0;
}

// y += (row `lane` of the slice's A) v over the slots first, first + step, ... below the slice's
// width.  BLK = 3: 3x3 blocks (9 values per slot); BLK = 1: one value per slot, the block being
// that value times the 3x3 identity.  get(col, v0, v1, v2) supplies v at a column.
template <typename R, int BLK, typename Get>
__device__ __forceinline__ void row_apply(const IeDev &d, int n, int first, int step, Get get, double *y) {
  const R *__restrict__ A = (const R *)d.A;
  // all lanes run to the slice width (padding slots hold zeros and the row's own column), so the
  // loop is uniform across the wavefront and can be unrolled to overlap its loads
  const int lane = n & 63, g0 = d.slice_off[n >> 6], width = d.slice_off[(n >> 6) + 1] - g0;
#pragma unroll 2
  for (int j = first; j < width; j += step) {
    const int col = d.bcol[(size_t)(g0 + j) * 64 + lane];
    double x0, x1, x2;
    get(col, x0, x1, x2);
    if (BLK == 3) {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        y[q] += (double)A[val_idx(g0 + j, 3 * q, lane)] * x0 + (double)A[val_idx(g0 + j, 3 * q + 1, lane)] * x1 +
                (double)A[val_idx(g0 + j, 3 * q + 2, lane)] * x2;
    } else {
      const double a = (double)A[(size_t)(g0 + j) * 64 + lane];
      y[0] += a * x0;
      y[1] += a * x1;
      y[2] += a * x2;
    }
  }
}

// Slot (within the row) of column `col`: the row's columns are ascending.
__device__ __forceinline__ int find_col(const int *__restrict__ bcol, int g0, int lane, int len, int col) {
  int lo = 0, hi = len - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (bcol[(size_t)(g0 + mid) * 64 + lane] < col) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// ---------------------------------------------------------------------------------------------
// Assembly.  For node n at corner i of an incident tet, with shape vectors c_m (rows of Dm^-1,
// c_0 = -(c_1 + c_2 + c_3)), g_m = F^-T c_m and V the rest volume, the stiffness block
// K(i,j)[d][e] = -d f_i[d] / d x_j[e] is
//   neo-Hookean: V [ mu (c_i . c_j) delta_de + (mu - lambda ln J) g_j[d] g_i[e] + lambda g_i[d] g_j[e] ]
//   stretch:     V [ 2 mu ((c_i . c_j) delta_de - sum_{k<l} (a^d_kl . c_i)(a^e_kl . c_j) / (s_k + s_l))
//                    + lambda ((2J - 1) J g_i[d] g_j[e] - (J - 1) J g_i[e] g_j[d]) ]
// with a^d_kl[b] = U_dk V_bl - U_dl V_bk (F = U diag(s) V^T): the closed form of the
// derivative the reference evaluates through the SVD and Xu et al. 2015's 2x2 solves
// (compute_dfdx, CUDAInterface.cu:101-219).  The elastic force of the corner comes from the same
// per-tet routine as the descent solver's.
// LACC: the row (`row`) is accumulated in LDS (one 64-row slice per workgroup, each lane its own
// column of slots, so no lane touches another's) and written to the matrix once; otherwise it is
// accumulated in place in the matrix.
// ---------------------------------------------------------------------------------------------
template <typename R, int MAT, bool LACC>
__global__ void __launch_bounds__(kBlock)
    k_ie_assemble(DevParams p, IeAsm a, IeDev d, const int4 *__restrict__ tets, const float *__restrict__ dmi,
                  const float *__restrict__ vol, const int *__restrict__ inc_off, const int *__restrict__ inc,
                  const R *__restrict__ xpos, const R *__restrict__ vel, const float *__restrict__ rest,
                  const float *__restrict__ mass, const float *__restrict__ gforce, const float *__restrict__ ext,
                  const int *__restrict__ mask, const float *__restrict__ inst_mu, const float *__restrict__ inst_lam) {
  extern __shared__ __align__(16) unsigned char ie_lds[];
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= d.n) return;
  R *__restrict__ A = (R *)d.A;
  const int N = p.nn, T = p.nt;
  const int lane = n & 63;
  const int g0 = d.slice_off[n >> 6];
  const int width = d.slice_off[(n >> 6) + 1] - g0;
  const int len = d.row_len[n];
  R *__restrict__ row = LACC ? (R *)ie_lds : A;
  auto ix = [&](int j, int q) -> size_t { return LACC ? ((size_t)j * 9 + q) * 64 + lane : val_idx(g0 + j, q, lane); };
  for (int j = 0; j < width; ++j)
#pragma unroll
    for (int q = 0; q < 9; ++q) row[ix(j, q)] = (R)0;
  const R mu = (R)inst_mu[0], lam = (R)inst_lam[0];
  R f[3] = {(R)0, (R)0, (R)0};
  for (int e = inc_off[n]; e < inc_off[n + 1]; ++e) {
    const int t = inc[e] >> 2, ci = inc[e] & 3;
    const int4 q4 = tets[t];
    const int qn[4] = {q4.x, q4.y, q4.z, q4.w};
    R Dmi[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) Dmi[k] = (R)dmi[(size_t)k * T + t];
    const R V = (R)vol[t];
    R X[4][3];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int k = 0; k < 3; ++k) X[c][k] = xpos[(size_t)k * N + qn[c]];
    R Ds[9], F[9];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      Ds[3 * k + 0] = X[1][k] - X[0][k];
      Ds[3 * k + 1] = X[2][k] - X[0][k];
      Ds[3 * k + 2] = X[3][k] - X[0][k];
    }
    mul3(Ds, Dmi, F);
    R f12[12], en;
    if (MAT == 0) neo_tet<R, false>(F, Dmi, V, mu, lam, f12, en, nullptr);
    else stretch_tet<R, false>(F, Dmi, V, mu, lam, f12, en, nullptr);
#pragma unroll
    for (int k = 0; k < 3; ++k) f[k] += f12[3 * ci + k];
    R C[9];
    const R J = adj3(F, C);
    const R iJ = (R)1 / J;
    R c[4][3], g[4][3];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      shape_vec(Dmi, m, c[m]);
#pragma unroll
      for (int k = 0; k < 3; ++k) g[m][k] = (c[m][0] * C[k] + c[m][1] * C[3 + k] + c[m][2] * C[6 + k]) * iJ;
    }
    R ci3[3], gi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // corner ci's vectors, selected without dynamic register indexing
      ci3[k] = ci == 0 ? c[0][k] : ci == 1 ? c[1][k] : ci == 2 ? c[2][k] : c[3][k];
      gi[k] = ci == 0 ? g[0][k] : ci == 1 ? g[1][k] : ci == 2 ? g[2][k] : g[3][k];
    }
    R k1, k2;          // coefficients of g_j[d] g_i[e] and g_i[d] g_j[e]
    R ai[3][3] = {};   // stretch: (a^d_kl . c_i) for the pairs kl = 01, 02, 12
    R aw[3] = {};      // stretch: 1 / (s_k + s_l)
    R U[9] = {}, Vv[9] = {};
    if (MAT == 0) {
      const R lj = dlog(J);
      k1 = mu - lam * lj;
      k2 = lam;
    } else {
      R S[3];
      svd3(F, U, S, Vv);
      k1 = -lam * (J - (R)1) * J;
      k2 = lam * ((R)2 * J - (R)1) * J;
      const int kk[3] = {0, 0, 1}, ll[3] = {1, 2, 2};
      const R lim = (sizeof(R) == 4 ? (R)1e-6 : (R)1e-12);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const R den = S[kk[q]] + S[ll[q]];
        aw[q] = (R)1 / (den > lim ? den : lim);
#pragma unroll
        for (int dd = 0; dd < 3; ++dd) {
          R acc = (R)0;
#pragma unroll
          for (int b = 0; b < 3; ++b)
            acc += (U[3 * dd + kk[q]] * Vv[3 * b + ll[q]] - U[3 * dd + ll[q]] * Vv[3 * b + kk[q]]) * ci3[b];
          ai[q][dd] = acc;
        }
      }
    }
    const R mu2 = (MAT == 0) ? mu : (R)2 * mu;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int slot_j = find_col(d.bcol, g0, lane, len, qn[m]);
      const R cc = ci3[0] * c[m][0] + ci3[1] * c[m][1] + ci3[2] * c[m][2];
      R aj[3][3];
      if (MAT != 0) {
        const int kk[3] = {0, 0, 1}, ll[3] = {1, 2, 2};
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
          for (int ee = 0; ee < 3; ++ee) {
            R acc = (R)0;
#pragma unroll
            for (int b = 0; b < 3; ++b)
              acc += (U[3 * ee + kk[q]] * Vv[3 * b + ll[q]] - U[3 * ee + ll[q]] * Vv[3 * b + kk[q]]) * c[m][b];
            aj[q][ee] = acc;
          }
      }
#pragma unroll
      for (int dd = 0; dd < 3; ++dd)
#pragma unroll
        for (int ee = 0; ee < 3; ++ee) {
          R kv = (dd == ee ? mu2 * cc : (R)0) + k1 * g[m][dd] * gi[ee] + k2 * gi[dd] * g[m][ee];
          if (MAT != 0) {
            R rot = (R)0;
#pragma unroll
            for (int q = 0; q < 3; ++q) rot += ai[q][dd] * aj[q][ee] * aw[q];
            kv -= mu2 * rot;
          }
          row[ix(slot_j, 3 * dd + ee)] += V * kv;
        }
    }
  }
  auto flush = [&]() {  // LDS row -> matrix
    if (LACC)
      for (int j = 0; j < width; ++j)
#pragma unroll
        for (int q = 0; q < 9; ++q) A[val_idx(g0 + j, q, lane)] = row[ix(j, q)];
  };
  if (a.raw) {
    flush();
    return;
  }
  // system matrix (h + beta) h K + (1 + alpha h) M (doBackEuler, CUDAInterface.cu:845-851)
  const R s1 = (R)a.h + (R)a.beta, s2 = (R)a.h;
  for (int j = 0; j < len; ++j)
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      const size_t i = ix(j, q);
      row[i] = row[i] * s1 * s2;
    }
  const R ms = (R)mass[n] * ((R)1 + (R)a.alpha * (R)a.h);
  const int ds = d.diag_slot[n];
  const int dj = (int)((ds >> 6) - g0);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = ix(dj, 4 * k);
    row[i] += ms;
    d.dinv[3 * (size_t)n + k] = 1.0 / (double)row[i];
  }
  flush();
  // right-hand side h f + m v (setRHSofLinearSystem :418-442) with the forces of
  // addFixContraintsAndGravity (:327-343): fixed nodes a 1e8 spring to the rest position
  const R h = (R)a.h;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = (size_t)k * N + n;
    R fk;
    if (mask[n]) {
      fk = (R)(1e8 * (double)((R)rest[i] - xpos[i]));
    } else {
      fk = f[k] + (R)gforce[i];
      if (a.has_ext) fk += (R)ext[i];
    }
    const R vk = vel[i];
    d.b[3 * (size_t)n + k] = (double)(fk * h + (R)mass[n] * vk);
    d.x[3 * (size_t)n + k] = a.warm ? (double)vk : 0.0;
  }
}

// Per-tet stiffness K = -df/dx (12 x 12, rows 3 a + d, columns 3 b + e over the tet's corners a,
// b and axes d, e) at the node-major positions x: the blocks of the closed form the assembly above
// accumulates, one thread per requested tet (IsotropicMaterial::computeStiffnessMatrixFromPos,
// IsotropicMaterial.cpp:503-552).  ids: solver tet ids; out: 144 FP32 values per requested tet.
template <typename R, int MAT>
__global__ void k_tet_stiffness(DevParams p, int num, const int *__restrict__ ids, const int4 *__restrict__ tets,
                                const float *__restrict__ dmi, const float *__restrict__ vol, const R *__restrict__ x,
                                const float *__restrict__ inst_mu, const float *__restrict__ inst_lam,
                                float *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= num) return;
  const int t = ids[k], T = p.nt;
  const int4 q4 = tets[t];
  const int qn[4] = {q4.x, q4.y, q4.z, q4.w};
  R Dmi[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) Dmi[i] = (R)dmi[(size_t)i * T + t];
  const R V = (R)vol[t];
  const R mu = (R)inst_mu[0], lam = (R)inst_lam[0];
  R X[4][3];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int d = 0; d < 3; ++d) X[c][d] = x[3 * (size_t)qn[c] + d];
  R Ds[9], F[9], C[9];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    Ds[3 * d + 0] = X[1][d] - X[0][d];
    Ds[3 * d + 1] = X[2][d] - X[0][d];
    Ds[3 * d + 2] = X[3][d] - X[0][d];
  }
  mul3(Ds, Dmi, F);
  const R J = adj3(F, C);
  const R iJ = (R)1 / J;
  R c[4][3], g[4][3];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    shape_vec(Dmi, m, c[m]);
#pragma unroll
    for (int d = 0; d < 3; ++d) g[m][d] = (c[m][0] * C[d] + c[m][1] * C[3 + d] + c[m][2] * C[6 + d]) * iJ;
  }
  R k1, k2, U[9] = {}, Vv[9] = {}, aw[3] = {};
  const int kk[3] = {0, 0, 1}, ll[3] = {1, 2, 2};
  if (MAT == 0) {
    const R lj = dlog(J);
    k1 = mu - lam * lj;
    k2 = lam;
  } else {
    R S[3];
    svd3(F, U, S, Vv);
    k1 = -lam * (J - (R)1) * J;
    k2 = lam * ((R)2 * J - (R)1) * J;
    const R lim = (sizeof(R) == 4 ? (R)1e-6 : (R)1e-12);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const R den = S[kk[q]] + S[ll[q]];
      aw[q] = (R)1 / (den > lim ? den : lim);
    }
  }
  const R mu2 = (MAT == 0) ? mu : (R)2 * mu;
  // a[m][q][d] = (a^d_kl . c_m) for the pairs kl = 01, 02, 12 (stretch material)
  R a[4][3][3] = {};
  if (MAT != 0)
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          R acc = (R)0;
#pragma unroll
          for (int b = 0; b < 3; ++b)
            acc += (U[3 * d + kk[q]] * Vv[3 * b + ll[q]] - U[3 * d + ll[q]] * Vv[3 * b + kk[q]]) * c[m][b];
          a[m][q][d] = acc;
        }
  float *o = out + 144 * (size_t)k;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const R cc = c[i][0] * c[m][0] + c[i][1] * c[m][1] + c[i][2] * c[m][2];
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          R kv = (d == e ? mu2 * cc : (R)0) + k1 * g[m][d] * g[i][e] + k2 * g[i][d] * g[m][e];
          if (MAT != 0) {
            R rot = (R)0;
#pragma unroll
            for (int q = 0; q < 3; ++q) rot += a[i][q][d] * a[m][q][e] * aw[q];
            kv -= mu2 * rot;
          }
          o[12 * (3 * i + d) + 3 * m + e] = (float)(V * kv);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Conjugate gradients.  An iteration is three launches, and the two inner products are finished by
// the launch that needs them: every block of k_ie_dir sums the partials of r.z that k_ie_res left,
// every block of k_ie_res those of p.Ap that k_ie_spmv left, each in the same fixed order, so no
// launch of its own stands between two vector passes.  The partials, the control block and the
// block's first vector entries are all requested before any of them is waited for.  The control
// block is double-buffered: a launch reads the one and its block 0 writes the other, so no block
// reads what another one of the same launch has written.
//
// z = D^-1 r is the only residual kept (r.z = z.z / D^-1), and x += alpha p is done by the pass that
// reads p anyway, so the vectors cost 9 passes over 3N doubles per iteration.  Per iteration, 5
// launches and 11 passes before: 20 K tets 20.3 -> 11.9 us (backward Euler), 729 K 29.5 -> 18.9 us
// (projective dynamics), 1.5 M 55.6 -> 44.8 us, 6.3 M 229 -> 210 us; launches and their start-up
// bound the first, the matrix's bytes the last.
// ---------------------------------------------------------------------------------------------
// Vector passes: at most kVecBlocks blocks, each one contiguous range of 3N / blocks entries
// (multiples of 64), so that few blocks have the SpMV's partials to sum and every block the same
// work (both passes at 6.3 M tets with 512, 1024, 2048 blocks: 52.4, 53.4, 59.7 us);
// XCD-contiguous as the SpMV's rows.
constexpr int kVec = 4;  // entries a thread has in flight
__device__ __forceinline__ void vec_range(const IeDev &d, int &i0, int &i1) {
  const int b = xcd_block(blockIdx.x, gridDim.x);
  i0 = d.vec_unit * (b * d.vec_per + min(b, d.vec_rem));
  i1 = min(i0 + d.vec_unit * (d.vec_per + (b < d.vec_rem ? 1 : 0)), 3 * d.n);
}
// The thread's kVec entries of v from i on, kBlock apart (past the end: the range's last).
__device__ __forceinline__ void vec_load(const double *__restrict__ v, int i, int i1, double (&t)[kVec]) {
#pragma unroll
  for (int u = 0; u < kVec; ++u) t[u] = v[i + u * kBlock < i1 ? i + u * kBlock : i1 - 1];
}

// z = D^-1 (b - A x0); partials r.z, b.D^-1.b.  The stopping test uses the Jacobi-scaled norms
// |D^-1/2 r| = sqrt(r.z) and |D^-1/2 b|: fixed nodes carry a 1e8 mass and spring, and in the plain
// 2-norm their rows would swamp the free nodes' residual.
template <typename R, int BLK> __global__ void __launch_bounds__(kBlock) k_ie_start(IeDev d) {
  __shared__ double lds[4];
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int n = blk * kBlock + threadIdx.x;
  double rz = 0.0, bb = 0.0;
  if (n < d.n) {
    double y[3] = {0.0, 0.0, 0.0};
    const double *__restrict__ xv = d.x;
    row_apply<R, BLK>(d, n, 0, 1, [&](int col, double &x0, double &x1, double &x2) {
      x0 = xv[3 * (size_t)col];
      x1 = xv[3 * (size_t)col + 1];
      x2 = xv[3 * (size_t)col + 2];
    }, y);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const size_t i = 3 * (size_t)n + k;
      const double b = d.b[i];
      const double r = b - y[k];
      const double z = d.dinv[i] * r;
      d.z[i] = z;
      rz += r * z;
      bb += b * b * d.dinv[i];
    }
  }
  rz = block_sum256(rz, lds);
  bb = block_sum256(bb, lds);
  if (threadIdx.x == 0) {
    d.part_rz[blk] = rz;
    d.part_pap[blk] = bb;
  }
}

__global__ void __launch_bounds__(1024) k_ie_start_ctrl(IeDev d, int nb) {
  __shared__ double lds[2][16];
  PartialSum<1024> a, b;
  a.load(d.part_rz, nb);
  b.load(d.part_pap, nb);
  const double rz = a.sum(d.part_rz, nb, lds[0]), bb = b.sum(d.part_pap, nb, lds[1]);
  if (threadIdx.x == 0) {
    IeCtrl c = {};
    c.rz = rz;
    c.rz0 = rz;
    c.bb = bb;
    c.converged = (rz <= d.tol2 * bb) ? 1 : 0;
    c.done = c.converged || d.maxit <= 0;
    d.ctrl[0] = c;
  }
}

// x += alpha p (the step of the iteration before), p = z + beta p.
__global__ void __launch_bounds__(kBlock) k_ie_dir(IeDev d) {
  __shared__ double lds[4];
  int i0, i1;
  vec_range(d, i0, i1);
  int i = i0 + threadIdx.x;
  double *__restrict__ p = d.p, *__restrict__ x = d.x;
  PartialSum<kBlock> part;
  part.load(d.part_rz, gridDim.x);
  const IeCtrl in = d.ctrl[0];
  double zv[kVec], pv[kVec], xv[kVec];
  vec_load(d.z, i, i1, zv);
  vec_load(p, i, i1, pv);
  vec_load(x, i, i1, xv);
  __builtin_amdgcn_sched_barrier(0);  // all of them requested before the first is used
  const bool first = in.k == 0;
  const double sum = part.sum(d.part_rz, gridDim.x, lds);
  const double rz = first || in.done ? in.rz : sum, beta = first || in.done ? in.beta : sum / in.rz;
  const int converged = first || in.done ? in.converged : rz <= d.tol2 * in.bb;
  if (blockIdx.x == 0 && threadIdx.x == 0)
    d.ctrl[1] = {rz, in.pAp, in.alpha, beta, in.bb, in.rz0, in.k, in.done || converged || in.k >= d.maxit, converged,
                 in.indefinite};
  if (in.done) return;
  const double alpha = in.alpha;
  while (true) {
#pragma unroll
    for (int u = 0; u < kVec; ++u)
      if (i + u * kBlock < i1) {
        if (!first) x[i + u * kBlock] = xv[u] + alpha * pv[u];
        p[i + u * kBlock] = first ? zv[u] : zv[u] + beta * pv[u];
      }
    i += kVec * kBlock;
    if (i - (int)threadIdx.x >= i1) break;
    vec_load(d.z, i, i1, zv);
    vec_load(p, i, i1, pv);
    vec_load(x, i, i1, xv);
  }
}

// Ap = A p, partial p . Ap.  One 64-row slice per block, its 4 waves sharing the slots (wave w takes
// w, w + 4, ...; the shares are added in wave order): 4 times the loads in flight of one wave per
// slice.  At 6.3 M tets 147 us instead of 161 (3x3) and 49 instead of 64 (scalar), 5.1 TB/s with
// the padding; at 20 K tets 4.2 instead of 9 us.  Unrolled 4 instead of 2 slots: no faster.
template <typename R, int BLK> __global__ void __launch_bounds__(kBlock) k_ie_spmv(IeDev d) {
  __shared__ double lds[4];
  __shared__ double share[4][3][64];
  if (d.ctrl[1].done) return;
  const int sl = xcd_block(blockIdx.x, gridDim.x);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double *__restrict__ p = d.p;
  const int n = sl * 64 + lane;
  double y[3] = {0.0, 0.0, 0.0};
  if (n < d.n)
    row_apply<R, BLK>(d, n, w, 4, [&](int col, double &x0, double &x1, double &x2) {
      x0 = p[3 * (size_t)col];
      x1 = p[3 * (size_t)col + 1];
      x2 = p[3 * (size_t)col + 2];
    }, y);
#pragma unroll
  for (int q = 0; q < 3; ++q) share[w][q][lane] = y[q];
  __syncthreads();
  double pap = 0.0;
  if (w < 3) {  // 192 row components, one per thread of the first three waves
    const int e = 64 * w + lane, row = e / 3, q = e % 3;
    const double a = ((share[0][q][row] + share[1][q][row]) + share[2][q][row]) + share[3][q][row];
    const int i = 192 * sl + e;
    if (i < 3 * d.n) {
      d.Ap[i] = a;
      pap = p[i] * a;
    }
  }
  pap = block_sum256(pap, lds);
  if (threadIdx.x == 0) d.part_pap[sl] = pap;
}

// alpha = r.z / p.Ap, z -= alpha D^-1 Ap; partial r.z.
__global__ void __launch_bounds__(kBlock) k_ie_res(IeDev d) {
  __shared__ double lds[4];
  int i0, i1;
  vec_range(d, i0, i1);
  int i = i0 + threadIdx.x;
  double *__restrict__ z = d.z;
  PartialSum<kBlock> part;
  load_pap(d, part);
  const IeCtrl in = d.ctrl[1];
  double zv[kVec], av[kVec], dv[kVec];
  vec_load(z, i, i1, zv);
  vec_load(d.Ap, i, i1, av);
  vec_load(d.dinv, i, i1, dv);
  __builtin_amdgcn_sched_barrier(0);  // all of them requested before the first is used
  const double pap = part.sum(d.part_pap, d.vec_unit == 192 ? d.vec_blocks : d.nslice, lds);
  // not positive definite (or a non-finite value): stop without a step
  const bool indefinite = !in.done && !(pap > 0.0), go = !in.done && !indefinite;
  const double alpha = go ? in.rz / pap : indefinite ? 0.0 : in.alpha;
  // (the control block is written field by field: a copy modified under conditions would become a
  // private array, which the compiler moves to LDS at an index it computes from the dispatch packet
  // in host memory, and those reads cost a launch of 383 blocks 12 us)
  if (blockIdx.x == 0 && threadIdx.x == 0)
    d.ctrl[0] = {in.rz, go ? pap : in.pAp, alpha, in.beta, in.bb, in.rz0, in.k + (go ? 1 : 0), in.done || indefinite,
                 in.converged, in.indefinite || indefinite};
  if (!go) return;
  double rz = 0.0;
  while (true) {
#pragma unroll
    for (int u = 0; u < kVec; ++u)
      if (i + u * kBlock < i1) {
        const double zi = zv[u] - dv[u] * (alpha * av[u]);
        z[i + u * kBlock] = zi;
        rz += zi * zi * (1.0 / dv[u]);
      }
    i += kVec * kBlock;
    if (i - (int)threadIdx.x >= i1) break;
    vec_load(z, i, i1, zv);
    vec_load(d.Ap, i, i1, av);
    vec_load(d.dinv, i, i1, dv);
  }
  __syncthreads();  // part.sum's slots are read
  rz = block_sum256(rz, lds);
  if (threadIdx.x == 0) d.part_rz[xcd_block(blockIdx.x, gridDim.x)] = rz;
}

// ---------------------------------------------------------------------------------------------
// The same iterations as one resident kernel, for systems whose launches cost more than their work.
// A workgroup owns one or two blocks of the vector passes, that is 1 to 8 slices; its entries of x, p,
// z and D^-1 stay in registers, and so does its part of the matrix; the directions that its rows
// touch are in LDS.  An iteration waits for the other workgroups twice (pbs_exchange.h): for the
// partials of p.Ap, and for those of r.z together with the neighbours' z, from which each workgroup
// forms the neighbours' new directions itself.  All sums are formed as the three launches form them,
// term by term, so iterates and counts are bitwise theirs.
//
// Bound: the two waits, 5,000 to 8,000 cycles each (a store and a read through the memory side, and
// the slowest workgroup), of 15,000 to 25,000 an iteration; launches took 11 to 18 us an iteration.
// A step, launches -> resident, backward Euler (projective dynamics in brackets), FP32: 20 K tets 3.3
// -> 2.0 ms (2.3 -> 1.6), 99 K 5.3 -> 3.8 (4.7 -> 3.5), 338 K 7.6 -> 6.5 (7.1 -> 5.8), 729 K (9.3 ->
// 7.0).  With the matrix read from memory in every iteration, by 8 waves per CU, backward Euler on
// 729 K tets took 24 ms instead of 11: hence registers, and the launches where they do not suffice.
//
// Slots.  Each exchange has 2, iteration k uses slot k mod 2.  A workgroup that has all partials of
// r.z of iteration k knows that those of p.Ap of k have been consumed, with all of p.Ap of k + 1 that
// z and r.z of k have been, and clears its own.  Both clearings are waited for before it publishes
// the next r.z, and a slot is polled again only by who has that one, or the p.Ap that follows it.
// ---------------------------------------------------------------------------------------------
// Clears the exchange buffers (n times 16 bytes, at least one for each of the 3N entries of x) and keeps
// the start vector in p, which k_cg does not use: where some workgroups give up in the last iteration
// and others do not, the latter have written their part of x, and the launches begin again from p.
__global__ void k_cg_fill(IeDev d, uint4 *__restrict__ xch, long n, int *__restrict__ abort) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xch[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  if (i < 3 * (long)d.n) d.p[i] = d.x[i];
  if (i == 0) *abort = 0;
}

// The first four waves: sum of nb <= 512 published partials, as PartialSum<256> adds them, of which
// they leave 4 terms in total, to be added in order after a barrier.
__device__ __forceinline__ void published_sum(const double *v, int nb, double *total, int polls, int *abort,
                                              int *gave_up) {
  const int tid = threadIdx.x;
  if (tid >= 256) return;
  unsigned long long t[2];
  int spin = 0;
  while (true) {
#pragma unroll
    for (int u = 0; u < 2; ++u) t[u] = u * 256 + tid < nb ? poll(v + u * 256 + tid) : 0;
    if (t[0] != Bits<double>::none && t[1] != Bits<double>::none) break;
    if (give_up(spin, polls, abort)) {
      *gave_up = 1;
      break;
    }
  }
  double a = 0.0;
#pragma unroll
  for (int u = 0; u < 2; ++u) a += u * 256 + tid < nb ? __builtin_bit_cast(double, t[u]) : 0.0;
  a = wave_sum(a);
  if ((tid & 63) == 0) total[tid >> 6] = a;
}

// SH: shares of a slice per wave (a slice has four; 8 / (4 / SH) slices per workgroup at most).
template <typename R, int BLK, int SH> __global__ void __launch_bounds__(kCgThreads) k_cg(IeDev d, CgDev c) {
  extern __shared__ double lp[];         // directions of the local rows, x y z of each
  __shared__ double share[2 * SH][4][3][64];  // Ap of each slice in four shares
  __shared__ double csum[8][3], zsum[2][4], tot[2][4];
  __shared__ int gave_up;
  constexpr int NU = 3, GH = cg_ghost_entries(SH), WS = 4 / SH, NJ = kCgWidth / 4, NV = BLK * BLK;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int g = xcd_block(blockIdx.x, c.nparts);
  IeCtrl in = d.ctrl[0];
  if (in.done) return;
  if (tid == 0) gave_up = 0;
  const int vb0 = g * c.per_part, vb1 = min(vb0 + c.per_part, d.vec_blocks);
  const int s0 = first_slice(d, vb0), nsl = first_slice(d, vb1) - s0;
  const int n0 = 64 * s0, own = min(64 * nsl, d.n - n0);
  // this thread's vector entries: wave w holds chunks w % 4, + 4, + 8 (of 64 entries) of its block
  const int vb = vb0 + (w >> 2), q = w & 3;
  const int vs = vb < vb1 ? first_slice(d, vb) : 0, vn = vb < vb1 ? 3 * (first_slice(d, vb + 1) - vs) : 0;
  int ei[NU];
  double x[NU], p[NU], z[NU], di[NU], ri[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int ch = q + 4 * u, i = 192 * vs + 64 * ch + lane;
    ei[u] = ch < vn && i < 3 * d.n ? i : -1;
    const int k = ei[u] < 0 ? 0 : i;
    x[u] = d.x[k];
    z[u] = d.z[k];
    di[u] = d.dinv[k];
    ri[u] = 1.0 / di[u];
    p[u] = 0.0;
  }
  // ghost components: entry, z, direction
  const int goff = c.ghost_off[g], gcnt = c.ghost_off[g + 1] - goff;
  int gi[GH];
  double gz[GH], gp[GH];
#pragma unroll
  for (int u = 0; u < GH; ++u) {
    const int e = tid + u * kCgThreads;
    gi[u] = e < 3 * gcnt ? 3 * c.ghost[goff + e / 3] + e % 3 : -1;
    gz[u] = gi[u] >= 0 ? d.z[gi[u]] : 0.0;
    gp[u] = 0.0;
  }
  // the product: WS waves per slice; this wave's shares of its slice in registers
  const int sl = w / WS, sub = w % WS;
  const bool mul = sl < nsl;
  const int g0 = mul ? d.slice_off[s0 + sl] : 0, width = mul ? d.slice_off[s0 + sl + 1] - g0 : 0;
  const R *__restrict__ A = (const R *)d.A;
  R av[SH][NJ][NV];
  int ac[SH][NJ];
#pragma unroll
  for (int h = 0; h < SH; ++h)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int jj = sub + WS * h + 4 * j;
      if (jj < width) {
        ac[h][j] = 3 * (int)c.lcol[(size_t)(g0 + jj) * 64 + lane];
#pragma unroll
        for (int v = 0; v < NV; ++v) av[h][j][v] = BLK == 3 ? A[val_idx(g0 + jj, v, lane)] : A[(size_t)(g0 + jj) * 64 + lane];
      }
    }
  const bool row = mul && 64 * (s0 + sl) + lane < d.n;
  double rz = in.rz, alpha = in.alpha, beta = in.beta, pap = in.pAp;
  int k = in.k, converged = in.converged, indefinite = 0;
  __syncthreads();
  for (int it = 0;; ++it) {
    const int slot = it & 1;
    double *pz = c.z + (size_t)slot * 3 * d.n;
    // as k_ie_dir
    if (it > 0) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += tot[1][i];
      beta = sum / rz;
      rz = sum;
      converged = rz <= d.tol2 * in.bb;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (it > 0) x[u] = x[u] + alpha * p[u];
      p[u] = it > 0 ? z[u] + beta * p[u] : z[u];
      if (ei[u] >= 0) lp[ei[u] - 3 * n0] = p[u];
    }
    if (converged || k >= d.maxit) break;
#pragma unroll
    for (int u = 0; u < GH; ++u) {
      gp[u] = it > 0 ? gz[u] + beta * gp[u] : gz[u];
      if (gi[u] >= 0) lp[3 * own + tid + u * kCgThreads] = gp[u];
    }
    __syncthreads();
    // as k_ie_spmv
#pragma unroll
    for (int h = 0; h < SH; ++h) {
      double y[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (sub + WS * h + 4 * j < width) {
          const double *v = lp + ac[h][j];
          const double x0 = v[0], x1 = v[1], x2 = v[2];
          // (FP32 values stay so: converted here, not once before the loop into twice the registers)
          if constexpr (sizeof(R) == 4) {
#pragma unroll
            for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(av[h][j][i]));
          }
          if (BLK == 3) {
#pragma unroll
            for (int r = 0; r < 3; ++r)
              y[r] += (double)av[h][j][3 * r] * x0 + (double)av[h][j][3 * r + 1] * x1 + (double)av[h][j][3 * r + 2] * x2;
          } else {
            const double a = (double)av[h][j][0];
            y[0] += a * x0;
            y[1] += a * x1;
            y[2] += a * x2;
          }
        }
      if (mul) {
#pragma unroll
        for (int r = 0; r < 3; ++r) share[sl][sub + WS * h][r][lane] = row ? y[r] : 0.0;
      }
    }
    __syncthreads();
    double ap[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int ch = q + 4 * u;
      if (ch >= vn) continue;
      const int s = vs - s0 + ch / 3, e = 64 * (ch % 3) + lane, rw = e / 3, r = e % 3;
      ap[u] = ((share[s][0][r][rw] + share[s][1][r][rw]) + share[s][2][r][rw]) + share[s][3][r][rw];
      const double t = wave_sum(ei[u] >= 0 ? p[u] * ap[u] : 0.0);
      if (lane == 0) csum[s][ch % 3] = t;
    }
    __syncthreads();
    if (tid < vb1 - vb0) {
      const int a = first_slice(d, vb0 + tid) - s0, n = first_slice(d, vb0 + tid + 1) - s0 - a;
      double v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = i < n ? (csum[a + i][0] + csum[a + i][1]) + (csum[a + i][2] + 0.0) : 0.0;
      publish(c.pap + (size_t)slot * d.vec_blocks + vb0 + tid, ((v[0] + v[1]) + v[2]) + v[3]);
    }
    published_sum(c.pap + (size_t)slot * d.vec_blocks, d.vec_blocks, tot[0], 2 * it < c.from ? kPolls : c.polls, c.abort, &gave_up);
    __syncthreads();
    if (gave_up) break;
    if (it > 0) {
#pragma unroll
      for (int u = 0; u < NU; ++u)
        if (ei[u] >= 0) clear(c.z + (size_t)(slot ^ 1) * 3 * d.n + ei[u]);
      if (tid < vb1 - vb0) clear(c.rz + (size_t)(slot ^ 1) * d.vec_blocks + vb0 + tid);
    }
    // as k_ie_res
    {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += tot[0][i];
      indefinite = !(sum > 0.0);
      alpha = indefinite ? 0.0 : rz / sum;
      if (indefinite) break;
      pap = sum;
      ++k;
    }
    double zz = 0.0;
#pragma unroll
    for (int u = 0; u < NU; ++u)
      if (ei[u] >= 0) {
        const double zi = z[u] - di[u] * (alpha * ap[u]);
        z[u] = zi;
        publish(pz + ei[u], zi);
        zz += zi * zi * ri[u];
      }
    const int polls = 2 * it + 1 < c.from ? kPolls : c.polls;
    zz = wave_sum(zz);
    if (lane == 0) zsum[w >> 2][q] = zz;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // clearings are complete
    __syncthreads();
    if (tid < vb1 - vb0)
      publish(c.rz + (size_t)slot * d.vec_blocks + vb0 + tid, (zsum[tid][0] + zsum[tid][1]) + (zsum[tid][2] + zsum[tid][3]));
    published_sum(c.rz + (size_t)slot * d.vec_blocks, d.vec_blocks, tot[1], polls, c.abort, &gave_up);
    {
      unsigned long long t[GH];
      int spin = 0;
      while (true) {
        bool wait = false;
#pragma unroll
        for (int u = 0; u < GH; ++u) t[u] = gi[u] >= 0 ? poll(pz + gi[u]) : 0;
#pragma unroll
        for (int u = 0; u < GH; ++u) wait = wait || t[u] == Bits<double>::none;
        if (!wait) break;
        if (give_up(spin, polls, c.abort)) {
          gave_up = 1;
          break;
        }
      }
#pragma unroll
      for (int u = 0; u < GH; ++u) gz[u] = __builtin_bit_cast(double, t[u]);
    }
    __syncthreads();
    if (gave_up) break;
    if (tid < vb1 - vb0) clear(c.pap + (size_t)slot * d.vec_blocks + vb0 + tid);
  }
  if (gave_up) {
    if (tid == 0) __hip_atomic_store(c.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (ei[u] >= 0) d.x[ei[u]] = x[u];
  if (blockIdx.x == 0 && tid == 0) d.ctrl[0] = {rz, pap, alpha, beta, in.bb, in.rz0, k, 1, converged, indefinite};
}

// v = solution, x += h v for every node (cublasSaxpy in doBackEuler, CUDAInterface.cu:873).
template <typename R>
__global__ void k_ie_finish(DevParams p, float h, IeDev d, R *__restrict__ xpos, R *__restrict__ vel) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= d.n) return;
  const bool zero = d.ctrl[0].bb == 0.0;  // b = 0: the solution is 0 whatever the start
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = (size_t)k * p.nn + n;
    const R v = zero ? (R)0 : (R)d.x[3 * (size_t)n + k];
    vel[i] = v;
    xpos[i] = xpos[i] + (R)h * v;
  }
}

// ---------------------------------------------------------------------------------------------
// Projective dynamics (ProjDynamic.cpp).  The global matrix (buildGlobalSolverMatrix, :46-96) is
// G = M / t^2 + sum_k w_k Ac_k^T Ac_k with w_k = stiffness * vol_k; Ac_k^T Ac_k couples corners i, j
// of tet k by (c_i . c_j) times the 3x3 identity, so G is stored with one value per slot.
// ---------------------------------------------------------------------------------------------
template <typename R>
__global__ void __launch_bounds__(kBlock)
    k_pd_matrix(DevParams p, float stiffness, IeDev d, const int4 *__restrict__ tets, const float *__restrict__ dmi,
                const float *__restrict__ vol, const int *__restrict__ inc_off, const int *__restrict__ inc,
                const float *__restrict__ mass) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= d.n) return;
  R *__restrict__ A = (R *)d.A;
  const int T = p.nt;
  const int lane = n & 63;
  const int g0 = d.slice_off[n >> 6];
  const int width = d.slice_off[(n >> 6) + 1] - g0;
  const int len = d.row_len[n];
  for (int j = 0; j < width; ++j) A[(size_t)(g0 + j) * 64 + lane] = (R)0;
  for (int e = inc_off[n]; e < inc_off[n + 1]; ++e) {
    const int t = inc[e] >> 2, ci = inc[e] & 3;
    const int4 q4 = tets[t];
    const int qn[4] = {q4.x, q4.y, q4.z, q4.w};
    R Dmi[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) Dmi[k] = (R)dmi[(size_t)k * T + t];
    const R w = (R)stiffness * (R)vol[t];
    R c[4][3];
#pragma unroll
    for (int m = 0; m < 4; ++m) shape_vec(Dmi, m, c[m]);
    R cs[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) cs[k] = ci == 0 ? c[0][k] : ci == 1 ? c[1][k] : ci == 2 ? c[2][k] : c[3][k];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int slot_g = g0 + find_col(d.bcol, g0, lane, len, qn[m]);
      A[(size_t)slot_g * 64 + lane] += w * (cs[0] * c[m][0] + cs[1] * c[m][1] + cs[2] * c[m][2]);
    }
  }
  const R h = (R)p.h;
  const R t2inv = (R)1 / (h * h);
  const int ds = d.diag_slot[n];
  A[ds] += (R)mass[n] * t2inv;
  const double di = 1.0 / (double)A[ds];
#pragma unroll
  for (int k = 0; k < 3; ++k) d.dinv[3 * (size_t)n + k] = di;
}

// Momentum term of doProjDynamics (ProjDynamic.cpp:442-460): s = (x + t v + t^2 m^-1 f_ext) m / t^2
// with f_ext = gravity + external forces (TetMesh::computeExternalForces; fixed nodes have
// m^-1 = 0); the iterate starts at x.
template <typename R>
__global__ void k_pd_begin(DevParams p, IeDev d, double *__restrict__ srhs, const R *__restrict__ xpos,
                           const R *__restrict__ vel, const float *__restrict__ mass, const float *__restrict__ gforce,
                           const float *__restrict__ ext, int has_ext, const int *__restrict__ mask) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= d.n) return;
  const R t = (R)p.h, m = (R)mass[n];
  const R im = mask[n] ? (R)0 : (R)1 / m;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = (size_t)k * p.nn + n;
    R f = (R)gforce[i];
    if (has_ext) f += (R)ext[i];
    const R y = xpos[i] + t * vel[i] + t * t * im * f;
    srhs[3 * (size_t)n + k] = (double)(y * m / (t * t));
    d.x[3 * (size_t)n + k] = (double)xpos[i];
  }
}

// The projection rotation of one tet: R = U V^T of F's SVD with the signs the reference fixes
// (ProjDynamic.cpp:359-368: a column of U or V whose determinant is negative is negated, column 0
// of the singular values sorted in decreasing order).  With svd3's rotations U, V and the sign of
// det F on the last singular value this is U V^T for det F >= 0 and U diag(-1, 1, -1) V^T otherwise.
template <typename R> __device__ __forceinline__ void pd_rotation(const R *F, R *Rot) {
  // det F > 0: U V^T is the rotation of the polar decomposition (scaled Newton iteration)
  if (polar_rotation(F, Rot)) return;
  R U[9], S[3], V[9];
  svd3(F, U, S, V);
  const R s0 = S[2] < (R)0 ? (R)-1 : (R)1;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) Rot[3 * i + j] = s0 * U[3 * i] * V[3 * j] + U[3 * i + 1] * V[3 * j + 1] + s0 * U[3 * i + 2] * V[3 * j + 2];
}

// Local step (projectLocalConstraints2, ProjDynamic.cpp:223-308), in two passes like the
// reference's: k_pd_tet evaluates each tet once -- F from the iterate pos (3N node-major
// doubles), the SVD, R -- and writes its four corner projections w_k R_k c_i to rec (12 values
// per tet); k_pd_gather sums each node's corner records over its tets in ascending order,
// out = s + sum (s may be null: the projection alone).
template <typename R>
__global__ void __launch_bounds__(kBlock)
    k_pd_tet(DevParams p, float stiffness, const double *__restrict__ pos, const int4 *__restrict__ tets,
             const float *__restrict__ dmi, const float *__restrict__ vol, const int *__restrict__ inc_pos,
             R *__restrict__ rec) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int T = p.nt;
  if (t >= T) return;
  const int4 q4 = tets[t];
  const int qn[4] = {q4.x, q4.y, q4.z, q4.w};
  R X[4][3];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int k = 0; k < 3; ++k) X[c][k] = (R)pos[3 * (size_t)qn[c] + k];
  R Dmi[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) Dmi[k] = (R)dmi[(size_t)k * T + t];
  R Ds[9], F[9], Rot[9];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    Ds[3 * k + 0] = X[1][k] - X[0][k];
    Ds[3 * k + 1] = X[2][k] - X[0][k];
    Ds[3 * k + 2] = X[3][k] - X[0][k];
  }
  mul3(Ds, Dmi, F);
  pd_rotation(F, Rot);
  const R w = (R)stiffness * (R)vol[t];
#pragma unroll
  for (int ci = 0; ci < 4; ++ci) {
    R c[3];
    shape_vec(Dmi, ci, c);
    R *o = rec + 3 * (size_t)inc_pos[4 * (size_t)t + ci];  // the (tet, corner) slot of its node's run
#pragma unroll
    for (int k = 0; k < 3; ++k) o[k] = w * (Rot[3 * k] * c[0] + Rot[3 * k + 1] * c[1] + Rot[3 * k + 2] * c[2]);
  }
}

template <typename R>
__global__ void __launch_bounds__(kBlock)
    k_pd_gather(int n_nodes, const int *__restrict__ inc_off, const R *__restrict__ rec,
                const double *__restrict__ srhs, double *__restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n_nodes) return;
  R acc[3] = {(R)0, (R)0, (R)0};
  for (int e = inc_off[n]; e < inc_off[n + 1]; ++e) {  // the node's run, in ascending tet order
    const R *r = rec + 3 * (size_t)e;
#pragma unroll
    for (int k = 0; k < 3; ++k) acc[k] += r[k];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = 3 * (size_t)n + k;
    out[i] = srhs ? (double)((R)srhs[i] + acc[k]) : (double)acc[k];
  }
}

// v = damping (x_new - x) / t, x = x_new (ProjDynamic.cpp:477-478), every node.
template <typename R>
__global__ void k_pd_finish(DevParams p, float damping, IeDev d, R *__restrict__ xpos, R *__restrict__ vel) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= d.n) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = (size_t)k * p.nn + n;
    const R xn = (R)d.x[3 * (size_t)n + k];
    vel[i] = (xn - xpos[i]) / (R)p.h * (R)damping;
    xpos[i] = xn;
  }
}

inline int nb_of(int n) { return (n + kBlock - 1) / kBlock; }

}  // namespace

template <typename R>
void IeLaunch<R>::tet_stiffness(const DevMesh<R> &m, const DevParams &p, const float *inst_mu, const float *inst_lam,
                                const R *x, int num, const int *ids, float *out, hipStream_t st) {
  if (num <= 0) return;
  const int blocks = (num + 63) / 64;
  if (p.material == 0)
    hipLaunchKernelGGL((k_tet_stiffness<R, 0>), dim3(blocks), dim3(64), 0, st, p, num, ids, m.tets, m.dmi, m.vol, x,
                       inst_mu, inst_lam, out);
  else
    hipLaunchKernelGGL((k_tet_stiffness<R, 1>), dim3(blocks), dim3(64), 0, st, p, num, ids, m.tets, m.dmi, m.vol, x,
                       inst_mu, inst_lam, out);
}
template <typename R>
void IeLaunch<R>::assemble(const DevMesh<R> &m, const TileDev &td, const DevParams &p, const IeDev &d,
                           const IeAsm &a, int max_width, hipStream_t st) {
  // rows accumulated in LDS when the widest slice fits in 96 KB per workgroup, else in place
  // (6.3M-tet bar, 15 slots per row: FP32 5.8 -> 3.1 ms, FP64 8.5 -> 4.6 ms)
  const size_t lds = (size_t)max_width * 9 * 64 * sizeof(R);
  if (lds <= 98304) {
    const dim3 grid((d.n + 63) / 64), blk(64);
    if (p.material == 0)
      hipLaunchKernelGGL((k_ie_assemble<R, 0, true>), grid, blk, lds, st, p, a, d, m.tets, m.dmi, m.vol, m.inc_off,
                         m.inc, m.xpos, m.v, m.rest, m.mass, m.gforce, m.ext, m.mask, td.inst_mu, td.inst_lam);
    else
      hipLaunchKernelGGL((k_ie_assemble<R, 1, true>), grid, blk, lds, st, p, a, d, m.tets, m.dmi, m.vol, m.inc_off,
                         m.inc, m.xpos, m.v, m.rest, m.mass, m.gforce, m.ext, m.mask, td.inst_mu, td.inst_lam);
    return;
  }
  if (p.material == 0)
    hipLaunchKernelGGL((k_ie_assemble<R, 0, false>), dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, a, d, m.tets, m.dmi,
                       m.vol, m.inc_off, m.inc, m.xpos, m.v, m.rest, m.mass, m.gforce, m.ext, m.mask, td.inst_mu,
                       td.inst_lam);
  else
    hipLaunchKernelGGL((k_ie_assemble<R, 1, false>), dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, a, d, m.tets, m.dmi,
                       m.vol, m.inc_off, m.inc, m.xpos, m.v, m.rest, m.mass, m.gforce, m.ext, m.mask, td.inst_mu,
                       td.inst_lam);
}

template <typename R> void IeLaunch<R>::start(const IeDev &d, hipStream_t st) {
  if (d.scalar) hipLaunchKernelGGL((k_ie_start<R, 1>), dim3(nb_of(d.n)), dim3(kBlock), 0, st, d);
  else hipLaunchKernelGGL((k_ie_start<R, 3>), dim3(nb_of(d.n)), dim3(kBlock), 0, st, d);
  hipLaunchKernelGGL(k_ie_start_ctrl, dim3(1), dim3(1024), 0, st, d, nb_of(d.n));
}

void ie_vec_split(IeDev &d) {
  d.vec_unit = 64;
  const int groups = (3 * d.n + 63) / 64;
  const long most = (3 * (long)d.n + kVec * kBlock - 1) / (kVec * kBlock);
  d.vec_blocks = (int)std::min<long>(most, kVecBlocks);
  d.vec_per = groups / d.vec_blocks;
  d.vec_rem = groups % d.vec_blocks;
}

// e0 set: the launch records the dispatch's start and end in e0, e1 (as a kernel trace times it)
template <typename F, typename... Args>
static void ie_launch(F kernel, dim3 grid, dim3 block, hipStream_t st, hipEvent_t e0, hipEvent_t e1, Args... args) {
  if (e0) hipExtLaunchKernelGGL(kernel, grid, block, 0u, st, e0, e1, 0u, args...);
  else hipLaunchKernelGGL(kernel, grid, block, 0, st, args...);
}
template <typename R> void IeLaunch<R>::dir(const IeDev &d, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  ie_launch(k_ie_dir, dim3(d.vec_blocks), dim3(kBlock), st, e0, e1, d);
}
template <typename R> void IeLaunch<R>::spmv(const IeDev &d, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if (d.scalar) ie_launch(k_ie_spmv<R, 1>, dim3(d.nslice), dim3(kBlock), st, e0, e1, d);
  else ie_launch(k_ie_spmv<R, 3>, dim3(d.nslice), dim3(kBlock), st, e0, e1, d);
}
template <typename R> void IeLaunch<R>::res(const IeDev &d, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  ie_launch(k_ie_res, dim3(d.vec_blocks), dim3(kBlock), st, e0, e1, d);
}

template <typename R, int BLK> static const void *cg_kernel_of(int shares) {
  return shares == 1 ? (const void *)k_cg<R, BLK, 1> : shares == 2 ? (const void *)k_cg<R, BLK, 2> : (const void *)k_cg<R, BLK, 4>;
}
template <typename R> static const void *cg_kernel(const CgDev &c, int scalar) {
  // (the 3 x 3 blocks are held for as many shares as the registers take, see resident_fits)
  if (scalar) return cg_kernel_of<R, 1>(c.shares);
  return c.shares == 1 ? (const void *)k_cg<R, 3, 1> : (const void *)k_cg<R, 3, 2>;
}
static size_t cg_lds(const CgDev &c) { return sizeof(double) * 3 * (size_t)c.local_max; }
template <typename R> bool IeLaunch<R>::resident_fits(const CgDev &c, int scalar, int device) {
  // at most 126 registers of matrix values (7 slots of 9 values per share): FP32 up to two shares,
  // about 65,000 nodes, FP64 one, about 32,000; scalar values always
  if (!scalar && c.shares * (int)sizeof(R) > 8) return false;
  int coop = 0, cus = 0;
  if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess || !coop) return false;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < c.nparts) return false;
  int per = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, cg_kernel<R>(c, scalar), kCgThreads, cg_lds(c)) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return per > 0;
}
template <typename R> hipError_t IeLaunch<R>::resident(const IeDev &d, const CgDev &c, hipStream_t st) {
  const long n16 = c.xch_bytes / 16;
  hipLaunchKernelGGL(k_cg_fill, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st, d, (uint4 *)c.z, n16, c.abort);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  IeDev dd = d;
  CgDev cc = c;
  void *args[] = {&dd, &cc};
  return hipLaunchCooperativeKernel(cg_kernel<R>(c, d.scalar), dim3(c.nparts), dim3(kCgThreads), args, (unsigned)cg_lds(c), st);
}

template <typename R>
void IeLaunch<R>::finish(const DevMesh<R> &m, const DevParams &p, float h, const IeDev &d, hipStream_t st) {
  hipLaunchKernelGGL(k_ie_finish<R>, dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, h, d, m.xpos, m.v);
}

template <typename R>
void IeLaunch<R>::pd_matrix(const DevMesh<R> &m, const DevParams &p, float stiffness, const IeDev &d, hipStream_t st) {
  hipLaunchKernelGGL(k_pd_matrix<R>, dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, stiffness, d, m.tets, m.dmi, m.vol,
                     m.inc_off, m.inc, m.mass);
}
template <typename R>
void IeLaunch<R>::pd_begin(const DevMesh<R> &m, const DevParams &p, const IeDev &d, double *srhs, int has_ext,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_pd_begin<R>, dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, d, srhs, m.xpos, m.v, m.mass, m.gforce,
                     m.ext, has_ext, m.mask);
}
template <typename R>
void IeLaunch<R>::pd_local(const DevMesh<R> &m, const DevParams &p, float stiffness, const int *inc_pos,
                           const double *pos, const double *srhs, double *out, hipStream_t st) {
  // the per-tet force records of the standalone calls (12 R per tet) serve as the staging array,
  // filled in incidence order
  hipLaunchKernelGGL(k_pd_tet<R>, dim3(nb_of(p.nt)), dim3(kBlock), 0, st, p, stiffness, pos, m.tets, m.dmi, m.vol,
                     inc_pos, m.frec);
  hipLaunchKernelGGL(k_pd_gather<R>, dim3(nb_of(p.nn)), dim3(kBlock), 0, st, p.nn, m.inc_off, (const R *)m.frec, srhs,
                     out);
}
template <typename R>
void IeLaunch<R>::pd_finish(const DevMesh<R> &m, const DevParams &p, float damping, const IeDev &d, hipStream_t st) {
  hipLaunchKernelGGL(k_pd_finish<R>, dim3(nb_of(d.n)), dim3(kBlock), 0, st, p, damping, d, m.xpos, m.v);
}

template struct IeLaunch<float>;
template struct IeLaunch<double>;

}  // namespace pbs
