// pbs_pass.h -- device code shared by the kernels of the descent pass: the rest shape and force of
// one tet, the Chebyshev schedule and the loop control.  The launches of a pass (pbs_kernels.hip)
// and the resident descent kernel (pbs_persist.hip) evaluate the same functions, so their iterates
// agree bitwise while the loop's decisions do.
#pragma once
#include <type_traits>

#include "pbs_device.h"
#include "pbs_internal.h"

namespace pbs {

// Chebyshev schedule of the reference (CUDAInterface.cu:967-986; DescentOptimize.cpp:156-175).
__device__ __forceinline__ void cheb_schedule(const DevParams &p, int k, float &rho, float &omega) {
  if (k == 0) {
    rho = 0.0f;
    omega = 1.0f;
  }
  omega = 4.0f / (4.0f - rho * rho * omega);
  for (int i = 0; i < p.profile_n; ++i) {
    if (k == p.profile_k[i] - 1) {
      rho = 0.0f;
      omega = 1.0f;
    }
    if (k == p.profile_k[i]) {
      rho = p.profile_rho[i];
      omega = 2.0f / (2.0f - rho * rho);
      break;
    }
  }
}

// x / 6, correctly rounded as the division (checked over all 2^23 mantissas): the quotient's
// estimate and one correction by its exact remainder, 3 instructions instead of the division's 10.
__device__ __forceinline__ float div6(float x) {
  const float q = x * (1.0f / 6.0f);
  return fmaf(fmaf(-6.0f, q, x), 1.0f / 6.0f, q);
}

// Contraction is off for the rest shape so that Dm^-1, volumes and masses round exactly as the FP32
// reference formulas written out without fused multiply-adds; below it is allowed within a
// statement only, so that a function rounds the same in every kernel.
#pragma clang fp contract(off)
// Dm^-1 (row-major) and the volume |det Dm| / 6 of a rest tet from its corners' rest positions
// r[c][k] (compute_DmInv_ANs_Mass, CUDAInterface.cu:273-325; TetMesh.cpp:189-216); returns det Dm.
// The setup kernel and the tile pass both call this, so the tile pass's values are bitwise the
// stored ones.
__device__ __forceinline__ float rest_shape(const float r[4][3], float Dmi[9], float &V) {
  float Dm[9], C[9];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float x0 = r[0][k];
    Dm[3 * k + 0] = r[1][k] - x0;
    Dm[3 * k + 1] = r[2][k] - x0;
    Dm[3 * k + 2] = r[3][k] - x0;
  }
  // adjugate and determinant written out here so that the no-contraction pragma applies
  C[0] = Dm[4] * Dm[8] - Dm[7] * Dm[5];
  C[1] = Dm[7] * Dm[2] - Dm[1] * Dm[8];
  C[2] = Dm[1] * Dm[5] - Dm[4] * Dm[2];
  C[3] = Dm[5] * Dm[6] - Dm[3] * Dm[8];
  C[4] = Dm[0] * Dm[8] - Dm[2] * Dm[6];
  C[5] = Dm[2] * Dm[3] - Dm[0] * Dm[5];
  C[6] = Dm[3] * Dm[7] - Dm[4] * Dm[6];
  C[7] = Dm[1] * Dm[6] - Dm[0] * Dm[7];
  C[8] = Dm[0] * Dm[4] - Dm[1] * Dm[3];
  const float det = Dm[0] * C[0] + Dm[3] * C[1] + Dm[6] * C[2];
  V = div6(fabsf(det));
  const float inv = 1.0f / det;
#pragma unroll
  for (int i = 0; i < 9; ++i) Dmi[i] = C[i] * inv;
  return det;
}

#pragma clang fp contract(on)

// ---------------------------------------------------------------------------------------------
// Loop control of the reference (CUDAInterface.cu:917-1003) applied on the device after the
// pass over iterate x_k: E = incremental potential at x_k (FP64), g2 = |g(x_k)|^2.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void control_apply(const DevParams &p, Ctrl &C, double E, double g2) {
  const double g = sqrt(g2);
  C.g = g;
  if (C.first) {
    if (C.g0 < 0.0) C.g0 = g;
    C.first = 0;
  }
  // (mixed mode: convergence is only declared on a pass with FP64 forces)
  if (p.relgrad_tol > 0.0 && !p.f32math && g <= p.relgrad_tol * C.g0) {
    C.converged = 1;
    C.done = 1;
    C.passes++;
    return;
  }
  int rb = 0;
  const bool robust = p.relgrad_tol > 0.0;
  if (C.check_now) {
    C.E = E;
    // Rel-grad mode (no reference counterpart) also rejects a non-finite energy.
    const bool worse = robust ? !(E <= C.E_old) : (E > C.E_old);
    if (C.k != 0 && worse) {  // rollback (CUDAInterface.cu:946-958)
      C.alpha *= p.alpha_decay;
      if (robust) C.kc = C.k;  // rel-grad mode: keep the budget, restart Chebyshev at k
      else C.budget -= C.k - p.energy_check;
      C.cur = C.old;
      C.rollbacks++;
      rb = 1;
    } else {
      C.E_old = E;
      C.old = C.cur;
    }
  }
  if (!rb) {
    C.rho = C.rho_next;
    C.omega = C.omega_next;
    C.last = C.cur;
    C.cur = C.nxt;
    int f = 0;
    while (f == C.cur || f == C.last || f == C.old) ++f;
    C.nxt = f;
    C.k++;
  }
  C.passes++;
  if (C.alpha < p.alpha_min || !(C.k < C.budget)) {
    C.done = 1;
  } else {
    C.hd_now = (C.k % p.hd_refresh) == 0;
    C.check_now = (C.k % p.energy_check) == 0;
    float rho = C.rho, om = C.omega;
    cheb_schedule(p, C.k - C.kc, rho, om);
    C.rho_next = rho;
    C.omega_next = om;
    C.cheb_now = om != 1.0f;
  }
}

// adj3 and mul3 of pbs_device.h, rounded the same in every kernel (there the compiler may contract
// across statements, and does so differently from one caller to the next).
template <typename R> __device__ __forceinline__ R pass_adj3(const R *A, R *C) {
  C[0] = A[4] * A[8] - A[7] * A[5];
  C[1] = A[7] * A[2] - A[1] * A[8];
  C[2] = A[1] * A[5] - A[4] * A[2];
  C[3] = A[5] * A[6] - A[3] * A[8];
  C[4] = A[0] * A[8] - A[2] * A[6];
  C[5] = A[2] * A[3] - A[0] * A[5];
  C[6] = A[3] * A[7] - A[4] * A[6];
  C[7] = A[1] * A[6] - A[0] * A[7];
  C[8] = A[0] * A[4] - A[1] * A[3];
  return A[0] * C[0] + A[3] * C[1] + A[6] * C[2];
}
template <typename R> __device__ __forceinline__ void pass_mul3(const R *A, const R *B, R *C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[3 * i + j] = A[3 * i] * B[j] + A[3 * i + 1] * B[3 + j] + A[3 * i + 2] * B[6 + j];
}

// FP64 neo-Hookean corner forces without forming F or P.  With Ds, Dr the deformed and rest edges, V
// the rest volume, F = Ds Dr^-1 and P = mu F + (lambda ln J - mu) F^-T:
//   F Dr^-T = Ds S with S = Dr^-1 Dr^-T (symmetric), and F^-T Dr^-T = Ds^-T, so
//   G = -V P Dr^-T = -V mu Ds S + V (mu - lambda ln J) Ds^-T
// takes the adjugate of Ds, six entries of S and one 3x3 product, where F, F^-1, P and P Dr^-T take
// three products.  Both terms have the size of the old ones, so near rest they cancel alike.
// neo_corners: f12 from Ds, its adjugate C, k = V (mu - lambda ln J) / det Ds and Sm = -V mu S
// (entries 00 01 02 11 12 22).
template <typename R>
__device__ __forceinline__ void neo_corners(const R *Ds, const R *C, R k, const R *Sm, R *f12) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const R x = Ds[3 * a], y = Ds[3 * a + 1], z = Ds[3 * a + 2];
    const R g0 = fma(z, Sm[2], fma(y, Sm[1], fma(x, Sm[0], k * C[a])));
    const R g1 = fma(z, Sm[4], fma(y, Sm[3], fma(x, Sm[1], k * C[3 + a])));
    const R g2 = fma(z, Sm[5], fma(y, Sm[4], fma(x, Sm[2], k * C[6 + a])));
    f12[3 + a] = g0;
    f12[6 + a] = g1;
    f12[9 + a] = g2;
    f12[a] = -(g0 + g1 + g2);
  }
}
// Sm = s A A^T for the rows of A.
template <typename R> __device__ __forceinline__ void scaled_gram(const R *A, R s, R *Sm) {
  Sm[0] = s * (A[0] * A[0] + A[1] * A[1] + A[2] * A[2]);
  Sm[1] = s * (A[0] * A[3] + A[1] * A[4] + A[2] * A[5]);
  Sm[2] = s * (A[0] * A[6] + A[1] * A[7] + A[2] * A[8]);
  Sm[3] = s * (A[3] * A[3] + A[4] * A[4] + A[5] * A[5]);
  Sm[4] = s * (A[3] * A[6] + A[4] * A[7] + A[5] * A[8]);
  Sm[5] = s * (A[6] * A[6] + A[7] * A[7] + A[8] * A[8]);
}
// What the forces need of a tet's rest shape (r: its corners' rest positions).  FP64: S and det Dm^-1 from the stored FP32 Dm^-1 (so F is the one the other calls use).
template <typename R> struct NeoRest;
template <> struct NeoRest<double> {
  double Sm[6], dinv, V;
  __device__ __forceinline__ NeoRest() {}
  __device__ __forceinline__ NeoRest(const float r[4][3], double mu) {
    float Dmf[9], Vf;
    rest_shape(r, Dmf, Vf);
    double D[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) D[i] = (double)Dmf[i];
    V = (double)Vf;
    scaled_gram(D, -V * mu, Sm);
    dinv = D[0] * (D[4] * D[8] - D[7] * D[5]) + D[3] * (D[7] * D[2] - D[1] * D[8]) + D[6] * (D[1] * D[5] - D[4] * D[2]);
  }
};
// FP32: Dm^-1 and V themselves; the forces are neo_tet's, from F and P (the rounding of Dm^-1 and of
// F is part of what the FP32 trajectories of the reference are compared with).
template <> struct NeoRest<float> {
  float D[9], V;
  __device__ __forceinline__ NeoRest() {}
  __device__ __forceinline__ NeoRest(const float r[4][3], float) { rest_shape(r, D, V); }
};
// Corner forces from Ds.  FP64: J = det Ds det Dm^-1.
__device__ __forceinline__ void neo_force(const double *Ds, const NeoRest<double> &n, double mu, double lam, double *f12) {
  double C[9];
  const double det = pass_adj3(Ds, C);
  const double lj = log_f64(det * n.dinv);
  double q = __builtin_amdgcn_rcp(det);  // 1 / det Ds: the hardware's estimate and two Newton steps
  q = fma(fma(-det, q, 1.0), q, q);
  q = fma(fma(-det, q, 1.0), q, q);
  neo_corners(Ds, C, n.V * (mu - lam * lj) * q, n.Sm, f12);
}
__device__ __forceinline__ void neo_force(const float *Ds, const NeoRest<float> &n, float mu, float lam, float *f12) {
  float F[9], C[9], P[9];
  pass_mul3(Ds, n.D, F);
  const float J = pass_adj3(F, C), iJ = 1.0f / J, ll = lam * dlog(J);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float fit = C[3 * c + a] * iJ;  // (F^-T)[a][c]
      P[3 * a + c] = (F[3 * a + c] - fit) * mu + ll * fit;
    }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float g0 = -n.V * (P[3 * a] * n.D[0] + P[3 * a + 1] * n.D[1] + P[3 * a + 2] * n.D[2]);
    const float g1 = -n.V * (P[3 * a] * n.D[3] + P[3 * a + 1] * n.D[4] + P[3 * a + 2] * n.D[5]);
    const float g2 = -n.V * (P[3 * a] * n.D[6] + P[3 * a + 1] * n.D[7] + P[3 * a + 2] * n.D[8]);
    f12[3 + a] = g0;
    f12[6 + a] = g1;
    f12[9 + a] = g2;
    f12[a] = -(g0 + g1 + g2);
  }
}
// psi V as neo_tet forms it (check passes).  I1 and J both come from the one rounded F: near rest
// their rounding errors then cancel, where those of an F and a det Ds det Dm^-1 would not.
template <typename R>
__device__ __forceinline__ R neo_energy(const R *Ds, const float r[4][3], R mu, R lam) {
  float Dmf[9], Vf;
  rest_shape(r, Dmf, Vf);
  R D[9], F[9], C[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) D[i] = (R)Dmf[i];
  pass_mul3(Ds, D, F);
  const R lj = dlog(pass_adj3(F, C));
  R I1 = (R)0;
#pragma unroll
  for (int i = 0; i < 9; ++i) I1 += F[i] * F[i];
  return ((R)0.5 * mu * (I1 - (R)3) - mu * lj + (R)0.5 * lam * lj * lj) * (R)Vf;
}

// One tet of a tile: positions from LDS (stride 4 R per local node), rest positions from get_r(r),
// the neo-Hookean forces' rest shape from get_neo(), the material response, and its four corner
// contributions written to their slots of the LDS array rec (W values each): forces on phase 0 (plus the clamped energy on check passes), Hessian-diagonal
// entries rounded to FP32 on phase 1.  The arithmetic type C is R, or FP32 on FP64 positions (the
// mixed mode).  Mixed mode: F is formed in R; the energy of check passes is evaluated in R from
// that F (the same value the FP64 passes compute, so the line search compares like with like);
// the neo-Hookean force is evaluated in FP32 from the displacement gradient H = F - I, whose FP32
// rounding is relative to the strain instead of to 1; contributions are stored as FP32.
template <typename R, typename C, int MAT, int PHASE, typename GetR, typename GetNeo>
__device__ __forceinline__ void tile_tet(const uint4 lp, GetR get_r, GetNeo get_neo, const R *__restrict__ sx,
                                         C *__restrict__ rec, C mu, C lam, int chk, int clamp, double &e_el) {
  constexpr int W = ContribWidth<C>::value;
  constexpr bool MIX = sizeof(C) < sizeof(R);
  const R *p0 = sx + 4 * (lp.x & 0xffff), *p1 = sx + 4 * (lp.x >> 16), *p2 = sx + 4 * (lp.y & 0xffff),
          *p3 = sx + 4 * (lp.y >> 16);
  typedef typename std::conditional<MIX, R, C>::type FT;  // type F is formed in
  const unsigned q[4] = {lp.z & 0xffff, lp.z >> 16, lp.w & 0xffff, lp.w >> 16};
  FT Ds[9];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const R x0 = p0[k];
    Ds[3 * k + 0] = (FT)(p1[k] - x0);
    Ds[3 * k + 1] = (FT)(p2[k] - x0);
    Ds[3 * k + 2] = (FT)(p3[k] - x0);
  }
  C f12[12], h12[12], en = (C)0;
  auto store = [&](const C *v) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      C *o = rec + W * q[c];
      o[0] = v[3 * c];
      o[1] = v[3 * c + 1];
      o[2] = v[3 * c + 2];
    }
  };
  auto count = [&](R er) {
    if (clamp == 1) er = er > (R)0 ? er : (R)0;          // CUDAInterface.cu:549
    else if (clamp == 2) er = er > (R)1e-6 ? er : (R)0;  // IsotropicNeohookeanMaterial.cpp:129
    e_el += (double)er;
  };
  if constexpr (!MIX && MAT == 0 && PHASE == 0) {
    neo_force(Ds, get_neo(), mu, lam, f12);
    store(f12);
    if (chk) {
      float r[4][3];
      get_r(r);
      count(neo_energy(Ds, r, mu, lam));
    }
    return;
  }
  float r[4][3], Dmf[9], Vf;
  get_r(r);
  rest_shape(r, Dmf, Vf);
  FT Dm[9], Fw[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) Dm[k] = (FT)Dmf[k];
  pass_mul3(Ds, Dm, Fw);
  C F[9], Dmi[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    Dmi[k] = (C)Dmf[k];
    F[k] = (C)Fw[k];
  }
  const C V = (C)Vf;
  if constexpr (PHASE == 0) {
    if constexpr (MAT == 0) {  // the mixed mode
      C H[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) H[k] = (C)(Fw[k] - ((k & 3) == 0 ? (FT)1 : (FT)0));
      neo_tet_disp<C>(H, Dmi, V, mu, lam, f12);
    } else {
      stretch_tet<C, false, true>(F, Dmi, V, mu, lam, f12, en, h12);
    }
    store(f12);
    if (chk) count(MIX ? tet_energy<R, MAT>((const R *)Fw, (R)Vf, (R)mu, (R)lam) : (R)en);
  } else if constexpr (MAT == 0) {
    // the neo-Hookean stiffness diagonal of neo_tet<C, true>, written corner by corner as it is
    // formed (the 12 values are never all live: this phase sets the kernel's register count)
    C Cf[9];
    const C J = pass_adj3(F, Cf);
    const C iJ = (C)1 / J;
    C Fi[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) Fi[i] = Cf[i] * iJ;
    const C k2 = mu + lam - lam * dlog(J);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      C c3[3];
      if (n == 0) {
#pragma unroll
        for (int j = 0; j < 3; ++j) c3[j] = -((C)Dmf[j] + (C)Dmf[3 + j] + (C)Dmf[6 + j]);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j) c3[j] = (C)Dmf[3 * (n - 1) + j];
      }
      const C cc = c3[0] * c3[0] + c3[1] * c3[1] + c3[2] * c3[2];
      C h[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const C sd = c3[0] * Fi[d] + c3[1] * Fi[3 + d] + c3[2] * Fi[6 + d];
        h[d] = V * (mu * cc + k2 * sd * sd);
      }
      C *o = rec + W * q[n];
      o[0] = (C)(float)h[0];
      o[1] = (C)(float)h[1];
      o[2] = (C)(float)h[2];
      // FP64: the store stays here (sunk to the end of the loop it would hold all 12 values)
      if constexpr (sizeof(C) == 8) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    stretch_tet<C, true>(F, Dmi, V, mu, lam, f12, en, h12);
#pragma unroll
    for (int i = 0; i < 12; ++i) h12[i] = (C)(float)h12[i];
    store(h12);
  }
}

}  // namespace pbs
