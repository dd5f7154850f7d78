// pbs_learn.hip -- kernels of the learned warm start (no reference counterpart; PhyBS has no
// learned component).
//
// A per-vertex network (18 features -> 64 -> 64 -> 64 -> 3, SiLU) predicts the displacement of
// the converged step from the inertial target y = x + h v + h^2 g.  Inference runs on the matrix
// cores: BF16 weights and activations, FP32 accumulation, v_mfma_f32_16x16x16_bf16 with the
// layers written transposed (H_{l+1}^T = act(W_l^T H_l^T + b)), so that the accumulator tile of one
// layer is already the B-operand tile of the next and nothing is shuffled through LDS.  Training
// (on the matrix cores too: forward in BF16 as inference, backward in FP32) produces per-workgroup
// gradient partials that are reduced in a fixed order; Adam updates FP32 master weights.
//
// The warm start is a guess, never a replacement: both the plain guess and the learned one are
// evaluated with one gradient pass each, and the descent starts from the learned guess only if its
// gradient norm is not larger (the plain norm stays the rel-grad denominator).
#include "pbs_device.h"
#include "pbs_internal.h"

namespace pbs {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest, ties to even.
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ float bfround(float f) { return bf2f(f2bf(f)); }
__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }

// Layer table: inputs, outputs, 16-row output tiles, 16-wide input blocks, offsets of the
// A-operand arrangement, of the packed weights and of the packed biases.
struct Layer {
  int in, out, mt, kb, wa, pw, pb;
};
__constant__ Layer kLayers[4] = {{18, 64, 4, 2, 0, 0, 1152},
                                 {64, 64, 4, 4, 2048, 1216, 5312},
                                 {64, 64, 4, 4, 6144, 5376, 9472},
                                 {64, 3, 1, 4, 10240, 9536, 9728}};

// A operand of tile (mt, kb) for lane (q, r) = 4 BF16: W^T[16 mt + r][16 kb + 4 q + i], i = 0..3,
// i.e. W[16 kb + 4 q + i][16 mt + r], zero outside the layer.
__global__ void k_mlp_arrange(const float *__restrict__ params, unsigned short *__restrict__ wA) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_WA) return;
  int l = 3;
  while (l > 0 && e < kLayers[l].wa) --l;
  const Layer L = kLayers[l];
  const int el = e - L.wa, blk = el >> 8, lane = (el >> 2) & 63, i = el & 3;
  const int mt = blk / L.kb, kb = blk % L.kb, q = lane >> 4, r = lane & 15;
  const int o = 16 * mt + r, k = 16 * kb + 4 * q + i;
  wA[e] = (o < L.out && k < L.in) ? f2bf(params[L.pw + k * L.out + o]) : (unsigned short)0;
}

// Forward pass of one 16-sample tile by one wave.  feat: FP32 features (18 per sample); samples
// base .. base+15 (those >= n read as zero).  On return, lanes 0..15 hold the three normalised
// outputs of sample base + lane in o[0..2].
__device__ __forceinline__ void mlp_tile(const unsigned short *__restrict__ sW, const MlpDev &net,
                                         const float *__restrict__ feat, int base, int n, float o[3]) {
  const int lane = threadIdx.x & 63, q = lane >> 4, r = lane & 15;
  const int sidx = base + r;
  const bool valid = sidx < n;
  bf16x4 x[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 16 * kb + 4 * q + i;
      const float f = (valid && k < 18) ? feat[(size_t)sidx * 18 + k] * net.inv_s[k / 3] : 0.0f;
      x[kb][i] = (short)f2bf(f);
    }
  bf16x4 h[4], hn[4];
  const float *P = net.params;
  // layer 1: 18 (2 blocks) -> 64
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 c;
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = P[1152 + 16 * mt + 4 * q + i];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const bf16x4 a = *(const bf16x4 *)(sW + 0 + (mt * 2 + kb) * 256 + lane * 4);
      c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, x[kb], c, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) h[mt][i] = (short)f2bf(silu(c[i]));
  }
  // layers 2 and 3: 64 -> 64
#pragma unroll
  for (int l = 1; l < 3; ++l) {
    const int wa = l == 1 ? 2048 : 6144, pb = l == 1 ? 5312 : 9472;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      f32x4 c;
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = P[pb + 16 * mt + 4 * q + i];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const bf16x4 a = *(const bf16x4 *)(sW + wa + (mt * 4 + kb) * 256 + lane * 4);
        c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, h[kb], c, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) hn[mt][i] = (short)f2bf(silu(c[i]));
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) h[mt] = hn[mt];
  }
  // layer 4: 64 -> 3 (rows 3..15 of the tile are zero weights)
  f32x4 c;
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = (4 * q + i < 3) ? P[9728 + 4 * q + i] : 0.0f;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const bf16x4 a = *(const bf16x4 *)(sW + 10240 + kb * 256 + lane * 4);
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, h[kb], c, 0, 0, 0);
  }
  o[0] = c[0];
  o[1] = c[1];
  o[2] = c[2];
}

__device__ __forceinline__ void load_wA(const unsigned short *__restrict__ wA, unsigned short *sW) {
  const uint4 *src = (const uint4 *)wA;
  uint4 *dst = (uint4 *)sW;
  for (int i = threadIdx.x; i < MLP_WA / 8; i += blockDim.x) dst[i] = src[i];
  __syncthreads();
}

__global__ void __launch_bounds__(256) k_mlp_forward(MlpDev net, const float *__restrict__ feat, int n,
                                                     float *__restrict__ out) {
  __shared__ __align__(16) unsigned short sW[MLP_WA];
  load_wA(net.wA, sW);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int tile = blockIdx.x * 4 + wave; tile * 16 < n; tile += gridDim.x * 4) {
    float o[3];
    mlp_tile(sW, net, feat, tile * 16, n, o);
    const int sidx = tile * 16 + lane;
    if (lane < 16 && sidx < n) {
      out[(size_t)sidx * 3 + 0] = o[0];
      out[(size_t)sidx * 3 + 1] = o[1];
      out[(size_t)sidx * 3 + 2] = o[2];
    }
  }
}

// Features at the step start (x = current positions, v = current velocities):
//   u = x - X, h v, s = h v + h^2 g, and the 1-ring means of (u, h v, s) minus the node's own;
// fixed nodes get zeros.  Also writes the inertial target y = x + s.
template <typename R>
__global__ void k_features(DevParams p, const R *__restrict__ x, const R *__restrict__ v, const float *__restrict__ rest,
                           const int *__restrict__ mask, const int *__restrict__ adj_off, const int *__restrict__ adj,
                           float *__restrict__ feat, R *__restrict__ y) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int N = p.nn;
  if (n >= N) return;
  const R h = (R)p.h;
  R u[3], hv[3], s[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const size_t i = (size_t)d * N + n;
    u[d] = x[i] - (R)rest[i];
    hv[d] = h * v[i];
    s[d] = hv[d] + h * h * (R)p.grav[d];
    y[i] = x[i] + s[d];
  }
  float *f = feat + (size_t)n * 18;
  if (mask[n]) {
#pragma unroll
    for (int k = 0; k < 18; ++k) f[k] = 0.0f;
    return;
  }
  R mu[3] = {0, 0, 0}, mv[3] = {0, 0, 0}, ms[3] = {0, 0, 0};
  const int e0 = adj_off[n], e1 = adj_off[n + 1];
  for (int e = e0; e < e1; ++e) {
    const int m = adj[e];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const size_t i = (size_t)d * N + m;
      const R hvm = h * v[i];
      mu[d] += x[i] - (R)rest[i];
      mv[d] += hvm;
      ms[d] += hvm + h * h * (R)p.grav[d];
    }
  }
  const R c = (R)(e1 - e0 > 0 ? e1 - e0 : 1);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    f[d] = (float)u[d];
    f[3 + d] = (float)hv[d];
    f[6 + d] = (float)s[d];
    f[9 + d] = (float)(mu[d] / c - u[d]);
    f[12 + d] = (float)(mv[d] / c - hv[d]);
    f[15 + d] = (float)(ms[d] / c - s[d]);
  }
}

// Learned guess: ring.b[1] = y + out * scale for free nodes, ring.b[0] for fixed nodes.
template <typename R>
__global__ void __launch_bounds__(256) k_guess(DevParams p, MlpDev net, const float *__restrict__ feat,
                                               const R *__restrict__ y, const int *__restrict__ mask,
                                               const R *__restrict__ plain, R *__restrict__ out, float s_out) {
  __shared__ __align__(16) unsigned short sW[MLP_WA];
  load_wA(net.wA, sW);
  const int N = p.nn;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int tile = blockIdx.x * 4 + wave; tile * 16 < N; tile += gridDim.x * 4) {
    float o[3];
    mlp_tile(sW, net, feat, tile * 16, N, o);
    const int n = tile * 16 + lane;
    if (lane < 16 && n < N) {
      const bool fixed = mask[n] != 0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const size_t i = 3 * (size_t)n + d;
        out[i] = fixed ? plain[i] : y[(size_t)d * N + n] + (R)(o[d] * s_out);
      }
    }
  }
}

// Smoothing of the learned correction d = learned - plain over the node graph (fixed nodes pinned
// at 0): d'[n] = d[n] / 2 + (mean of d over the 1-ring) / 2.  The network's per-node errors are
// uncorrelated between neighbours, and such rough errors dominate the gradient norm through the
// stiff elastic forces; a few averaging sweeps keep the smooth part of the correction.  The
// correction is a heuristic guess (the gradient test decides whether it is used), so the sweeps
// run on FP32 xyz(w) quadruples: one 16-byte load per neighbour instead of three plane loads.
template <typename R>
__global__ void k_corr_diff(int N, const int *__restrict__ mask, const R *__restrict__ learned, const R *__restrict__ plain,
                            float4 *__restrict__ d) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  float v[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = 3 * (size_t)n + k;
    v[k] = mask[n] ? 0.0f : (float)(learned[i] - plain[i]);
  }
  d[n] = make_float4(v[0], v[1], v[2], 0.0f);
}
// One sweep; the neighbours come from SELL-64 slices (one coalesced index load per slot for the
// whole wavefront, a uniform loop to the slice width; padding slots hold the node itself).
__global__ void k_corr_smooth(int N, const int *__restrict__ mask, const int *__restrict__ adj_off,
                              const int *__restrict__ sell_off, const int *__restrict__ sell_col,
                              const float4 *__restrict__ d, float4 *__restrict__ dn) {
  // XCD-contiguous blocks (block i runs on XCD i % 8): a node's neighbours, mostly in the same or
  // the adjacent blocks in Morton order, stay in that XCD's L2
  const int per = (gridDim.x + 7) >> 3, xcd = blockIdx.x & 7, full = gridDim.x - 8 * (per - 1);
  const int blk = (xcd < full ? xcd * per : full * per + (xcd - full) * (per - 1)) + (blockIdx.x >> 3);
  const int n = blk * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int e0 = adj_off[n], e1 = adj_off[n + 1];
  const int g0 = sell_off[n >> 6], width = sell_off[(n >> 6) + 1] - g0, lane = n & 63;
  float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
#pragma unroll 2
  for (int j = 0; j < width; ++j) {
    const int m = sell_col[(size_t)(g0 + j) * 64 + lane];
    const float4 v = d[m];
    if (m != n) {  // neighbours ascending as in the adjacency list; padding is the node itself
      a0 += v.x;
      a1 += v.y;
      a2 += v.z;
    }
  }
  const float ic = 1.0f / (float)(e1 - e0 > 0 ? e1 - e0 : 1);
  const float4 s = d[n];
  dn[n] = mask[n] ? make_float4(0.0f, 0.0f, 0.0f, 0.0f)
                  : make_float4(0.5f * s.x + 0.5f * (a0 * ic), 0.5f * s.y + 0.5f * (a1 * ic), 0.5f * s.z + 0.5f * (a2 * ic),
                                0.0f);
}
// Candidate ring.b[1] = ring.b[0] + beta d, with beta from the argument or (beta < 0) the
// control block's chosen step.
template <typename R>
__global__ void k_corr_apply(int N, const Ctrl *__restrict__ ctrl, float beta, const R *__restrict__ plain,
                             const float4 *__restrict__ d, R *__restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N || ctrl->done) return;
  const R b = (R)(beta < 0.0f ? ctrl->ws_beta : beta);
  const float4 v = d[n];
  const float dv[3] = {v.x, v.y, v.z};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const size_t i = 3 * (size_t)n + k;
    out[i] = plain[i] + b * (R)dv[k];
  }
}

// Warm-start selection around gradient passes (k_tile + k_node<R, true>, no Hessian refresh or
// energy):  stage 0 starts, 1 records |g(plain)|^2, 2 records |g(candidate beta)|^2 and keeps the
// best beta, 3 starts the descent from the best candidate iff |g| <= |g(plain)| (the plain norm
// stays the rel-grad denominator).
__global__ void __launch_bounds__(1024) k_ws_stage(Ctrl *__restrict__ ctrl, const double *__restrict__ npart, int nnb,
                                                   int stage, float beta) {
  __shared__ double lg[1024];
  if (ctrl->done) return;
  const int tid = threadIdx.x;
  double c = 0.0;
  if (stage == 1 || stage == 2)
    for (int i = tid; i < nnb; i += 1024) c += npart[2 * i + 1];
  lg[tid] = c;
  __syncthreads();
  for (int st = 512; st > 0; st >>= 1) {
    if (tid < st) lg[tid] += lg[tid + st];
    __syncthreads();
  }
  if (tid == 0) {
    Ctrl C = *ctrl;
    if (stage == 0) {
      C.hd_now = 0;
      C.check_now = 0;
      C.cur = 0;
      C.g_learned = -1.0;
      C.ws_beta = 0.0f;
    } else if (stage == 1) {
      C.g_plain = lg[0];
      C.cur = 1;
    } else if (stage == 2) {
      if (C.g_learned < 0.0 || lg[0] < C.g_learned) {
        C.g_learned = lg[0];
        C.ws_beta = beta;
      }
    } else {
      const bool use = C.g_learned >= 0.0 && C.g_learned <= C.g_plain;
      C.cur = use ? 1 : 0;
      C.nxt = use ? 0 : 1;
      C.used_learned = use ? 1 : 0;
      // (a rejected guess leaves g0 to the first pass, which is then the plain step's own)
      if (use) C.g0 = sqrt(C.g_plain);
      C.hd_now = 1;
      C.check_now = 1;
    }
    *ctrl = C;
  }
}

// Appends (features, x_new - y) of free nodes: sample base + free_rank[n].
template <typename R>
__global__ void k_collect(DevParams p, const R *__restrict__ xnew, const float *__restrict__ feat, const R *__restrict__ y,
                          const int *__restrict__ free_rank, long base, int stride, int phase,
                          float *__restrict__ ds_x, float *__restrict__ ds_y) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int N = p.nn;
  if (n >= N) return;
  const int r = free_rank[n];
  if (r < 0 || r % stride != phase) return;
  const size_t j = (size_t)(base + r / stride);
#pragma unroll
  for (int k = 0; k < 18; ++k) ds_x[j * 18 + k] = feat[(size_t)n * 18 + k];
#pragma unroll
  for (int d = 0; d < 3; ++d) ds_y[j * 3 + d] = (float)(xnew[(size_t)d * N + n] - y[(size_t)d * N + n]);
}

// ---------------------------------------------------------------------------------------------
// Training.  Loss = mean over (sample, component) of (out - t / scale)^2 with the mean taken over
// the whole batch; the inference path's BF16 roundings (inputs, weights, hidden activations) with
// straight-through gradients.  Every product is on the matrix cores: the forward ones in BF16 with
// FP32 accumulation (their factors are BF16 values), the backward ones, whose deltas are FP32, in
// FP32 (v_mfma_f32_16x16x4_f32), so nothing is rounded further than by the loss itself.
//
// A workgroup takes tiles of 64 samples, 16 per wave.  Forward and delta propagation stay in the
// wave's registers in the transposed form of mlp_tile: an accumulator tile (rows 4 q + i, column r)
// is the next product's B operand, an FP32 product taking rows 4 q + j, j = 0..3, in its 4 steps.
// The weight gradients contract over samples, which are the lanes: activations and deltas go
// through LDS (rows of 64 samples, padded to 68 so that 16 rows start in different banks), and
// each wave accumulates 11 of the 44 gradient tiles in registers over all tiles of the workgroup.
// At most 256 workgroups (one per CU: the arrays take 126 KB of LDS) write one gradient partial each.
//
// A batch of 8192 samples: 166 -> 23 us (on the vector units, both factors of each multiply-add
// came from LDS; 20 us without the activations formed again in FP64), and its reduction, Adam step and arrangement 77 -> 4.7 us in one launch
// (k_mlp_step).  128 workgroups of 4 waves: what is left is the chain of one tile (weights 38 KB
// and samples in, 192 exponentials per sample, 308 FP32 products per wave).  With the weights
// converted one load at a time and the biases read where they are used it took 31 us.
// ---------------------------------------------------------------------------------------------
constexpr int TS = 64;         // samples per tile
constexpr int SP = TS + 4;     // padded row of samples
constexpr int kTrainWGs = 256;
struct TrainLds {
  unsigned short wA[MLP_WA];                // forward A operands
  unsigned short wB[2][64][SP];             // layers 2 and 3, BF16 [in][out], padded likewise
  float w4[64][4];                          // layer 4 [in][out], column 3 zero
  float bias[4][64];
  unsigned short h0[32][SP], h[3][64][SP];  // BF16 inputs (18 rows used) and activations [unit][sample]
  float dz[3][64][SP], dz4[16][SP];         // deltas [unit][sample] (3 rows of dz4 used)
  double red[4];
};

__device__ __forceinline__ f32x4 bf4(bf16x4 v) {
  f32x4 f;
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = bf2f((unsigned short)v[i]);
  return f;
}
// SiLU and its derivative from one exponential: s = 1 / (1 + e^-z), refined to the last bit or two.  Zero
// below -85, where s leaves the normal numbers (e^-z is capped there), so that any finite z gives 0 and
// 0; above 17, s is 1 and the quotient needs no refinement, which infinity would not survive.
__device__ __forceinline__ void silu_both(float z, float &s, float &v, float &dv) {
  const float d = 1.0f + fminf(expf(-z), 1e37f);
  s = __builtin_amdgcn_rcpf(d);
  s = fmaf(fmaf(-d, s, 1.0f), s, s);
  s = z < -85.0f ? 0.0f : s;
  v = z * s;
  if (d > 1.0f) v = fmaf(fmaf(-v, d, z), s, v);  // the quotient z / d to the last bit: it is rounded to BF16 next
  dv = s * fmaf(z, 1.0f - s, 1.0f);
}

// Whether a hidden activation v = SiLU(z), z = z0 + z1 + z2 + z3, is as near to the middle of two BF16
// values as its own rounding error: z's, 1.5e-7 of the sum of |z_i|, times SiLU's slope, and the
// exponential's, which reaches 1 - s of v (about 1 in 2000 are, saturated units among them; without the
// slope nine in ten are at z = -10, and a batch of such units takes 11 times as long as a usual one).  One
// rounded to the other neighbour of an exact evaluation's changes the sample's gradient in the third
// digit, far more than FP32 rounding does, so those are formed again in FP64, by the whole wave (each by
// its own lane alone: 28 instead of 23 us a batch; without it 20).  Relative error of the gradient
// against 64 bits, 30 seeds each of 65 to 30,000 samples: at most 1.7e-7, without it up to 7e-5; a bound
// of 1e-7 instead of 1.5e-7 misses a few.
__device__ __forceinline__ bool near_middle(float s, float v, float dv, float z0, float z1, float z2, float z3) {
  const float mid = __builtin_bit_cast(float, (__builtin_bit_cast(unsigned, v) & 0xffff0000u) | 0x8000u);
  const float sum = fabsf(z0) + fabsf(z1) + fabsf(z2) + fabsf(z3);
  return fabsf(v - mid) <= 1.5e-7f * fmaf(fabsf(dv), sum, 2.0f * (1.0f - s) * fabsf(v));
}

__global__ void __launch_bounds__(256) k_mlp_train(MlpDev net, const float *__restrict__ ds_x,
                                                   const float *__restrict__ ds_y, const int *__restrict__ idx, int n,
                                                   int batch, float *__restrict__ grad_part,
                                                   float *__restrict__ loss_part) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  TrainLds &S = *(TrainLds *)smem_raw;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, q = lane >> 4, r = lane & 15;
  const float *P = net.params;
  // the lane's sample of a tile: 8 scaled features (inputs 4 q + i and 16 + 4 q + i) and, q = 0, the
  // targets; zeros past the end
  auto load_sample = [&](int tile, f32x4 (&x)[2], float (&t)[3]) {
    const int j = tile * TS + 16 * w + r;
    const bool valid = j < n;
    const size_t row = valid ? idx[j] : 0;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 16 * kb + 4 * q + i;
        x[kb][i] = (valid && k < 18) ? ds_x[row * 18 + k] * net.inv_s[k / 3] : 0.0f;
      }
#pragma unroll
    for (int i = 0; i < 3; ++i) t[i] = valid && q == 0 ? ds_y[row * 3 + i] * net.inv_s[6] : 0.0f;
  };
  // weights: every load is issued before the first is waited for
  f32x4 x[2];
  float t[3];
  load_sample(blockIdx.x, x, t);
  {
    uint4 u[6];
    f32x4 f[8];
#pragma unroll
    for (int i = 0; i < 6; ++i) u[i] = ((const uint4 *)net.wA)[min(tid + 256 * i, MLP_WA / 8 - 1)];
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // rows of 64 outputs, 4 per load
      const int e = 4 * (tid + 256 * i), l = e >> 12;
      const float *v = P + kLayers[1 + l].pw + (e & 4095);
#pragma unroll
      for (int c = 0; c < 4; ++c) f[i][c] = v[c];
    }
    const float w4 = (tid & 3) < 3 ? bfround(P[9536 + (tid >> 2) * 3 + (tid & 3)]) : 0.0f;
    const float bias = w < 3 ? P[kLayers[w].pb + lane] : lane < 3 ? P[9728 + lane] : 0.0f;
#pragma unroll
    for (int i = 0; i < 6; ++i)
      if (tid + 256 * i < MLP_WA / 8) ((uint4 *)S.wA)[tid + 256 * i] = u[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = 4 * (tid + 256 * i);
      bf16x4 v;
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = (short)f2bf(f[i][c]);
      *(bf16x4 *)&S.wB[e >> 12][(e >> 6) & 63][e & 63] = v;
    }
    S.w4[tid >> 2][tid & 3] = w4;
    S.bias[w][lane] = bias;
  }
  // gradient tiles of this wave: rows (inputs) of tile mt, columns (outputs) of tile ot; layers 2
  // and 3: mt = w, ot = 0..3; layer 1: mt = w & 1, ot = 2 (w >> 1) + 0..1; layer 4: mt = w
  f32x4 g1[2] = {}, g2[4] = {}, g3[4] = {}, g4 = {};
  float gb[3] = {0.0f, 0.0f, 0.0f}, gb4 = 0.0f;  // bias gradients: unit lane, samples 16 w .. 16 w + 15
  double se = 0.0;
  __syncthreads();
  for (int tile = blockIdx.x; tile * TS < n; tile += gridDim.x) {
    const int j = tile * TS + 16 * w + r;  // the lane's sample
    const bool valid = j < n;
    bf16x4 h[4], hn[4];
    f32x4 ds[3][4];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h[kb][i] = (short)f2bf(x[kb][i]);
        S.h0[16 * kb + 4 * q + i][16 * w + r] = (unsigned short)h[kb][i];
      }
    // forward, hidden layers
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int nkb = l == 0 ? 2 : 4, wa = l == 0 ? 0 : l == 1 ? 2048 : 6144;
      unsigned again = 0;  // activations to form again, bit 4 mt + i
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        f32x4 c[4] = {*(const f32x4 *)&S.bias[l][16 * mt + 4 * q], {}, {}, {}};
#pragma unroll
        for (int kb = 0; kb < nkb; ++kb) {
          const bf16x4 a = *(const bf16x4 *)(S.wA + wa + (mt * nkb + kb) * 256 + lane * 4);
          c[kb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, h[kb], c[kb], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float s, v, dv;
          silu_both((c[0][i] + c[1][i]) + (c[2][i] + c[3][i]), s, v, dv);
          ds[l][mt][i] = dv;
          hn[mt][i] = (short)f2bf(v);
          again |= (near_middle(s, v, dv, c[0][i], c[1][i], c[2][i], c[3][i]) ? 1u : 0u) << (4 * mt + i);
          S.h[l][16 * mt + 4 * q + i][16 * w + r] = (unsigned short)hn[mt][i];
        }
      }
      // the whole wave forms each of them, lane k the product of input k; inputs and results in LDS
      const unsigned short(*in)[SP] = l == 0 ? S.h0 : S.h[l > 0 ? l - 1 : 0];
      const bool redo = again != 0;
      for (unsigned long long left = __ballot(redo); left; left = __ballot(again != 0)) {
        const int src = __ffsll(left) - 1, e = __ffs(__builtin_amdgcn_readlane((int)again, src)) - 1;
        const int mt = e >> 2, row = 4 * (src >> 4) + (e & 3), col = 16 * w + (src & 15);
        double z = 0.0;
        if (lane < 16 * nkb) {
          const int at = wa + (mt * nkb + (lane >> 4)) * 256 + (16 * ((lane >> 2) & 3) + row) * 4 + (lane & 3);
          z = (double)bf2f(S.wA[at]) * (double)bf2f(in[lane][col]);
        }
        z = wave_sum(z) + (double)S.bias[l][16 * mt + row];
        const unsigned short v = f2bf((float)(z / (1.0 + exp(-z))));
        if (lane == src) {
          S.h[l][16 * mt + row][col] = v;
          again &= again - 1;
        }
      }
      if (redo) {
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) hn[mt][i] = (short)S.h[l][16 * mt + 4 * q + i][16 * w + r];
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) h[mt] = hn[mt];
    }
    // output layer, loss and output delta: rows 0..2 of the tile, i.e. lanes with q = 0
    f32x4 c = *(const f32x4 *)&S.bias[3][4 * q];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const bf16x4 a = *(const bf16x4 *)(S.wA + 10240 + kb * 256 + lane * 4);
      c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, h[kb], c, 0, 0, 0);
    }
    float d4[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float diff = c[i] - t[i];
      d4[i] = valid && q == 0 ? (2.0f / (3.0f * (float)batch)) * diff : 0.0f;
      if (valid && q == 0) {
        se += (double)diff * (double)diff;
      }
      if (q == 0) S.dz4[i][16 * w + r] = d4[i];
    }
    const float e1 = __shfl(d4[1], r, 64), e2 = __shfl(d4[2], r, 64);
    const float b4 = q == 0 ? d4[0] : q == 1 ? e1 : q == 2 ? e2 : 0.0f;
    f32x4 d[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
      d[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(S.w4[16 * mt + r][q], b4, z, 0, 0, 0) * ds[2][mt];
    }
#pragma unroll
    for (int l = 2; l >= 0; --l) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) S.dz[l][16 * mt + 4 * q + i][16 * w + r] = d[mt][i];
      if (l == 0) break;
      f32x4 dn[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ob = 0; ob < 4; ++ob) {
          const f32x4 a = bf4(*(const bf16x4 *)&S.wB[l - 1][16 * mt + r][16 * ob + 4 * q]);
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[jj], d[ob][jj], acc, 0, 0, 0);
        }
        dn[mt] = acc * ds[l - 1][mt];
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) d[mt] = dn[mt];
    }
    __syncthreads();
    if ((tile + (int)gridDim.x) * TS < n) load_sample(tile + gridDim.x, x, t);
    // weight gradients: sum over the 64 samples of h_in[k] dz[o]
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      const int s0 = 16 * sb + 4 * q;
      const f32x4 a1 = bf4(*(const bf16x4 *)&S.h0[16 * (w & 1) + r][s0]), a2 = bf4(*(const bf16x4 *)&S.h[0][16 * w + r][s0]),
                  a3 = bf4(*(const bf16x4 *)&S.h[1][16 * w + r][s0]), a4 = bf4(*(const bf16x4 *)&S.h[2][16 * w + r][s0]);
#pragma unroll
      for (int ot = 0; ot < 2; ++ot) {
        const f32x4 bz = *(const f32x4 *)&S.dz[0][16 * (2 * (w >> 1) + ot) + r][s0];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) g1[ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[jj], bz[jj], g1[ot], 0, 0, 0);
      }
#pragma unroll
      for (int ot = 0; ot < 4; ++ot) {
        const f32x4 b2 = *(const f32x4 *)&S.dz[1][16 * ot + r][s0], b3 = *(const f32x4 *)&S.dz[2][16 * ot + r][s0];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          g2[ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[jj], b2[jj], g2[ot], 0, 0, 0);
          g3[ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(a3[jj], b3[jj], g3[ot], 0, 0, 0);
        }
      }
      const f32x4 bo = *(const f32x4 *)&S.dz4[r][s0];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) g4 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[jj], bo[jj], g4, 0, 0, 0);
      // bias gradients: samples 16 w + 4 sb .. + 3 of unit `lane`
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        const f32x4 v = *(const f32x4 *)&S.dz[l][lane][16 * w + 4 * sb];
        gb[l] += (v[0] + v[1]) + (v[2] + v[3]);
      }
      if (lane < 3) {
        const f32x4 v = *(const f32x4 *)&S.dz4[lane][16 * w + 4 * sb];
        gb4 += (v[0] + v[1]) + (v[2] + v[3]);
      }
    }
    __syncthreads();
  }
  // the workgroup's partial
  float *gp = grad_part + (size_t)blockIdx.x * MLP_NPARAM;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k1 = 16 * (w & 1) + 4 * q + i, k = 16 * w + 4 * q + i;
#pragma unroll
    for (int ot = 0; ot < 2; ++ot)
      if (k1 < 18) gp[k1 * 64 + 16 * (2 * (w >> 1) + ot) + r] = g1[ot][i];
#pragma unroll
    for (int ot = 0; ot < 4; ++ot) {
      gp[1216 + k * 64 + 16 * ot + r] = g2[ot][i];
      gp[5376 + k * 64 + 16 * ot + r] = g3[ot][i];
    }
    if (r < 3) gp[9536 + k * 3 + r] = g4[i];
  }
  float(*sb)[4][64] = (float(*)[4][64])S.dz;  // bias shares of the 4 waves
#pragma unroll
  for (int l = 0; l < 3; ++l) sb[l][w][lane] = gb[l];
  sb[3][w][lane] = gb4;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) se += __shfl_down(se, off, 64);
  if (lane == 0) S.red[w] = se;
  __syncthreads();
  const float bsum = (sb[w][0][lane] + sb[w][1][lane]) + (sb[w][2][lane] + sb[w][3][lane]);
  if (w < 3) gp[kLayers[w].pb + lane] = bsum;
  else if (lane < 3) gp[9728 + lane] = bsum;
  if (tid == 0) loss_part[blockIdx.x] = (float)((S.red[0] + S.red[1]) + (S.red[2] + S.red[3]));
}

// grad[p] = sum over the workgroups of the partials (4 interleaved shares, each in order, then the
// shares in order; 8 loads in flight per thread); loss_acc += sum of squared errors.  With `update`
// also Adam (beta1 = 0.9, beta2 = 0.999, eps = 1e-8; b1t, b2t = beta^t) and the parameter's place in
// the BF16 A-operand arrangement, which were two launches of their own.
__global__ void __launch_bounds__(256) k_mlp_step(const float *__restrict__ grad_part, const float *__restrict__ loss_part,
                                                  int nwg, float *__restrict__ grad, double *__restrict__ loss_acc,
                                                  int update, float *__restrict__ params, float *__restrict__ m1,
                                                  float *__restrict__ m2, unsigned short *__restrict__ wA, float lr,
                                                  float b1t, float b2t) {
  __shared__ float share[4][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, p = blockIdx.x * 64 + lane;
  const float *v = grad_part + min(p, MLP_NPARAM - 1);
  float a = 0.0f;
  for (int i = w; i < nwg; i += 32) {
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = v[(size_t)(i + 4 * u < nwg ? i + 4 * u : i) * MLP_NPARAM];
#pragma unroll
    for (int u = 0; u < 8; ++u) a += i + 4 * u < nwg ? t[u] : 0.0f;
  }
  share[w][lane] = a;
  __syncthreads();
  if (blockIdx.x == 0 && w == 1) {
    double l = 0.0;
    for (int i = lane; i < nwg; i += 64) l += (double)loss_part[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off, 64);
    if (lane == 0) *loss_acc += l;
  }
  if (w != 0 || p >= MLP_NPARAM) return;
  const float g = (share[0][lane] + share[1][lane]) + (share[2][lane] + share[3][lane]);
  grad[p] = g;
  if (!update) return;
  const float a1 = 0.9f * m1[p] + 0.1f * g;
  const float a2 = 0.999f * m2[p] + 0.001f * g * g;
  m1[p] = a1;
  m2[p] = a2;
  const float mh = a1 / (1.0f - b1t), vh = a2 / (1.0f - b2t);
  const float np = params[p] - lr * mh / (sqrtf(vh) + 1e-8f);
  params[p] = np;
  int l = 3;
  while (l > 0 && p < kLayers[l].pw) --l;
  const Layer L = kLayers[l];
  if (p >= L.pb) return;  // a bias
  const int k = (p - L.pw) / L.out, o = (p - L.pw) % L.out;
  wA[L.wa + (((o >> 4) * L.kb + (k >> 4)) * 64 + ((k >> 2) & 3) * 16 + (o & 15)) * 4 + (k & 3)] = f2bf(np);
}

// ---- launch wrappers ----
static inline unsigned nb(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <typename R>
void LearnLaunch<R>::features(const DevMesh<R> &m, const DevParams &p, const int *adj_off, const int *adj, float *feat,
                              R *y, hipStream_t st) {
  hipLaunchKernelGGL((k_features<R>), dim3(nb(p.nn, 256)), dim3(256), 0, st, p, (const R *)m.xpos, (const R *)m.v,
                     m.rest, m.mask, adj_off, adj, feat, y);
}
template <typename R>
void LearnLaunch<R>::guess(const DevMesh<R> &m, const DevParams &p, const MlpDev &net, const float *feat, const R *y,
                           hipStream_t st) {
  const long tiles = (p.nn + 15) / 16;
  const unsigned grid = (unsigned)std::min<long>((tiles + 3) / 4, 2048);
  hipLaunchKernelGGL((k_guess<R>), dim3(grid), dim3(256), 0, st, p, net, feat, y, m.mask, (const R *)m.ring.b[0],
                     m.ring.b[1], 1.0f / net.inv_s[6]);
}
template <typename R>
void LearnLaunch<R>::select(const DevMesh<R> &m, const TileDev &td, const DevParams &p, const int *adj_off,
                            const int *adj, const int *sell_off, const int *sell_col, int iters, const float *betas,
                            int nbeta, float *sm, hipStream_t st) {
  const unsigned g = nb(p.nn, 256);
  const int nnb = (int)nb(p.nn, 256);
  float4 *sm4[2] = {(float4 *)sm, (float4 *)sm + p.nn};
  hipLaunchKernelGGL((k_corr_diff<R>), dim3(g), dim3(256), 0, st, p.nn, m.mask, (const R *)m.ring.b[1],
                     (const R *)m.ring.b[0], sm4[0]);
  for (int k = 0; k < iters; ++k)
    hipLaunchKernelGGL(k_corr_smooth, dim3(g), dim3(256), 0, st, p.nn, m.mask, adj_off, sell_off, sell_col,
                       (const float4 *)sm4[k & 1], sm4[(k + 1) & 1]);
  const float4 *d = sm4[iters & 1];
  hipLaunchKernelGGL(k_ws_stage, dim3(1), dim3(1024), 0, st, m.ctrl, td.npart, nnb, 0, 0.0f);
  Launch<R>::tile_pass(m, td, p, st);
  Launch<R>::grad_pass(m, td, p, st);
  hipLaunchKernelGGL(k_ws_stage, dim3(1), dim3(1024), 0, st, m.ctrl, td.npart, nnb, 1, 0.0f);
  for (int j = 0; j < nbeta; ++j) {
    hipLaunchKernelGGL((k_corr_apply<R>), dim3(g), dim3(256), 0, st, p.nn, (const Ctrl *)m.ctrl, betas[j],
                       (const R *)m.ring.b[0], d, m.ring.b[1]);
    Launch<R>::tile_pass(m, td, p, st);
    Launch<R>::grad_pass(m, td, p, st);
    hipLaunchKernelGGL(k_ws_stage, dim3(1), dim3(1024), 0, st, m.ctrl, td.npart, nnb, 2, betas[j]);
  }
  hipLaunchKernelGGL((k_corr_apply<R>), dim3(g), dim3(256), 0, st, p.nn, (const Ctrl *)m.ctrl, -1.0f,
                     (const R *)m.ring.b[0], d, m.ring.b[1]);
  hipLaunchKernelGGL(k_ws_stage, dim3(1), dim3(1024), 0, st, m.ctrl, td.npart, nnb, 3, 0.0f);
}
template <typename R>
void LearnLaunch<R>::collect(const DevMesh<R> &m, const DevParams &p, const float *feat, const R *y,
                             const int *free_rank, long base, int stride, int phase, float *ds_x, float *ds_y,
                             hipStream_t st) {
  hipLaunchKernelGGL((k_collect<R>), dim3(nb(p.nn, 256)), dim3(256), 0, st, p, (const R *)m.xpos, feat, y, free_rank,
                     base, stride, phase, ds_x, ds_y);
}
template struct LearnLaunch<float>;
template struct LearnLaunch<double>;

void mlp_arrange(const float *params, unsigned short *wA, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_arrange, dim3(nb(MLP_WA, 256)), dim3(256), 0, st, params, wA);
}
void mlp_forward(const MlpDev &net, const float *feat, int n, float *out, hipStream_t st) {
  if (n <= 0) return;
  const long tiles = (n + 15) / 16;
  const unsigned grid = (unsigned)std::min<long>((tiles + 3) / 4, 2048);
  hipLaunchKernelGGL(k_mlp_forward, dim3(grid), dim3(256), 0, st, net, feat, n, out);
}
int mlp_train_wgs(int n) { return std::min((n + TS - 1) / TS, kTrainWGs); }
void mlp_train_partials(const MlpDev &net, const float *ds_x, const float *ds_y, const int *idx, int n, int batch,
                        float *grad_part, float *loss_part, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mlp_train, dim3(mlp_train_wgs(n)), dim3(256), sizeof(TrainLds), st, net, ds_x, ds_y, idx, n, batch,
                     grad_part, loss_part);
}
void mlp_step(const float *grad_part, const float *loss_part, int nwg, float *grad, double *loss_acc, bool update,
              float *params, float *m1, float *m2, unsigned short *wA, float lr, float b1t, float b2t, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_step, dim3(nb(MLP_NPARAM, 64)), dim3(256), 0, st, grad_part, loss_part, nwg, grad, loss_acc,
                     update ? 1 : 0, params, m1, m2, wA, lr, b1t, b2t);
}

}  // namespace pbs
