// surrogate_mlp.hip -- the reflectance surrogate's MLP: BF16 matrix-core
// kernels (forward, backward, Adam) and their host driver.
//
// No counterpart in the reference.  Layout: activations are row-major
// [batch][width] with the batch and the widths padded to multiples of 64 (the
// pads hold zeros and stay zero: padded weights and biases are zero and
// receive zero gradients).  Layer l keeps FP32 master weights
// W[N][K] (N = out, K = in), their BF16 copy for the products, the FP32 bias,
// Adam moments, and from the forward pass the FP32 pre-activation Z and the
// BF16 input A of the layer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "fdtd_hip.h"
#include "fdtd_internal.h"
#include "mpifdtd_surrogate.h"

#define HIPCHK(x)                                                                                    \
  do {                                                                                               \
    hipError_t e_ = (x);                                                                             \
    if (e_ != hipSuccess) return fdtd_fail(FDTD_EHIP, "%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

typedef unsigned short bf16_t;
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16_t v) { return __uint_as_float((unsigned)v << 16); }
// round to nearest even (finite inputs)
__device__ __forceinline__ bf16_t f2bf(float f)
{
  const unsigned u = __float_as_uint(f);
  return (bf16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// GELU(z) = z Phi(z), Phi the standard normal CDF; GELU'(z) = Phi(z) + z phi(z)
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z)
{
  const float Phi = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
  const float phi = 0.39894228040143268f * expf(-0.5f * z * z);
  return Phi + z * phi;
}

enum { EPI_F32 = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2 };

struct GemmOut {
  float *c;           // FP32 result [M][ldc]
  bf16_t *h;          // EPI_BIAS_GELU: BF16 GELU(z)
  const float *bias;  // EPI_BIAS, EPI_BIAS_GELU: [N]
  int ldc;
};

// C[M][N] = sum_k A(m, k) B(k, n): A(m, k) = a[m lda + k] (TA 0) or a[k lda + m]
// (TA 1); B(k, n) = b[n ldb + k] (TB 0) or b[k ldb + n] (TB 1).  One workgroup
// per 64 x 64 tile of C, four wavefronts of 32 x 32, each 2 x 2 products of
// v_mfma_f32_16x16x16 bf16 per 16-deep slice; the operands pass through LDS
// as [row][k] tiles 32 deep.  M, N multiples of 64, K of 32 (the caller pads).  Runs
// mlp_gemm_bf16 and the forward pass of networks too wide for k_mlp_forward.
template <int TA, int TB, int EPI>
__global__ __launch_bounds__(256) void k_gemm(const bf16_t *__restrict__ a, int lda, const bf16_t *__restrict__ b,
                                              int ldb, int K, GemmOut o)
{
  __shared__ __attribute__((aligned(16))) bf16_t sa[64][40];  // 32 k + 8 pad
  __shared__ __attribute__((aligned(16))) bf16_t sb[64][40];
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 32) {
    if (TA == 0) {  // 64 rows of 32 k: 4 chunks of 8 per row
      const int r = tid >> 2, c = (tid & 3) * 8;
      *(uint4 *)&sa[r][c] = *(const uint4 *)&a[(size_t)(m0 + r) * lda + k0 + c];
    } else {  // 32 rows of k, 64 m each: 8 chunks of 8 per row, transposed into LDS
      const int kr = tid >> 3, c = (tid & 7) * 8;
      const uint4 v = *(const uint4 *)&a[(size_t)(k0 + kr) * lda + m0 + c];
      const bf16_t *pv = (const bf16_t *)&v;
#pragma unroll
      for (int j = 0; j < 8; j++) sa[c + j][kr] = pv[j];
    }
    if (TB == 0) {
      const int r = tid >> 2, c = (tid & 3) * 8;
      *(uint4 *)&sb[r][c] = *(const uint4 *)&b[(size_t)(n0 + r) * ldb + k0 + c];
    } else {
      const int kr = tid >> 3, c = (tid & 7) * 8;
      const uint4 v = *(const uint4 *)&b[(size_t)(k0 + kr) * ldb + n0 + c];
      const bf16_t *pv = (const bf16_t *)&v;
#pragma unroll
      for (int j = 0; j < 8; j++) sb[c + j][kr] = pv[j];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 32; kk += 16) {
      // 16x16x16 operands: lane l holds row (l mod 16), k = 4 (l / 16) + 0..3
      bf16x4 af[2], bq[2];
#pragma unroll
      for (int i = 0; i < 2; i++) af[i] = *(const bf16x4 *)&sa[wm + i * 16 + (lane & 15)][kk + 4 * (lane >> 4)];
#pragma unroll
      for (int j = 0; j < 2; j++) bq[j] = *(const bf16x4 *)&sb[wn + j * 16 + (lane & 15)][kk + 4 * (lane >> 4)];
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(af[i], bq[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // result lane l, element r: row 4 (l / 16) + r, column l mod 16 of each 16 x 16 block
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + wm + i * 16 + 4 * (lane >> 4) + r, n = n0 + wn + j * 16 + (lane & 15);
        const size_t idx = (size_t)m * o.ldc + n;
        float v = acc[i][j][r];
        if (EPI == EPI_F32) {
          o.c[idx] = v;
        } else if (EPI == EPI_BIAS) {
          o.c[idx] = v + o.bias[n];
        } else {  // EPI_BIAS_GELU
          v += o.bias[n];
          o.c[idx] = v;
          o.h[idx] = f2bf(gelu(v));
        }
      }
}

// Workgroup barrier ordering LDS accesses only: the loads of the next slab stay in flight.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ------------------------------------------------------------------ training products
//
// Every product of a training step has its two operands with the summed index
// contiguous (C[m][n] = sum_k a[m][k] b[n][k]): the forward activations and the
// gradients are also stored transposed by the kernel that makes them, the BF16
// weights by Adam.  Tiles of 32 x BN (BN 64, or 32 for the weight gradients, whose
// 512 x 512 results would otherwise leave half of the compute units idle), slabs of
// 64 along k through two LDS buffers, the next slab's loads in flight meanwhile.
// The products are summed slice by slice of 16 in order, as k_gemm sums them.
// Bound by latency at these sizes (a 1024 x 512 x 512 product is 0.5 GFLOP): the
// weight gradient of a 512 x 512 layer over 1024 rows took 30.6 us with the
// operands transposed on their way into LDS and no load in flight.
enum { T_GELU = 0, T_MSE = 1, T_DW = 2, T_DA = 3 };

struct TrainOut {
  float *c;           // T_GELU: z; the others: the gradient in FP32  [M][ldc]
  bf16_t *h, *ht;     // T_GELU: GELU(z); T_MSE, T_DA: the gradient; [M][ldc] and its transpose [N][ldt]
  const float *bias;
  const float *zp;    // T_DA: pre-activation of the layer below [M][ldc]
  int ldc, ldt;
  // T_MSE: targets t[perm[row]][d] (perm null: row), B x d real outputs, the loss's sum
  const float *t;
  const int *perm;
  int B, d;
  float *loss;
};

template <int BN, int EPI>
__device__ __forceinline__ void train_tile(const bf16_t *__restrict__ a, const bf16_t *__restrict__ b, int K, int m0, int n0,
                                           const TrainOut &o, bf16_t *lds)
{
  constexpr int KS = 64, LD = KS + 8, CB = BN / 32;  // 16-byte chunks of b per thread
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = (w >> 1) * 16, wn = (w & 1) * (BN / 2);
  constexpr int NJ = BN / 32;
  bf16_t *sa = lds, *sb = lds + 2 * 32 * LD;
  const int r = tid >> 3, c = (tid & 7) * 8;
  const bf16_t *ga = a + (size_t)(m0 + r) * K + c;
  const bf16_t *gb = b + (size_t)(n0 + r) * K + c;
  uint4 va, vb[CB];
  auto fetch = [&](int k0) {
    va = *(const uint4 *)(ga + k0);
#pragma unroll
    for (int q = 0; q < CB; q++) vb[q] = *(const uint4 *)(gb + (size_t)32 * q * K + k0);
  };
  f32x4 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  for (int k0 = 0, p = 0; k0 < K; k0 += KS, p ^= 1) {
    bf16_t *ta = sa + p * 32 * LD, *tb = sb + p * BN * LD;
    *(uint4 *)&ta[r * LD + c] = va;
#pragma unroll
    for (int q = 0; q < CB; q++) *(uint4 *)&tb[(r + 32 * q) * LD + c] = vb[q];
    lds_barrier();
    if (k0 + KS < K) fetch(k0 + KS);
#pragma unroll
    for (int kk = 0; kk < KS; kk += 16) {
      const bf16x4 af = *(const bf16x4 *)&ta[(wm + (lane & 15)) * LD + kk + 4 * (lane >> 4)];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const bf16x4 bq = *(const bf16x4 *)&tb[(wn + j * 16 + (lane & 15)) * LD + kk + 4 * (lane >> 4)];
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(af, bq, acc[j], 0, 0, 0);
      }
    }
  }
  // lane l, element q: row 4 (l / 16) + q, column l mod 16 of each 16 x 16 block
  float loss = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int n = n0 + wn + j * 16 + (lane & 15), mb = m0 + wm + 4 * (lane >> 4);
    bf16_t hv[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = mb + q;
      const size_t idx = (size_t)m * o.ldc + n;
      float v = acc[j][q];
      if (EPI == T_DW) {
        o.c[idx] = v;
      } else if (EPI == T_GELU) {
        v += o.bias[n];
        o.c[idx] = v;
        hv[q] = f2bf(gelu(v));
      } else if (EPI == T_MSE) {
        v += o.bias[n];
        float g = 0.f;
        if (m < o.B && n < o.d) {
          const float e = v - o.t[(size_t)(o.perm ? o.perm[m] : m) * o.d + n];
          loss += e * e;
          g = 2.f * e / ((float)o.B * (float)o.d);
        }
        o.c[idx] = g;
        hv[q] = f2bf(g);
      } else {
        v *= gelu_d(o.zp[idx]);
        o.c[idx] = v;
        hv[q] = f2bf(v);
      }
      if (EPI != T_DW) o.h[idx] = hv[q];
    }
    if (EPI != T_DW) {
      ushort4 t4 = make_ushort4(hv[0], hv[1], hv[2], hv[3]);
      *(ushort4 *)&o.ht[(size_t)n * o.ldt + mb] = t4;
    }
  }
  if (EPI == T_MSE) {
    for (int q = 32; q > 0; q >>= 1) loss += __shfl_down(loss, q, 64);
    if (lane == 0) atomicAdd(o.loss, loss / ((float)o.B * (float)o.d));
  }
}

#define TRAIN_LDS(BN) (2 * (32 + (BN)) * 72)

template <int EPI>
__global__ __launch_bounds__(256) void k_train_fwd(const bf16_t *__restrict__ a, const bf16_t *__restrict__ b, int K, TrainOut o)
{
  __shared__ __attribute__((aligned(16))) bf16_t lds[TRAIN_LDS(64)];
  train_tile<64, EPI>(a, b, K, blockIdx.y * 32, blockIdx.x * 64, o, lds);
}

// The backward products of one layer in one launch (they share the gradient G alone):
// workgroups [0, ndw) the weight gradient, then nda of the layer below's gradient,
// then the bias gradient: the columns of G summed row by row in order (another order
// moves the biases by a rounding, which Adam and the BF16 activations carry into
// every weight).  A column's chain of additions is short work once its values are
// near: three wavefronts' loads go ahead of the one that adds, through LDS, beside
// the products' workgroups.  As a launch of one thread per column, each waiting for
// its own loads, it took 229 us, three quarters of a training step.
struct BwdArgs {
  const bf16_t *gt, *at;  // G^T [Np][Bp], A^T [Kp][Bp]: dW = G^T A
  const bf16_t *g, *wt;   // G [Bp][Np], W^T [Kp][Np]: dA = G W
  TrainOut dw, da;
  int Np, Kp, Bp, ndw, nda;
  const float *gf;        // G in FP32 [Bp][Np]
  float *db;
};

__global__ __launch_bounds__(256) void k_train_bwd(BwdArgs p)
{
  __shared__ __attribute__((aligned(16))) bf16_t lds[TRAIN_LDS(64)];
  int id = blockIdx.x;
  if (id < p.ndw) {
    const int nx = p.Kp / 32;
    train_tile<32, T_DW>(p.gt, p.at, p.Bp, id / nx * 32, id % nx * 32, p.dw, lds);
    return;
  }
  id -= p.ndw;
  if (id < p.nda) {
    const int nx = p.Kp / 64;
    train_tile<64, T_DA>(p.g, p.wt, p.Np, id / nx * 32, id % nx * 64, p.da, lds);
    return;
  }
  // 64 columns per workgroup, 32 rows at a time (Bp is a multiple of 64)
  float *buf = (float *)lds;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, n = (id - p.nda) * 64 + lane;
  float v[8], s = 0.f;
  auto fetch = [&](int r0) {
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = p.gf[(size_t)(r0 + w + 4 * q) * p.Np + n];
  };
  fetch(0);
  for (int r0 = 0, h = 0; r0 < p.Bp; r0 += 32, h ^= 1) {
    float *t = buf + h * 32 * 64 + lane;
#pragma unroll
    for (int q = 0; q < 8; q++) t[(w + 4 * q) * 64] = v[q];
    lds_barrier();
    if (r0 + 32 < p.Bp) fetch(r0 + 32);
    if (w == 0) {
#pragma unroll
      for (int r = 0; r < 32; r++) s += t[r * 64];
    }
  }
  if (w == 0) p.db[n] = s;
}

// rows perm[0..B) (perm null: 0..B) of x[.][d] (FP32) -> X[Bp][dp] (BF16, zero pads) and its transpose XT[dp][Bp]
__global__ __launch_bounds__(256) void k_pack(const float *x, const int *perm, int B, int d, bf16_t *X, bf16_t *XT, int Bp, int dp)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)Bp * dp) return;
  const int r = (int)(i / dp), c = (int)(i % dp);
  const bf16_t v = (r < B && c < d) ? f2bf(x[(size_t)(perm ? perm[r] : r) * d + c]) : (bf16_t)0;
  X[i] = v;
  XT[(size_t)c * Bp + r] = v;
}

// Adam (Kingma and Ba 2015) with bias correction c1 = 1 - beta1^t, c2 = 1 - beta2^t
__device__ __forceinline__ float adam(float *w, const float *g, float *m, float *v, size_t i, float lr, float c1, float c2)
{
  const float gi = g[i];
  const float mi = 0.9f * m[i] + 0.1f * gi, vi = 0.999f * v[i] + 0.001f * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
  w[i] = wi;
  return wi;
}

// One launch updates every layer: workgroup tiles of 32 x 32 weights, whose BF16 copy
// is written as [N][K] and, through LDS, as [K][N]; then the biases, 256 a workgroup.
#define MLP_MAX_LAYERS 8
struct AdamLayer {
  float *w, *dw, *mw, *vw, *b, *db, *mb, *vb;
  bf16_t *wh, *wt;
  int Np, Kp, first, tiles;  // first workgroup of the layer, its weight tiles
};
struct AdamArgs {
  AdamLayer l[MLP_MAX_LAYERS];
  int n, update;  // update 0: only refresh the BF16 copies
  float lr, c1, c2;
};

__global__ __launch_bounds__(256) void k_adam(AdamArgs a)
{
  __shared__ bf16_t tile[32][34];
  int q = a.n - 1;
  while (q > 0 && (int)blockIdx.x < a.l[q].first) q--;
  const AdamLayer &y = a.l[q];
  const int id = (int)blockIdx.x - y.first;
  if (id >= y.tiles) {
    const int n = (id - y.tiles) * 256 + threadIdx.x;
    if (n < y.Np && a.update) adam(y.b, y.db, y.mb, y.vb, n, a.lr, a.c1, a.c2);
    return;
  }
  const int nx = y.Kp / 32, n0 = id / nx * 32, k0 = id % nx * 32, c = threadIdx.x & 31;
#pragma unroll
  for (int r = threadIdx.x >> 5; r < 32; r += 8) {
    const size_t i = (size_t)(n0 + r) * y.Kp + k0 + c;
    const bf16_t h = f2bf(a.update ? adam(y.w, y.dw, y.mw, y.vw, i, a.lr, a.c1, a.c2) : y.w[i]);
    y.wh[i] = h;
    tile[r][c] = h;
  }
  __syncthreads();
#pragma unroll
  for (int r = threadIdx.x >> 5; r < 32; r += 8) y.wt[(size_t)(k0 + r) * y.Np + n0 + c] = tile[c][r];
}

// ------------------------------------------------------------------ inference
//
// The whole network for 16 rows per workgroup: the activations stay in LDS from layer
// to layer and the weights come from a copy in the order of the matrix operands
// (wp[n / 16][k / 32][lane][8]: a wavefront's load is 1 KB in a row).  Bound by the
// weights' way from L2 into each compute unit (1.25 MB for 13-512-512-512-180, about
// 8 us at 64 B a clock).  The sums run slice by slice of 16 as in k_gemm: same bits.
struct FwdLayer {
  const bf16_t *wp;
  const float *b;
  int Kp, Np, N;
};
struct FwdArgs {
  FwdLayer l[MLP_MAX_LAYERS];
  int n, B, d0, ld;  // ld: LDS row length of an activation buffer
  const float *x;
  float *y;
};
#define FWD_WAVES 8

__global__ __launch_bounds__(64 * FWD_WAVES) void k_mlp_forward(FwdArgs a)
{
  extern __shared__ __attribute__((aligned(16))) bf16_t act[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, row0 = blockIdx.x * 16, ld = a.ld;
  bf16_t *in = act, *out = act + 16 * ld;
  for (int i = tid; i < 16 * a.l[0].Kp; i += 64 * FWD_WAVES) {
    const int r = i / a.l[0].Kp, c = i % a.l[0].Kp;
    in[r * ld + c] = row0 + r < a.B && c < a.d0 ? f2bf(a.x[(size_t)(row0 + r) * a.d0 + c]) : (bf16_t)0;
  }
  __syncthreads();
  for (int l = 0; l < a.n; l++) {
    const FwdLayer &y = a.l[l];
    const int nt = y.Np / 16, kp = y.Kp / 32;
    const bool last = l + 1 == a.n;
    const bf16_t *ar = in + (lane & 15) * ld + 4 * (lane >> 4);
    for (int t0 = 4 * w; t0 < nt; t0 += 4 * FWD_WAVES) {  // Np is a multiple of 64: whole groups of 4 tiles
      f32x4 acc[4];
#pragma unroll
      for (int j = 0; j < 4; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      const uint4 *wp = (const uint4 *)y.wp + (size_t)t0 * kp * 64 + lane;
#pragma unroll 4
      for (int k = 0; k < kp; k++) {
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = wp[((size_t)j * kp + k) * 64];
        const bf16x4 a0 = *(const bf16x4 *)(ar + 32 * k), a1 = *(const bf16x4 *)(ar + 32 * k + 16);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bf16x4 *bv = (const bf16x4 *)&v[j];
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0, bv[0], acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, bv[1], acc[j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int n = (t0 + j) * 16 + (lane & 15);
        const float bias = y.b[n];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int r = 4 * (lane >> 4) + q;
          const float v = acc[j][q] + bias;
          if (!last) out[r * ld + n] = f2bf(gelu(v));
          else if (n < y.N && row0 + r < a.B) a.y[(size_t)(row0 + r) * y.N + n] = v;
        }
      }
    }
    __syncthreads();
    bf16_t *t = in;
    in = out;
    out = t;
  }
}

// wp of a layer from its BF16 weights [Np][Kp]: one 16-byte entry per thread
__global__ __launch_bounds__(256) void k_pack_w(const bf16_t *wh, int Np, int Kp, bf16_t *wp)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)Np * Kp / 8) return;
  const int lane = (int)(i & 63), kp = Kp / 32;
  const size_t q = i >> 6;
  const int n = (int)(q / kp) * 16 + (lane & 15), k = (int)(q % kp) * 32 + 4 * (lane >> 4);
  const ushort4 lo = *(const ushort4 *)&wh[(size_t)n * Kp + k], hi = *(const ushort4 *)&wh[(size_t)n * Kp + k + 16];
  ushort4 *o = (ushort4 *)wp + 2 * i;
  o[0] = lo;
  o[1] = hi;
}

// y[B][d] (FP32, real sizes) from Y[Bp][dp]
__global__ __launch_bounds__(256) void k_unpack(const float *Y, int dp, int B, int d, float *y)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)B * d) return;
  y[i] = Y[(i / d) * dp + (i % d)];
}

// ------------------------------------------------------------------ host

struct MlpLayer {
  int K, N, Kp, Np;  // real and padded (multiples of 64) in / out widths
  float *w, *b, *dw, *db, *mw, *vw, *mb, *vb;
  bf16_t *wh, *wt, *wp;  // BF16 weights: [Np][Kp], transposed, and in k_mlp_forward's order
  float *z;              // [Bp][Np] pre-activation (FP32)
  bf16_t *a, *at;        // input of the layer (BF16): [Bp][Kp] and transposed
};

struct mlp_net {
  int L, Bmax;
  MlpLayer l[MLP_MAX_LAYERS];
  int maxW;            // widest padded width
  bool packed;         // wp holds the current weights
  bf16_t *gh[2], *ght[2];  // gradient w.r.t. a layer's output [Bp][Np] and transposed; the layer below's
  float *gf[2];            // and in FP32
  float *loss;   // device losses, one per batch of the current epoch
  int nloss;
  int *perm;       // device permutation of an epoch
  int nperm;
  long step;
};

static inline int pad_to(int v, int q) { return (v + q - 1) / q * q; }

template <int TA, int TB, int EPI>
static void gemm(const bf16_t *a, int lda, const bf16_t *b, int ldb, int M, int N, int K, const GemmOut &o)
{
  hipLaunchKernelGGL((k_gemm<TA, TB, EPI>), dim3(N / 64, M / 64), dim3(256), 0, 0, a, lda, b, ldb, K, o);
}

static uint64_t sm64(uint64_t &s)
{
  s += 0x9E3779B97F4A7C15ull;
  uint64_t z = s;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

template <typename T>
static int dalloc(T **p, size_t n)
{
  HIPCHK(hipMalloc(p, std::max<size_t>(1, n) * sizeof(T)));
  HIPCHK(hipMemset(*p, 0, std::max<size_t>(1, n) * sizeof(T)));
  return FDTD_OK;
}

static void free_net(mlp_net *n)
{
  for (int i = 0; i < n->L; i++) {
    MlpLayer &y = n->l[i];
    for (float *p : {y.w, y.b, y.dw, y.db, y.mw, y.vw, y.mb, y.vb, y.z}) (void)hipFree(p);
    for (bf16_t *p : {y.wh, y.wt, y.wp, y.a, y.at}) (void)hipFree(p);
  }
  for (int i = 0; i < 2; i++) {
    (void)hipFree(n->gh[i]);
    (void)hipFree(n->ght[i]);
    (void)hipFree(n->gf[i]);
  }
  (void)hipFree(n->loss);
  (void)hipFree(n->perm);
  delete n;
}

// one k_adam launch over layers [l0, l1): an Adam step, or (update 0) only the BF16 copies
static void launch_adam(mlp_net *n, int l0, int l1, int update, float lr, float c1, float c2)
{
  AdamArgs a = {};
  int blocks = 0;
  a.n = l1 - l0;
  a.update = update;
  a.lr = lr;
  a.c1 = c1;
  a.c2 = c2;
  for (int i = l0; i < l1; i++) {
    MlpLayer &y = n->l[i];
    const int tiles = (y.Np / 32) * (y.Kp / 32);
    a.l[i - l0] = AdamLayer{y.w, y.dw, y.mw, y.vw, y.b, y.db, y.mb, y.vb, y.wh, y.wt, y.Np, y.Kp, blocks, tiles};
    blocks += tiles + (y.Np + 255) / 256;
  }
  hipLaunchKernelGGL(k_adam, dim3(blocks), dim3(256), 0, 0, a);
  n->packed = false;
}

extern "C" int mlp_create(int nlayers, const int *dims, int batch_max, unsigned long long seed, mlp_net **out)
{
  if (!dims || !out || nlayers < 1 || nlayers > MLP_MAX_LAYERS || batch_max < 1)
    return fdtd_fail(FDTD_EINVAL, "mlp_create: bad argument");
  for (int i = 0; i <= nlayers; i++)
    if (dims[i] < 1 || dims[i] > 4096) return fdtd_fail(FDTD_EINVAL, "mlp_create: width %d out of range", dims[i]);
  mlp_net *n = new mlp_net();
  n->L = nlayers;
  n->Bmax = pad_to(batch_max, 64);
  // every width padded to 64: a layer's padded output is the next layer's padded input
  int maxW = 0;
  uint64_t s = seed;
  int rc = FDTD_OK;
  for (int i = 0; i < nlayers && rc == FDTD_OK; i++) {
    MlpLayer &y = n->l[i];
    y.K = dims[i];
    y.N = dims[i + 1];
    y.Kp = pad_to(y.K, 64);
    y.Np = pad_to(y.N, 64);
    maxW = std::max(maxW, std::max(y.Np, y.Kp));
    const size_t nw = (size_t)y.Np * y.Kp;
    if ((rc = dalloc(&y.w, nw)) || (rc = dalloc(&y.dw, nw)) || (rc = dalloc(&y.mw, nw)) || (rc = dalloc(&y.vw, nw)) ||
        (rc = dalloc(&y.wh, nw)) || (rc = dalloc(&y.wt, nw)) || (rc = dalloc(&y.wp, nw)) || (rc = dalloc(&y.b, y.Np)) || (rc = dalloc(&y.db, y.Np)) ||
        (rc = dalloc(&y.mb, y.Np)) || (rc = dalloc(&y.vb, y.Np)) || (rc = dalloc(&y.z, (size_t)n->Bmax * y.Np)) ||
        (rc = dalloc(&y.a, (size_t)n->Bmax * y.Kp)) || (rc = dalloc(&y.at, (size_t)n->Bmax * y.Kp)))
      break;
    std::vector<float> hw(nw, 0.f);
    const double bound = 1.0 / std::sqrt((double)y.K);
    for (int r = 0; r < y.N; r++)
      for (int c = 0; c < y.K; c++)
        hw[(size_t)r * y.Kp + c] = (float)((2.0 * (double)(sm64(s) >> 11) / 9007199254740992.0 - 1.0) * bound);
    if (hipMemcpy(y.w, hw.data(), nw * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
      rc = fdtd_fail(FDTD_EHIP, "mlp_create: upload failed");
      break;
    }
    launch_adam(n, i, i + 1, 0, 0.f, 1.f, 1.f);
  }
  if (rc == FDTD_OK) {
    const size_t ng = (size_t)n->Bmax * maxW;
    n->nloss = 1;
    n->maxW = maxW;
    for (int i = 0; i < 2 && rc == FDTD_OK; i++)
      (rc = dalloc(&n->gh[i], ng)) || (rc = dalloc(&n->ght[i], ng)) || (rc = dalloc(&n->gf[i], ng));
    if (rc == FDTD_OK && (rc = dalloc(&n->loss, 1)) == FDTD_OK && hipDeviceSynchronize() != hipSuccess)
      rc = fdtd_fail(FDTD_EHIP, "mlp_create: init failed");
  }
  if (rc) {
    free_net(n);
    return rc;
  }
  *out = n;
  return FDTD_OK;
}

extern "C" int mlp_destroy(mlp_net *net)
{
  if (!net) return FDTD_EINVAL;
  (void)hipDeviceSynchronize();
  free_net(net);
  return FDTD_OK;
}

// rows of an activation buffer in k_mlp_forward's LDS: the widest layer and a pad that
// spreads the rows over the banks; both buffers have to fit 64 KiB (widths up to 960)
static int fwd_ld(const mlp_net *n) { return n->maxW + 8; }
static bool fwd_fits(const mlp_net *n) { return 2u * 16 * fwd_ld(n) * sizeof(bf16_t) <= 65536; }

// Whether k_mlp_forward's workgroups, which read and write 16 rows each in any order, may
// run on these buffers: y apart from x, or row for row in its place.
static bool fwd_apart(const float *x, size_t nx, const float *y, size_t ny)
{
  const uintptr_t a = (uintptr_t)x, b = (uintptr_t)y;
  return b >= a + nx * sizeof(float) || a >= b + ny * sizeof(float) || (a == b && nx == ny);
}

extern "C" int mlp_forward(mlp_net *n, const float *x, int B, float *y)
{
  if (!n || !x || !y || B < 1 || B > n->Bmax) return fdtd_fail(FDTD_EINVAL, "mlp_forward: bad argument");
  if (fwd_fits(n) && fwd_apart(x, (size_t)B * n->l[0].K, y, (size_t)B * n->l[n->L - 1].N)) {
    FwdArgs a = {};
    a.n = n->L;
    a.B = B;
    a.d0 = n->l[0].K;
    a.ld = fwd_ld(n);
    a.x = x;
    a.y = y;
    for (int i = 0; i < n->L; i++) {
      MlpLayer &l = n->l[i];
      if (!n->packed)
        hipLaunchKernelGGL(k_pack_w, dim3((unsigned)(((size_t)l.Np * l.Kp / 8 + 255) / 256)), dim3(256), 0, 0, l.wh, l.Np,
                           l.Kp, l.wp);
      a.l[i] = FwdLayer{l.wp, l.b, l.Kp, l.Np, l.N};
    }
    n->packed = true;
    hipLaunchKernelGGL(k_mlp_forward, dim3((B + 15) / 16), dim3(64 * FWD_WAVES), 2 * 16 * fwd_ld(n) * sizeof(bf16_t), 0, a);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return FDTD_OK;
  }
  // layer by layer: layer i's input is l[i].a, its output the next layer's input
  // (BF16 GELU) or l[L-1].z (the linear output)
  const int Bp = pad_to(B, 64);
  MlpLayer &l0 = n->l[0];
  const size_t np = (size_t)Bp * l0.Kp;
  hipLaunchKernelGGL(k_pack, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, 0, x, (const int *)nullptr, B, l0.K, l0.a,
                     l0.at, Bp, l0.Kp);
  for (int i = 0; i < n->L; i++) {
    MlpLayer &l = n->l[i];
    GemmOut o = {};
    o.c = l.z;
    o.bias = l.b;
    o.ldc = l.Np;
    if (i + 1 < n->L) {
      o.h = n->l[i + 1].a;
      gemm<0, 0, EPI_BIAS_GELU>(l.a, l.Kp, l.wh, l.Kp, Bp, l.Np, l.Kp, o);
    } else {
      gemm<0, 0, EPI_BIAS>(l.a, l.Kp, l.wh, l.Kp, Bp, l.Np, l.Kp, o);
    }
  }
  MlpLayer &o = n->l[n->L - 1];
  const size_t ny = (size_t)B * o.N;
  hipLaunchKernelGGL(k_unpack, dim3((unsigned)((ny + 255) / 256)), dim3(256), 0, 0, o.z, o.Np, B, o.N, y);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  return FDTD_OK;
}

// gradients of a batch (rows perm[0..B) of x and t, or 0..B) into the layers' dW / db,
// the batch's loss into *loss_dev (accumulated: the caller zeroes it); no synchronisation
static int grads_async(mlp_net *n, const float *x, const float *t, const int *perm, int B, float *loss_dev)
{
  const int Bp = pad_to(B, 64);
  MlpLayer &l0 = n->l[0];
  const size_t np = (size_t)Bp * l0.Kp;
  hipLaunchKernelGGL(k_pack, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, 0, x, perm, B, l0.K, l0.a, l0.at, Bp, l0.Kp);
  for (int i = 0; i < n->L; i++) {
    MlpLayer &y = n->l[i];
    TrainOut o = {};
    o.c = i + 1 < n->L ? y.z : n->gf[0];
    o.bias = y.b;
    o.ldc = y.Np;
    o.ldt = Bp;
    const dim3 grid(y.Np / 64, Bp / 32);
    if (i + 1 < n->L) {
      o.h = n->l[i + 1].a;
      o.ht = n->l[i + 1].at;
      hipLaunchKernelGGL(k_train_fwd<T_GELU>, grid, dim3(256), 0, 0, y.a, y.wh, y.Kp, o);
    } else {
      o.h = n->gh[0];
      o.ht = n->ght[0];
      o.t = t;
      o.perm = perm;
      o.B = B;
      o.d = y.N;
      o.loss = loss_dev;
      hipLaunchKernelGGL(k_train_fwd<T_MSE>, grid, dim3(256), 0, 0, y.a, y.wh, y.Kp, o);
    }
  }
  for (int i = n->L - 1, p = 0; i >= 0; i--, p ^= 1) {
    MlpLayer &y = n->l[i];
    BwdArgs b = {};
    b.gt = n->ght[p];
    b.at = y.at;
    b.g = n->gh[p];
    b.wt = y.wt;
    b.Np = y.Np;
    b.Kp = y.Kp;
    b.Bp = Bp;
    b.gf = n->gf[p];
    b.db = y.db;
    b.dw.c = y.dw;
    b.dw.ldc = y.Kp;
    b.ndw = (y.Np / 32) * (y.Kp / 32);
    if (i > 0) {
      // times GELU'(z) of the layer below: that layer's output gradient
      b.nda = (Bp / 32) * (y.Kp / 64);
      b.da.h = n->gh[p ^ 1];
      b.da.ht = n->ght[p ^ 1];
      b.da.zp = n->l[i - 1].z;
      b.da.c = n->gf[p ^ 1];
      b.da.ldc = y.Kp;
      b.da.ldt = Bp;
    }
    hipLaunchKernelGGL(k_train_bwd, dim3(b.ndw + b.nda + y.Np / 64), dim3(256), 0, 0, b);
  }
  HIPCHK(hipGetLastError());
  return FDTD_OK;
}

static int adam_async(mlp_net *n, float lr)
{
  n->step++;
  const float c1 = (float)(1.0 - std::pow(0.9, (double)n->step)), c2 = (float)(1.0 - std::pow(0.999, (double)n->step));
  launch_adam(n, 0, n->L, 1, lr, c1, c2);
  HIPCHK(hipGetLastError());
  return FDTD_OK;
}

extern "C" int mlp_grads(mlp_net *n, const float *x, const float *t, int B, float *loss)
{
  if (!n || !x || !t || B < 1 || B > n->Bmax) return fdtd_fail(FDTD_EINVAL, "mlp_grads: bad argument");
  HIPCHK(hipMemset(n->loss, 0, sizeof(float)));
  int rc = grads_async(n, x, t, nullptr, B, n->loss);
  if (rc) return rc;
  if (loss) HIPCHK(hipMemcpy(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost));
  HIPCHK(hipDeviceSynchronize());
  return FDTD_OK;
}

extern "C" int mlp_train_step(mlp_net *n, const float *x, const float *t, int B, float lr, float *loss)
{
  if (!n || !x || !t || B < 1 || B > n->Bmax) return fdtd_fail(FDTD_EINVAL, "mlp_train_step: bad argument");
  HIPCHK(hipMemset(n->loss, 0, sizeof(float)));
  int rc = grads_async(n, x, t, nullptr, B, n->loss);
  if (rc || (rc = adam_async(n, lr))) return rc;
  if (loss) HIPCHK(hipMemcpy(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost));
  HIPCHK(hipDeviceSynchronize());
  return FDTD_OK;
}

extern "C" int mlp_train_epoch(mlp_net *n, const float *x, const float *t, int rows, int batch, unsigned long long seed,
                               float lr, float *loss)
{
  if (!n || !x || !t || rows < 1 || batch < 1 || batch > n->Bmax) return fdtd_fail(FDTD_EINVAL, "mlp_train_epoch: bad argument");
  // Fisher-Yates shuffle from a SplitMix64 stream of `seed`
  std::vector<int> perm(rows);
  for (int i = 0; i < rows; i++) perm[i] = i;
  uint64_t s = seed;
  for (int i = rows - 1; i > 0; i--) std::swap(perm[i], perm[(int)(sm64(s) % (uint64_t)(i + 1))]);
  if (n->nperm < rows) {
    (void)hipFree(n->perm);
    n->perm = nullptr;
    n->nperm = 0;
    HIPCHK(hipMalloc(&n->perm, (size_t)rows * sizeof(int)));
    n->nperm = rows;
  }
  const int nb = (rows + batch - 1) / batch;
  if (n->nloss < nb) {
    (void)hipFree(n->loss);
    n->loss = nullptr;
    n->nloss = 0;
    HIPCHK(hipMalloc(&n->loss, (size_t)nb * sizeof(float)));
    n->nloss = nb;
  }
  HIPCHK(hipMemcpy(n->perm, perm.data(), (size_t)rows * sizeof(int), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(n->loss, 0, (size_t)nb * sizeof(float)));
  for (int b = 0; b < nb; b++) {
    const int B = std::min(batch, rows - b * batch);
    int rc = grads_async(n, x, t, n->perm + b * batch, B, n->loss + b);
    if (rc || (rc = adam_async(n, lr))) return rc;
  }
  std::vector<float> lb(nb);
  HIPCHK(hipMemcpy(lb.data(), n->loss, (size_t)nb * sizeof(float), hipMemcpyDeviceToHost));
  HIPCHK(hipDeviceSynchronize());
  if (loss) {
    double acc = 0.0;
    for (int b = 0; b < nb; b++) acc += (double)lb[b] * std::min(batch, rows - b * batch);
    *loss = (float)(acc / rows);
  }
  return FDTD_OK;
}

static int copy_layer(mlp_net *n, int l, float *w, float *b, const float *dw_src, const float *db_src)
{
  MlpLayer &y = n->l[l];
  std::vector<float> h((size_t)y.Np * y.Kp), hb(y.Np);
  HIPCHK(hipMemcpy(h.data(), dw_src, h.size() * sizeof(float), hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(hb.data(), db_src, hb.size() * sizeof(float), hipMemcpyDeviceToHost));
  for (int r = 0; r < y.N; r++)
    for (int c = 0; c < y.K; c++) w[(size_t)r * y.K + c] = h[(size_t)r * y.Kp + c];
  for (int r = 0; r < y.N; r++) b[r] = hb[r];
  return FDTD_OK;
}

extern "C" int mlp_get_params(mlp_net *n, int l, float *w, float *b)
{
  if (!n || l < 0 || l >= n->L || !w || !b) return fdtd_fail(FDTD_EINVAL, "mlp_get_params: bad argument");
  return copy_layer(n, l, w, b, n->l[l].w, n->l[l].b);
}

extern "C" int mlp_get_grads(mlp_net *n, int l, float *dw, float *db)
{
  if (!n || l < 0 || l >= n->L || !dw || !db) return fdtd_fail(FDTD_EINVAL, "mlp_get_grads: bad argument");
  return copy_layer(n, l, dw, db, n->l[l].dw, n->l[l].db);
}

extern "C" int mlp_set_params(mlp_net *n, int l, const float *w, const float *b)
{
  if (!n || l < 0 || l >= n->L || !w || !b) return fdtd_fail(FDTD_EINVAL, "mlp_set_params: bad argument");
  MlpLayer &y = n->l[l];
  std::vector<float> h((size_t)y.Np * y.Kp, 0.f), hb(y.Np, 0.f);
  for (int r = 0; r < y.N; r++)
    for (int c = 0; c < y.K; c++) h[(size_t)r * y.Kp + c] = w[(size_t)r * y.K + c];
  for (int r = 0; r < y.N; r++) hb[r] = b[r];
  HIPCHK(hipMemcpy(y.w, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(y.b, hb.data(), hb.size() * sizeof(float), hipMemcpyHostToDevice));
  launch_adam(n, l, l + 1, 0, 0.f, 1.f, 1.f);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  return FDTD_OK;
}

extern "C" int mlp_gemm_bf16(const unsigned short *a, const unsigned short *b, float *c, int M, int N, int K, int ta, int tb)
{
  if (!a || !b || !c || M <= 0 || N <= 0 || K <= 0 || M % 64 || N % 64 || K % 32 || (ta & ~1) || (tb & ~1))
    return fdtd_fail(FDTD_EINVAL, "mlp_gemm_bf16: sizes must be multiples of 64 (M, N) and 32 (K)");
  GemmOut o = {};
  o.c = c;
  o.ldc = N;
  const int lda = ta ? M : K, ldb = tb ? N : K;
  if (!ta && !tb)
    gemm<0, 0, EPI_F32>(a, lda, b, ldb, M, N, K, o);
  else if (!ta && tb)
    gemm<0, 1, EPI_F32>(a, lda, b, ldb, M, N, K, o);
  else if (ta && !tb)
    gemm<1, 0, EPI_F32>(a, lda, b, ldb, M, N, K, o);
  else
    gemm<1, 1, EPI_F32>(a, lda, b, ldb, M, N, K, o);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  return FDTD_OK;
}
