// fdt_mlp.hip -- kernels of the learned initialiser: a BF16 MFMA GEMM with a
// fused bias/GELU epilogue and the element-wise passes of training
// (GELU backward, bias gradients, Adam, loss) and of inference (signal
// normalisation, decoding of the network outputs into chain start values and
// proposal widths, the fallback test).
//
// GEMM: C[M x N] = A[M x K] . B[K x N] in v_mfma_f32_16x16x32_bf16 (FP32
// accumulation).  Each operand is stored with k contiguous or with m (n)
// contiguous, so X.W, dZ.W^T and X^T.dZ are one kernel (a transposed A with a
// k-contiguous B is no product of the network and refused).
#include "fdt_device.h"
#include "fdt_mlp.h"

namespace fdt {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (finite inputs)
FDT_DEV uint16_t f2bf(float x) {
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
FDT_DEV float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
FDT_DEV float gelu_grad(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// A 256-thread workgroup computes a TM x TN tile, each of its 2 x 2 waves a
// quadrant in 16 x 16 blocks, K in steps of 64.  What bounds it: the forward
// of 65,536 rows is memory- and LDS-fed MFMA work (128 x 128 tiles reuse every
// staged element 128 times; 64 x 64 tiles with 2-byte loads, as before, ran
// 50 TFLOP/s), a training step's products are a few hundred thousand outputs
// and bound by latency, so their tiles shrink until every CU has one.  The
// next step's global loads (16 bytes a lane) are in flight while a step
// multiplies; LDS rows are 144 bytes, which spreads a wave's 16-byte reads
// over all banks.  An operand with m (n) contiguous is transposed on its way
// to LDS in pairs of k.  Every output is the same chain of 32-wide products
// in k order for every tile.
constexpr int GK = 64;   // K step
constexpr int GLD = 72;  // LDS row stride in bf16

typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// one operand's tile of T rows (m or n) by GK: fetched to registers, then stored to LDS [row][k]
template <int T, bool KC>
struct Stage {
  static constexpr int UNITS = T * GK / 8;  // of 8 elements
  static constexpr int NU = KC || UNITS >= 512 ? UNITS / 256 : 2;  // per thread
  static_assert(KC ? UNITS >= 256 : UNITS >= 256 && T % 32 == 0, "tile too small");
  // a tile of 32 rows has pairs for half of the threads only
  static FDT_DEV bool mine() { return KC || UNITS >= 512 || threadIdx.x < UNITS / 2; }
  u16x8 v[NU];
  // unit u: KC: row u / 8, k (u % 8) * 8.  Otherwise units come in pairs (k, k + 1) of 8 rows: four 8-row groups
  // and 16 k pairs per wave (64-byte runs of global memory, two lanes per LDS bank)
  static FDT_DEV void where(int i, int& row, int& k) {
    const int t = threadIdx.x;
    if constexpr (KC) {
      const int u = t + 256 * i;
      row = u >> 3;
      k = (u & 7) * 8;
    } else {
      const int p = t + 256 * (i >> 1);  // T / 8 * GK / 2 pairs
      const int g = p >> 6;              // wave-sized block: T / 32 row blocks, then two k halves
      row = ((g % (T / 32)) * 4 + (p & 3)) * 8;
      k = ((g / (T / 32)) * 16 + ((p >> 2) & 15)) * 2 + (i & 1);
    }
  }
  FDT_DEV void fetch(const GemmOperand& o, int row0, int rows, int k0, int K) {
    if (!mine()) return;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      int r, k;
      where(i, r, k);
      r += row0;
      k += k0;
      const uint16_t* p = o.p + (KC ? (size_t)r * o.ld + k : (size_t)k * o.ld + r);
      const bool whole = KC ? (r < rows && k + 8 <= K) : (k < K && r + 8 <= rows);
      if (whole && o.vec) v[i] = *reinterpret_cast<const u16x8*>(p);
      else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int re = KC ? r : r + e, ke = KC ? k + e : k;
          uint16_t x = 0;
          if (ke < K) {
            if (re < rows) x = p[e];
            else if (re == rows && o.ones) x = 0x3F80;  // bf16 1
          }
          v[i][e] = x;
        }
      }
    }
  }
  FDT_DEV void store(uint16_t* lds) const {
    if (!mine()) return;
#pragma unroll
    for (int i = 0; i < NU; i += KC ? 1 : 2) {
      int r, k;
      where(i, r, k);
      if constexpr (KC) *reinterpret_cast<u16x8*>(&lds[r * GLD + k]) = v[i];
      else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          *reinterpret_cast<uint32_t*>(&lds[(r + e) * GLD + k]) = (uint32_t)v[i][e] | ((uint32_t)v[i + 1][e] << 16);
      }
    }
  }
};

template <int TM, int TN, bool AK, bool BK>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[TM * GLD];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[TN * GLD];  // [n][k]
  constexpr int MB = TM / 32, NB = TN / 32;                       // 16 x 16 blocks of a wave's quadrant
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rows = g.M + (g.a.ones ? 1 : 0);
  // The n tiles of one m tile follow each other on one XCD (workgroups go
  // round robin over the 8), so that its L2 holds the A rows they share
  const int nt = (g.N + TN - 1) / TN, mt = (rows + TM - 1) / TM;
  int b = blockIdx.x, tm, tn;
  if (b < (mt >> 3) * 8 * nt) { tm = (b >> 3) / nt * 8 + (b & 7); tn = (b >> 3) % nt; }
  else { tm = b / nt; tn = b % nt; }
  const int m0 = tm * TM, n0 = tn * TN;
  const int qm = (wave >> 1) * (TM / 2), qn = (wave & 1) * (TN / 2);
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  Stage<TM, AK> sa;
  Stage<TN, BK> sb;
  sa.fetch(g.a, m0, g.M, 0, g.K);
  sb.fetch(g.b, n0, g.N, 0, g.K);
  const int r = lane & 15, kb = (lane >> 4) * 8;
  for (int k0 = 0; k0 < g.K; k0 += GK) {
    sa.store(As);
    sb.store(Bs);
    __syncthreads();
    if (k0 + GK < g.K) {
      sa.fetch(g.a, m0, g.M, k0 + GK, g.K);
      sb.fetch(g.b, n0, g.N, k0 + GK, g.K);
    }
#pragma unroll
    for (int h = 0; h < GK; h += 32) {
      if (k0 + h >= g.K) break;
      bf16x8 a[MB], bb[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i) a[i] = *reinterpret_cast<const bf16x8*>(&As[(qm + 16 * i + r) * GLD + h + kb]);
#pragma unroll
      for (int j = 0; j < NB; ++j) bb[j] = *reinterpret_cast<const bf16x8*>(&Bs[(qn + 16 * j + r) * GLD + h + kb]);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bb[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // lane holds C[(lane / 16) * 4 + v][lane % 16] of each 16x16 block
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + qn + 16 * j + (lane & 15);
    if (n >= g.N) continue;
    const float bias = g.bias ? g.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + qm + 16 * i + (lane >> 4) * 4 + v;
        if (m >= rows) continue;
        float x = acc[i][j][v];
        const size_t ci = (size_t)m * g.ldc + n;
        if (g.bias) x += bias;
        if (g.C) g.C[ci] = x;
        if (g.Cb) g.Cb[ci] = f2bf(g.act == GEMM_GELU ? gelu(x) : g.act == GEMM_GELU_BWD ? x * gelu_grad(g.Z[ci]) : x);
      }
  }
}

// Adam (Kingma & Ba 2015) on FP32 master weights, with a BF16 copy for the GEMMs
__global__ void adam_kernel(float* w, float* m, float* v, const float* g, uint16_t* wb, size_t n, float lr, float b1,
                            float b2, float eps, float c1, float c2) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.0f - b1) * gi;
  float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ void to_bf16_kernel(const float* x, uint16_t* y, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// Network input: the voxel's signal over the mean of its b=0 volumes (the
// volumes with b <= b0_max), one 16-lane row per voxel; rows of X are ldx long,
// zero beyond N.  Bound by the read of the signals (one thread per voxel read
// them in 4-byte strides: 170 us per 65,536 voxels of 288 volumes).
__global__ __launch_bounds__(256) void normalize_kernel(const float* data, int N, int nvox, const float* bvals,
                                                        float b0_max, uint16_t* X, int ldx, float* S0) {
  const int v = blockIdx.x * 16 + (threadIdx.x >> 4), rl = threadIdx.x & 15;
  if (v >= nvox) return;
  const float* y = data + (size_t)v * N;
  double s = 0.0;
  int nb = 0;
  for (int i = rl; i < N; i += 16)
    if (bvals[i] <= b0_max) { s += y[i]; ++nb; }
  s = row_sum16_d(s);
  nb = (int)row_sum16((float)nb);
  float s0 = nb ? (float)(s / nb) : 1.0f;
  if (!(s0 > 0.0f)) s0 = 1.0f;
  float inv = 1.0f / s0;
  for (int i = rl; i < ldx; i += 16) X[(size_t)v * ldx + i] = i < N ? f2bf(y[i] * inv) : (uint16_t)0;
  if (S0 && rl == 0) S0[v] = s0;
}

// Loss on the network outputs O [M][SG_OUT] against targets T [M][SG_OUT] and
// its gradient dO (bf16 [M][SG_LDO], zero padded; the last layer has no activation).  Targets: f_k (3),
// dyads x_k (3 x 3, sign-free: loss |p|^4 - 2 (p.x)^2 + 1 = ||p p^T - x x^T||^2
// weighted by f_k), 1000 d, 1000 d_std, log proposal widths (weight w_lw,
// zero where the target slot is unused, marked by a target >= 1e29).
__global__ void sg_loss_kernel(const float* O, const float* T, int M, uint16_t* dO, float* loss_part, float w_lw) {
  int m = blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.0f;
  if (m < M) {
    const float* o = O + (size_t)m * SG_OUT;
    const float* t = T + (size_t)m * SG_OUT;
    float g[SG_LDO];
    for (int i = 0; i < SG_LDO; ++i) g[i] = 0.0f;
    for (int k = 0; k < 3; ++k) {
      float e = o[k] - t[k];
      l += e * e;
      g[k] = 2.0f * e;
    }
    for (int k = 0; k < 3; ++k) {
      const float* p = o + 3 + 3 * k;
      const float* x = t + 3 + 3 * k;
      float w = fmaxf(t[k], 0.0f);
      float pp = p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
      float px = p[0] * x[0] + p[1] * x[1] + p[2] * x[2];
      l += w * (pp * pp - 2.0f * px * px + 1.0f);
      for (int c = 0; c < 3; ++c) g[3 + 3 * k + c] = w * (4.0f * pp * p[c] - 4.0f * px * x[c]);
    }
    for (int i = 12; i < 14; ++i) {
      float e = o[i] - t[i];
      l += e * e;
      g[i] = 2.0f * e;
    }
    for (int i = 14; i < SG_OUT; ++i) {
      if (t[i] >= 1e29f) continue;
      float e = o[i] - t[i];
      l += w_lw * e * e;
      g[i] = 2.0f * w_lw * e;
    }
    for (int i = 0; i < SG_LDO; ++i) dO[(size_t)m * SG_LDO + i] = i < SG_OUT ? f2bf(g[i] / (float)M) : (uint16_t)0;
  }
  // block partial sums of the loss (fixed order within the block)
  __shared__ float red[256];
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0];
}

// Network outputs -> chain start [S0, d, (d_std), f_k, th_k, ph_k] and the
// proposal widths of the slots (f0, d, d_std, R, S0, th/ph/f of each fibre);
// also the predicted principal direction (for the fallback test).
__global__ void sg_decode_kernel(SgDecodeArgs a) {
  int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= a.nvox) return;
  const float* o = a.O + (size_t)v * SG_OUT;
  float f[3];
  float fs = 0.0f;
  for (int k = 0; k < 3; ++k) { f[k] = fminf(fmaxf(o[k], 0.01f), 0.95f); fs += f[k]; }
  if (fs > 0.95f) for (int k = 0; k < 3; ++k) f[k] *= 0.95f / fs;
  float* P = a.params + (size_t)v * a.np;
  const int fb = a.model >= 2 ? 3 : 2;
  P[0] = a.S0[v];
  P[1] = fminf(fmaxf(o[12] * 1e-3f, 1e-5f), 0.0049f);
  if (a.model >= 2) {
    float up = a.model == 3 ? 0.0039f : 0.0099f;
    P[2] = fminf(fmaxf(o[13] * 1e-3f, 1e-5f), up);
  }
  for (int k = 0; k < a.K; ++k) {
    const float* p = o + 3 + 3 * k;
    float n2 = p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
    float x0 = p[0], x1 = p[1], x2 = p[2];
    if (!(n2 > 1e-20f)) { x0 = 0.0f; x1 = 0.0f; x2 = 1.0f; }
    float th = atan2f(sqrtf(x0 * x0 + x1 * x1), x2), ph = atan2f(x1, x0);
    P[fb + 3 * k] = f[k];
    P[fb + 3 * k + 1] = th;
    P[fb + 3 * k + 2] = ph;
    if (k == 0 && a.dir) {
      float inv = n2 > 1e-20f ? rsqrtf(n2) : 1.0f;
      a.dir[3 * v] = x0 * inv; a.dir[3 * v + 1] = x1 * inv; a.dir[3 * v + 2] = x2 * inv;
    }
  }
  if (a.f0) P[a.np - 1] = 0.001f;
  if (a.widths) {
    float* w = a.widths + (size_t)v * 16;
    for (int s = 0; s < 16; ++s) w[s] = -1.0f;  // default width
    const int slot_of[14] = {0, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14};
    // slot 0 (f0) keeps the default width: the training targets carry no f0
    for (int i = 1; i < 14; ++i) {
      float lw = fminf(fmaxf(o[14 + i], -20.0f), 5.0f);
      w[slot_of[i]] = expf(lw);
    }
  }
}

// Fallback test after the short chain: the voxel is rerun the plain way when
// its final sum of squares exceeds chi2_max * N * sigma^2 (sigma^2 from the
// spread of its b=0 volumes; flag bit 1) or the predicted direction of fibre 1
// lies more than ang_max from every posterior mean dyad (flag bit 2).
__global__ void sg_fallback_kernel(SgFallbackArgs a) {
  int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= a.nvox) return;
  const float* y = a.data + (size_t)v * a.N;
  double s = 0.0, s2 = 0.0;
  int nb = 0;
  for (int i = 0; i < a.N; ++i)
    if (a.bvals[i] <= a.b0_max) { s += y[i]; s2 += (double)y[i] * y[i]; ++nb; }
  double var = nb > 1 ? (s2 - s * s / nb) / (nb - 1) : 0.0;
  int why = 0;
  if (var > 0.0 && a.energy[v] > a.chi2_max * a.N * var) why |= 1;
  // the predicted direction of fibre 1 against the closest posterior mean dyad
  float c = 0.0f;
  for (int k = 0; k < a.K; ++k) {
    const float* dy = a.dyads + (size_t)k * 3 * a.nvox + v;  // [K][3][nvox]
    c = fmaxf(c, fabsf(dy[0] * a.dir[3 * v] + dy[(size_t)a.nvox] * a.dir[3 * v + 1] +
                       dy[(size_t)2 * a.nvox] * a.dir[3 * v + 2]));
  }
  if (c < a.cos_min) why |= 2;
  if (a.flag) a.flag[v] = (unsigned char)why;
  if (why) a.list[atomicAdd(a.count, 1)] = v;
}

}  // namespace fdt

namespace {
template <int TM, int TN, bool AK, bool BK>
hipError_t launch_tile(const fdt::GemmArgs* g, hipStream_t s) {
  const int rows = g->M + (g->a.ones ? 1 : 0);
  const dim3 grid((unsigned)(((rows + TM - 1) / TM) * ((g->N + TN - 1) / TN))), block(256);
  hipLaunchKernelGGL((fdt::gemm_bf16_kernel<TM, TN, AK, BK>), grid, block, 0, s, *g);
  return hipGetLastError();
}
// The largest tile that still gives each of the 256 CUs a workgroup
template <bool BK>
hipError_t launch_sized(const fdt::GemmArgs* g, hipStream_t s) {
  auto tiles = [&](int tm, int tn) { return (long)((g->M + tm - 1) / tm) * ((g->N + tn - 1) / tn); };
  if constexpr (!BK)  // outputs of at most 32 columns do not fill wider tiles
    if (g->N <= 32) return tiles(128, 32) >= 256 ? launch_tile<128, 32, true, BK>(g, s) : launch_tile<32, 32, true, BK>(g, s);
  if (tiles(128, 128) >= 256) return launch_tile<128, 128, true, BK>(g, s);
  if (tiles(64, 64) >= 256) return launch_tile<64, 64, true, BK>(g, s);
  return launch_tile<32, 32, true, BK>(g, s);
}
}  // namespace

// Weight gradients (A with m contiguous) have at most 513 x 512 outputs, so that
// no tile but the smallest comes near a workgroup per CU: they have that one only.
extern "C" hipError_t fdt_launch_gemm_bf16(const fdt::GemmArgs* g, hipStream_t s) {
  if (g->M <= 0 || g->N <= 0) return hipSuccess;
  if (g->a.kc) return g->a.ones ? hipErrorInvalidValue : g->b.kc ? launch_sized<true>(g, s) : launch_sized<false>(g, s);
  return g->b.kc ? hipErrorInvalidValue : launch_tile<32, 32, false, false>(g, s);
}

extern "C" hipError_t fdt_launch_to_bf16(const float* x, uint16_t* y, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(fdt::to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, y, n);
  return hipGetLastError();
}

extern "C" hipError_t fdt_launch_adam(float* w, float* m, float* v, const float* g, uint16_t* wb, size_t n, float lr,
                                      float b1, float b2, float eps, int step, hipStream_t s) {
  float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(fdt::adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w, m, v, g, wb, n, lr, b1, b2,
                     eps, c1, c2);
  return hipGetLastError();
}

extern "C" hipError_t fdt_launch_normalize(const float* data, int N, int nvox, const float* bvals, float b0_max,
                                           uint16_t* X, int ldx, float* S0, hipStream_t s) {
  if (nvox <= 0) return hipSuccess;
  hipLaunchKernelGGL(fdt::normalize_kernel, dim3((nvox + 15) / 16), dim3(256), 0, s, data, N, nvox, bvals, b0_max, X, ldx,
                     S0);
  return hipGetLastError();
}

extern "C" hipError_t fdt_launch_sg_loss(const float* O, const float* T, int M, uint16_t* dO, float* loss_part,
                                         float w_lw, hipStream_t s) {
  hipLaunchKernelGGL(fdt::sg_loss_kernel, dim3((M + 255) / 256), dim3(256), 0, s, O, T, M, dO, loss_part, w_lw);
  return hipGetLastError();
}

extern "C" hipError_t fdt_launch_sg_decode(const fdt::SgDecodeArgs* a, hipStream_t s) {
  if (a->nvox <= 0) return hipSuccess;
  hipLaunchKernelGGL(fdt::sg_decode_kernel, dim3((a->nvox + 255) / 256), dim3(256), 0, s, *a);
  return hipGetLastError();
}

extern "C" hipError_t fdt_launch_sg_fallback(const fdt::SgFallbackArgs* a, hipStream_t s) {
  if (a->nvox <= 0) return hipSuccess;
  hipLaunchKernelGGL(fdt::sg_fallback_kernel, dim3((a->nvox + 255) / 256), dim3(256), 0, s, *a);
  return hipGetLastError();
}
