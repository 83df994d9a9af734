// fdt_mlp.h -- argument blocks of the learned-initialiser kernels (plain data).
#pragma once
#include <stdint.h>
#include <stddef.h>

namespace fdt {

constexpr int SG_OUT = 28;     // 3 f + 3x3 directions + d + d_std + 14 log proposal widths
constexpr int SG_LAYERS = 4;   // N -> 512 -> 512 -> 256 -> 28
constexpr int SG_HID0 = 512, SG_HID1 = 512, SG_HID2 = 256;

constexpr int SG_LDO = 32;     // row length of the output gradients (zero padded)

// An operand of the GEMM, bf16, rows along m (A) or n (B): element (row, k) at
// p[row * ld + k] (kc) or p[k * ld + row]; vec: p and ld are 16-byte multiples.
// ones (A, not kc): row M of A is all ones, so that row M of C is the column
// sum of B
struct GemmOperand {
  const uint16_t* p;
  long ld;
  bool kc, vec, ones;
};
enum { GEMM_LINEAR = 0, GEMM_GELU = 1, GEMM_GELU_BWD = 2 };
// C[m][n] (row-major, leading dimension ldc) = sum_k A(m,k) B(n,k) (+ bias[n])
// -> C (fp32, optional) and act of it -> Cb (bf16, optional, same indexing);
// GEMM_GELU_BWD: C gelu'(Z)
struct GemmArgs {
  int M, N, K;
  GemmOperand a, b;
  float* C;
  uint16_t* Cb;
  long ldc;
  const float* bias;
  int act;
  const float* Z;
};

struct SgDecodeArgs {
  const float* O;     // [nvox][SG_OUT]
  const float* S0;    // [nvox]
  int nvox, model, K, f0, np;
  float* params;      // [nvox][np] chain start
  float* widths;      // [nvox][16] proposal widths per slot (< 0: default), optional
  float* dir;         // [nvox][3] predicted direction of fibre 1, optional
};

struct SgFallbackArgs {
  const float* data;
  int N, nvox;
  const float* bvals;
  float b0_max;
  const float* energy;  // final sum of squares of each chain
  const float* dyads;   // [K][3][nvox]
  int K;
  const float* dir;     // [nvox][3]
  float chi2_max, cos_min;
  unsigned char* flag;  // reason per voxel: 1 sum of squares, 2 direction (optional)
  int* list;
  int* count;
};

}  // namespace fdt
