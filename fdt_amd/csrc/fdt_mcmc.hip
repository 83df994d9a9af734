// fdt_mcmc.hip -- the persistent MCMC launch over one volume: one chain per
// 16-lane row, 16 chains per 256-thread workgroup, the whole nburn + njumps
// loop in one launch.  The chain itself is run_chain (fdt_chain.h).
#include "fdt_chain.h"

namespace fdt {

// XCD-aware tile order.  The dispatcher deals workgroups round-robin over the
// 8 XCDs, each with its own L2; renumbered this way each XCD runs one
// contiguous range of tiles, so the 64-byte record runs of neighbouring
// workgroups (16 voxels x 4 B per sample and quantity) meet in one L2 and
// leave it as whole lines.  A bijection of [0, nb) for every nb.
__device__ inline int xcd_tile(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, x = b & 7, l = b >> 3;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + l;
}

// VPL volumes per lane in ROWS rows per voxel: a tile of VPL ROWS.
// Waves per SIMD: two where the state allows it, and above that as many as a
// kernel's registers let in (four up to 128 of them, three up to 168): from 33 to
// 160 volumes the chains are short series of dependent operations, which other
// waves fill.  60,000 voxels, 250 sweeps, held to two waves -> not: 33 volumes,
// model 2, K=1, 4.45 -> 3.65 ms; 69 volumes, K=3, 10.36 -> 9.73; 100 volumes, K=3,
// 13.4 -> 11.8 (Rician 30.6 -> 25.8, --gradnonlin 14.5 -> 13.6); 145 volumes, K=3,
// 17.5 -> 15.6.  Nothing changes above 168 registers: Rician chains and
// zeppelins of three fibres at 145 volumes, and all above 160 volumes but model 2
// with one fibre (200 volumes: 11.3 -> 9.6).
template <int K, int VPL, bool RIC, bool GN>
constexpr int MIN_WAVES = VPL <= 18 || (K == 1 && !RIC && !GN) ? 2 : 1;
template <int K, int VPL, int MODEL, bool RIC, bool GN, bool FULL, int ROWS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MIN_WAVES<K, VPL, RIC, GN>, 4))) void mcmc_kernel(McmcArgs a) {
  constexpr bool SMALL = Chain<K, VPL, MODEL, RIC, GN, FULL, ROWS>::SMALL;  // state in registers
  constexpr int TILE = VPL * ROWS;
  __shared__ float4 sacq[16 * TILE];
  __shared__ float sba[SMALL ? 1 : 4 * K * VPL * 64];
  __shared__ int ssh[GN ? 1 : 16 * TILE];
  __shared__ float sshb[16];
  __shared__ float siso[GN ? 1 : 16 * 16];
  __shared__ float sbp[GN ? 16 * 16 * VPL : 1];
  __shared__ float sgd[GN ? 16 * 9 : 1];
  __shared__ float svol[GN || SMALL ? 1 : 4 * VPL * 64];
  constexpr bool ZS = ZERO_SLOT<TILE>;
  __shared__ int sperm[ZS ? 16 * TILE : 1];
  __shared__ int szc[ZS ? ZC_CHUNKS : 1];
  const ChainLds L{sacq, sba, GN ? nullptr : ssh, sshb, siso, sbp, sgd, GN ? nullptr : svol, ZS ? sperm : nullptr,
                   ZS ? szc : nullptr};
  stage_acq<TILE>(a, L);
  __syncthreads();
  const int i = xcd_tile(blockIdx.x, gridDim.x) * (16 / ROWS) + (threadIdx.x >> 4) / ROWS;
  if (i < a.nvox) run_chain<K, VPL, MODEL, RIC, GN, FULL, ROWS>(a, a.list ? a.list[i] : i, L);
}

}  // namespace fdt

// Up to six translation units per tile FDT_VPL, built in parallel, each with its
// own compiler options and loaded with its first launch: -DFDT_MCMC_UNIT=0 holds
// the launcher and the Gaussian kernels with one row per voxel, 1 the Rician
// ones, 2 the kernels with two rows (the iterative scheduler of the others
// crashes on their row swap); 3, 4 and 5 are 0, 1 and 2 for acquisitions that
// fill the tile.  K = 1..3 and models 1..3 have a kernel each (one that held all
// models at once took 128 KB of code at K = 3 and 98 scalar registers more than
// there are), with the shared acquisition or per-voxel ones (--gradnonlin,
// a->acqv set; its stride must cover 16 * FDT_VPL volumes; units 0 and 1).
#ifndef FDT_VPL
#define FDT_VPL 18
#endif
#ifndef FDT_MCMC_UNIT
#define FDT_MCMC_UNIT 0
#endif
#define FDT_CAT2_(a, b) a##b
#define FDT_CAT2(a, b) FDT_CAT2_(a, b)

#define FDT_CAN_TWO (FDT_VPL % 2 == 0 && FDT_VPL >= 10)

namespace {
constexpr bool FULL = FDT_MCMC_UNIT >= 3;
constexpr int ROWS = FDT_MCMC_UNIT % 3 == 2 ? 2 : 1;
template <int K, int MODEL, bool RIC>
hipError_t launch_model(const fdt::McmcArgs* a, hipStream_t s) {
  const dim3 grid((a->nvox + 16 / ROWS - 1) / (16 / ROWS)), block(256);
  if constexpr (!FULL && ROWS == 1) {
    if (a->acqv) {
      hipLaunchKernelGGL((fdt::mcmc_kernel<K, FDT_VPL, MODEL, RIC, true, false, 1>), grid, block, 0, s, *a);
      return hipGetLastError();
    }
  }
  if constexpr (ROWS == 2 || fdt::mcmc_one_row(FDT_VPL, K, RIC)) {
    hipLaunchKernelGGL((fdt::mcmc_kernel<K, FDT_VPL / ROWS, MODEL, RIC, false, FULL, ROWS>), grid, block, 0, s, *a);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
template <int K, bool RIC>
hipError_t launch_k(const fdt::McmcArgs* a, hipStream_t s) {
  if (a->model == 1) return launch_model<K, 1, RIC>(a, s);
  if (a->model == 2) return launch_model<K, 2, RIC>(a, s);
  if (a->model == 3) return launch_model<K, 3, RIC>(a, s);
  return hipErrorInvalidValue;
}
template <bool RIC>
hipError_t launch(const fdt::McmcArgs* a, int K, hipStream_t s) {
  if (K == 1) return launch_k<1, RIC>(a, s);
  if (K == 2) return launch_k<2, RIC>(a, s);
  if (K == 3) return launch_k<3, RIC>(a, s);
  return hipErrorInvalidValue;
}
}  // namespace

#define FDT_UNIT(u) FDT_CAT2(FDT_CAT2(FDT_CAT2(fdt_launch_mcmc_unit, u), _vpl), FDT_VPL)
#define FDT_UNIT_ARGS (const fdt::McmcArgs* a, int K, int rician, hipStream_t s)
extern "C" {
#if FDT_MCMC_UNIT
hipError_t FDT_UNIT(FDT_MCMC_UNIT) FDT_UNIT_ARGS {
#if FDT_MCMC_UNIT == 1 || FDT_MCMC_UNIT == 4
  return launch<true>(a, K, s);
#elif FDT_MCMC_UNIT == 3
  return launch<false>(a, K, s);
#else
  return rician ? launch<true>(a, K, s) : launch<false>(a, K, s);
#endif
}
#else
hipError_t FDT_UNIT(1) FDT_UNIT_ARGS;
hipError_t FDT_UNIT(2) FDT_UNIT_ARGS;
hipError_t FDT_UNIT(3) FDT_UNIT_ARGS;
hipError_t FDT_UNIT(4) FDT_UNIT_ARGS;
hipError_t FDT_UNIT(5) FDT_UNIT_ARGS;
hipError_t FDT_CAT2(fdt_launch_mcmc_vpl, FDT_VPL) FDT_UNIT_ARGS {
  if (a->nvox <= 0) return hipSuccess;
  if (a->acqv && a->acqv_stride < 16 * FDT_VPL) return hipErrorInvalidValue;
  // An acquisition of 16 FDT_VPL volumes leaves no padding slot: kernels without
  // the masks.  Measured masked -> without at 48, 80, 112, 160, 224, 288, 384, 448
  // and 512 volumes, every model and K: Gaussian 0.2 to 5% faster (288 volumes,
  // K=3, model 2, 24,000 voxels, 250 sweeps: 11.05 -> 10.89 ms), Rician 4 to 7%
  // (31.8 -> 30.1, model 3), two rows 1 to 9% (4.24 -> 3.93 at 2,000 voxels).  The
  // --gradnonlin kernels keep the masks.
  const bool full = !a->acqv && a->N == 16 * FDT_VPL;
#if FDT_CAN_TWO
  if (fdt::mcmc_rows(*a, FDT_VPL, K, rician) == 2)
    return full ? FDT_UNIT(5)(a, K, rician, s) : FDT_UNIT(2)(a, K, rician, s);
#endif
#if FDT_VPL <= 28
  if (full && !rician) return FDT_UNIT(3)(a, K, rician, s);
#endif
#if FDT_VPL <= 18
  if (full) return FDT_UNIT(4)(a, K, rician, s);
#endif
  return rician ? FDT_UNIT(1)(a, K, rician, s) : launch<false>(a, K, s);
}
#endif
}
