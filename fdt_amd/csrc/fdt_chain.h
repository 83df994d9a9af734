// fdt_chain.h -- one Metropolis-Hastings chain of the ball-and-sticks models
// per 16-lane row on gfx950, shared by the per-volume kernel (fdt_mcmc.hip)
// and the batched queue kernel (fdt_queue.hip).
//
// Semantics follow the reference GPU MCMC: init_Fibres_Multifibres_kernel
// (CUDA/runmcmc_kernels.cu:193-505) and runmcmc_kernel (:507-1474), with the
// burn-in and record launches (CUDA/runmcmc.cu:108-316) fused into one loop of
// nburn + njumps sweeps.  Layout: one voxel per 16-lane DPP row, four voxels
// per wave64.  Lane l of a row holds volumes l, l+16, l+32, ... (VPL volumes
// per lane) and keeps, in VGPRs,
//   the residual r = y - S0*M (Gaussian) or the terms of the volumes (Rician),
//   the mixture M = sum_k f_k s_k + (1 - f0 - sum_k f_k) iso + f0,
//   the isotropic signal iso and the stick signals s_k;
// one of these arrays and the arguments b (g.x_k)^2 of the stick signals live
// in LDS (one block per wave, lane-interleaved), and K=3 at 18 volumes per
// lane fits two waves per SIMD.
// The kernel is bound by VALU issue (99% of the SIMD cycles before, on the
// 250,968-voxel multi-shell volume at K=3), so what counts is instructions per
// sweep: evaluating what belongs to a slot once per sweep in its own lane,
// keeping the stick arguments for the diffusivity moves and each proposal's
// per-volume changes for its acceptance took 5,107 VALU instructions per wave
// and sweep to 4,154, and one kernel per model (128 KB of code to 54, no
// spilled vector registers) let the launch follow: 1,247 to 1,013 ms.  Masks
// compiled out where the acquisition fills the tile (here 288 volumes), the
// draws' products from one instruction and no question about a slot or a sweep
// number inside a sweep: 973 ms.
// A proposal evaluates only what it changes; its likelihood change is
// summed over the row with DPP adds.  For Gaussian noise a move of every
// residual by -c*q gives the change of the sum of squares c*(c*sum q^2 -
// 2*sum r*q), and the energy difference (N/2)*log1p(dSSR/SSR) keeps full
// relative precision (the reference differences two FP32 energies).  The
// acquisition (gx,gy,gz,b) is staged in LDS.  Draws: lane l of the row
// computes the Philox block of proposal slot l for the current jump; DPP
// row_newbcast hands it to the row.
#pragma once
#include "fdt_device.h"
#include "fdt_kernels.h"
#include <utility>

namespace fdt {

constexpr float L2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
FDT_DEV float ex2(float x) { return __builtin_amdgcn_exp2f(x); }
FDT_DEV float lg2(float x) { return __builtin_amdgcn_logf(x); }
FDT_DEV float flog(float x) { return lg2(x) * LN2; }

// sin and cos of a float angle of any magnitude.  Width adaptation drives the
// angles of unsupported fibres to 1e8..1e11 rad, and the reference evaluates
// them as sin/cos(double(angle)) with a full-range reduction
// (CUDA/runmcmc_kernels.cu:340, :1165, :1177-1182).  Here the angle is turned
// into revolutions x/(2 pi) and reduced to its fraction in double, with
// 1/(2 pi) split into two doubles: the first FMA forms x * HI exactly before
// subtracting the nearest integer, so the fraction is accurate to ~2^-53 for
// |x| < 2^60.  The hardware sin/cos take revolutions (valid in [-256, 256]).
FDT_DEV void sincos_full(float x, float& s, float& c) {
  constexpr double R_HI = 0x1.45f306dc9c883p-3, R_LO = -0x1.6b01ec5417056p-57;
  const double xd = (double)x;
  const double n = __builtin_rint(xd * R_HI);
  double fr = __builtin_fma(xd, R_HI, -n);
  fr = __builtin_fma(xd, R_LO, fr);
  const float f = (float)fr;
  s = __builtin_amdgcn_sinf(f);
  c = __builtin_amdgcn_cosf(f);
}

// draw slots (fixed per parameter)
enum { SL_F0 = 0, SL_TAU = 1, SL_D = 2, SL_DSTD = 3, SL_R = 4, SL_S0 = 5, SL_FIB = 6 };

// Tiles whose chains stage b = 0 volumes first and skip their slot (see
// stage_acq): the 14- and 18-volume tiles, where it saves 3-4% of the chain time.  In
// the smaller tiles the uniform branch around slot 0 costs more than it saves
// (it splits the few volumes a lane interleaves); at 24 and 32 volumes per
// lane in one row (one wave per SIMD) it saved nothing (N = 384 with 24 b = 0
// volumes) and cost 1.4% (N = 432).
template <int VPL> constexpr bool ZERO_SLOT = VPL == 14 || VPL == 18;

// Signal forms with row-uniform coefficients (compute_signal /
// compute_iso_signal, CUDA/runmcmc_kernels.cu:67-95):
//   kind 0: exp(-d*u)                        model 1
//   kind 1: (1 + w)^(-d^2/dstd^2), w = (dstd^2/d) u   model 2 (gamma diffusivities);
//           below d_std 1e-5 the reference switches to exp(-d*u), which the
//           same expression evaluates with c0 = 2^-64, c1 = -d 2^64: then
//           1 + w rounds to 1, lg2 of it is 0, and the recovered rounding
//           error is w = c0 u exactly (a power-of-two scaling), so the
//           exponent is c1 w / ln2 = -d u / ln2 with the roundings of the
//           exponential form.  Rows on either side of the switch share one
//           code path (a wave whose rows took different forms would run both).
//   kind 2: exp(-3 d invR ((1-R) b a + R b))  model 3 zeppelin, u = b a
// Kind 1 in FP32: u1 = fl(1 + w) keeps w only to 2^-24 absolute, and the
// exponent d^2/dstd^2 multiplies that error (1e-3 relative signal error at
// dstd/d ~ 0.01; the reference evaluates these signals in double).  The
// rounding error e = (1 + w) - u1 is recovered with one FMA and
// lg2(1 + w) = lg2(u1) + lg2(1 + e/u1) ~ lg2(u1) + e/ln2; the dropped 1/u1
// factor leaves an exponent error below d u 2^-24 for every w (e <= half an
// ulp of u1, and (d^2/dstd^2) w = d u).
struct SigC {
  float c0, c1;
};
// the stick and isotropic forms of a model (model 3: zeppelins with the
// gamma-distributed isotropic term)
template <int MODEL> constexpr int STICK_KIND = MODEL - 1;
template <int MODEL> constexpr int ISO_KIND = MODEL == 1 ? 0 : 1;
FDT_DEV SigC gamma_coef(float d, float dstd) {
  SigC c;
  if (dstd < 1e-5f) { c.c0 = 0x1p-64f; c.c1 = -d * 0x1p64f; }
  else { const float s2 = dstd * dstd; c.c0 = s2 / d; c.c1 = -(d * d / s2); }
  return c;
}
template <int MODEL>
FDT_DEV SigC aniso_coef(float d, float dstd, float R) {
  if constexpr (MODEL == 1) return SigC{-d * L2E, 0.0f};
  else if constexpr (MODEL == 2) return gamma_coef(d, dstd);
  else {
    float iR = 1.0f / (2.0f * R + 1.0f);
    float k = -3.0f * d * iR * L2E;
    return SigC{k * (1.0f - R), k * R};
  }
}
template <int MODEL>
FDT_DEV SigC iso_coef(float d, float dstd) {
  if constexpr (MODEL == 1) return SigC{-d * L2E, 0.0f};
  else return gamma_coef(d, dstd);
}
template <int SK>
FDT_DEV float sig(const SigC& c, float u, float b) {
  if constexpr (SK == 0) return ex2(c.c0 * u);
  else if constexpr (SK == 1) {
    const float u1 = fmaf(c.c0, u, 1.0f);
    const float e = fmaf(c.c0, u, 1.0f - u1);  // (1 + w) - u1 (1 - u1 is exact)
    return ex2(c.c1 * fmaf(e, L2E, lg2(u1)));
  }
  else return ex2(fmaf(c.c0, u, c.c1 * b));
}
// log I0 by Abramowitz-Stegun 9.8.1/9.8.2 (fibre.h:29-48, CUDA/runmcmc_kernels.cu:126-145)
FDT_DEV float logI0f(float x) {
  float b = fabsf(x);
  float a = x * (1.0f / 3.75f);
  a *= a;
  float ys = 1.0f + a * (3.5156229f + a * (3.0899424f + a * (1.2067492f + a * (0.2659732f + a * (0.0360768f + a * 0.0045813f)))));
  float Ls = flog(ys);
  float c = 3.75f * __builtin_amdgcn_rcpf(b);
  float pl = 0.39894228f + c * (0.01328592f + c * (0.00225319f + c * (-0.00157565f + c * (0.00916281f + c * (-0.02057706f + c * (0.02635537f + c * (-0.01647633f + c * 0.00392377f)))))));
  // one logarithm of the selected branch: log ys, or b + log(pl / sqrt b)
  const bool sm = b < 3.75f;
  return flog(sm ? ys : pl * __builtin_amdgcn_rsqf(b)) + (sm ? 0.0f : b);
}
// log I0 above 3.75 alone, the same operations
FDT_DEV float logI0_large(float x) {
  const float b = fabsf(x);
  float c = 3.75f * __builtin_amdgcn_rcpf(b);
  float pl = 0.39894228f + c * (0.01328592f + c * (0.00225319f + c * (-0.00157565f + c * (0.00916281f + c * (-0.02057706f + c * (0.02635537f + c * (-0.01647633f + c * 0.00392377f)))))));
  return flog(pl * __builtin_amdgcn_rsqf(b)) + b;
}
// Rician log-likelihood term of one volume (fibre.h:949-953),
//   log y - tau (y^2 + p^2) / 2 + log I0(tau p y),
// without the part that does not depend on the model signal p: log y and
// -tau y^2 / 2 cancel from every energy difference except the tau move's,
// which adds -(tau' - tau) sum y^2 / 2 itself; the energy of a state adds
// both back (sum log y - tau sum y^2 / 2)
FDT_DEV float ell_of(float y, float p, float tau) {
  const float tp = tau * p;
  return fmaf(-0.5f * tp, p, logI0f(tp * y));
}

// Gaussian likelihood change when every residual moves by -c*q_t:
// sum (r - c q)^2 - r^2 = c (c sum q^2 - 2 sum r q); two FMAs per volume and
// two row sums
struct Quad {
  float A = 0.0f, B = 0.0f;
  FDT_DEV void add(float r, float q) { A = fmaf(r, q, A); B = fmaf(q, q, B); }
  FDT_DEV float delta(float c) {
    A = row_sum16(A);
    B = row_sum16(B);
    return c * fmaf(c, B, -2.0f * A);
  }
};
// Compiler-only memory barrier: keeps the acquisition table in LDS (re-read
// per proposal) instead of letting the loop-invariant loads be hoisted into
// ~4*VPL VGPRs for the whole chain.
FDT_DEV void reload_acq() { asm volatile("" ::: "memory"); }
// x^2 rounded on its own: not contracted into a sum, with padding masks or without
FDT_DEV float square(float x) {
#pragma clang fp contract(off)
  return x * x;
}
FDT_DEV float product(float x, float y) {
#pragma clang fp contract(off)
  return x * y;
}

// One chain per 16-lane row.  Volume state lives in registers per lane;
// everything that belongs to a proposal slot -- the parameter value, its
// proposal width, its acceptance counters (acc + rej << 16) and its current
// prior energy -- lives in the lane of that slot (sval/sprop/scnt/sprior) and
// is read by a row broadcast.  Slots: f0 0, tau 1, d 2, d_std 3, R 4, S0 5,
// theta_k 6+3k, phi_k 7+3k, f_k 8+3k (the theta prior sits in the theta slot).
// GN (--gradnonlin): the voxel sees gradient g through its deviation M = I+L
// as direction Mg/|Mg| and b value |Mg|^2 b, so b'(g'.x)^2 = b (g.M^T x)^2:
// the stick signals use the shared acquisition with the fibre directions
// mapped by M^T, and the isotropic signal (and the model-3 R term) the
// voxel's own b values, kept per row in LDS.
// ROWS (1 or 2): a voxel's volumes spread over that many consecutive rows of
// the wave, VPL in each lane; every row holds the slots' state and makes the
// same decisions.  A sum over volumes runs through the lanes of the first row
// and on through those of the second, so that it is the one-row sum to the last
// bit.
template <int K, int VPL, int MODEL, bool RIC, bool GN = false, bool FULL = false, int ROWS = 1>
struct Chain {
  // lane-resident volume state, volume i = rl + 16 t.  One per-volume
  // array lives in the wave's LDS block `vol` instead of registers (18
  // VGPRs at 18 volumes per lane, the difference between spilling and not):
  // the isotropic signal of the Gaussian chain, the data of the Rician one.
  // The --gradnonlin kernels keep both in registers (their LDS holds the
  // rows' b values).
  // Tiles of up to 5 volumes per lane keep everything in registers, the
  // acquisition and the stick arguments too: their proposals are short chains
  // of dependent operations, where each LDS read adds its latency (2,000
  // voxels of 69 volumes, model 1: 5.5 -> 4.5 ms).  At 10 volumes per lane and
  // K=3 the registers run out (48 spilled).
  static constexpr bool SMALL = VPL <= 5;
  static constexpr bool ISO_LDS = !GN && !RIC && !SMALL, Y_LDS = !GN && RIC && !SMALL;
  float r[Y_LDS ? 1 : VPL];  // Gaussian: y - S0*M; Rician: -2 y
  float M[VPL];
  float iso_r[ISO_LDS ? 1 : VPL];
  float s[K][VPL];
  float* vol;   // wave's LDS block: vol[t*64]
  // The wave's LDS block sk[(k*VPL+t)*64] holds the arguments b (g.x_k)^2 of
  // the stick signals (U_LDS): the diffusivity proposals read them there and
  // keep their candidate signals in registers.  Where the registers do not
  // allow that, it holds the candidate signals, and the arguments are formed
  // from the fibre directions again.
  static constexpr int HELD = VPL * (2 * K + 3 + !ISO_LDS + RIC);  // floats a lane holds in a diffusivity proposal
  static constexpr bool U_LDS = HELD <= (RIC ? 130 : 162) * (VPL > 18 ? 2 : 1);
  float* sk;
  float ur[SMALL ? K : 1][SMALL ? VPL : 1];
  float4 ga[SMALL ? VPL : 1];
  float ell[RIC ? VPL : 1];
  // isotropic signal per b-shell (acquisitions with <= 16 distinct b values):
  // sh[i] is the shell of volume i, shb[l] its b value, isot the row's table
  const int* sh;
  const float* shb;
  float* isot;
  int nshell;
  float sval, sprop, sprior;
  int scnt;
  // sin and cos of the slot's angle (theta_k / phi_k slots), kept with the value
  float ssin, scos;
  // The slots' candidates of the current sweep (propose): a slot's value and
  // width change only with its own proposal, so every candidate, its sine and
  // cosine and its prior are known when the sweep begins and each lane
  // evaluates its own slot's once, instead of the whole row at every proposal.
  float sxn, ssn, scn, sprn, sdp;
  uint32_t accm;  // slots accepted in the current sweep (bit: slot), settled at its end
  int rejinc;     // what a rejection adds to the slot's counters (0: not sampled)
  // row-uniform copies of the parameters that other slots' proposals read
  float S0, tau, d, dstd, Rr, f0, fk[K], fsum;
  SigC ca;        // stick-signal coefficients of the current state
  double like;  // Gaussian: SSR; Rician: sum of ell
  int nv;       // slots of this lane that hold a real volume (rl + 16 t < N)
  int rl;
  // slot 0 holds b = 0 volumes only (see stage_acq): the moves that leave
  // their signals at 1 skip it (ZERO_SLOT tiles only)
  bool z0;
  bool th;   // a theta slot's lane
  float pw;  // weight of the slot's log prior (see prior_weight)
  FDT_DEV bool skip(int t) const { return ROWS == 1 && ZERO_SLOT<VPL> && t == 0 && z0; }
  // two rows: this lane's slot t is in the slot of b = 0 volumes
  FDT_DEV bool zero(int t) const { return ROWS > 1 && ZERO_SLOT<VPL * ROWS> && t == 0 && z0; }
  // A running sum handed from the first row to the second (0 to the first): the
  // gfx950 row swap exchanges the odd rows of its first operand with the even
  // rows of its second; clang 22 gives the first result for the second one too,
  // so only the first is used.
  static FDT_DEV float next_row(float a) {
    const auto w = __builtin_amdgcn_permlane16_swap(0, __builtin_bit_cast(int, a), false, false);
    return __builtin_bit_cast(float, w[0]);
  }
  // a total that every lane of the second row holds, to both rows (two voxels per wave)
  static FDT_DEV float from_last(float a) {
    const float lo = fdt::rl(a, 16), hi = fdt::rl(a, 48);
    return __lane_id() < 32 ? lo : hi;
  }
  // sum over the voxel's volumes of the row-wise chain f(t, sum so far)
  // (ALL: slot 0 of b = 0 volumes too)
  template <bool ALL = false, class F>
  FDT_DEV float chain_sum(F&& f) const {
    float a = 0.0f;
#pragma unroll
    for (int h = 0; h < ROWS; ++h) {
      if (h) a = next_row(a);
#pragma unroll
      for (int t = 0; t < VPL; ++t)
        if (ALL || !skip(t)) a = f(t, a);
    }
    a = row_sum16(a);
    if constexpr (ROWS > 1) a = from_last(a);
    return a;
  }
  template <class F>
  FDT_DEV double chain_sum_d(F&& f) const {
    double a = 0.0;
#pragma unroll
    for (int h = 0; h < ROWS; ++h) {
      if (h) {
        const int2 b = __builtin_bit_cast(int2, a);
        a = __builtin_bit_cast(double, make_int2(__builtin_bit_cast(int, next_row(__builtin_bit_cast(float, b.x))),
                                                 __builtin_bit_cast(int, next_row(__builtin_bit_cast(float, b.y)))));
      }
#pragma unroll
      for (int t = 0; t < VPL; ++t) a = f(t, a);
    }
    a = row_sum16_d(a);
    if constexpr (ROWS > 1) {
      const int2 b = __builtin_bit_cast(int2, a);
      a = __builtin_bit_cast(double, make_int2(__builtin_bit_cast(int, from_last(__builtin_bit_cast(float, b.x))),
                                               __builtin_bit_cast(int, from_last(__builtin_bit_cast(float, b.y)))));
    }
    return a;
  }
  // Gaussian likelihood change when every residual moves by -c q(t); ALL: slot 0
  // of b = 0 volumes too
  template <bool ALL = false, class Q>
  FDT_DEV float quad(Q&& q, float c) const {
    if constexpr (ROWS == 1) {
      Quad qd;
#pragma unroll
      for (int t = 0; t < VPL; ++t)
        if (ALL || !skip(t)) qd.add(r[t], q(t));
      return qd.delta(c);
    } else {
      float A = 0.0f, B = 0.0f;
#pragma unroll
      for (int h = 0; h < ROWS; ++h) {
        if (h) { A = next_row(A); B = next_row(B); }
#pragma unroll
        for (int t = 0; t < VPL; ++t) { A = fmaf(r[t], q(t), A); B = fmaf(q(t), q(t), B); }
      }
      A = from_last(row_sum16(A));
      B = from_last(row_sum16(B));
      return c * fmaf(c, B, -2.0f * A);
    }
  }
  // options
  bool incf0, ardf0, can_ard;
  bool lam[K];
  float fudge, halfN, Nf, Rmean, Rstd, Rfudge;
  const float4* acq;
  const float* bp;  // GN: the voxel's b values, bp[rl + 16 t] (LDS)
  const float* gd;  // GN: the voxel's 9 deviation values L(i,j) = gd[3j+i] (LDS)

  // b of slot t for the isotropic signal and the model-3 R term
  FDT_DEV float bv(int t, const float4& g) const {
    if constexpr (GN) return bp[rl + 16 * t];
    else return g.w;
  }
  // fibre direction as the voxel's gradients see it: x -> M^T x
  FDT_DEV void xform(float& x0, float& x1, float& x2) const {
    if constexpr (GN) {
      float y0 = x0 + fmaf(gd[0], x0, fmaf(gd[1], x1, gd[2] * x2));
      float y1 = x1 + fmaf(gd[3], x0, fmaf(gd[4], x1, gd[5] * x2));
      float y2 = x2 + fmaf(gd[6], x0, fmaf(gd[7], x1, gd[8] * x2));
      x0 = y0; x1 = y1; x2 = y2;
    }
  }

  static constexpr int TH(int k) { return SL_FIB + 3 * k; }
  static constexpr int PH(int k) { return SL_FIB + 3 * k + 1; }
  static constexpr int FK(int k) { return SL_FIB + 3 * k + 2; }
  template <int SL> FDT_DEV float cand() const { return row_bcast<SL>(sxn); }    // the slot's candidate
  template <int SL> FDT_DEV float dprior() const { return row_bcast<SL>(sdp); }  // its prior energy change
  template <int SL> FDT_DEV void accept() { accm |= 1u << SL; }

  FDT_DEV float& ldsk(int k, int t) const { return sk[(k * VPL + t) * 64]; }
  // stick-signal argument of fibre k at slot t
  FDT_DEV float& arg(int k, int t) {
    if constexpr (SMALL) return ur[k][t];
    else return ldsk(k, t);
  }
  // acquisition of slot t
  FDT_DEV float4 grad(int t) const {
    if constexpr (SMALL) return ga[t];
    else return acq[rl + 16 * t];
  }
  FDT_DEV static void fence() { if constexpr (!SMALL) reload_acq(); }
  FDT_DEV float& isov(int t) {
    if constexpr (ISO_LDS) return vol[t * 64];
    else return iso_r[t];
  }
  FDT_DEV float isov(int t) const {
    if constexpr (ISO_LDS) return vol[t * 64];
    else return iso_r[t];
  }
  // the Rician chain's data of slot t, held as -2 y (exact): with h = -tau p / 2
  // the argument of log I0 is h (-2 y) and the quadratic part h p
  FDT_DEV float ym2(int t) const {
    if constexpr (Y_LDS) return vol[t * 64];
    else return r[t];
  }
  FDT_DEV float yv(int t) const { return -0.5f * ym2(t); }
  float yy;  // Rician: sum of y^2 over the row's volumes
  // unit directions of the row's fibres (from the theta / phi slots)
  struct Dirs {
    float x[K][3];
  };
  FDT_DEV Dirs dirs() const {
    Dirs D;
    sfor<K>([&](auto kc) {
      constexpr int k = kc;
      const float st = row_bcast<TH(k)>(ssin), ct = row_bcast<TH(k)>(scos);
      const float sp = row_bcast<PH(k)>(ssin), cp = row_bcast<PH(k)>(scos);
      D.x[k][0] = st * cp; D.x[k][1] = st * sp; D.x[k][2] = ct;
      xform(D.x[k][0], D.x[k][1], D.x[k][2]);
    });
    return D;
  }
  // Contribution of slot t: zero where the slot is padding (volume >= N).
  // Padding slots see g = 0 and b = 0 in every acquisition table (shared,
  // per-voxel, b-shell), so their isotropic and stick signals are exactly 1
  // for every parameter value.  The Gaussian chain keeps their residual at
  // exactly 0 (masked where it is formed and where S0 or the mixture moves),
  // so the f0, f and angle proposals, whose per-volume change is then exactly
  // 0 there, need no mask; the S0 and diffusivity proposals, where the
  // mixture at a padding slot moves by rounding, and every Rician term do.
  // FULL: the tile has no padding (N = 16 VPL).
  FDT_DEV float mask(int t, float x) const { return FULL || t < nv ? x : 0.0f; }
  // sum of the fractions (f0 first, the order of the reference's sums)
  FDT_DEV float sum_fractions() const {
    float q = f0;
    sfor<K>([&](auto kc) { q += fk[kc]; });
    return q;
  }
  // energy change of the likelihood from a row-summed change `dl`
  FDT_DEV float dlik(float dl) const {
    if constexpr (RIC) return -dl;
    else {
      // log1p(x): log of u = fl(1 + x) plus the rounding error of u,
      // x - (u - 1) (exact for x in [-1/2, 1]; outside, its error is below an
      // ulp of u against |log u| > 0.4); the dropped factor 1/u leaves an
      // error below 2^-24 |x| (the same device as the gamma-form signal)
      const float x = dl * __builtin_amdgcn_rcpf((float)like);
      const float u = 1.0f + x;
      return halfN * fmaf(lg2(u), LN2, x - (u - 1.0f));
    }
  }
  // theta prior -log(|sin t| / 2) from st = sin t (fibre.h:283-290)
  FDT_DEV static float theta_prior(float t, float st) {
    return t == 0.0f ? 0.0f : -flog(fabsf(st) * 0.5f);
  }
  // R prior (fibre.h:816-843) at diffusivity d; false outside its support
  FDT_DEV bool r_prior(float Rv, float d, float& pr) const {
    float upper = 2.0f * Rmean, lower = Rmean - 2.0f * Rstd;
    if (Rmean > 0.5f) upper = 1.0f;
    if (lower < 0.0f) lower = 1e-8f;
    if (Rfudge > 0.0f && d > UPPERDIFF_F / 2.0f) {
      if (Rv < 1e-8f || Rv > upper) return false;
      pr = Rfudge * flog(Rv);
      return true;
    }
    if (Rv <= lower || Rv > upper) return false;
    pr = (Rv - Rmean) * (Rv - Rmean) / (Rstd * Rstd);
    return true;
  }
  // mixture of slot t from the stored signals
  FDT_DEV float mix(int t) const {
    float m = fmaf(1.0f - fsum, isov(t), f0);
#pragma unroll
    for (int k = 0; k < K; ++k) m = fmaf(fk[k], s[k][t], m);
    return m;
  }

  // rebuild M and the residual (or the Rician terms) from the stored signals
  FDT_DEV void rebuild(const float* y) {
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      float m = mix(t);
      M[t] = m;
      if constexpr (RIC) ell[t] = ell_of(yv(t), S0 * m, tau);
      else r[t] = mask(t, y[t] - S0 * m);
    }
    like = chain_sum_d([&](int t, double ss) {
      if constexpr (RIC) return ss + (double)mask(t, ell[t]);
      else return ss + (double)(r[t] * r[t]);
    });
  }

  // A candidate out of its range is refused with the energy's own test: a
  // branch of its own saves the evaluation only where all four rows of a wave
  // are out of range at once (the wavefronts over 1,440 voxels at 69 volumes:
  // 215.6 -> 210.3 ms without it).  The Rician terms are dear enough to keep it.
  static constexpr bool EARLY = RIC;

  // The prior energy of a slot is pw log(x), x the candidate or, for a theta
  // slot, half the size of its sine: one weight per lane, fixed before the
  // first sweep.  Asking which slot a lane is, and two remainders for the sweep
  // numbers, cost about 50 scalar instructions and six branches per sweep, which
  // the other waves of a SIMD do not hide and a single one waits for: 237.5 ->
  // 215.6 ms for the wavefronts over 1,440 voxels at 69 volumes, 1,262 -> 1,242 ms
  // for a run of 250,968 voxels at 288.
  FDT_DEV void prior_weight() {
    th = rl >= SL_FIB && (rl - SL_FIB) % 3 == 0;
    pw = th ? -1.0f : 0.0f;
    if (rl == SL_DSTD || (rl == SL_F0 && ardf0)) pw = 1.0f;
    sfor<K>([&](auto kc) {
      if (rl == FK(kc) && can_ard && lam[kc]) pw = fudge;
    });
  }

  // ---------------------------------------------------------- proposals
  // The candidates of every slot from the sweep's normal draws, lane l for
  // slot l (the R slot's prior depends on d and is formed at its proposal).
  // The prior changes keep one rounding where the whole expression is one FMA.
  FDT_DEV void propose(float n) {
    sxn = sval + n * sprop;
    sincos_full(sxn, ssn, scn);
    const float lg = lg2(th ? fabsf(ssn) * 0.5f : sxn);
    const float L = lg * LN2;
    float p = pw == 0.0f || (th && sxn == 0.0f) ? 0.0f : product(pw, L);
    if (MODEL == 3 && rl == SL_D) p = fmaf(sxn, 4000.0f, -(L + L));
    sprn = p;
    sdp = rl == SL_DSTD ? fmaf(lg, LN2, -sprior) : p - sprior;
    accm = 0;
  }
  // end of the sweep: accepted slots take their candidate
  FDT_DEV void settle() {
    const bool acc = (accm >> rl) & 1u;
    scnt += acc ? 1 : rejinc;
    sval = acc ? sxn : sval;
    sprior = acc ? sprn : sprior;
    ssin = acc ? ssn : ssin;
    scos = acc ? scn : scos;
  }
  // lu: log of the uniform draw of the slot.
  // f0 (CUDA/runmcmc_kernels.cu:842-888)
  FDT_DEV void prop_f0(float lu) {
    const float f0n = cand<SL_F0>();
    const float fsn = fsum - f0 + f0n;
    const bool in = !(f0n <= 0.0f || f0n >= 1.0f || fsn > 1.0f);
    if (EARLY && !in) return;
    const float df = f0n - f0;
    float a, en[RIC ? VPL : 1], qv[VPL];
#pragma unroll
    for (int t = 0; t < VPL; ++t)
      if (!skip(t)) qv[t] = 1.0f - isov(t);
    if constexpr (RIC) a = ric_terms<false>([&](int t) { return S0 * fmaf(df, qv[t], M[t]); }, tau, en);
    else a = quad([&](int t) { return qv[t]; }, S0 * df);
    if (in & (dlik(a) + dprior<SL_F0>() < -lu)) {
      const float c = S0 * df;
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        if (skip(t)) continue;
        M[t] = fmaf(df, qv[t], M[t]);
        if constexpr (RIC) ell[t] = en[t]; else r[t] = fmaf(-c, qv[t], r[t]);
      }
      like += (double)a;
      f0 = f0n;
      fsum = sum_fractions();
      accept<SL_F0>();
    }
  }
  // tau (:890-922), Rician only
  FDT_DEV void prop_tau(float lu) {
    if constexpr (RIC) {
      const float tn = cand<SL_TAU>();
      if (tn <= 0.0f) return;
      float en[VPL];
      const float a = ric_terms<true>([&](int t) { return S0 * M[t]; }, tn, en);  // change of the stored terms
      // the -tau y^2 / 2 part of the full terms moves with tau too
      float dE = -Nf * (flog(tn) - flog(tau)) - fmaf(-0.5f * (tn - tau), yy, a);
      if (dE < -lu) {
#pragma unroll
        for (int t = 0; t < VPL; ++t) ell[t] = en[t];
        like += (double)a;
        tau = tn;
        accept<SL_TAU>();
      }
    }
  }
  // S0 (:1125-1155)
  FDT_DEV void prop_S0(float lu) {
    const float Sn = cand<SL_S0>();
    const bool in = !(Sn < 0.0f);
    if (EARLY && !in) return;
    const float dS = Sn - S0;
    float a, en[RIC ? VPL : 1];
    if constexpr (RIC) a = ric_terms<true>([&](int t) { return Sn * M[t]; }, tau, en);
    else a = quad<true>([&](int t) { return mask(t, M[t]); }, dS);
    if (in & (dlik(a) < -lu)) {
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        if constexpr (RIC) ell[t] = en[t]; else r[t] -= dS * mask(t, M[t]);
      }
      like += (double)a;
      S0 = Sn;
      accept<SL_S0>();
    }
  }
  // candidate isotropic signal of every shell into the row's table (lane l: shell l)
  template <int SI>
  FDT_DEV void fill_iso(const SigC& ci) const {
    float b = shb[rl];
    isot[rl] = sig<SI>(ci, b, b);
  }
  // run f(SH) with SH = true when the isotropic signal changes and the
  // acquisition has a shell table (the loop over slots is then the table
  // variant only; no per-slot branch)
  template <bool NI, class F>
  FDT_DEV void by_shells(F&& f) const {
    if constexpr (NI && !GN && !(SMALL && MODEL == 1)) {
      if (nshell) f(std::true_type{});
      else f(std::false_type{});
    } else f(std::false_type{});
  }
  // the Rician terms of every slot at the signals p(t) and precision tv into
  // en[], and their change into a.  Both series of log I0 cost 26 operations,
  // the one above 3.75 alone 14; x = tau p y is ~SNR^2, so most slots of most
  // waves need only that one: a vote over each group of slots takes it where
  // no volume of the wave is below 3.75 (the results are the same).
  static constexpr int RG = 3;
  // ALL: also slot 0 of b = 0 volumes (the S0 and tau moves).
  template <bool ALL, class P>
  FDT_DEV float ric_terms(P&& p, float tv, float (&en)[RIC ? VPL : 1]) const {
    const float th = -0.5f * tv;
    float a = 0.0f;
#pragma unroll
    for (int t0 = 0; t0 < VPL; t0 += RG) {
      float q[RG], h[RG], x[RG];
      bool sm = false;
      auto out = [&](int t) { return t >= VPL || (!ALL && skip(t)); };
#pragma unroll
      for (int i = 0; i < RG; ++i) {
        const int t = t0 + i;
        q[i] = h[i] = x[i] = 0.0f;
        if (out(t)) continue;
        q[i] = p(t);
        h[i] = th * q[i];
        x[i] = h[i] * ym2(t);
        sm = sm || ((FULL || t < nv) && fabsf(x[i]) < 3.75f);
      }
      if (__builtin_amdgcn_ballot_w64(sm)) {
#pragma unroll
        for (int i = 0; i < RG; ++i)
          if (t0 + i < VPL) x[i] = logI0f(x[i]);
      } else {
#pragma unroll
        for (int i = 0; i < RG; ++i)
          if (t0 + i < VPL) x[i] = logI0_large(x[i]);
      }
#pragma unroll
      for (int i = 0; i < RG; ++i) {
        const int t = t0 + i;
        if (out(t)) continue;
        en[t] = fmaf(h[i], q[i], x[i]);
        if constexpr (ROWS == 1) a += mask(t, en[t] - ell[t]);
      }
    }
    if constexpr (ROWS == 1) return row_sum16(a);
    else return chain_sum([&](int t, float z) { return z + mask(t, en[t] - ell[t]); });
  }
  // all stick signals and/or iso change: d (:924-985), d_std (:987-1051), R
  // (:1053-1122).  NA: the stick signals change, NI: the isotropic signal.
  template <int SL>
  FDT_DEV void prop_global(float lu) {
    constexpr bool NA = !(SL == SL_DSTD && MODEL == 3), NI = SL != SL_R;
    constexpr int SA = STICK_KIND<MODEL>, SI = ISO_KIND<MODEL>;
    float dn = d, dsn = dstd, Rn = Rr;
    bool in;
    if constexpr (SL == SL_D) {
      dn = cand<SL>();
      in = !(dn < 0.0f || dn > UPPERDIFF_F);
    } else if constexpr (SL == SL_DSTD) {
      dsn = cand<SL>();
      in = !(dsn <= 0.0f || dsn > (MODEL == 3 ? 0.004f : 0.01f));
    } else {
      Rn = cand<SL>();
      float prn = 0.0f;
      in = r_prior(Rn, d, prn);
      if (rl == SL_R && in) { sprn = prn; sdp = prn - sprior; }
    }
    if (EARLY && !in) return;
    const SigC cn = aniso_coef<MODEL>(dn, dsn, Rn), ci = iso_coef<MODEL>(dn, dsn);
    fence();
    constexpr bool KEEP_M = U_LDS || RIC;
    constexpr bool KEEP_Q = !RIC && ROWS > 1;
    float a, mn[KEEP_M ? VPL : 1], en[RIC ? VPL : 1], sn[U_LDS ? K : 1][VPL], qv[KEEP_Q ? VPL : 1];
    Dirs D;
    if constexpr (NA && !U_LDS) D = dirs();
    Quad qd;
    by_shells<NI>([&](auto SHc) {
      constexpr bool SH = decltype(SHc)::value;
      if constexpr (SH) fill_iso<SI>(ci);
      // slot t's reads are issued one slot ahead (the shell index two), so
      // that they return while the slot before it computes
      float u[NA && U_LDS ? K : 1][VPL], iso[VPL], b[VPL];
      float4 g[NA && !U_LDS ? VPL : 1];
      int si[SH ? VPL : 1];
      auto index = [&](int t) {
        if constexpr (SH) { if (t < VPL) si[t] = sh[rl + 16 * t]; }
      };
      auto fetch = [&](int t) {
        if (t >= VPL) return;
        if constexpr (NA && U_LDS) {
#pragma unroll
          for (int k = 0; k < K; ++k) u[k][t] = arg(k, t);
        }
        if constexpr (NA && !U_LDS) g[t] = grad(t);
        if constexpr ((NA && SA == 2) || (NI && !SH)) b[t] = bv(t, grad(t));
        if constexpr (SH) iso[t] = isot[si[t]];
        else if constexpr (!NI) iso[t] = isov(t);
      };
      index(0);
      index(1);
      fetch(0);
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        index(t + 2);
        fetch(t + 1);
        if (skip(t)) continue;
        if constexpr (NI && !SH) iso[t] = sig<SI>(ci, b[t], b[t]);
        float m = fmaf(1.0f - fsum, iso[t], f0);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          float sk_ = s[k][t];
          if constexpr (NA && U_LDS) sk_ = sn[k][t] = sig<SA>(cn, u[k][t], b[t]);
          if constexpr (NA && !U_LDS) {
            const float dp = fmaf(g[t].x, D.x[k][0], fmaf(g[t].y, D.x[k][1], g[t].z * D.x[k][2]));
            ldsk(k, t) = sk_ = sig<SA>(cn, g[t].w * dp * dp, b[t]);
          }
          m = fmaf(fk[k], sk_, m);
        }
        if (zero(t)) m = M[t];
        if constexpr (KEEP_M) mn[t] = m;
        if constexpr (KEEP_Q) qv[t] = mask(t, m - M[t]);
        else if constexpr (!RIC) qd.add(r[t], mask(t, m - M[t]));
        // the gamma form has several temporaries per volume and signal: keep
        // the scheduler from overlapping many volumes of it (register spills)
        if constexpr ((NA && SA == 1) || (NI && SI == 1)) fence();
      }
    });
    if constexpr (RIC) a = ric_terms<false>([&](int t) { return S0 * mn[t]; }, tau, en);
    else if constexpr (KEEP_Q) a = quad([&](int t) { return qv[t]; }, S0);
    else a = qd.delta(S0);
    if (in & (dlik(a) + dprior<SL>() < -lu)) {
      fence();
      by_shells<NI>([&](auto SHc) {
#pragma unroll
        for (int t = 0; t < VPL; ++t) {
          if (skip(t)) continue;
          if constexpr (NI) {
            if constexpr (decltype(SHc)::value) isov(t) = isot[sh[rl + 16 * t]];
            else {
              const float b = bv(t, grad(t));
              isov(t) = sig<SI>(ci, b, b);
            }
          }
          if constexpr (NA) {
#pragma unroll
            for (int k = 0; k < K; ++k) s[k][t] = U_LDS ? sn[U_LDS ? k : 0][t] : ldsk(k, t);
          }
        }
      });
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        if (skip(t)) continue;
        const float m = KEEP_M ? mn[KEEP_M ? t : 0] : (zero(t) ? M[t] : mix(t));  // mix(t) repeats the candidate's expression
        if constexpr (RIC) ell[t] = en[t]; else r[t] -= S0 * mask(t, m - M[t]);
        M[t] = m;
      }
      like += (double)a;
      if constexpr (SL == SL_D) d = dn;
      else if constexpr (SL == SL_DSTD) dstd = dsn;
      else Rr = Rn;
      ca = cn;
      accept<SL>();
    }
  }
  // theta_k / phi_k (:1157-1265); st..cp: sin and cos of fibre k's current
  // angles, updated with an accepted move
  template <int k, bool IS_TH>
  FDT_DEV void prop_angle(float lu, float& st, float& ct, float& sp, float& cp) {
    constexpr int SL = IS_TH ? TH(k) : PH(k);
    const float sa = row_bcast<SL>(ssn), cs = row_bcast<SL>(scn);
    const float st_ = IS_TH ? sa : st, ct_ = IS_TH ? cs : ct;
    const float sp_ = IS_TH ? sp : sa, cp_ = IS_TH ? cp : cs;
    float x0 = st_ * cp_, x1 = st_ * sp_, x2 = ct_;
    xform(x0, x1, x2);
    fence();
    float sn[VPL], un[U_LDS ? VPL : 1], qv[VPL], en[RIC ? VPL : 1];
    float a;
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      if (skip(t)) continue;
      const float4 g = grad(t);
      float dp = fmaf(g.x, x0, fmaf(g.y, x1, g.z * x2));
      const float u = g.w * dp * dp;
      if constexpr (U_LDS) un[t] = u;
      sn[t] = sig<STICK_KIND<MODEL>>(ca, u, bv(t, g));
    }
#pragma unroll
    for (int t = 0; t < VPL; ++t)
      if (!skip(t)) qv[t] = sn[t] - s[k][t];
    if constexpr (RIC) a = ric_terms<false>([&](int t) { return S0 * fmaf(fk[k], qv[t], M[t]); }, tau, en);
    else a = quad([&](int t) { return qv[t]; }, S0 * fk[k]);
    if (dlik(a) + (IS_TH ? dprior<SL>() : 0.0f) < -lu) {
      const float c = S0 * fk[k];
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        if (skip(t)) continue;
        M[t] = fmaf(fk[k], qv[t], M[t]);
        if constexpr (RIC) ell[t] = en[t]; else r[t] = fmaf(-c, qv[t], r[t]);
        s[k][t] = sn[t];
        if constexpr (U_LDS) arg(k, t) = un[t];
      }
      like += (double)a;
      if constexpr (IS_TH) { st = sa; ct = cs; } else { sp = sa; cp = cs; }
      accept<SL>();
    }
  }
  // f_k (:1267-1322)
  template <int k>
  FDT_DEV void prop_f(float lu) {
    constexpr int SL = FK(k);
    const float fn = cand<SL>();
    const float fsn = fsum - fk[k] + fn;
    const bool in = !(fn <= 0.0f || fn >= 1.0f || fsn > 1.0f);
    if (EARLY && !in) return;
    const float df = fn - fk[k];
    float a, en[RIC ? VPL : 1], qv[VPL];
#pragma unroll
    for (int t = 0; t < VPL; ++t)
      if (!skip(t)) qv[t] = s[k][t] - isov(t);
    if constexpr (RIC) a = ric_terms<false>([&](int t) { return S0 * fmaf(df, qv[t], M[t]); }, tau, en);
    else a = quad([&](int t) { return qv[t]; }, S0 * df);
    if (in & (dlik(a) + dprior<SL>() < -lu)) {
      const float c = S0 * df;
#pragma unroll
      for (int t = 0; t < VPL; ++t) {
        if (skip(t)) continue;
        M[t] = fmaf(df, qv[t], M[t]);
        if constexpr (RIC) ell[t] = en[t]; else r[t] = fmaf(-c, qv[t], r[t]);
      }
      like += (double)a;
      fk[k] = fn;
      fsum = sum_fractions();
      accept<SL>();
    }
  }

  // proposal-width adaptation every upe jumps (:1341-1395), all slots of the
  // row in parallel; slots of parameters that are not sampled keep counters
  // 0/0 and are never read
  FDT_DEV void update_proposals() {
    float acc = (float)(scnt & 0xFFFF), rej = (float)(scnt >> 16);
    sprop *= sqrtf((acc + 1.0f) / (rej + 1.0f));
    sprop = fminf(sprop, MAXPROP_F);
    scnt = 0;
  }
};

// LDS of a chain workgroup: the acquisition table, the stick-signal arguments per wave, the
// b-shell index of each volume and the shells' b values, the rows' isotropic
// shell tables
struct ChainLds {
  float4* acq;
  float* sk;
  int* sh;     // null without a shell table (--gradnonlin)
  float* shb;
  float* iso;
  float* bp;   // --gradnonlin: [16 rows][16 VPL] b values of the rows' voxels
  float* gd;   // --gradnonlin: [16 rows][9] deviation values
  float* vol;  // [4 waves][VPL][64] per-volume array of the chains (null for --gradnonlin)
  int* perm;   // [16 VPL] volume held by each slot position (null: identity)
  int* zc;     // [ZC_CHUNKS] b = 0 volumes per 64-volume chunk of the acquisition
};

// Volumes with b = 0 have stick and isotropic signals of exactly 1 in every
// model, so an angle, fraction or f0 move leaves their mixture, residual and
// likelihood term unchanged, and a diffusivity move changes their mixture by
// rounding only.  When the acquisition has at least 16 of them, the staging
// puts them first (a stable partition: b = 0 volumes in order, then the others
// in order, padding last), so that slot 0 of every row holds b = 0 volumes
// only, and those proposals skip slot 0.  The likelihood is the same sum over
// the same volumes; with fewer than 16 the order is the acquisition's.  Only
// the 14- and 18-volume tiles do this (ZERO_SLOT).  With --gradnonlin the per-voxel
// b values are b |(I+L) g|^2, zero exactly where the shared table's are, and
// the rows read them in the staged order.
constexpr int ZC_CHUNKS = 8;  // 64-volume chunks of the largest table (16 x 32)

// stage the acquisition of `a` (16*VPL volumes, zero padded) into LDS; the
// caller synchronises the workgroup afterwards.  The block size is a multiple
// of 64.
template <int VPL>
FDT_DEV void stage_acq(const McmcArgs& a, const ChainLds& L) {
  constexpr int NV = 16 * VPL, NCH = (NV + 63) / 64;
  static_assert(NCH <= ZC_CHUNKS, "acquisition table larger than the chunk counts");
  if (!ZERO_SLOT<VPL> || !L.perm) {
    for (int i = threadIdx.x; i < NV; i += blockDim.x) {
      L.acq[i] = a.acq[i];
      if (L.sh) L.sh[i] = a.nshell ? a.shell[i] : 0;
    }
  } else {
    // b = 0 count per 64-volume chunk (one wave per chunk), then each volume's
    // position from the counts of the chunks before it and a ballot
    const int lane = __lane_id(), w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int ch = w; ch < NCH; ch += nw) {
      const int i = 64 * ch + lane;
      bool z = false;
      if (i < a.N) z = a.acq[i].w == 0.0f;
      const uint64_t m = __builtin_amdgcn_ballot_w64(z);
      if (lane == 0) L.zc[ch] = __builtin_popcountll(m);
    }
    __syncthreads();
    int nz = 0;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) nz += L.zc[ch];
    const bool part = nz >= 16;
    for (int ch = w; ch < NCH; ch += nw) {
      const int i = 64 * ch + lane;
      const float4 g = i < NV ? a.acq[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const bool z = i < a.N && g.w == 0.0f;
      const uint64_t m = __builtin_amdgcn_ballot_w64(z);
      int before = __builtin_popcountll(m & ((1ull << lane) - 1ull));  // b = 0 volumes below i
#pragma unroll
      for (int c = 0; c < NCH; ++c) before += c < ch ? L.zc[c] : 0;
      const int pos = (!part || i >= a.N) ? i : (z ? before : nz + i - before);
      if (i < NV) {
        L.perm[pos] = i;
        L.acq[pos] = g;
        if (L.sh) L.sh[pos] = a.nshell ? a.shell[i] : 0;
      }
    }
  }
  if (threadIdx.x < 16) L.shb[threadIdx.x] = a.nshell ? a.shell_b[threadIdx.x] : 0.0f;
}
// slot 0 of every row holds b = 0 volumes only (after the caller's
// synchronisation); uniform over the workgroup
template <int VPL>
FDT_DEV bool zero_slot0(const ChainLds& L) {
  constexpr int NCH = (16 * VPL + 63) / 64;
  if (!ZERO_SLOT<VPL> || !L.perm) return false;
  int nz = 0;
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) nz += L.zc[ch];
  return __builtin_amdgcn_readfirstlane(nz) >= 16;
}

// The whole chain of voxel `vox` on this thread's 16-lane row: initialisation
// (init_Fibres_Multifibres_kernel, CUDA/runmcmc_kernels.cu:193-505), nburn +
// njumps sweeps with recording and proposal adaptation (runmcmc_kernel,
// :507-1474, run twice by CUDA/runmcmc.cu:108-316).  GN (--gradnonlin): the
// chain reads its voxel's own corrected acquisition from a.acqv (the reference
// indexes per-voxel bvals/alpha/beta with posBV, :266, :711).
template <int K, int VPL, int MODEL, bool RIC, bool GN = false, bool FULL = false, int ROWS = 1>
FDT_DEV void run_chain(const McmcArgs& a, int vox, const ChainLds& L) {
  using C = Chain<K, VPL, MODEL, RIC, GN, FULL, ROWS>;
  static_assert(ROWS == 1 || (ROWS == 2 && !GN), "rows per voxel");
  constexpr bool ZS = ZERO_SLOT<VPL * ROWS>;
  const int lane = __lane_id();
  const int rl = lane & 15;
  const int h = ROWS > 1 ? (lane >> 4) % ROWS : 0;  // which of the voxel's rows
  const int v0 = h * 16 * VPL;                       // its first volume
  const float4* sacq = L.acq + v0;
  C c;
  c.rl = rl;
  c.acq = sacq;
  c.sk = L.sk + (threadIdx.x >> 6) * (K * VPL * 64) + lane;
  c.vol = L.vol ? L.vol + (threadIdx.x >> 6) * (VPL * 64) + lane : nullptr;
  if constexpr (C::SMALL) {
#pragma unroll
    for (int t = 0; t < VPL; ++t) c.ga[t] = sacq[rl + 16 * t];
  }
  c.sh = GN ? nullptr : L.sh + v0;
  c.shb = L.shb;
  c.isot = GN ? L.iso : L.iso + (threadIdx.x >> 4) * 16;
  c.nshell = GN ? 0 : a.nshell;
  if constexpr (GN) {
    // the row's b values (from the corrected acquisition table) and deviations
    float* bp = L.bp + (threadIdx.x >> 4) * (16 * VPL);
    float* gd = L.gd + (threadIdx.x >> 4) * 9;
    const float4* av = a.acqv + (size_t)vox * a.acqv_stride;
    const int* pm = ZS ? L.perm : nullptr;  // the staged order of the shared table
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      const int i = rl + 16 * t;
      bp[i] = av[pm ? pm[i] : i].w;
    }
    if (rl < 9) gd[rl] = a.gdev[(size_t)vox * 9 + rl];
    c.bp = bp;
    c.gd = gd;
  }
  c.incf0 = a.f0 != 0;
  c.ardf0 = a.ardf0 != 0;
  c.can_ard = a.no_ard == 0;
  c.fudge = a.fudge;
  c.halfN = 0.5f * (float)a.N;
  c.Nf = (float)a.N;
  c.Rmean = a.Rmean; c.Rstd = a.Rstd; c.Rfudge = a.Rfudge;
  c.nv = a.N - v0 > rl ? min(VPL, (a.N - v0 - rl + 15) >> 4) : 0;
#pragma unroll
  for (int k = 0; k < K; ++k) c.lam[k] = (k == 0) ? (a.all_ard != 0) : (a.no_ard == 0);

  // ---- data (with the Rician non-positive replacement, CUDA/xfibres_gpu.cu:350-367)
  float y[VPL];
  const float* yrow = a.data + (size_t)vox * a.N;
  const int* perm = ZS ? L.perm : nullptr;  // volume of each slot position (null: identity)
  c.z0 = zero_slot0<VPL * ROWS>(L) && h == 0;
#pragma unroll
  for (int t = 0; t < VPL; ++t) {
    int i = v0 + rl + 16 * t;
    y[t] = i < a.N ? yrow[perm ? perm[i] : i] : 0.0f;
  }
  if (RIC) {
    float mn = 3.0e38f, mx = -3.0e38f, mnp = 3.0e38f;
#pragma unroll
    for (int t = 0; t < VPL; ++t)
      if (v0 + rl + 16 * t < a.N) { mn = fminf(mn, y[t]); mx = fmaxf(mx, y[t]); if (y[t] > 0.0f) mnp = fminf(mnp, y[t]); }
    mn = row_min16(mn); mx = row_max16(mx); mnp = row_min16(mnp);
    if constexpr (ROWS > 1) {
      mn = fminf(mn, __shfl_xor(mn, 16)); mx = fmaxf(mx, __shfl_xor(mx, 16)); mnp = fminf(mnp, __shfl_xor(mnp, 16));
    }
    bool san = (mn <= 0.0f && mx > 0.0f);
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      if (san && y[t] <= 0.0f) y[t] = mnp;
      if (v0 + rl + 16 * t >= a.N) y[t] = 1.0f;
    }
  }

  // ---- chain initialisation (init_Fibres_Multifibres_kernel, :265-504):
  // every lane loads the parameter of its slot and evaluates its prior
  const float* P = a.params + (size_t)vox * a.np;
  const int add = MODEL >= 2 ? 1 : 0;
  float d = P[1];
  if (d < 0.0f || d > UPPERDIFF_F) d = 2e-3f;
  float dstd = 0.0f, Rr = 0.0f;
  if (MODEL >= 2) {
    dstd = P[2];
    float up = MODEL == 3 ? 0.004f : 0.01f;
    if (dstd < 0.0f || dstd > up) dstd = d / 10.0f;
    if (MODEL == 3) Rr = a.Rmean;
  }
  float val = 0.0f, pr = 0.0f, wd = 0.2f;  // f0 and the fibre slots start at width 0.2 (:497-503)
  float vs = 0.0f, vc = 1.0f;              // sin / cos of an angle slot's value
  if (rl == SL_F0) {
    val = c.incf0 ? P[a.np - 1] : 0.0f;
    if (c.incf0 && c.ardf0 && val > 0.0f && val < 1.0f) pr = flog(val);
  } else if (rl == SL_TAU) {
    val = (RIC && a.tau) ? a.tau[vox] : 0.0f;
    wd = val / 2.0f;
  } else if (rl == SL_D) {
    val = d;
    if (MODEL == 3) pr = (1.0f - 3.0f) * flog(d) + 4000.0f * d;
    wd = d / 10.0f;
  } else if (rl == SL_DSTD) {
    val = dstd;
    float up = MODEL == 3 ? 0.004f : 0.01f;
    if (MODEL >= 2 && dstd > 0.0f && dstd <= up) pr = flog(dstd);
    wd = dstd / 10.0f;
  } else if (rl == SL_R) {
    val = Rr;
    float q;
    if (MODEL == 3 && c.r_prior(Rr, d, q)) pr = q;
    wd = Rr / 10.0f;
  } else if (rl == SL_S0) {
    val = P[0];
    wd = val / 10.0f;
  } else if (rl < SL_FIB + 3 * K) {
    int k = (rl - SL_FIB) / 3, w = (rl - SL_FIB) % 3;
    if (w == 0) { val = P[3 + 3 * k + add]; sincos_full(val, vs, vc); pr = C::theta_prior(val, vs); }
    else if (w == 1) { val = P[4 + 3 * k + add]; sincos_full(val, vs, vc); }
    else {
      val = P[2 + 3 * k + add];
      bool lk = (k == 0) ? (a.all_ard != 0) : (a.no_ard == 0);
      pr = (val <= 0.0f || val >= 1.0f) ? 0.0f : a.fudge * (lk ? flog(val) : 0.0f);
    }
  }
  if (a.widths_in) {
    float w = a.widths_in[(size_t)vox * 16 + rl];
    if (w > 0.0f) wd = w;
  }
  c.sval = val;
  c.sprior = pr;
  c.sprop = wd;
  c.ssin = vs;
  c.scos = vc;
  c.scnt = 0;
  c.rejinc = 0;
  if (rl == SL_D || rl == SL_S0 || (rl >= SL_FIB && rl < SL_FIB + 3 * K) || (rl == SL_F0 && c.incf0) ||
      (rl == SL_TAU && RIC) || (rl == SL_DSTD && MODEL >= 2) || (rl == SL_R && MODEL == 3))
    c.rejinc = 1 << 16;
  c.S0 = row_bcast<SL_S0>(val);
  c.tau = row_bcast<SL_TAU>(val);
  c.d = d; c.dstd = dstd; c.Rr = Rr;
  c.f0 = row_bcast<SL_F0>(val);
  sfor<K>([&](auto kc) { c.fk[kc] = row_bcast<C::FK(kc)>(val); });
  c.fsum = c.sum_fractions();
  {
    c.ca = aniso_coef<MODEL>(d, dstd, Rr);
    const SigC ci = iso_coef<MODEL>(d, dstd);
    const typename C::Dirs D = c.dirs();
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      const float4 g = c.grad(t);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        float dp = fmaf(g.x, D.x[k][0], fmaf(g.y, D.x[k][1], g.z * D.x[k][2]));
        const float u = g.w * dp * dp;
        if constexpr (C::U_LDS) c.arg(k, t) = u;
        c.s[k][t] = sig<STICK_KIND<MODEL>>(c.ca, u, c.bv(t, g));
      }
    }
#pragma unroll
    for (int t = 0; t < VPL; ++t) { float b = c.bv(t, c.grad(t)); c.isov(t) = sig<ISO_KIND<MODEL>>(ci, b, b); }
  }
  if constexpr (RIC) {
#pragma unroll
    for (int t = 0; t < VPL; ++t) {
      if constexpr (C::Y_LDS) c.vol[t * 64] = -2.0f * y[t];
      else c.r[t] = -2.0f * y[t];
    }
    c.yy = c.template chain_sum<true>([&](int t, float z) { return z + c.mask(t, square(y[t])); });
  }
  c.rebuild(y);

  // record destination of the lane's slot (:1326-1339)
  float* rec_base = nullptr;
  size_t rec_stride = (size_t)a.vstride;  // per sample
  if (rl == SL_F0) rec_base = a.f0s;
  else if (rl == SL_TAU) rec_base = a.taus;
  else if (rl == SL_D) rec_base = a.d;
  else if (rl == SL_DSTD) rec_base = a.dstd;
  else if (rl == SL_R) rec_base = a.R;
  else if (rl == SL_S0) rec_base = a.S0;
  else if (rl < SL_FIB + 3 * K) {
    int k = (rl - SL_FIB) / 3, w = (rl - SL_FIB) % 3;
    float* arr = w == 0 ? a.th : (w == 1 ? a.ph : a.f);
    if (arr) rec_base = arr + (size_t)k * a.nsamples * a.vstride;
  }
  if (h) rec_base = nullptr;
  if (rec_base) rec_base += vox;

  const uint64_t gvox = a.vox_offset + (uint64_t)vox;
  const int total = a.nburn + a.njumps;
  c.prior_weight();
  // sweeps to the next record and to the next change of the widths (counted
  // down: see prior_weight)
  int to_record = a.se, to_widths = a.upe, smp = 0;
  for (int j = 0; j < total; ++j) {
    float nl, lul;
    draw<!RIC>(a.seed, gvox, (uint32_t)j, (uint32_t)rl, nl, lul);
    c.propose(nl);
    if (c.incf0) c.prop_f0(row_bcast<SL_F0>(lul));
    if (RIC) c.prop_tau(row_bcast<SL_TAU>(lul));
    c.template prop_global<SL_D>(row_bcast<SL_D>(lul));
    if (MODEL >= 2) {
      c.template prop_global<SL_DSTD>(row_bcast<SL_DSTD>(lul));
      if (MODEL == 3) c.template prop_global<SL_R>(row_bcast<SL_R>(lul));
    }
    c.prop_S0(row_bcast<SL_S0>(lul));
    sfor<K>([&](auto kc) {
      constexpr int k = kc;
      float st = row_bcast<C::TH(k)>(c.ssin), ct = row_bcast<C::TH(k)>(c.scos);
      float sp = row_bcast<C::PH(k)>(c.ssin), cp = row_bcast<C::PH(k)>(c.scos);
      c.template prop_angle<k, true>(row_bcast<C::TH(k)>(lul), st, ct, sp, cp);
      c.template prop_angle<k, false>(row_bcast<C::PH(k)>(lul), st, ct, sp, cp);
      c.template prop_f<k>(row_bcast<C::FK(k)>(lul));
    });
    c.settle();

    // record: the lane of each sampled slot writes its value
    if (a.se > 0 && j >= a.nburn && --to_record == 0) {
      to_record = a.se;
      if (smp < a.nsamples && rec_base) rec_base[(size_t)smp * rec_stride] = c.sval;
      ++smp;
    }
    if (--to_widths == 0) {
      to_widths = a.upe;
      c.update_proposals();
      // Re-anchor the incremental state with the widths: the mixtures, the
      // residuals (Gaussian: from the data, re-read) and the running
      // likelihood recomputed from the stored signals, so rounding in the
      // per-move updates cannot accumulate over the whole chain (the
      // reference recomputes its likelihood at every proposal).
      if constexpr (RIC) c.rebuild(nullptr);
      else {
        float yr[VPL];
#pragma unroll
        for (int t = 0; t < VPL; ++t) {
          const int i = v0 + rl + 16 * t;
          yr[t] = i < a.N ? yrow[perm ? perm[i] : i] : 0.0f;
        }
        c.rebuild(yr);
      }
    }
  }
  if (a.energy) {
    const float tau = c.tau;
    double e = c.like;
    if constexpr (RIC) {
      // the model-independent part of the Rician terms
      const double sl = c.chain_sum_d([&](int t, double z) { return z + (double)c.mask(t, flog(c.yv(t))); });
      const double sy = c.chain_sum_d([&](int t, double z) {
        const double yd = (double)c.yv(t);
        return z + (t < c.nv ? yd * yd : 0.0);
      });
      e = -(double)a.N * (double)flog(tau) - (c.like + sl - 0.5 * (double)tau * sy);
    }
    if (rl == 0 && h == 0) a.energy[vox] = (float)e;
  }
  if (a.ssr) {  // sum of squares of the final state's residuals (the Rician chain keeps the data in r)
    double ss;
    if constexpr (RIC) {
      const float S0 = c.S0;
      ss = (double)c.template chain_sum<true>([&](int t, float z) {
        const float e = c.yv(t) - S0 * c.M[t];
        return z + c.mask(t, square(e));
      });
    } else {
      ss = c.like;
    }
    if (rl == 0 && h == 0) a.ssr[vox] = (float)ss;
  }
  if (a.widths_out && h == 0) a.widths_out[(size_t)vox * 16 + rl] = c.sprop;
}


}  // namespace fdt
