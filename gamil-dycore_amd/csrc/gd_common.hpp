// gd_common.hpp -- device helpers shared by the row kernels and the polar
// filter: XCD-aware tile mapping, deterministic workgroup sums, tendency
// loads/stores in the compute type and the predictor/corrector epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gd_device.hpp"

namespace gd {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ int xcd_tile(int ntiles) {
  const int b = blockIdx.x, nb = gridDim.x;  // nb is a multiple of kXcd
  const int per = nb / kXcd;
  const int t = (b % kXcd) * per + b / kXcd;
  return t < ntiles ? t : -1;
}

// Thread index within a tile of kBlock threads.  A workgroup of the wide
// phase launch holds several such tiles side by side (tile threadIdx.x /
// kBlock); in every other launch the workgroup is one tile.
__device__ __forceinline__ int ltid() { return (int)(threadIdx.x & (kBlock - 1)); }

// x of another lane by a DPP move (CTRL: the DPP control of the move; every
// lane active).
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double x) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true));
}

// The wave butterfly l <-> l ^ 32, 16, 8, 4, 2, 1 without LDS.  fold32(a, b):
// in the lower half a's sums over l, l ^ 32, in the upper half b's
// (v_permlane32_swap exchanges a's upper half with b's lower); fold16
// likewise by rows of 16 (even rows a's, odd rows b's).  fold_row adds over l
// ^ 8, 4, 2, 1: a rotation within the row of 16 gives lane l ^ n's value, since
// the sums before it repeat with period 2 n.
__device__ __forceinline__ double fold32(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double fold_row(double v) {
  v += dpp_mov<0x128>(v);  // row_ror:8
  v += dpp_mov<0x124>(v);
  v += dpp_mov<0x122>(v);
  v += dpp_mov<0x121>(v);
  return v;
}

// Sum over the 64 lanes of a wave, the same in every lane.
__device__ __forceinline__ double wave_sum(double v) {
  v = fold32(v, v);
  v = fold16(v, v);
  return fold_row(v);
}

// The sums of K values over the wave, left in dst[0..K-1] (LDS) by the lanes
// that hold them; four values to a butterfly.
template <int K>
__device__ __forceinline__ void wave_sums_to(const double (&v)[K], double *dst) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < K; q += 4) {
    const int q1 = q + 1 < K ? q + 1 : q, q2 = q + 2 < K ? q + 2 : q, q3 = q + 3 < K ? q + 3 : q1;
    const double s = fold_row(fold16(fold32(v[q], v[q1]), fold32(v[q2], v[q3])));
    // lanes 0, 16, 32, 48 hold values q, q + 2, q + 1, q + 3
    const int k = q + ((lane >> 4) & 1) * 2 + (lane >> 5);
    if ((lane & 15) == 0 && k < K) dst[k] = s;
  }
}

// One wave holding a whole row: v[k] are the values of the lanes of wave k of a
// tile; their total as block_sum adds it, the same in every lane.
__device__ __forceinline__ double row_total(const double (&v)[4]) {
  const double s = fold_row(fold16(fold32(v[0], v[1]), fold32(v[2], v[3])));
  auto at = [s](int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(s), lane),
                            __builtin_amdgcn_readlane(__double2loint(s), lane));
  };
  return ((at(0) + at(32)) + at(16)) + at(48);
}

// Deterministic sum over the kBlock threads of a tile (fixed butterfly +
// fixed cross-wave order); every thread of the tile returns the same value.
// The barriers are the workgroup's, so every tile of a workgroup calls it
// at the same point, each with its own `red`.
__device__ __forceinline__ double block_sum(double v, double *red) {
  v = wave_sum(v);
  const int w = (threadIdx.x >> 6) & (kBlock / 64 - 1);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = red[0];
  for (int k = 1; k < kBlock / 64; ++k) s += red[k];
  return s;
}

// Deterministic tile sums of K values at once (one pair of barriers);
// `red` holds 4*K doubles.  Every thread of the tile returns the same sums.
template <int K>
__device__ __forceinline__ void block_sum_n(double (&v)[K], double *red) {
  const int w = (threadIdx.x >> 6) & (kBlock / 64 - 1);
  __syncthreads();
  wave_sums_to<K>(v, red + w * K);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q) {
    double s = red[q];
    for (int k = 1; k < kBlock / 64; ++k) s += red[k * K + q];
    v[q] = s;
  }
}

__device__ __forceinline__ const double *fld_ptr(const Member &mb, int slot, int comp) {
  return mb.st(slot, comp == CDU ? FU : (comp == CDV ? FV : FGD));
}

__device__ __forceinline__ double fld_base(const Member &mb, int slot, int comp, size_t o) {
  return mb.st(slot, comp == CDU ? FU : (comp == CDV ? FV : FGD))[o];
}

// Stored tendencies Tb, Tc are FP64 in every precision mode: the FP32
// values of mixed mode widen exactly, filtered rows keep the FP64 rescale,
// and the wider loads measured faster than FP32 ones in the corrector.
__device__ __forceinline__ double tend_load(const Member &mb, bool tb, int comp, size_t o) {
  return (tb ? mb.tb(comp) : mb.tc(comp))[o];
}

__device__ __forceinline__ void tend_store(const Member &mb, bool tb, int comp, size_t o, double v) {
  (tb ? mb.tb(comp) : mb.tc(comp))[o] = v;
}

// Phase A of a call may form its own state from the call before it, X' = X +
// dt beta Tc (k_update's expression), wherever it reads it, in place of a
// k_update launch (FOLD).  fold_step: dt beta of that call, from the member's
// partials in k_update's order (thread tid adds entries tid, tid + kBlock, ...),
// by every tile for itself.  `red` holds 24 doubles; ends with barriers.
__device__ __forceinline__ double fold_step(const Args &a, const Member &mb, double *red) {
  const int n = a.M * a.nseg, tid = ltid();
  double q[6] = {0, 0, 0, 0, 0, 0};
  for (int k0 = 0; k0 < n; k0 += 3 * kBlock) {
    double2 x[3][3];
    bool in[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int k = k0 + u * kBlock + tid;
      in[u] = k < n;
      const int kk = in[u] ? k : 0, row = kk / a.nseg, sg = kk - row * a.nseg;
#pragma unroll
      for (int c = 0; c < 3; ++c) x[u][c] = *(const double2 *)(mb.part() + ((size_t)(row * 3 + c) * a.nseg + sg) * 2);
    }
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        q[2 * c] += in[u] ? x[u][c].x : 0.0;
        q[2 * c + 1] += in[u] ? x[u][c].y : 0.0;
      }
  }
  block_sum_n<6>(q, red);
  const double ip1 = (q[0] + q[2]) + q[4];
  const double ip2 = (q[1] + q[3]) + q[5];
  const double beta = (a.fold_qcon && ip1 != 0.0 && ip2 != 0.0) ? ip1 / ip2 : 1.0;
  return a.fold_dt * beta;
}

// The epilogue of one tendency value of a predict/correct phase (not
// diffusion), split in two so a kernel can issue the load early: the value
// phase_store needs (state s0 for the predictors, Tb for phase C) ...
template <typename CT>
__device__ __forceinline__ double phase_pre(const Args &a, const Member &mb, int comp, size_t o) {
  if (a.phase == PH_A || a.phase == PH_B) return fld_base(mb, a.s0, comp, o);
  if (a.phase == PH_C) return tend_load(mb, true, comp, o);
  return 0.0;
}

// ... and the stores given that value: S_out = s0 + dt/2 T for the
// predictors (phase B also keeps T as Tb), T as Tc for phase C with the
// (Tb T w, T T w) products of the beta partials.
template <typename CT>
__device__ __forceinline__ void phase_store(const Args &a, const Member &mb, int comp, size_t o, double T,
                                            double pre, double w, double &p1, double &p2) {
  const int f = comp == CDU ? FU : (comp == CDV ? FV : FGD);
  if (a.phase == PH_A || a.phase == PH_B) {
    mb.st(a.s_out, f)[o] = pre + a.hdt * T;
    if (a.phase == PH_B) tend_store(mb, true, comp, o, T);
  } else {
    tend_store(mb, false, comp, o, T);
    if (a.phase == PH_C) {
      p1 += pre * T * w;
      p2 += T * T * w;
    }
  }
}

}  // namespace gd
