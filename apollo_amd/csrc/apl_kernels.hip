// apl_kernels.hip -- instantiates the RHS kernels of one polynomial order.
// Compiled once per order with -DAPL_ORDER=<N> (see Makefile), so the eight
// orders build in parallel.
#include "apl_adj_eo.h"
#include "apl_adjoint.h"
#include "apl_device.h"
#include "apl_eo.h"
#include "apl_eo_linear.h"
#include "apl_limiter.h"
#include "apl_valu.h"

#ifndef APL_ORDER
#error "compile with -DAPL_ORDER=<N>"
#endif

namespace apl {

template <typename K>
static bool allow_lds(K kern, size_t lds) {
  return lds <= 65536 || hipFuncSetAttribute((const void *)kern,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds) == hipSuccess;
}

// Launch `kern` over `nbatches` 16-element batches in workgroups of W waves
// (one batch per wave, LDS_DOUBLES doubles of LDS per wave).
template <int LDS_DOUBLES, int W, typename K, typename A>
static int launch_batches(K kern, hipStream_t s, const A &a, int nbatches) {
  const size_t lds = sizeof(double) * (size_t)LDS_DOUBLES * W;
  if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((nbatches + W - 1) / W), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// The vector-ALU cubature kernel: groups of 64 elements, W waves each.
template <int N, int EQN, int FLUX, typename T, int W>
static int launch_valu(hipStream_t s, const RhsArgs &a) {
  auto kern = rhs_valu_kernel<N, EQN, FLUX, T, W>;
  const size_t lds = sizeof(double) * (size_t)ValuLds<N, EQN, T, W>::doubles;
  if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((a.K + 63) / 64), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// The even-odd kernel: groups of 32 elements, W waves each.
template <int N, int EQN, int FLUX, int W, bool VTX = false>
static int launch_eo(hipStream_t s, const RhsArgs &a) {
  auto kern = rhs_eo_kernel<N, EQN, FLUX, W, VTX>;
  const size_t lds = sizeof(double) * (size_t)EoCfg<N, EQN, W>::LDS;
  if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((a.K + 31) / 32), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// The even-odd nodal kernel: groups of 64 / EO_LPE elements, W waves each.
template <int N, int EQN, int FLUX, int W>
static int launch_eo_linear(hipStream_t s, const RhsArgs &a) {
  using C = EoLinCfg<N, EQN, W>;
  auto kern = rhs_eo_linear_kernel<N, EQN, FLUX, W>;
  const size_t lds = sizeof(double) * (size_t)C::LDS;
  if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((a.K + C::EL - 1) / C::EL), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// kind: 0 the cubature form on MFMA, 1 the nodal form (linear fluxes) on
// MFMA, 2 the cubature form on the VALU kernel (N <= 3, FP32), 3 the nodal
// form on the VALU kernel (TM, FP64 and FP32), 4 the cubature form on the
// even-odd kernel (FP64, eo_order), 5 the nodal form on the even-odd kernel
// (FP64)
template <int N, int EQN, int FLUX, typename T>
static int launch_typed(int kind, hipStream_t s, const RhsArgs &a, int nblocks) {
  if constexpr ((EQN == APL_EQN_PHMAXWELL8 || EQN == APL_EQN_MAXWELL_TM3) && sizeof(T) == 8) {
    if (kind == 5) {
      // Four waves per group while a CU's LDS holds its share of the groups,
      // at most two (us per stage, 4 / 2 waves: 8-variable N = 4, K = 5000,
      // 14.5 / 17.7; K = 9800, 20.6 / 19.5); then two.  At N <= 4 one, without
      // the reduction, from four groups per CU on (N = 4: K = 16200 24.5 / 29.5
      // with one, K = 28800 38.9 / 35.1, K = 180000 212 / 188; N = 5, where one
      // wave leaves no room for a second one's registers, 241 / 261).
      const int groups = (a.K + 15) / 16;
      constexpr int fit = 163840 / (EoLinCfg<N, EQN, 4>::LDS * 8);
      if constexpr (EQN == APL_EQN_MAXWELL_TM3) {
        return launch_eo_linear<N, EQN, FLUX, 4>(s, a);
      } else {
        if constexpr (fit > 0)
          if (groups <= 256 * (fit < 2 ? fit : 2)) return launch_eo_linear<N, EQN, FLUX, 4>(s, a);
        if constexpr (N <= 4)
          if (groups > 1024) return launch_eo_linear<N, EQN, FLUX, 1>(s, a);
        return launch_eo_linear<N, EQN, FLUX, 2>(s, a);
      }
    }
  }
  if constexpr (EQN == APL_EQN_PHMAXWELL8 || EQN == APL_EQN_MAXWELL_TM3) {
    if (kind == 1)
      return launch_batches<LinLds<N, EQN, T>::doubles, LinGroup<N, EQN, T>::W>(
          rhs_linear_kernel<N, EQN, FLUX, T>, s, a, nblocks);
  }
  if constexpr (EQN == APL_EQN_MAXWELL_TM3 && sizeof(T) != 1) {
    if (kind == 3) {
      // 64 elements per workgroup
      auto kern = rhs_valu_linear_kernel<N, EQN, FLUX, T>;
      const size_t lds = sizeof(double) * (size_t)ValuLinLds<N, EQN, T>::doubles;
      if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
      hipLaunchKernelGGL(kern, dim3((a.K + 63) / 64), dim3(64 * ValuLinCfg<N, EQN>::W), lds, s, a);
      return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
    }
  }
  if (kind == 1 || kind == 3) return APL_ERR_ARG;
  if (kind == 4) {
    if constexpr (eo_order(N, Vars<EQN>::M) && sizeof(T) == 8) {
      if constexpr (EQN == APL_EQN_EULER5 || EQN == APL_EQN_EULER4)
        if (a.vortex) return launch_eo<N, EQN, FLUX, 4, true>(s, a);
      // One wave per group once the waves fill the card's 1024 SIMDs twice
      // over (no reduction; us per stage, 1 against 4 waves: Euler N = 4,
      // 16384 groups 404 / 494; 5-variable N = 4, 4096 groups 162 / 240);
      // below that the last round of long waves costs more than the split
      // (N = 3, 4096 groups 74 / 67; N = 4, 2500 groups 96 / 78), unless a
      // CU's LDS holds only one four-wave group.  At N = 1 and, with five
      // variables or more, N = 2 the waves are short and the reduction is more of
      // a group's work: one from 1536 groups on (N = 1: TM, 3906 groups 21.7 /
      // 27.1, Euler, 1600 17.0 / 18.0; N = 2, 5 variables HLL, 1600 groups 35.7 /
      // 38.1, 1156 33.3 / 29.1), for eight variables at N = 1 from 1024 on (16.8 /
      // 18.2).  Eight while a CU gets at most one group (256 groups, N = 4: 15.4 /
      // 16.4 with four).
      const int groups = (a.K + 31) / 32;
      constexpr bool PAIR = 2 * EoCfg<N, EQN, 4>::LDS * 8 <= 163840;
      constexpr int M = Vars<EQN>::M;
      constexpr int ONE = N == 1 && M == 8 ? 1024 : N == 1 || (N == 2 && M >= 5) ? 1536
                          : (PAIR ? 2 * EoWaves<N, EQN, 1>::value : 1) * 1024;
      if (groups >= ONE) return launch_eo<N, EQN, FLUX, 1>(s, a);
      if constexpr (EoCfg<N, EQN, 8>::LDS * 8 <= 163840)
        if (groups <= 256) return launch_eo<N, EQN, FLUX, 8>(s, a);
      return launch_eo<N, EQN, FLUX, 4>(s, a);
    } else {
      return APL_ERR_UNSUPPORTED;
    }
  }
  if (kind == 2) {
    if constexpr (N <= 3 && (sizeof(T) == 4 || (sizeof(T) == 8 && valu_fp64_order(EQN, N)))) {
      // 64 elements per workgroup of four waves, or of eight on small meshes
      const int groups = (a.K + 63) / 64;
      if constexpr (sizeof(T) == 4)
        if (groups < VALU_SMALL_GROUPS && ValuLds<N, EQN, T, 8>::doubles * 8 <= 163840)
          return launch_valu<N, EQN, FLUX, T, 8>(s, a);
      return launch_valu<N, EQN, FLUX, T, 4>(s, a);
    } else {
      return APL_ERR_UNSUPPORTED;
    }
  }
  return launch_batches<Lds<N, EQN, T>::doubles, RhsGroup<N, EQN, T>::W>(rhs_kernel<N, EQN, FLUX, T>, s,
                                                                          a, nblocks);
}

template <int N, int EQN, int FLUX>
static int launch_prec(int prec, int kind, hipStream_t s, const RhsArgs &a, int nblocks) {
  switch (prec) {
    case APL_PREC_FP64: return launch_typed<N, EQN, FLUX, double>(kind, s, a, nblocks);
    case APL_PREC_FP32_MFMA: return launch_typed<N, EQN, FLUX, float>(kind, s, a, nblocks);
    case APL_PREC_BF16X3: return launch_typed<N, EQN, FLUX, Bf16x3>(kind, s, a, nblocks);
    default: return APL_ERR_UNSUPPORTED;
  }
}

template <int N>
int launch_rhs(int eqn, int flux, int prec, int linear, hipStream_t s, const RhsArgs &a,
               int nblocks) {
  switch (eqn) {
    case APL_EQN_EULER5:
      if (flux == APL_FLUX_HLL) return launch_prec<N, APL_EQN_EULER5, APL_FLUX_HLL>(prec, linear, s, a, nblocks);
      if (flux == APL_FLUX_ROE) return launch_prec<N, APL_EQN_EULER5, APL_FLUX_ROE>(prec, linear, s, a, nblocks);
      if (flux == APL_FLUX_WAVE) return launch_prec<N, APL_EQN_EULER5, APL_FLUX_WAVE>(prec, linear, s, a, nblocks);
      return launch_prec<N, APL_EQN_EULER5, APL_FLUX_LF>(prec, linear, s, a, nblocks);
    case APL_EQN_EULER4:
      if (flux == APL_FLUX_HLL) return launch_prec<N, APL_EQN_EULER4, APL_FLUX_HLL>(prec, linear, s, a, nblocks);
      if (flux == APL_FLUX_ROE) return launch_prec<N, APL_EQN_EULER4, APL_FLUX_ROE>(prec, linear, s, a, nblocks);
      if (flux == APL_FLUX_WAVE) return launch_prec<N, APL_EQN_EULER4, APL_FLUX_WAVE>(prec, linear, s, a, nblocks);
      return launch_prec<N, APL_EQN_EULER4, APL_FLUX_LF>(prec, linear, s, a, nblocks);
    case APL_EQN_PHMAXWELL8:
      return launch_prec<N, APL_EQN_PHMAXWELL8, APL_FLUX_LF>(prec, linear, s, a, nblocks);
    case APL_EQN_MAXWELL_TM3:
      if (flux == APL_FLUX_UPWIND)
        return launch_prec<N, APL_EQN_MAXWELL_TM3, APL_FLUX_UPWIND>(prec, linear, s, a, nblocks);
      return launch_prec<N, APL_EQN_MAXWELL_TM3, APL_FLUX_LF>(prec, linear, s, a, nblocks);
    default: return APL_ERR_ARG;
  }
}

template int launch_rhs<APL_ORDER>(int, int, int, int, hipStream_t, const RhsArgs &, int);

template <int N, int EQN, int FLUX, int W, bool VTX = false>
static int launch_adj_eo(hipStream_t s, const AdjArgs &a) {
  auto kern = a.mode == 1 ? adj_eo_kernel<N, EQN, FLUX, W, true, VTX> : adj_eo_kernel<N, EQN, FLUX, W, false, VTX>;
  const size_t lds = sizeof(double) * (size_t)AdjEoCfg<N, EQN, W>::LDS;
  if (!allow_lds(kern, lds)) return APL_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((a.K + 31) / 32), dim3(64 * W), lds, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

template <int N, int EQN, int FLUX>
static int launch_adjoint_typed(hipStream_t s, const AdjArgs &a, int nblocks) {
  if constexpr (adj_eo_order(N, Vars<EQN>::M)) {
    const int groups = (a.K + 31) / 32;
    if (a.face_pass) {
      hipLaunchKernelGGL((adj_mu_kernel<N, EQN>), dim3(groups), dim3(64), 0, s, a);
      if (hipGetLastError() != hipSuccess) return APL_ERR_HIP;
    }
    if constexpr (EQN == APL_EQN_EULER5 || EQN == APL_EQN_EULER4)
      if (a.vortex) return launch_adj_eo<N, EQN, FLUX, 4, true>(s, a);
    // as launch_eo, with a later change to one wave, since the larger units
    // make its last round longer (us, 1 against 4 waves: adjoint RHS, Euler
    // N = 3, 4096 groups 133 / 122; 5-variable N = 3, 2500 groups, where
    // four-wave groups fill a CU's LDS one at a time, 137 / 164)
    constexpr bool PAIR = 2 * AdjEoCfg<N, EQN, 4>::LDS * 8 <= 163840;
    if (groups >= (PAIR ? 3 * AdjEoWaves<N, EQN, 1>::value : 1) * 1024)
      return launch_adj_eo<N, EQN, FLUX, 1>(s, a);
    if constexpr (AdjEoCfg<N, EQN, 8>::LDS * 8 <= 163840)
      if (groups <= 256) return launch_adj_eo<N, EQN, FLUX, 8>(s, a);
    return launch_adj_eo<N, EQN, FLUX, 4>(s, a);
  } else {
  if (a.face_pass) {
    const int rc = launch_batches<AdjFaceLds<N, EQN>::doubles, AdjFaceGroup<N, EQN>::W>(
        adj_face_kernel<N, EQN>, s, a, nblocks);
    if (rc) return rc;
  }
  if (a.mode == 1)
    return launch_batches<AdjLds<N, EQN>::doubles, AdjGroup<N, EQN>::W>(
        adj_rhs_kernel<N, EQN, FLUX, true>, s, a, nblocks);
  return launch_batches<AdjLds<N, EQN>::doubles, AdjGroup<N, EQN>::W>(
      adj_rhs_kernel<N, EQN, FLUX, false>, s, a, nblocks);
  }
}

template <int N>
int launch_adjoint(int eqn, int flux, hipStream_t s, const AdjArgs &a, int nblocks) {
  switch (eqn) {
    case APL_EQN_EULER5: return launch_adjoint_typed<N, APL_EQN_EULER5, APL_FLUX_LF>(s, a, nblocks);
    case APL_EQN_EULER4: return launch_adjoint_typed<N, APL_EQN_EULER4, APL_FLUX_LF>(s, a, nblocks);
    case APL_EQN_PHMAXWELL8:
      return launch_adjoint_typed<N, APL_EQN_PHMAXWELL8, APL_FLUX_LF>(s, a, nblocks);
    case APL_EQN_MAXWELL_TM3:
      if (flux == APL_FLUX_UPWIND)
        return launch_adjoint_typed<N, APL_EQN_MAXWELL_TM3, APL_FLUX_UPWIND>(s, a, nblocks);
      return launch_adjoint_typed<N, APL_EQN_MAXWELL_TM3, APL_FLUX_LF>(s, a, nblocks);
    default: return APL_ERR_ARG;
  }
}

template <int N>
int launch_objective(int m, hipStream_t s, const ObjArgs &a, int nblocks) {
  switch (m) {
    case 3: hipLaunchKernelGGL((objective_kernel<N, 3>), dim3(nblocks), dim3(64), 0, s, a); break;
    case 4: hipLaunchKernelGGL((objective_kernel<N, 4>), dim3(nblocks), dim3(64), 0, s, a); break;
    case 5: hipLaunchKernelGGL((objective_kernel<N, 5>), dim3(nblocks), dim3(64), 0, s, a); break;
    case 8: hipLaunchKernelGGL((objective_kernel<N, 8>), dim3(nblocks), dim3(64), 0, s, a); break;
    default: return APL_ERR_ARG;
  }
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

template int launch_adjoint<APL_ORDER>(int, int, hipStream_t, const AdjArgs &, int);
template int launch_objective<APL_ORDER>(int, hipStream_t, const ObjArgs &, int);

template <int N, int EQN>
static int launch_limiter_typed(hipStream_t s, const LimArgs &a) {
  const int gt = lim_gradient_threads<N>(a.K);
  const dim3 wgrid((a.K + LE - 1) / LE), rgrid((a.K + LER - 1) / LER), wave(64);
  hipLaunchKernelGGL((lim_average_kernel<N, EQN>), wgrid, wave, 0, s, a);
  hipLaunchKernelGGL((lim_gradient_kernel<N, EQN>), dim3((a.K + gt - 1) / gt), dim3(gt), 0, s, a);
  hipLaunchKernelGGL((lim_reconstruct_kernel<N, EQN>), rgrid, wave, 0, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

template <int N>
int launch_limiter(int eqn, hipStream_t s, const LimArgs &a) {
  if constexpr (N > 4) {
    return APL_ERR_UNSUPPORTED;
  } else {
    switch (eqn) {
      case APL_EQN_EULER5: return launch_limiter_typed<N, APL_EQN_EULER5>(s, a);
      case APL_EQN_EULER4: return launch_limiter_typed<N, APL_EQN_EULER4>(s, a);
      default: return APL_ERR_UNSUPPORTED;
    }
  }
}

template int launch_limiter<APL_ORDER>(int, hipStream_t, const LimArgs &);

#if APL_ORDER == 1
__global__ void __launch_bounds__(256) lim_patch_kernel(LimArgs a) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.K) return;
  const double *ave = a.tab, *vk = a.vert + e * 6;
  // J from the vertices as the geometry computes it (wxnodaldggeometry2d.cc:412-426)
  const double xr = (vk[2] - vk[0]) / 2, xs = (vk[4] - vk[0]) / 2;
  const double yr = (vk[3] - vk[1]) / 2, ys = (vk[5] - vk[1]) / 2;
  const double J = -xs * yr + xr * ys;
  double xc = 0.0, yc = 0.0, A0 = 0.0;
#pragma unroll
  for (int kk = 0; kk < 3; ++kk) {
    xc += ave[kk] * vk[2 * kk];
    yc += ave[kk] * vk[2 * kk + 1];
    A0 += 2. / 3. * ave[kk] * J;
  }
  double *o = a.avg + e * 8;
  o[5] = xc;
  o[6] = yc;
  o[7] = A0;
}

int launch_limiter_patch(hipStream_t s, const LimArgs &a) {
  hipLaunchKernelGGL(lim_patch_kernel, dim3((a.K + 255) / 256), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

__global__ void advance_time_kernel(double *t, double dt) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *t = *t + dt;
}

int launch_advance_time(hipStream_t s, double *t, double dt) {
  hipLaunchKernelGGL(advance_time_kernel, dim3(1), dim3(64), 0, s, t, dt);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// One workgroup of 1024 lanes: strided maxima, eight loads of a lane in
// flight at once, then a tree over LDS.  A host copy of the per-batch maxima
// and of the flags took two transfers and two synchronisations (RHS of the
// 8-variable Maxwell system, N = 4, K = 45000: 73 us per call, of which 48
// the RHS kernel).
__global__ void __launch_bounds__(1024) report_kernel(const double *in, int n, unsigned *err, double *pin) {
  __shared__ double part[16];
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += 8 * 1024) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = i + k * 1024 < n ? in[i + k * 1024] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = v[k] > m ? v[k] : m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)blockDim.x / 64; ++w) m = part[w] > m ? part[w] : m;
    pin[0] = m;
    *(unsigned *)(pin + 1) = *err;
    *err = 0u;
  }
}

int launch_report(hipStream_t s, const double *in, int n, unsigned *err, double *pin) {
  hipLaunchKernelGGL(report_kernel, dim3(1), dim3(n > 64 ? 1024 : 64), 0, s, in, n, err, pin);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// One workgroup: the partials that are not zero, packed in their order, to
// pinned memory, for a sum on the host in index order (the zeros of a disc's
// objective change no sum).  Added here, by the one lane that such a sum allows,
// a partial took 9 ns (N = 1, K = 524288, a disc over the domain: 116 us per
// call with gradient, 56 here; N = 3, K = 131072, 7% of it: 38.1 against
// 35.8).
__global__ void __launch_bounds__(1024) pack_report_kernel(const double *in, int n, double *pin) {
  __shared__ int cnt[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int done = 0;
  for (int b = 0; b < n; b += 4096) {
    double v[4];
    unsigned long long some[4];
    int mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = b + wave * 256 + j * 64 + lane;
      v[j] = i < n ? in[i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      some[j] = __ballot(!(v[j] == 0.0));
      mine += __popcll(some[j]);
    }
    if (lane == 0) cnt[wave] = mine;
    __syncthreads();
    int at = done;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) at += cnt[w];
      done += cnt[w];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (some[j] >> lane & 1) pin[1 + at + __popcll(some[j] & ((1ull << lane) - 1))] = v[j];
      at += __popcll(some[j]);
    }
  }
  if (threadIdx.x == 0) pin[0] = done;
}

int launch_pack_report(hipStream_t s, const double *in, int n, double *pin) {
  hipLaunchKernelGGL(pack_report_kernel, dim3(1), dim3(1024), 0, s, in, n, pin);
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}

// Roe speeds of each node's state against itself (wxnodaldg2dmethod.cc:201-213,
// wxeulereqn.cc:95-234), squared, with the operations and the order of the
// host's loop; a NaN speed does not count, as there.  A pass over the state,
// bound by memory; on the host it took a copy of the state and a serial loop
// (N = 1, K = 15842: 300 us, here 12).
template <int M>
__global__ void __launch_bounds__(256) roe_speed_kernel(const double *q, long nodes, double gamma, double *part) {
#pragma clang fp contract(off)
  __shared__ double wm[4];
  const double g1 = gamma - 1.0;
  double m = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < nodes; i += (long)gridDim.x * 256) {
    const double *d = q + i * M;
    const double rho = d[0], mu = d[1], mv = d[2], mw = M == 5 ? d[3] : 0.0, E = d[M - 1];
    const double pr = g1 * (E - 0.5 * (mu * mu + mv * mv + mw * mw) / rho);
    const double u = mu / rho, v = mv / rho, w = mw / rho;
    const double enth = (E + pr) / rho;
    const double a = sqrt(g1 * (enth - 0.5 * (u * u + v * v + w * w)));
    const double s[6] = {u - a, u, u + a, v - a, v, v + a};
#pragma unroll
    for (int k = 0; k < 6; ++k) m = m < s[k] * s[k] ? s[k] * s[k] : m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k) m = wm[k] > m ? wm[k] : m;
    part[blockIdx.x] = m;
  }
}

int launch_roe_speed(hipStream_t s, const double *q, long nodes, int m, double gamma, double *part, int *nparts) {
  const int nb = (int)((nodes + 255) / 256 < SPEED_BLOCKS ? (nodes + 255) / 256 : SPEED_BLOCKS);
  if (m == 5) hipLaunchKernelGGL(roe_speed_kernel<5>, dim3(nb), dim3(256), 0, s, q, nodes, gamma, part);
  else hipLaunchKernelGGL(roe_speed_kernel<4>, dim3(nb), dim3(256), 0, s, q, nodes, gamma, part);
  *nparts = nb;
  return hipGetLastError() == hipSuccess ? APL_OK : APL_ERR_HIP;
}
#endif

}  // namespace apl
