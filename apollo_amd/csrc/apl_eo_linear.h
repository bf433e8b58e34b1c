// apl_eo_linear.h -- the nodal RHS of the linear (Maxwell) fluxes in FP64 by the
// mirror symmetry of the reference triangle (gfx950).
//
// The nodal form of rhs_linear_kernel (apl_device.h) with the symmetry of
// apl_eo.h: nodes a <-> b and face nodes k <-> k' (bottom <-> left side,
// hypotenuse onto itself) under r <-> s, Dt_s[a, n] = Dt_r[b, n'], so that
//   Re, Ro = sum_n De, Do[., n] (Phi_r(n) +- Phi_s(n'))     Np Np products
//          - sum_k Le, Lo[., k] (S(k) +- S(k'))             3 Nfp Np / 2
// per variable instead of 2 Np Np + 3 Nfp Np, with Phi_r, Phi_s the contravariant
// fluxes at the nodes.  The FP64 matrix instructions that rhs_linear_kernel runs
// them on share their pipe with the vector ALU and pad every product to 16
// rows; here the operators are scalar operands without padding.
//
// Four lanes share an element: each evaluates the fluxes of one node of a unit
// (two mirrored pairs) with all variables, read from the LDS copy of the
// state, and holds ceil(M / 4) variables of the residual, between which
// v_permlane32_swap and v_permlane16_swap transpose.  A wave holds 16 elements
// and Np ceil(M / 4) residuals per lane, few enough for many waves, whose
// number decides how much of the memory latency shows (two lanes per element:
// 8-variable N = 4, K = 45000, 68.7 against 56.8 us a call).
//
// Measured, us per LSERK4 stage, rhs_linear_kernel -> here:
//   8 variables  K    1152         16200         45000          180000
//     N = 2      11.7 ->  8.2   14.8 -> 12.5   28.9 -> 24.2      71 -> 64.7
//     N = 4      16.9 -> 10.6   29.5 -> 24.1   59.1 -> 56.2     215 ->  173
//     N = 6      27.3 -> 14.8   57.9 -> 43.8    134 -> 97.5     427 ->  319
//     N = 8      44.7 -> 29.0    140 -> 98.5    296 ->  228     917 ->  708
//   TM           K    1152          5000
//     N = 3       9.1 ->  7.9   10.0 ->  8.8
//     N = 5      13.5 ->  9.7   15.1 -> 11.3
//     N = 7      19.2 -> 13.8   19.3 -> 14.2 (K = 3200)
// Bound: K < 8192 the chain load -> fluxes -> products -> store; above it the
// FP64 pipe from N = 5 on and the memory latency at two or three waves per
// SIMD below.
#pragma once

#include "apl_eo.h"

namespace apl {

constexpr int EO_LPE = 4;   // lanes per element

// Whether the kernel takes a mesh of K elements.  The 3 TM variables leave a
// quarter of the lanes without one, so rhs_linear_kernel is ahead once its
// waves fill the card (us per stage, rhs_linear_kernel / here: N = 3, K =
// 16200, 11.4 / 11.6; N = 4, K = 32768, 19 / 22); below, the split of an
// element over four waves gives the shorter chain.  The line is two groups of
// 16 elements per CU, or one at N = 8, where a CU's LDS holds one (K = 7200:
// 25.7 / 30.9).
inline bool eo_linear_takes(int eqn, int N, int K) {
  return eqn == APL_EQN_PHMAXWELL8 || (K + 15) / 16 <= (N <= 7 ? 512 : 256);
}

// ax F(q) + ay G(q) of the linear systems (phys_flux without its zero rows).
template <int EQN>
__device__ __forceinline__ void linear_flux(const PhysParams &P, double ax, double ay, const double *q,
                                            double *o) {
  const double c2 = P.c0 * P.c0;
  if constexpr (EQN == APL_EQN_MAXWELL_TM3) {
    o[0] = c2 * (ay * q[1] - ax * q[2]);
    o[1] = ay * q[0];
    o[2] = -ax * q[0];
  } else {
    const double chi = P.chi, g = P.gph;
    const double xc = ax * c2, yc = ay * c2;
    o[0] = chi * xc * q[6] - yc * q[5];
    o[1] = xc * q[5] + chi * yc * q[6];
    o[2] = yc * q[3] - xc * q[4];
    o[3] = g * ax * q[7] + ay * q[2];
    o[4] = g * ay * q[7] - ax * q[2];
    o[5] = ax * q[1] - ay * q[0];
    o[6] = chi * (ax * q[0] + ay * q[1]);
    o[7] = g * (xc * q[3] + yc * q[4]);
  }
}

// num_flux of the linear systems: the flux is linear, so it acts on the sum of
// the traces once.
template <int EQN, int FLUX>
__device__ __forceinline__ void linear_num_flux(const PhysParams &P, double l, double nx, double ny,
                                                const double *qM, const double *qP, double *f) {
  constexpr int M = Vars<EQN>::M;
  double s[M], d[M];
#pragma unroll
  for (int v = 0; v < M; ++v) {
    s[v] = qM[v] + qP[v];
    d[v] = qM[v] - qP[v];
  }
  linear_flux<EQN>(P, nx, ny, s, f);
  if constexpr (FLUX == APL_FLUX_UPWIND && EQN == APL_EQN_MAXWELL_TM3) {
    const double jb = nx * d[1] + ny * d[2];
    d[1] -= nx * jb;
    d[2] -= ny * jb;
  }
#pragma unroll
  for (int v = 0; v < M; ++v) f[v] = 0.5 * (f[v] + l * d[v]);
}

// Exchange lanes 16..31 of x with 0..15 of y, and 48..63 with 32..47.
__device__ __forceinline__ void swap_rows(double &x, double &y) {
  const unsigned long long ux = __builtin_bit_cast(unsigned long long, x);
  const unsigned long long uy = __builtin_bit_cast(unsigned long long, y);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ux, (unsigned)uy, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ux >> 32), (unsigned)(uy >> 32), false, false);
  x = __builtin_bit_cast(double, (unsigned long long)lo[0] | ((unsigned long long)hi[0] << 32));
  y = __builtin_bit_cast(double, (unsigned long long)lo[1] | ((unsigned long long)hi[1] << 32));
}

// All variables at the lane's own node -> the lane's variables at the unit's
// four nodes.
template <int M, int MH>
__device__ __forceinline__ void spread(const double (&p)[M], double (&y)[4][MH]) {
#pragma unroll
  for (int j = 0; j < MH; ++j) {
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k][j] = k * MH + j < M ? p[k * MH + j < M ? k * MH + j : 0] : 0.0;
    swap_halves(y[0][j], y[2][j]);
    swap_halves(y[1][j], y[3][j]);
    swap_rows(y[0][j], y[1][j]);
    swap_rows(y[2][j], y[3][j]);
  }
}

template <int N, int EQN, int W_>
struct EoLinCfg {
  using O = Order<N>;
  using E = EoNodes<N>;
  static constexpr int LPE = EO_LPE, W = W_, EL = 64 / LPE;      // lanes per element, elements per group
  static constexpr int M = Vars<EQN>::M, MH = (M + LPE - 1) / LPE;
  static constexpr int Np = O::Np, Nfp = O::Nfp, NE = E::NE, NO = E::NO;
  static constexpr int ES = Np * M, ESP = ES | 1;
  static constexpr int PPU = LPE / 2;                          // mirrored pairs per unit
  static constexpr int NVU = (NE + PPU - 1) / PPU;             // volume units
  static constexpr int NLP = Nfp + (Nfp + 1) / 2;              // mirrored face-node pairs
  static constexpr int NFU = (NLP + PPU - 1) / PPU;            // face units
  static constexpr int VW = 2 * Np, FW = Np;                   // table row of a pair
  static constexpr int CV = 2 * PPU * Np * MH + 12 * M, CF = PPU * Np * MH + 16 * M;
  // the waves of a group take contiguous shares of the units, volume first,
  // of about equal cost
  static constexpr int cost(int u) { return u < NVU ? u * CV : NVU * CV + (u - NVU) * CF; }
  static constexpr int ub(int w) {
    int u = 0;
    while (u < NVU + NFU && cost(u) + (u < NVU ? CV : CF) / 2 <= cost(NVU + NFU) * w / W) ++u;
    return w >= W ? NVU + NFU : u;
  }
  // A wave hands the others' pairs over, [dst W][src W - 1][rows of dst][64];
  // this and the result lie over the states, which are no longer needed then.
  static constexpr int RPW = 2 * ((NE + W - 1) / W) * MH;
  static constexpr int RED = W > 1 ? W * (W - 1) * RPW * 64 : 0;
  // per-unit node list: [NVU][LPE] nodes, then [NFU][LPE] face nodes f Nfp + i
  static constexpr int TAB = (NVU + NFU) * LPE;
  static constexpr int LDS = EL * ESP > RED ? EL * ESP : RED;
};

// Waves per SIMD the residual registers leave room for.
template <int N, int EQN>
struct EoLinWaves {
  static constexpr int NR = Order<N>::Np * ((Vars<EQN>::M + EO_LPE - 1) / EO_LPE);
  static constexpr int value =
      Vars<EQN>::M == 8 ? (NR <= 6 ? 4 : NR <= 20 ? 3 : 2) : (NR <= 21 ? 4 : NR <= 36 ? 3 : 2);
};

// The lane's face node kf = f Nfp + i of a unit: its face's code and geometry,
// the own node's offset, and the neighbour's values (its node
// Fmask[nf][Nfp-1-i]).
template <int M>
struct EoFaceNode {
  int code, own;
  double nx, ny, sj, qP[M];
};

template <int N, int M>
__device__ __forceinline__ void eo_face_node(const double *q, const double *gk, int kf,
                                             int code0, int code1, int code2, long ge, EoFaceNode<M> &F) {
  constexpr int Np = Order<N>::Np, Nfp = N + 1;
  const int f = kf / Nfp, i = kf - f * Nfp;
  F.code = f == 0 ? code0 : (f == 1 ? code1 : code2);
  F.nx = gk[G_NX + f];
  F.ny = gk[G_NY + f];
  F.sj = gk[G_SJ + f];
  F.own = face_node<N>(f, i) * M;
  const int nf = F.code >= 0 ? (F.code & 3) : 0;
  const double *src = q + ((F.code >= 0 ? (long)(F.code >> 2) : ge) * Np + face_node<N>(nf, Nfp - 1 - i)) * M;
#pragma unroll
  for (int v = 0; v < M; ++v) F.qP[v] = src[v];
}

template <int N, int EQN, int FLUX, int W>
__global__ void __launch_bounds__(64 * W, (EoLinWaves<N, EQN>::value))
    rhs_eo_linear_kernel(RhsArgs a) {
  using C = EoLinCfg<N, EQN, W>;
  constexpr int LPE = C::LPE, M = C::M, MH = C::MH, Np = C::Np, Nfp = C::Nfp, NE = C::NE, NO = C::NO, EL = C::EL;
  constexpr int ES = C::ES, ESP = C::ESP, NVU = C::NVU, NFU = C::NFU, PPU = C::PPU, NT = 64 * W;
  constexpr EoNodes<N> ND{};

  const cptr_t<double> TD = (cptr_t<double>)a.A1;     // [NVU PPU][VW]: De Do (a) | De Do (b) or, on the axis, the correction
  const cptr_t<double> TL = (cptr_t<double>)a.A3;     // [NFU PPU][FW]: -Le -Lo
  const int *tab = (const int *)a.A2;                 // [TAB]

  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = W == 1 ? lane : (int)threadIdx.x;
  const int el = lane & (EL - 1), qd = lane / EL;
  const int grp = xcd_batch(blockIdx.x, gridDim.x);
  const long e0 = (long)grp * EL;
  const int cnt = (int)min((long)EL, (long)a.K - e0);
  const long ge = e0 + (el < cnt ? el : 0);

  extern __shared__ double lds_all[];
  double *QS = lds_all;                     // [EL][ESP] staged states, then the result [EL][ES]

  int ub = 0, ue = 0;                       // this wave's units
#pragma unroll
  for (int w = 0; w < W; ++w)
    if (wave == w) {
      ub = C::ub(w);
      ue = C::ub(w + 1);
    }

  const int code0 = a.fcode[ge * 3], code1 = a.fcode[ge * 3 + 1], code2 = a.fcode[ge * 3 + 2];
  const double *gk = a.geom + ge * G_WORDS;
  const double jrx = gk[G_JRX], jry = gk[G_JRY], jsx = gk[G_JSX], jsy = gk[G_JSY];
  const double invJ = gk[G_INVJ];

  // 1. the group's states (missing elements repeat element 0)
  using Out = EoOut<ES, NT, false, EL>;
  constexpr int NV2 = Out::NV2, NIT = Out::NIT;
  {
    const double *qb = a.q + e0 * ES;
    if (cnt == EL) {
      dbl2 buf[NIT];
      Out::load(a.q, e0 * ES, tid, buf);
#pragma unroll
      for (int j = 0; j < NIT; ++j) {
        const int idx = tid + NT * j;
        if (NT * (j + 1) <= NV2 || idx < NV2) {
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int i = 2 * idx + k, e = i / ES, w = i - e * ES;
            QS[e * ESP + w] = buf[j][k];
          }
        }
      }
    } else {
      for (int i = tid; i < EL * ES; i += NT) {
        const int e = i / ES, w = i - e * ES;
        QS[e * ESP + w] = e < cnt ? qb[i] : qb[w];
      }
    }
  }

  const int fb = max(ub - NVU, 0), fe = max(ue - NVU, 0);
  EoFaceNode<M> F;
  if (fb < fe) eo_face_node<N, M>(a.q, gk, tab[(NVU + fb) * C::LPE + qd], code0, code1, code2, ge, F);
  group_sync<W>();

  const double *qe = QS + el * ESP;
  double Re[NE][MH], Ro[NO][MH];
#pragma unroll
  for (int i = 0; i < NE; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) {
      Re[i][j] = 0.0;
      if (i < NO) Ro[i < NO ? i : 0][j] = 0.0;
    }

  // 2. volume
#pragma unroll 1
  for (int u = ub; u < min(ue, NVU); ++u) {
    const double *qn = qe + tab[u * LPE + qd] * M;
    double q[M], pr[M], ps[M], yr[LPE][MH], ys[LPE][MH];
#pragma unroll
    for (int v = 0; v < M; ++v) q[v] = qn[v];
    linear_flux<EQN>(a.ph, jrx, jry, q, pr);
    linear_flux<EQN>(a.ph, jsx, jsy, q, ps);
    spread<M, MH>(pr, yr);
    spread<M, MH>(ps, ys);
#pragma unroll
    for (int s = 0; s < PPU; ++s) {
      const cptr_t<double> td = TD + (u * PPU + s) * C::VW;
      // an axis node's second row acts on Phi_r - Phi_s and Phi_r + Phi_s, the
      // parts that the mirror symmetry leaves out
      const double sg = u * PPU + s < NO ? 1.0 : -1.0;
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double e1 = yr[2 * s][j] + ys[2 * s + 1][j], o1 = yr[2 * s][j] - ys[2 * s + 1][j];
        const double e2 = yr[2 * s + 1][j] + sg * ys[2 * s][j], o2 = yr[2 * s + 1][j] - sg * ys[2 * s][j];
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          Re[i][j] += td[i] * e1;
          Re[i][j] += td[Np + i] * e2;
        }
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          Ro[i][j] += td[NE + i] * o1;
          Ro[i][j] += td[Np + NE + i] * o2;
        }
      }
    }
  }

  // 3. surface
  const double ca = a.ph.chi * a.ph.c0, cb = a.ph.gph * a.ph.c0;
  const double lam = fmax(fmax(ca, cb), a.ph.c0);
#pragma unroll 1
  for (int u = fb; u < fe; ++u) {
    const EoFaceNode<M> G = F;
    if (u + 1 < fe)
      eo_face_node<N, M>(a.q, gk, tab[(NVU + u + 1) * C::LPE + qd], code0, code1, code2, ge, F);
    double qM[M], qP[M], f[M], y[LPE][MH];
#pragma unroll
    for (int v = 0; v < M; ++v) {
      qM[v] = qe[G.own + v];
      qP[v] = G.qP[v];
    }
    if (G.code < 0) boundary_state<EQN, false>(*a.bc, -G.code - 1, 0.0, 0.0, 0.0, G.nx, G.ny, qM, qP);
    linear_num_flux<EQN, FLUX>(a.ph, lam, G.nx, G.ny, qM, qP, f);
#pragma unroll
    for (int v = 0; v < M; ++v) f[v] *= G.sj;
    spread<M, MH>(f, y);
#pragma unroll
    for (int s = 0; s < PPU; ++s) {
      const cptr_t<double> tl = TL + (u * PPU + s) * C::FW;
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double ev = y[2 * s][j] + y[2 * s + 1][j], od = y[2 * s][j] - y[2 * s + 1][j];
#pragma unroll
        for (int i = 0; i < NE; ++i) Re[i][j] += tl[i] * ev;
#pragma unroll
        for (int i = 0; i < NO; ++i) Ro[i][j] += tl[NE + i] * od;
      }
    }
  }

  // 4. R / J to LDS in the state's layout (W > 1: summed over the waves in
  // wave order)
  int vo[MH];
#pragma unroll
  for (int j = 0; j < MH; ++j) vo[j] = qd * MH + j < M ? qd * MH + j : M - 1;
  unsigned ef = 0;
  if constexpr (W == 1) {
    wave_sync();
    double *o = QS + el * ES;
#pragma unroll
    for (int i = 0; i < NE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j)
        if (MH * LPE == M || qd * MH + j < M) {
          if (i < NO) {
            o[ND.a[i] * M + vo[j]] = (Re[i][j] + Ro[i < NO ? i : 0][j]) * invJ;
            o[ND.b[i] * M + vo[j]] = (Re[i][j] - Ro[i < NO ? i : 0][j]) * invJ;
          } else {
            o[ND.a[i] * M + vo[j]] = Re[i][j] * invJ;
          }
        }
    wave_sync();
  } else {
    constexpr int RPW = C::RPW * 64, SRC = (W - 1) * RPW;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; ++i)
      if (i % W != wave) {
        double *rd = lds_all + (i % W) * SRC + (wave - (wave > i % W ? 1 : 0)) * RPW + lane;
#pragma unroll
        for (int j = 0; j < MH; ++j) {
          rd[(2 * (i / W) * MH + j) * 64] = Re[i][j];
          if (i < NO) rd[((2 * (i / W) + 1) * MH + j) * 64] = Ro[i < NO ? i : 0][j];
        }
      }
    __syncthreads();
    const double *rs = lds_all + wave * SRC + lane;
#pragma unroll
    for (int i = 0; i < NE; ++i)
      if (i % W == wave) {
#pragma unroll
        for (int w = 0; w < W - 1; ++w)
#pragma unroll
          for (int j = 0; j < MH; ++j) {
            Re[i][j] += rs[w * RPW + (2 * (i / W) * MH + j) * 64];
            if (i < NO) Ro[i < NO ? i : 0][j] += rs[w * RPW + ((2 * (i / W) + 1) * MH + j) * 64];
          }
      }
    __syncthreads();
    double *o = QS + el * ES;
#pragma unroll
    for (int i = 0; i < NE; ++i)
      if (i % W == wave) {
#pragma unroll
        for (int j = 0; j < MH; ++j)
          if (MH * LPE == M || qd * MH + j < M) {
            const double ro = i < NO ? Ro[i < NO ? i : 0][j] : 0.0;
            o[ND.a[i] * M + vo[j]] = (Re[i][j] + ro) * invJ;
            if (i < NO) o[ND.b[i] * M + vo[j]] = (Re[i][j] - ro) * invJ;
          }
      }
    __syncthreads();
  }

  // 5. the stage update and the store; every element sees the same speed
  dbl2 none[NIT];
  ef |= Out::write(a, QS, e0, cnt, tid, none, none);
  for (int off = 32; off > 0; off >>= 1) ef |= __shfl_xor(ef, off);
  if (lane == 0 && ef) atomicOr(a.err, ef);
  if (tid == 0 && a.speed_part)
    for (int b = 0; b < EL / 16; ++b)
      if (e0 + 16 * b < a.K) a.speed_part[e0 / 16 + b] = lam;
}

}  // namespace apl
