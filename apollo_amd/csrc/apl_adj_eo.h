// apl_adj_eo.h -- the discrete adjoint by the mirror symmetry of the
// reference triangle (FP64, gfx950).
//
// The transposed RHS of apl_adjoint.h with the products of apl_eo.h: two lanes
// per element, each with half of the variables for the products and one of
// two mirrored points for the pointwise work.  FP64 arithmetic bounds it, and
// the even and odd parts of the state and of lh = lam / J halve every product
// (E, O: sums over the even and odd parts with A_r's rows):
//   phi_r(c) = E(c) + O(c),  phi_s(c') = E(c) - O(c),  and with c' likewise;
//   out_a, out_b = Re +- Ro,  Re = sum Ve (qb(c) + qb(c')),
//                             Ro = sum Vo (qb(c) - qb(c')).
// The face weights Sb = -L^T lh are never stored: with mu = V V^T lh they are
// -gw I1D mu at the face's nodes, so a kernel writes mu (one state instead of
// 3 Ng M values per element) and reads it at its own and its neighbours' face
// nodes as it reads the state.  I_f^T touches the face's nodes only, so a face
// sums Nfp values and adds them to the residual once.
// Measured against the MFMA kernels it replaces at these orders (apl_adjoint.h),
// us: reverse stage, Euler N = 3, K = 131072 210 -> 110; adjoint RHS, both
// kernels and the call, Euler N = 3, K = 131072 215 -> 122, N = 4, K = 80000
// 236 -> 159, 5-variable N = 2, K = 20402 71 -> 39.
#pragma once

#include "apl_adjoint.h"
#include "apl_eo.h"

namespace apl {

// Orders and variable counts whose transposed RHS runs here: q, lh and the
// residual of a lane take 6 Np ceil(M / 2) registers, and above 180 they
// spill (5-variable Euler, N = 4: 315 us on MFMA, 558 here).
constexpr bool adj_eo_order(int N, int M) { return N <= 4 && (N + 1) * (N + 2) / 2 * ((M + 1) / 2) <= 30; }

// sqrt(x) as root() and 1 / (2 sqrt(x)) from the same iteration, for x >= 0
// (0 gives about 2^-500 and 2^499; trace_vjp reports the rest).
__device__ __forceinline__ double root_inv(double x, double &half_inv) {
  x = fmax(x, 0x1p-1000);
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  g = fma(fma(-g, g, x), h, g);
  e = fma(-h, g, 0.5);
  half_inv = fma(h, e, h);
  return g;
}

// The primitives a vector-Jacobian product needs (no floors).
template <int EQN>
struct EulerPoint {
  static constexpr int IE = Vars<EQN>::M - 1;
  double ir, u, v, w, k2, p, H;
  __device__ __forceinline__ EulerPoint(const PhysParams &P, const double *q) {
    ir = recip(q[0]);
    u = q[1] * ir;
    v = q[2] * ir;
    w = IE == 4 ? q[3] * ir : 0.0;
    k2 = u * u + v * v + w * w;
    p = (P.gamma - 1.0) * (q[IE] - 0.5 * q[0] * k2);
    H = (q[IE] + p) * ir;
  }
};

// qb = (dF/dq)^T Fb + (dG/dq)^T Gb at a cubature point (flux_vjp's Euler
// branch with its common factors formed once).
template <int EQN>
__device__ __forceinline__ void point_vjp(const PhysParams &P, const double *q, const double *Fb,
                                          const double *Gb, double *qb) {
  if constexpr (EQN == APL_EQN_EULER5 || EQN == APL_EQN_EULER4) {
    constexpr int IE = Vars<EQN>::M - 1;
    const EulerPoint<EQN> s(P, q);
    const double g1 = P.gamma - 1.0;
    double Sx = Fb[1] * s.u + Fb[2] * s.v, Sy = Gb[1] * s.u + Gb[2] * s.v;
    if constexpr (IE == 4) {
      Sx += Fb[3] * s.w;
      Sy += Gb[3] * s.w;
    }
    const double be = Fb[IE] * s.u + Gb[IE] * s.v;
    const double T = Fb[1] + Gb[2] + be, gT = g1 * T;
    qb[0] = 0.5 * s.k2 * gT - s.u * Sx - s.v * Sy - s.H * be;
    qb[1] = s.u * (Fb[1] - gT) + s.v * Gb[1] + (Fb[0] + Sx + Fb[IE] * s.H);
    qb[2] = s.u * Fb[2] + s.v * (Gb[2] - gT) + (Gb[0] + Sy + Gb[IE] * s.H);
    if constexpr (IE == 4) qb[3] = s.u * Fb[3] + s.v * Gb[3] - s.w * gT;
    qb[IE] = gT + be;
  } else {
#pragma unroll
    for (int c = 0; c < Vars<EQN>::M; ++c) qb[c] = 0.0;
    flux_vjp<EQN>(P, q, Fb, Gb, qb);
  }
}

// (d(nx F + ny G)/dq)^T b at one Euler trace.
template <int EQN>
__device__ __forceinline__ void euler_normal_vjp(double g1, const EulerPoint<EQN> &s, double nx,
                                                 double ny, const double *b, double *qb) {
  constexpr int IE = Vars<EQN>::M - 1;
  const double un = nx * s.u + ny * s.v;
  double S = b[1] * s.u + b[2] * s.v;
  if constexpr (IE == 4) S += b[3] * s.w;
  const double be = b[IE] * un, gT = g1 * (nx * b[1] + ny * b[2] + be);
  const double m = b[0] + S + b[IE] * s.H;
  qb[0] = 0.5 * s.k2 * gT - un * S - s.H * be;
  qb[1] = un * b[1] - s.u * gT + nx * m;
  qb[2] = un * b[2] - s.v * gT + ny * m;
  if constexpr (IE == 4) qb[3] = un * b[3] - s.w * gT;
  qb[IE] = gT + be;
}

// qMb = (dF*/dqM)^T nb and, with_p, qPb = (dF*/dqP)^T nb (num_flux_vjp; the
// speed's derivative goes to the faster trace, qP on a tie).  Returns whether
// a wave speed that enters does not exist (gamma p / rho negative or NaN), or
// has no derivative where that is used (gamma p / rho = 0): num_flux_vjp's
// square roots and quotients are NaN or infinite there, root_inv's are not.
// Compares alone, whose results are scalar masks: NaN and infinity carried
// through the root keep more values live (N = 4, one wave: 84 bytes of scratch
// against 56).
template <int EQN, int FLUX>
__device__ __forceinline__ bool trace_vjp(const PhysParams &P, double nx, double ny, const double *qM,
                                          const double *qP, const double *nb, bool with_p, double *qMb,
                                          double *qPb) {
  constexpr int M = Vars<EQN>::M;
  if constexpr (EQN == APL_EQN_EULER5 || EQN == APL_EQN_EULER4) {
    constexpr int IE = M - 1;
    const double g = P.gamma, g1 = g - 1.0;
    const EulerPoint<EQN> sM(P, qM), sP(P, qP);
    double hs, ha, hsP, haP;
    const double xM = g * sM.p * sM.ir, xP = g * sP.p * sP.ir;
    bool bad = !(xM >= 0.0) || !(xP >= 0.0);
    const bool noneM = !(xM > 0.0), noneP = !(xP > 0.0);
    const double spM = root_inv(sM.k2, hs), aM = root_inv(xM, ha);
    const double spP = root_inv(sP.k2, hsP), aP = root_inv(xP, haP);
    const double cM = spM + aM, cP = spP + aP;
    bad = bad || (cM > cP ? noneM : noneP && with_p);
    double b[M], jn = 0.0;
#pragma unroll
    for (int c = 0; c < M; ++c) {
      b[c] = 0.5 * nb[c];
      jn += (qM[c] - qP[c]) * b[c];
    }
    const double l = fmax(cM, cP);
    // jn dc/dq of one side
    auto speed = [&](const EulerPoint<EQN> &s, double sp, double a, double hsp, double hap, double jw,
                     double *o) {
      const double dap = g * s.ir * hap, dg = dap * g1, d = 2.0 * hsp * s.ir - dg;
      o[0] += jw * (0.5 * s.k2 * dg - (0.5 * a + sp) * s.ir);
      o[1] += jw * (s.u * d);
      o[2] += jw * (s.v * d);
      if constexpr (IE == 4) o[3] += jw * (s.w * d);
      o[IE] += jw * dg;
    };
    euler_normal_vjp<EQN>(g1, sM, nx, ny, b, qMb);
#pragma unroll
    for (int c = 0; c < M; ++c) qMb[c] += l * b[c];
    speed(sM, spM, aM, hs, ha, cM > cP ? jn : 0.0, qMb);
    if (with_p) {
      euler_normal_vjp<EQN>(g1, sP, nx, ny, b, qPb);
#pragma unroll
      for (int c = 0; c < M; ++c) qPb[c] -= l * b[c];
      speed(sP, spP, aP, hsP, haP, cM > cP ? 0.0 : jn, qPb);
    }
    return bad;
  } else {
#pragma unroll
    for (int c = 0; c < M; ++c) qMb[c] = qPb[c] = 0.0;
    num_flux_vjp<EQN, FLUX>(P, nx, ny, qM, qP, nb, qMb, qPb);
    return false;
  }
}

template <int N, int EQN, int W>
struct AdjEoCfg : EoCfg<N, EQN, W> {
  using B = EoCfg<N, EQN, W>;
  static constexpr int LDS = 2 * 32 * B::ESP + B::RED;
};

// Waves per SIMD: the even and odd parts of q and lh and the residual take
// 6 Np MH registers.
template <int N, int EQN, int W>
struct AdjEoWaves {
  static constexpr int value = Order<N>::Np * ((Vars<EQN>::M + 1) / 2) <= 12 && W < 8 ? 3 : 2;
};

// Even and odd parts of the lane's variables of one element in LDS, scaled.
template <int N, int M, int MH, int NE, int NO>
__device__ __forceinline__ void eo_parts(const double *x, const int (&vo)[MH], double sc,
                                         double (&e)[NE][MH], double (&o)[NO][MH]) {
  constexpr EoNodes<N> ND{};
#pragma unroll
  for (int i = 0; i < NE; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) {
      const double p = x[ND.a[i] * M + vo[j]] * sc;
      e[i][j] = p;
      if (i < NO) {
        const double m = x[ND.b[i] * M + vo[j]] * sc;
        e[i][j] = p + m;
        o[i < NO ? i : 0][j] = p - m;
      }
    }
}

// mu = V V^T x from the even and odd parts of x to LDS in the state's
// layout (rows i = wave, wave + W, ...).  TV: [NE][NE] even, [NO][NO] odd, then
// [NO] what the symmetry leaves out, of node MID's x.
template <int N, int M, int MH, int W, int NE, int NO>
__device__ __forceinline__ void eo_mass(const cptr_t<double> TV, const double (&e)[NE][MH],
                                        const double (&o)[NO][MH], const int (&vo)[MH], int wave,
                                        int hf, double *out) {
  constexpr EoNodes<N> ND{};
#pragma unroll
  for (int i = 0; i < NE; ++i)
    if (W == 1 || i % W == wave) {
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double me = 0.0, mo = i < NO ? TV[NE * NE + NO * NO + i] * e[EoNodes<N>::MID][j] : 0.0;
#pragma unroll
        for (int k = 0; k < NE; ++k) me += TV[i * NE + k] * e[k][j];
        if (i < NO) {
#pragma unroll
          for (int k = 0; k < NO; ++k) mo += TV[NE * NE + i * NO + k] * o[k][j];
        }
        if (MH * 2 == M || hf * MH + j < M) {
          out[ND.a[i] * M + vo[j]] = me + mo;
          if (i < NO) out[ND.b[i] * M + vo[j]] = me - mo;
        }
      }
    }
}

// mu = V V^T lam / J for every element: what the first transposed RHS of a
// sweep reads at the faces (mode 1: lam = rbar + b qbar).
template <int N, int EQN>
__global__ void __launch_bounds__(64) adj_mu_kernel(AdjArgs a) {
  using C = EoCfg<N, EQN, 1>;
  constexpr int M = C::M, MH = C::MH, NE = C::NE, NO = C::NO, ES = C::ES, ESP = C::ESP;
  __shared__ double L[32 * ESP];
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int el = lane & 31, hf = lane >> 5;
  const int grp = xcd_batch(blockIdx.x, gridDim.x);
  const long e0 = (long)grp * 32;
  const int cnt = (int)min((long)32, (long)a.K - e0);
  const double sc = el < cnt ? a.geom[(e0 + el) * G_WORDS + G_INVJ] : 0.0;
  for (int i = lane; i < cnt * ES; i += 64) {
    const int e = i / ES, w = i - e * ES;
    double v = a.lam[e0 * ES + i];
    if (a.mode == 1) v += a.rk_b * a.qbar[e0 * ES + i];
    L[e * ESP + w] = v;
  }
  for (int i = cnt * ES + lane; i < 32 * ES; i += 64) L[i / ES * ESP + i % ES] = 0.0;
  wave_sync();
  int vo[MH];
#pragma unroll
  for (int j = 0; j < MH; ++j) vo[j] = hf * MH + j < M ? hf * MH + j : M - 1;
  double e[NE][MH], o[NO][MH];
  eo_parts<N, M, MH, NE, NO>(L + el * ESP, vo, sc, e, o);
  wave_sync();
  eo_mass<N, M, MH, 1, NE, NO>((cptr_t<double>)a.TV, e, o, vo, 0, hf, L + el * ES);
  wave_sync();
  for (int i = lane; i < cnt * ES; i += 64) a.sbar[e0 * ES + i] = L[i];
}

// The transposed RHS.  STAGE: the reverse-LSERK4 stage (lam = rbar + b qbar,
// the stage update and the next stage's mu); otherwise out = J^T lam.
template <int N, int EQN, int FLUX, int W, bool STAGE, bool VTX>
__global__ void __launch_bounds__(64 * W, (AdjEoWaves<N, EQN, W>::value))
    adj_eo_kernel(AdjArgs a) {
  using C = AdjEoCfg<N, EQN, W>;
  constexpr int M = C::M, MH = C::MH, Np = C::Np, Nfp = C::Nfp, NE = C::NE, NO = C::NO;
  constexpr int ES = C::ES, ESP = C::ESP, HE = C::HE, HO = C::HO, NFU = C::NFU, NPR = C::NPR;
  constexpr int NT = 64 * W, NV2 = 32 * ES / 2, NIT = (NV2 + NT - 1) / NT;
  constexpr EoNodes<N> ND{};

  const cptr_t<double> TP = (cptr_t<double>)a.TP;     // rows of apl_eo.h
  const cptr_t<double> TX = TP + NPR * C::VW;
  const cptr_t<double> TD = TX + C::NAX * C::XW;      // [NV][2] what the symmetry leaves out of a
                                                      // unit's points, of node MID's weight
  const cptr_t<double> TI = (cptr_t<double>)a.TI;     // [NFU][Nfp] Ie Io, abscissae, weights [NFU]

  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = W == 1 ? lane : (int)threadIdx.x;
  const int el = lane & 31, hf = lane >> 5;
  const int grp = xcd_batch(blockIdx.x, gridDim.x);
  const long e0 = (long)grp * 32, base = e0 * ES;
  const int cnt = (int)min((long)32, (long)a.K - e0);
  const long ge = e0 + (el < cnt ? el : 0);

  extern __shared__ double lds_all[];
  double *QS = lds_all;                     // [32][ESP] states, then the result [32][ES]
  double *LT = lds_all + 32 * ESP;          // [32][ESP] lam, then the next stage's lam
  double *RED = LT + 32 * ESP;              // [W][Np MH][64] partial residuals

  int fb = 0, fe = 0, vb = 0, ve = 0;       // this wave's units
#pragma unroll
  for (int w = 0; w < W; ++w)
    if (wave == w) {
      fb = C::fb(w);
      fe = C::fe(w);
      vb = C::vb(w);
      ve = C::vb(w + 1);
    }
  const int code0 = a.fcode[ge * 3], code1 = a.fcode[ge * 3 + 1], code2 = a.fcode[ge * 3 + 2];
  const double *gk = a.geom + ge * G_WORDS;
  const double jrx = gk[G_JRX], jry = gk[G_JRY], jsx = gk[G_JSX], jsy = gk[G_JSY];
  const double sc = el < cnt ? gk[G_INVJ] : 0.0;   // no weight past the last element

  // 1. the group's states (missing elements repeat the first) and lam (zero)
  {
    const double *qb = a.q + base, *lb = a.lam + base, *kb = a.qbar + base;
    if (cnt == 32) {
      dbl2 buf[NIT], lam[NIT], kv[NIT];
#pragma unroll
      for (int j = 0; j < NIT; ++j) {
        const int idx = tid + NT * j;
        if (NT * (j + 1) <= NV2 || idx < NV2) {
          buf[j] = ((const dbl2 *)qb)[idx];
          lam[j] = ((const dbl2 *)lb)[idx];
          if (STAGE) kv[j] = ((const dbl2 *)kb)[idx];
        }
      }
#pragma unroll
      for (int j = 0; j < NIT; ++j) {
        const int idx = tid + NT * j;
        if (NT * (j + 1) <= NV2 || idx < NV2) {
          if (STAGE) lam[j] = lam[j] + a.rk_b * kv[j];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int i = 2 * idx + k, e = i / ES, w = i - e * ES;
            QS[e * ESP + w] = buf[j][k];
            LT[e * ESP + w] = lam[j][k];
          }
        }
      }
    } else {
      for (int i = tid; i < 32 * ES; i += NT) {
        const int e = i / ES, w = i - e * ES;
        QS[e * ESP + w] = e < cnt ? qb[i] : qb[w];
        double v = 0.0;
        if (e < cnt) v = STAGE ? lb[i] + a.rk_b * kb[i] : lb[i];
        LT[e * ESP + w] = v;
      }
    }
  }
  group_sync<W>();

  int vo[MH];
#pragma unroll
  for (int j = 0; j < MH; ++j) vo[j] = hf * MH + j < M ? hf * MH + j : M - 1;
  const double *qe = QS + el * ESP;
  double Re[NE][MH], Ro[NO][MH];
#pragma unroll
  for (int i = 0; i < NE; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) {
      Re[i][j] = 0.0;
      if (i < NO) Ro[i < NO ? i : 0][j] = 0.0;
    }

  // the neighbour's face nodes of the wave's first face, on their way
  const int f0 = fb / NFU;
  double PN[Nfp][MH];
  if (fb < fe)
    eo_gather<N, M, MH>(a.q, f0 == 0 ? code0 : (f0 == 1 ? code1 : code2), ge, vo, PN);

  // 2. volume
  {
    double Qe[NE][MH], Qo[NO][MH], Le[NE][MH], Lo[NO][MH];
    eo_parts<N, M, MH, NE, NO>(qe, vo, 1.0, Qe, Qo);
    eo_parts<N, M, MH, NE, NO>(LT + el * ESP, vo, sc, Le, Lo);
#pragma unroll 1
    for (int c = vb; c < min(ve, NPR); ++c) {
      const cptr_t<double> tv = TP + c * C::VW;
      double x[MH], y[MH], q[M], rx[MH], ry[MH], sx[MH], sy[MH];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double ev = 0.0, od = 0.0, e1 = 0.0, e2 = 0.0;
        double o1 = TD[2 * c] * Le[EoNodes<N>::MID][j], o2 = TD[2 * c + 1] * Le[EoNodes<N>::MID][j];
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          ev += tv[i] * Qe[i][j];
          e1 += tv[Np + i] * Le[i][j];
          e2 += tv[2 * Np + i] * Le[i][j];
        }
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          od += tv[NE + i] * Qo[i][j];
          o1 += tv[Np + NE + i] * Lo[i][j];
          o2 += tv[2 * Np + NE + i] * Lo[i][j];
        }
        x[j] = ev + od;
        y[j] = ev - od;
        rx[j] = e1 + o1;   // phi_r(c), phi_s(c')
        sy[j] = e1 - o1;
        ry[j] = e2 + o2;   // phi_r(c'), phi_s(c)
        sx[j] = e2 - o2;
      }
      double pr[M], ps[M], Fb[M], Gb[M], qb[M];
      to_point<M, MH>(x, y, q);
      to_point<M, MH>(rx, ry, pr);
      to_point<M, MH>(sx, sy, ps);
#pragma unroll
      for (int v = 0; v < M; ++v) {
        Fb[v] = jrx * pr[v] + jsx * ps[v];
        Gb[v] = jry * pr[v] + jsy * ps[v];
      }
      point_vjp<EQN>(a.ph, q, Fb, Gb, qb);
      to_vars<M, MH>(qb, x, y);
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double ev = x[j] + y[j], od = x[j] - y[j];
#pragma unroll
        for (int i = 0; i < NE; ++i) Re[i][j] += tv[i] * ev;
#pragma unroll
        for (int i = 0; i < NO; ++i) Ro[i][j] += tv[NE + i] * od;
      }
    }
#pragma unroll 1
    for (int c = max(vb, NPR); c < ve; ++c) {
      const cptr_t<double> tx = TX + (c - NPR) * C::XW, ta = tx + 2 * NE;
      double x[MH], y[MH], q[M], rx[MH], ry[MH], sx[MH], sy[MH];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double e1 = 0.0, e2 = 0.0;
        double o1 = TD[2 * c] * Le[EoNodes<N>::MID][j], o2 = TD[2 * c + 1] * Le[EoNodes<N>::MID][j];
        x[j] = y[j] = 0.0;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          x[j] += tx[i] * Qe[i][j];
          y[j] += tx[NE + i] * Qe[i][j];
          e1 += ta[i] * Le[i][j];
          e2 += ta[Np + i] * Le[i][j];
        }
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          o1 += ta[NE + i] * Lo[i][j];
          o2 += ta[Np + NE + i] * Lo[i][j];
        }
        rx[j] = e1 + o1;   // phi_r, phi_s of the first point
        sx[j] = e1 - o1;
        ry[j] = e2 + o2;   // and of the second
        sy[j] = e2 - o2;
      }
      double pr[M], ps[M], Fb[M], Gb[M], qb[M];
      to_point<M, MH>(x, y, q);
      to_point<M, MH>(rx, ry, pr);
      to_point<M, MH>(sx, sy, ps);
#pragma unroll
      for (int v = 0; v < M; ++v) {
        Fb[v] = jrx * pr[v] + jsx * ps[v];
        Gb[v] = jry * pr[v] + jsy * ps[v];
      }
      point_vjp<EQN>(a.ph, q, Fb, Gb, qb);
      to_vars<M, MH>(qb, x, y);
#pragma unroll
      for (int j = 0; j < MH; ++j)
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          Re[i][j] += tx[i] * x[j];
          Re[i][j] += tx[NE + i] * y[j];
        }
    }
  }

  // 3. surface
  unsigned ef = 0;
#pragma unroll 1
  for (int u0 = fb; u0 < fe;) {
    const int f = u0 / NFU, ue = min(fe, (f + 1) * NFU);
    const int code = f == 0 ? code0 : (f == 1 ? code1 : code2);
    const double nx = gk[G_NX + f], ny = gk[G_NY + f], sj = gk[G_SJ + f];
    // the weights' node values: own mu, less the neighbour's (its flux has
    // this trace as exterior state and the opposite normal; the fluxes the
    // adjoint covers are conservative, so one product serves both)
    double ZM[Nfp][MH], PM[Nfp][MH], PP[Nfp][MH];
    {
      double ZP[Nfp][MH];
      const double *mu = a.sbar + ge * ES;
      eo_gather<N, M, MH>(a.sbar, code, ge, vo, ZP);
      const double sn = code >= 0 ? a.geom[(long)(code >> 2) * G_WORDS + G_SJ + (code & 3)] : 0.0;
#pragma unroll
      for (int i = 0; i < Nfp; ++i) {
        const int fm = f == 0 ? eo_fmask(N, 0, i) : (f == 1 ? eo_fmask(N, 1, i) : eo_fmask(N, 2, i));
#pragma unroll
        for (int j = 0; j < MH; ++j) {
          PM[i][j] = qe[fm * M + vo[j]];
          ZM[i][j] = mu[fm * M + vo[j]];
        }
      }
#pragma unroll
      for (int i = 0; i < Nfp; ++i)
#pragma unroll
        for (int j = 0; j < MH; ++j) ZM[i][j] = sn * ZP[i][j] - sj * ZM[i][j];
    }
#pragma unroll
    for (int i = 0; i < HE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double m0 = PM[i][j], m1 = PM[Nfp - 1 - i][j], p0 = PN[i][j], p1 = PN[Nfp - 1 - i][j];
        const double z0 = ZM[i][j], z1 = ZM[Nfp - 1 - i][j];
        PM[i][j] = i < HO ? m0 + m1 : m0;
        PP[i][j] = i < HO ? p0 + p1 : p0;
        ZM[i][j] = i < HO ? z0 + z1 : z0;
        if (i < HO) {
          PM[Nfp - 1 - i][j] = m0 - m1;
          PP[Nfp - 1 - i][j] = p0 - p1;
          ZM[Nfp - 1 - i][j] = z0 - z1;
        }
      }
    if (ue < fe)   // the next face's
      eo_gather<N, M, MH>(a.q, f == 0 ? code1 : code2, ge, vo, PN);
    double S[Nfp][MH];   // the face's node sums, even and odd parts
#pragma unroll
    for (int i = 0; i < Nfp; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) S[i][j] = 0.0;
#pragma unroll 1
    for (int u = u0; u < ue; ++u) {
      const int g = u - f * NFU;
      const cptr_t<double> ti = TI + g * Nfp;
      double xM[MH], yM[MH], xP[MH], yP[MH], xZ[MH], yZ[MH];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double eM = 0.0, oM = 0.0, eP = 0.0, oP = 0.0, eZ = 0.0, oZ = 0.0;
#pragma unroll
        for (int i = 0; i < HE; ++i) {
          eM += ti[i] * PM[i][j];
          eP += ti[i] * PP[i][j];
          eZ += ti[i] * ZM[i][j];
        }
#pragma unroll
        for (int i = 0; i < HO; ++i) {
          oM += ti[HE + i] * PM[Nfp - 1 - i][j];
          oP += ti[HE + i] * PP[Nfp - 1 - i][j];
          oZ += ti[HE + i] * ZM[Nfp - 1 - i][j];
        }
        xM[j] = eM + oM;
        yM[j] = eM - oM;
        xP[j] = eP + oP;
        yP[j] = eP - oP;
        xZ[j] = eZ + oZ;
        yZ[j] = eZ - oZ;
      }
      double qM[M], qP[M], nb[M], qMb[M], qPb[M];
      to_point<M, MH>(xM, yM, qM);
      to_point<M, MH>(xP, yP, qP);
      to_point<M, MH>(xZ, yZ, nb);
      const double gw = TI[NFU * Nfp + NFU + g];
#pragma unroll
      for (int v = 0; v < M; ++v) nb[v] *= gw;
      if (code < 0) {
        const double *vk = a.vert + ge * 6;
        const int va = f, vb2 = f == 2 ? 0 : f + 1;
        const double z = TI[NFU * Nfp + g];
        const double sz = 0.5 * (1.0 + (hf ? -z : z));
        const double xg = vk[2 * va] + sz * (vk[2 * vb2] - vk[2 * va]);
        const double yg = vk[2 * va + 1] + sz * (vk[2 * vb2 + 1] - vk[2 * va + 1]);
        boundary_state<EQN, VTX>(*a.bc, -code - 1, a.t, xg, yg, nx, ny, qM, qP);
      }
      if (trace_vjp<EQN, FLUX>(a.ph, nx, ny, qM, qP, nb, code < 0, qMb, qPb)) ef |= EF_NAN;
      if (code < 0) boundary_vjp<EQN>(*a.bc, -code - 1, nx, ny, qPb, qMb);
      to_vars<M, MH>(qMb, xM, yM);
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double ev = xM[j] + yM[j], od = xM[j] - yM[j];
#pragma unroll
        for (int i = 0; i < HE; ++i) S[i][j] += ti[i] * ev;
#pragma unroll
        for (int i = 0; i < HO; ++i) S[Nfp - 1 - i][j] += ti[HE + i] * od;
      }
    }
    // to the residual's even and odd parts: node value s adds s / 2 to the
    // even part of its pair and +- s / 2 to the odd one
#pragma unroll
    for (int i = 0; i < HO; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double ev = S[i][j], od = S[Nfp - 1 - i][j];
        S[i][j] = ev + od;
        S[Nfp - 1 - i][j] = ev - od;
      }
#pragma unroll
    for (int ff = 0; ff < 3; ++ff)
      if (f == ff) {
#pragma unroll
        for (int i = 0; i < Nfp; ++i) {
          const int nd = eo_fmask(N, ff, i);
#pragma unroll
          for (int k = 0; k < NE; ++k)
#pragma unroll
            for (int j = 0; j < MH; ++j) {
              if (k >= NO && ND.a[k] == nd) Re[k][j] += S[i][j];
              if (k < NO && (ND.a[k] == nd || ND.b[k] == nd)) {
                Re[k][j] += 0.5 * S[i][j];
                Ro[k < NO ? k : 0][j] += (ND.a[k] == nd ? 0.5 : -0.5) * S[i][j];
              }
            }
        }
      }
    u0 = ue;
  }

  // 4. the residual in the state's layout
  if constexpr (W == 1) {
    wave_sync();
    double *o = QS + el * ES;
#pragma unroll
    for (int i = 0; i < NE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j)
        if (MH * 2 == M || hf * MH + j < M) {
          if (i < NO) {
            o[ND.a[i] * M + vo[j]] = Re[i][j] + Ro[i < NO ? i : 0][j];
            o[ND.b[i] * M + vo[j]] = Re[i][j] - Ro[i < NO ? i : 0][j];
          } else {
            o[ND.a[i] * M + vo[j]] = Re[i][j];
          }
        }
    wave_sync();
  } else {
    double *rd = RED + wave * Np * MH * 64 + lane;
#pragma unroll
    for (int i = 0; i < NE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        rd[(i * MH + j) * 64] = Re[i][j];
        if (i < NO) rd[((NE + i) * MH + j) * 64] = Ro[i < NO ? i : 0][j];
      }
    __syncthreads();
    double *o = QS + el * ES;
    const double *rs = RED + lane;
#pragma unroll
    for (int i = 0; i < NE; ++i)
      if (i % W == wave) {
#pragma unroll
        for (int j = 0; j < MH; ++j) {
          double re = 0.0, ro = 0.0;
#pragma unroll
          for (int w = 0; w < W; ++w) {
            re += rs[(w * Np * MH + i * MH + j) * 64];
            if (i < NO) ro += rs[(w * Np * MH + (NE + i) * MH + j) * 64];
          }
          if (MH * 2 == M || hf * MH + j < M) {
            o[ND.a[i] * M + vo[j]] = re + ro;
            if (i < NO) o[ND.b[i] * M + vo[j]] = re - ro;
          }
        }
      }
    __syncthreads();
  }

  // 5. out = J^T lam, or qbar += dt out, rbar = a lam and the next stage's
  // lam' = rbar + b' qbar (left in LT, zero past the last element)
  double *rbar = (double *)a.lam;
  if (cnt == 32) {
    dbl2 kv[NIT];
    if constexpr (STAGE) {
#pragma unroll
      for (int j = 0; j < NIT; ++j) {
        const int idx = tid + NT * j;
        if (NT * (j + 1) <= NV2 || idx < NV2) kv[j] = ((const dbl2 *)(a.qbar + base))[idx];
      }
    }
#pragma unroll
    for (int j = 0; j < NIT; ++j) {
      const int idx = tid + NT * j;
      if (NT * (j + 1) <= NV2 || idx < NV2) {
        const dbl2 v = dbl2{QS[2 * idx], QS[2 * idx + 1]};
        if (v[0] != v[0] || v[1] != v[1]) ef |= EF_NAN;
        if constexpr (!STAGE) {
          ((dbl2 *)(a.out + base))[idx] = v;
        } else {
          dbl2 lam;
          int at[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int i = 2 * idx + k, e = i / ES, w = i - e * ES;
            at[k] = e * ESP + w;
            lam[k] = LT[at[k]];
          }
          const dbl2 qn = kv[j] + a.dt * v, rn = a.rk_a * lam, ln = rn + a.rk_b_next * qn;
          ((dbl2 *)(a.qbar + base))[idx] = qn;
          ((dbl2 *)(rbar + base))[idx] = rn;
          LT[at[0]] = ln[0];
          LT[at[1]] = ln[1];
        }
      }
    }
  } else {
    for (int i = tid; i < cnt * ES; i += NT) {
      const int e = i / ES, w = i - e * ES;
      const double v = QS[i];
      if (v != v) ef |= EF_NAN;
      if constexpr (!STAGE) {
        a.out[base + i] = v;
      } else {
        const double qn = a.qbar[base + i] + a.dt * v, rn = a.rk_a * LT[e * ESP + w];
        a.qbar[base + i] = qn;
        rbar[base + i] = rn;
        LT[e * ESP + w] = rn + a.rk_b_next * qn;
      }
    }
  }
  if constexpr (STAGE) {
    if (a.sbar_out) {
      // the next reverse stage's mu of these elements
      group_sync<W>();
      double e[NE][MH], o[NO][MH];
      eo_parts<N, M, MH, NE, NO>(LT + el * ESP, vo, sc, e, o);
      eo_mass<N, M, MH, W, NE, NO>((cptr_t<double>)a.TV, e, o, vo, wave, hf, QS + el * ES);
      group_sync<W>();
      if (cnt == 32) {
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
          const int idx = tid + NT * j;
          if (NT * (j + 1) <= NV2 || idx < NV2) ((dbl2 *)(a.sbar_out + base))[idx] = dbl2{QS[2 * idx], QS[2 * idx + 1]};
        }
      } else {
        for (int i = tid; i < cnt * ES; i += NT) a.sbar_out[base + i] = QS[i];
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) ef |= __shfl_xor(ef, off);
  if (lane == 0 && ef) atomicOr(a.err, ef);
}

}  // namespace apl
