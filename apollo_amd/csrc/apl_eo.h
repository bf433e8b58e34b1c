// apl_eo.h -- the cubature-form RHS in FP64 by the mirror symmetry of the
// reference triangle (gfx950).
//
// The same RHS as rhs_kernel (apl_device.h), Apollo's over-integrated
// cubature form (src/subsolvers/wxnodaldg2dmethod.cc:320-510).  What bounds it
// is FP64 arithmetic: on gfx950 v_mfma_f64 and the FP64 vector ALU share one
// pipe (256 CUs x 8 waves: 4 waves of MFMA beside 4 of FMA take the sum of
// the two times, 952 us against 428 + 592), both at 32 flop per cycle and
// SIMD, so MFMA tiles only add their padding and fewer products is the one
// way to be faster.  The kernel halves the products of the volume term:
//
//   The nodes and the cubature points are symmetric under r <-> s (node a
//   <-> b, point c <-> c'), and A_s[a, c] = A_r[b, c'].  With the even and
//   odd parts qe = q_a + q_b, qo = q_a - q_b of a node pair,
//     q(c), q(c')  = sum Ve qe  +- sum Vo qo,
//     R_a, R_b     = Re +- Ro,   Re = sum_c Ae[., c] (Phi_r(c) + Phi_s(c')),
//                                Ro = sum_c Ao[., c] (Phi_r(c) - Phi_s(c')),
//   Ve = (V[c, a] + V[c, b]) / 2, Vo = (V[c, a] - V[c, b]) / 2, Ae and Ao
//   likewise from A_r: half the products of V_c Q and of A_r Phi_r + A_s Phi_s.
//   Nodes on the axis have no odd part; cubature points on it go two by two.
//
// Two lanes share an element (lane el and el + 32 of a wave of 32 elements):
// each holds half of the variables of Q and R for the products, whose
// operator entries are wave-uniform scalar operands, and evaluates the fluxes
// of one of the two mirrored points with all variables.  v_permlane32_swap
// turns "my variables at both points" into "all variables at my point" and
// back.  That halves the registers of the one-lane-per-element form (apl_valu.h),
// so more waves hide each other's latency and N = 4 fits.  On a face the two
// points are Gauss points g and Ng - 1 - g, whose traces split into even and
// odd parts the same way.
//
// W waves share a group of 32 elements: W = 1 where the mesh fills the card
// (no reduction), more on small meshes, where the waves split the points and
// sum their partial residuals through LDS in a fixed order.
#pragma once

#include "apl_device.h"
#include "apl_valu.h"

namespace apl {

// cubature points on the mirror axis of the rule of order N (checked at
// creation against the rule)
constexpr int eo_axis_points(int N) {
  return N == 1 ? 2 : N == 2 ? 5 : N == 3 ? 6 : N == 4 ? 6 : N == 5 ? 7 : N == 6 ? 7 : N == 7 ? 10 : 11;
}

// The even list: node pairs (a, b) first, then the nodes on the axis.
template <int N>
struct EoNodes {
  static constexpr int Np = Order<N>::Np;
  static constexpr int NX = N / 2 + 1;          // nodes on the axis
  static constexpr int NO = (Np - NX) / 2;      // pairs
  static constexpr int NE = NO + NX;
  static constexpr int MID = NO + (N + 1) / 3;  // the axis node nearest to the centroid
  int a[NE] = {}, b[NE] = {};
  constexpr EoNodes() {
    int k = 0;
    for (int j = 0; j <= N; ++j)
      for (int i = j + 1; i + j <= N; ++i) {
        a[k] = eo_node(N, i, j);
        b[k] = eo_node(N, j, i);
        ++k;
      }
    for (int i = 0; 2 * i <= N; ++i) {
      a[k] = b[k] = eo_node(N, i, i);
      ++k;
    }
  }
};

// Orders and variable counts whose FP64 cubature form runs here (us per stage:
// Euler N = 3, K = 131072 68 against 92 on the vector-ALU kernel's FP64 form that
// this kernel replaced; N = 4, K = 524288 404 against 585 on MFMA).  A lane holds
// the state and the residual of half the variables, and the 8-variable system at
// N = 4 spills 400-530 bytes: 4 LSERK4 steps (20 stages), here / on MFMA, K = 3200
// 752 / 706 us, K = 8192 909 / 727, K = 51200 5205 / 2677.
constexpr bool eo_order(int N, int M) { return N <= 3 || (N == 4 && M <= 5); }

template <int N, int EQN, int W_>
struct EoCfg {
  using O = Order<N>;
  using E = EoNodes<N>;
  static constexpr int W = W_;
  static constexpr int M = Vars<EQN>::M, MH = (M + 1) / 2;   // variables per lane
  static constexpr int Np = O::Np, Nc = O::Nc, Ng = O::Ng, Nfp = O::Nfp;
  static constexpr int NE = E::NE, NO = E::NO;
  static constexpr int ES = Np * M, ESP = ES | 1;            // LDS element stride (odd)
  static constexpr int NAX = (eo_axis_points(N) + 1) / 2;    // axis points, two by two
  static constexpr int NPR = (Nc - eo_axis_points(N)) / 2;   // point pairs
  static constexpr int NV = NPR + NAX;                       // volume units
  static constexpr int NFU = Nfp;                            // face units (Gauss pairs) per face
  static constexpr int VW = 3 * Np, XW = 2 * NE + 2 * Np, FW = 2 * Np;   // table rows
  static constexpr int HE = (Nfp + 1) / 2, HO = Nfp / 2;     // even, odd parts of a face
  // instructions of a unit (estimates that balance the waves of a group)
  static constexpr int CV = 3 * Np * MH + 6 * MH + 16 * M;
  static constexpr int CF = 2 * Nfp * MH + 4 * MH + 24 * M + 2 * Np * MH;
  // face units [fb, fe) of wave w, in the order of the 3 NFU units
  static_assert(W == 1 || W == 4 || W == 8, "the widths that the face units are split for");
  static constexpr int fb(int w) {
    return W == 1 ? 0
         : W == 4 ? (w < 3 ? w : 3) * NFU
                  : (w < 6 ? (w >> 1) * NFU + (w & 1) * ((NFU + 1) / 2) : 3 * NFU);
  }
  static constexpr int fe(int w) { return w + 1 < W ? fb(w + 1) : 3 * NFU; }
  // first volume unit of wave w: each wave's share tops its face units up to
  // the mean cost; what rounding leaves goes to the last wave
  static constexpr int vb(int w) {
    if (w >= W) return NV;
    const int mean = (NV * CV + 3 * NFU * CF) / W;
    int at = 0;
    for (int k = 0; k < w; ++k) {
      const int left = mean - (fe(k) - fb(k)) * CF;
      at += left > 0 ? (left + CV / 2) / CV : 0;
    }
    return at < NV ? at : NV;
  }
  static constexpr bool KEEP = W >= 8;   // the staged states stay in registers
  static constexpr int RED = W > 1 ? W * Np * MH * 64 : 0;   // partial residuals, doubles
  static constexpr int LDS = 32 * ESP + RED + W + (W + 1) / 2;
};

// Waves per SIMD asked of the register allocator: three where 168 registers
// hold a lane's state and residual.  The 5- and 8-variable systems at N = 2 spill
// 64-190 bytes there (4 LSERK4 steps, three / two waves: 5 variables HLL, K =
// 12800 350 / 310 us, K = 131072 1506 / 1341; 8 variables, K = 20000 576 / 411).
template <int N, int EQN, int W>
struct EoWaves {
  static constexpr int value = W < 8 && (N == 1 || (N <= 3 && Vars<EQN>::M <= 4)) ? 3 : 2;
};

// Exchange lanes 32..63 of x with lanes 0..31 of y.
__device__ __forceinline__ void swap_halves(double &x, double &y) {
  const unsigned long long ux = __builtin_bit_cast(unsigned long long, x);
  const unsigned long long uy = __builtin_bit_cast(unsigned long long, y);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ux, (unsigned)uy, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ux >> 32), (unsigned)(uy >> 32), false, false);
  x = __builtin_bit_cast(double, (unsigned long long)lo[0] | ((unsigned long long)hi[0] << 32));
  y = __builtin_bit_cast(double, (unsigned long long)lo[1] | ((unsigned long long)hi[1] << 32));
}

// The lane's variables at two points (x: first, y: second) -> all variables
// at the lane's own point (lanes 0..31: first, 32..63: second).
template <int M, int MH>
__device__ __forceinline__ void to_point(double (&x)[MH], double (&y)[MH], double (&q)[M]) {
#pragma unroll
  for (int j = 0; j < MH; ++j) {
    swap_halves(x[j], y[j]);
    q[j] = x[j];
    if (MH + j < M) q[MH + j] = y[j];
  }
}

// The inverse: all variables at the own point -> the lane's variables at both.
template <int M, int MH>
__device__ __forceinline__ void to_vars(const double (&q)[M], double (&x)[MH], double (&y)[MH]) {
#pragma unroll
  for (int j = 0; j < MH; ++j) {
    x[j] = q[j];
    y[j] = MH + j < M ? q[MH + j] : q[j];
    swap_halves(x[j], y[j]);
  }
}

// The group's result OUT[e*ES + w] (LDS) to memory: rhs (mode 0), the LSERK4
// stage (mode 1) or the SSP combination (mode 2), as write_batch does for 16
// elements.  KEEP: qv holds the group's states as they were staged, and the
// second operand rb was requested then; else both are read here.
template <int ES, int NT, bool KEEP, int EL = 32>
struct EoOut {
  static constexpr int NV2 = EL * ES / 2, NIT = (NV2 + NT - 1) / NT;
  static __device__ __forceinline__ bool second(const RhsArgs &a) {
    return a.mode == 1 ? a.rk_a != 0.0 : (a.mode == 2 && a.z != nullptr);
  }
  static __device__ __forceinline__ void load(const double *p, long base, int tid, dbl2 (&v)[NIT]) {
#pragma unroll
    for (int j = 0; j < NIT; ++j) {
      const int idx = tid + NT * j;
      if (NT * (j + 1) <= NV2 || idx < NV2) v[j] = ((const dbl2 *)(p + base))[idx];
    }
  }
  static __device__ __forceinline__ unsigned write(const RhsArgs &a, const double *OUT, long e0, int cnt,
                                                   int tid, dbl2 (&qv)[NIT], dbl2 (&rb)[NIT]) {
    const long base = e0 * ES;
    unsigned ef = 0;
    if (cnt == EL) {
      const bool two = second(a);
      // one path per mode, so that no select splits the stores
      if (a.mode == 0) {
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
          const int idx = tid + NT * j;
          if (NT * (j + 1) <= NV2 || idx < NV2) {
            const dbl2 v = dbl2{OUT[2 * idx], OUT[2 * idx + 1]};
            if (v[0] != v[0] || v[1] != v[1]) ef |= EF_NAN;
            ((dbl2 *)(a.out + base))[idx] = v;
          }
        }
      } else if (a.mode == 1) {
        dbl2 q1[NIT], r1[NIT];
        if constexpr (!KEEP) {
          if (two) load(a.res, base, tid, r1);
          load(a.q, base, tid, q1);
        }
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
          const int idx = tid + NT * j;
          if (NT * (j + 1) <= NV2 || idx < NV2) {
            const dbl2 v = dbl2{OUT[2 * idx], OUT[2 * idx + 1]};
            if (v[0] != v[0] || v[1] != v[1]) ef |= EF_NAN;
            const dbl2 r = two ? a.rk_a * (KEEP ? rb[j] : r1[j]) + a.dt * v : a.dt * v;
            ((dbl2 *)(a.res + base))[idx] = r;
            ((dbl2 *)(a.out + base))[idx] = (KEEP ? qv[j] : q1[j]) + a.rk_b * r;
          }
        }
      } else {
        dbl2 q1[NIT], r1[NIT];
        if constexpr (!KEEP) {
          if (two) load(a.z, base, tid, r1);
          load(a.q, base, tid, q1);
        }
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
          const int idx = tid + NT * j;
          if (NT * (j + 1) <= NV2 || idx < NV2) {
            const dbl2 v = dbl2{OUT[2 * idx], OUT[2 * idx + 1]};
            if (v[0] != v[0] || v[1] != v[1]) ef |= EF_NAN;
            dbl2 o = a.ca * (KEEP ? qv[j] : q1[j]) + a.cb * v;
            if (two) o = o + a.cz * (KEEP ? rb[j] : r1[j]);
            ((dbl2 *)(a.out + base))[idx] = o;
          }
        }
      }
    } else {
      for (int i = tid; i < cnt * ES; i += NT) {
        const double v = OUT[i];
        if (v != v) ef |= EF_NAN;
        double o = v;
        if (a.mode == 1) {
          const double r = (a.rk_a == 0.0) ? a.dt * v : a.rk_a * a.res[base + i] + a.dt * v;
          a.res[base + i] = r;
          o = a.q[base + i] + a.rk_b * r;
        } else if (a.mode == 2) {
          o = a.ca * a.q[base + i] + a.cb * v;
          if (a.z) o = o + a.cz * a.z[base + i];
        }
        a.out[base + i] = o;
      }
    }
    return ef;
  }
};

// The neighbour's values at face node i of a face with this code (its node
// Fmask[nf][Nfp-1-i]; the element's own on a boundary face, where they are
// not used), the lane's variables.
template <int N, int M, int MH>
__device__ __forceinline__ void eo_gather(const double *q, int code, long ge, const int (&vo)[MH],
                                          double (&P)[N + 1][MH]) {
  const int nf = code >= 0 ? (code & 3) : 0;
  const double *qn = q + (code >= 0 ? (long)(code >> 2) : ge) * (Order<N>::Np * M);
#pragma unroll
  for (int i = 0; i <= N; ++i) {
    const int nn = nf == 0 ? eo_fmask(N, 0, N - i) : (nf == 1 ? eo_fmask(N, 1, N - i) : eo_fmask(N, 2, N - i));
#pragma unroll
    for (int j = 0; j < MH; ++j) P[i][j] = qn[nn * M + vo[j]];
  }
}

template <int W>
__device__ __forceinline__ void group_sync() {
  if constexpr (W == 1) wave_sync();
  else __syncthreads();
}

// VTX: the handle has an isentropic-vortex boundary.
template <int N, int EQN, int FLUX, int W, bool VTX>
__global__ void __launch_bounds__(64 * W, (EoWaves<N, EQN, W>::value))
    rhs_eo_kernel(RhsArgs a) {
  using C = EoCfg<N, EQN, W>;
  constexpr int M = C::M, MH = C::MH, Np = C::Np, Nfp = C::Nfp, NE = C::NE, NO = C::NO;
  constexpr int ES = C::ES, ESP = C::ESP, HE = C::HE, HO = C::HO, NFU = C::NFU, NPR = C::NPR;
  constexpr int NT = 64 * W;
  constexpr EoNodes<N> ND{};

  // operator tables, read with wave-uniform indices (scalar loads)
  const cptr_t<double> TP = (cptr_t<double>)a.A1;     // [NPR][VW]: Ve Vo | Ae Ao (c) | Ae Ao (c')
  const cptr_t<double> TX = TP + NPR * C::VW;         // [NAX][XW]: Ve(c1) Ve(c2) | Ae Ao (c1) | Ae Ao (c2), then
                                                      // [Np]: the first axis point's correction
  const cptr_t<double> TF = (cptr_t<double>)a.A3;     // [3 NFU][FW]: -Le -Lo (g) | -Le -Lo (Ng-1-g)
  const cptr_t<double> TI = (cptr_t<double>)a.A2;     // [NFU][Nfp]: Ie Io (g), then the abscissae [NFU]

  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = W == 1 ? lane : (int)threadIdx.x;
  const int el = lane & 31, hf = lane >> 5;
  const int grp = xcd_batch(blockIdx.x, gridDim.x);
  const long e0 = (long)grp * 32;
  const int cnt = (int)min((long)32, (long)a.K - e0);
  const long ge = e0 + (el < cnt ? el : 0);

  extern __shared__ double lds_all[];
  double *QS = lds_all;                     // [32][ESP] staged states, then the result [32][ES]
  double *RED = lds_all + 32 * ESP;         // [W][Np MH][64] partial residuals
  double *SPD = RED + C::RED;               // [W] speed maxima
  unsigned *EFW = (unsigned *)(SPD + W);    // [W] flags

  // this wave's units
  int fb = 0, fe = 0, vb = 0, ve = 0;
#pragma unroll
  for (int w = 0; w < W; ++w)
    if (wave == w) {
      fb = C::fb(w);
      fe = C::fe(w);
      vb = C::vb(w);
      ve = C::vb(w + 1);
    }
  // element data on its way before the states
  const int code0 = a.fcode[ge * 3], code1 = a.fcode[ge * 3 + 1], code2 = a.fcode[ge * 3 + 2];
  const double *gk = a.geom + ge * G_WORDS;
  const double jrx = gk[G_JRX], jry = gk[G_JRY], jsx = gk[G_JSX], jsy = gk[G_JSY];
  const double invJ = gk[G_INVJ];

  // 1. the group's states (missing elements repeat element 0).  Groups of
  // several waves keep the few values a thread stages for the stage update,
  // and ask for the update's second operand now.
  using Out = EoOut<ES, NT, C::KEEP>;
  constexpr int NV2 = Out::NV2, NIT = Out::NIT;
  dbl2 buf[NIT], rb[NIT];
  {
    const double *qb = a.q + e0 * ES;
    if (cnt == 32) {
      Out::load(a.q, e0 * ES, tid, buf);
      if (C::KEEP && Out::second(a)) Out::load(a.mode == 1 ? a.res : a.z, e0 * ES, tid, rb);
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
      for (int i = tid; i < 32 * ES; i += NT) {
        const int e = i / ES, w = i - e * ES;
        QS[e * ESP + w] = e < cnt ? qb[i] : qb[w];
      }
    }
  }
  group_sync<W>();

  // offsets of the lane's variables within a node (a slot past the last
  // variable repeats it and is never written out)
  int vo[MH];
#pragma unroll
  for (int j = 0; j < MH; ++j) vo[j] = hf * MH + j < M ? hf * MH + j : M - 1;
  const double *qe = QS + el * ESP;

  double Re[NE][MH], Ro[NO][MH];
#pragma unroll
  for (int i = 0; i < NE; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) Re[i][j] = 0.0;
#pragma unroll
  for (int i = 0; i < NO; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) Ro[i][j] = 0.0;
  double lmax = 0.0;
  unsigned ef = 0;

  // the neighbour's face nodes of the wave's first face, on their way while
  // the volume runs
  const int f0 = fb / NFU;
  double PN[Nfp][MH];
  if (fb < fe)
    eo_gather<N, M, MH>(a.q, f0 == 0 ? code0 : (f0 == 1 ? code1 : code2), ge, vo, PN);

  // 2. volume: the wave's point pairs, then its axis points
  {
    double Qe[NE][MH], Qo[NO][MH];
#pragma unroll
    for (int i = 0; i < NO; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double x = qe[ND.a[i] * M + vo[j]], y = qe[ND.b[i] * M + vo[j]];
        Qe[i][j] = x + y;
        Qo[i][j] = x - y;
      }
#pragma unroll
    for (int i = NO; i < NE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) Qe[i][j] = qe[ND.a[i] * M + vo[j]];
#pragma unroll 1
    for (int c = vb; c < min(ve, NPR); ++c) {
      const cptr_t<double> tv = TP + c * C::VW;
      double x[MH], y[MH], q[M];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double ev = 0.0, od = 0.0;
#pragma unroll
        for (int i = 0; i < NE; ++i) ev += tv[i] * Qe[i][j];
#pragma unroll
        for (int i = 0; i < NO; ++i) od += tv[NE + i] * Qo[i][j];
        x[j] = ev + od;
        y[j] = ev - od;
      }
      to_point<M, MH>(x, y, q);
      double pr[M], ps[M];
      ef |= point_flux<EQN>(a.ph, jrx, jry, jsx, jsy, q, pr, ps);
      double rx[MH], ry[MH], sx[MH], sy[MH];
      to_vars<M, MH>(pr, rx, ry);
      to_vars<M, MH>(ps, sx, sy);
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double e1 = rx[j] + sy[j], o1 = rx[j] - sy[j];   // point c
        const double e2 = ry[j] + sx[j], o2 = ry[j] - sx[j];   // point c'
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          Re[i][j] += tv[Np + i] * e1;
          Re[i][j] += tv[2 * Np + i] * e2;
        }
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          Ro[i][j] += tv[Np + NE + i] * o1;
          Ro[i][j] += tv[2 * Np + NE + i] * o2;
        }
      }
    }
#pragma unroll 1
    for (int c = max(vb, NPR); c < ve; ++c) {
      const cptr_t<double> tx = TX + (c - NPR) * C::XW;
      double x[MH], y[MH], q[M];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        x[j] = y[j] = 0.0;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          x[j] += tx[i] * Qe[i][j];
          y[j] += tx[NE + i] * Qe[i][j];
        }
      }
      to_point<M, MH>(x, y, q);
      double pr[M], ps[M], pe[M], po[M];
      ef |= point_flux<EQN>(a.ph, jrx, jry, jsx, jsy, q, pr, ps);
#pragma unroll
      for (int v = 0; v < M; ++v) {
        pe[v] = pr[v] + ps[v];
        po[v] = pr[v] - ps[v];
      }
      double e1[MH], e2[MH], o1[MH], o2[MH];
      to_vars<M, MH>(pe, e1, e2);
      to_vars<M, MH>(po, o1, o2);
      const cptr_t<double> ta = tx + 2 * NE;
#pragma unroll
      for (int j = 0; j < MH; ++j) {
#pragma unroll
        for (int i = 0; i < NE; ++i) {
          Re[i][j] += ta[i] * e1[j];
          Re[i][j] += ta[Np + i] * e2[j];
        }
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          Ro[i][j] += ta[NE + i] * o1[j];
          Ro[i][j] += ta[Np + NE + i] * o2[j];
        }
      }
      if (c == NPR) {   // the parts that the mirror symmetry leaves out
        const cptr_t<double> tc = TX + C::NAX * C::XW;
#pragma unroll
        for (int j = 0; j < MH; ++j) {
#pragma unroll
          for (int i = 0; i < NE; ++i) Re[i][j] += tc[i] * o1[j];
#pragma unroll
          for (int i = 0; i < NO; ++i) Ro[i][j] += tc[NE + i] * e1[j];
        }
      }
    }
  }

  // 3. surface: the wave's Gauss pairs, face by face
#pragma unroll 1
  for (int u0 = fb; u0 < fe;) {
    const int f = u0 / NFU, ue = min(fe, (f + 1) * NFU);
    const int code = f == 0 ? code0 : (f == 1 ? code1 : code2);
    const double nx = gk[G_NX + f], ny = gk[G_NY + f], sj = gk[G_SJ + f];
    // own face nodes Fmask[f][i]; even and odd parts: i < HO even, Nfp-1-i
    // odd, the middle node even
    double PM[Nfp][MH], PP[Nfp][MH];
#pragma unroll
    for (int i = 0; i < Nfp; ++i) {
      const int fm = f == 0 ? eo_fmask(N, 0, i) : (f == 1 ? eo_fmask(N, 1, i) : eo_fmask(N, 2, i));
#pragma unroll
      for (int j = 0; j < MH; ++j) PM[i][j] = qe[fm * M + vo[j]];
    }
#pragma unroll
    for (int i = 0; i < HE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        const double m0 = PM[i][j], m1 = PM[Nfp - 1 - i][j], p0 = PN[i][j], p1 = PN[Nfp - 1 - i][j];
        PM[i][j] = i < HO ? m0 + m1 : m0;
        PP[i][j] = i < HO ? p0 + p1 : p0;
        if (i < HO) {
          PM[Nfp - 1 - i][j] = m0 - m1;
          PP[Nfp - 1 - i][j] = p0 - p1;
        }
      }
    if (ue < fe)   // the next face's
      eo_gather<N, M, MH>(a.q, f == 0 ? code1 : code2, ge, vo, PN);
#pragma unroll 1
    for (int u = u0; u < ue; ++u) {
      const int g = u - f * NFU;
      double xM[MH], yM[MH], xP[MH], yP[MH];
#pragma unroll
      for (int j = 0; j < MH; ++j) {
        double eM = 0.0, oM = 0.0, eP = 0.0, oP = 0.0;
#pragma unroll
        for (int i = 0; i < HE; ++i) {
          const double w = TI[g * Nfp + i];
          eM += w * PM[i][j];
          eP += w * PP[i][j];
        }
#pragma unroll
        for (int i = 0; i < HO; ++i) {
          const double w = TI[g * Nfp + HE + i];
          oM += w * PM[Nfp - 1 - i][j];
          oP += w * PP[Nfp - 1 - i][j];
        }
        xM[j] = eM + oM;
        yM[j] = eM - oM;
        xP[j] = eP + oP;
        yP[j] = eP - oP;
      }
      double qM[M], qP[M], fs[M], lam;
      to_point<M, MH>(xM, yM, qM);
      to_point<M, MH>(xP, yP, qP);
      if (code < 0) {
        const double *vk = a.vert + ge * 6;
        const int va = f, vb = f == 2 ? 0 : f + 1;
        const double z = TI[NFU * Nfp + g];
        const double sz = 0.5 * (1.0 + (hf ? -z : z));
        const double xg = vk[2 * va] + sz * (vk[2 * vb] - vk[2 * va]);
        const double yg = vk[2 * va + 1] + sz * (vk[2 * vb + 1] - vk[2 * va + 1]);
        const double tnow = (a.tptr ? *a.tptr : a.t) + a.tofs;
        boundary_state<EQN, VTX>(*a.bc, -code - 1, tnow, xg, yg, nx, ny, qM, qP);
      }
      ef |= num_flux<EQN, FLUX>(a.ph, nx, ny, qM, qP, fs, &lam);
      lmax = fmax(lmax, lam);
#pragma unroll
      for (int v = 0; v < M; ++v) fs[v] *= sj;
      double fx[MH], fy[MH];
      to_vars<M, MH>(fs, fx, fy);
      const cptr_t<double> tf = TF + u * C::FW;
#pragma unroll
      for (int i = 0; i < NE; ++i)
#pragma unroll
        for (int j = 0; j < MH; ++j) {
          Re[i][j] += tf[i] * fx[j];
          Re[i][j] += tf[Np + i] * fy[j];
        }
#pragma unroll
      for (int i = 0; i < NO; ++i)
#pragma unroll
        for (int j = 0; j < MH; ++j) {
          Ro[i][j] += tf[NE + i] * fx[j];
          Ro[i][j] += tf[Np + NE + i] * fy[j];
        }
    }
    u0 = ue;
  }

  // 4. R / J to LDS in the state's layout.  W > 1: every wave leaves its
  // partial residual and sums the pairs i = wave, wave + W, ... of all waves
  // in wave order.
  if constexpr (W == 1) {
    wave_sync();
    double *o = QS + el * ES;
#pragma unroll
    for (int i = 0; i < NE; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j)
        if (MH * 2 == M || hf * MH + j < M) {
          if (i < NO) {
            o[ND.a[i] * M + vo[j]] = (Re[i][j] + Ro[i < NO ? i : 0][j]) * invJ;
            o[ND.b[i] * M + vo[j]] = (Re[i][j] - Ro[i < NO ? i : 0][j]) * invJ;
          } else {
            o[ND.a[i] * M + vo[j]] = Re[i][j] * invJ;
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
            o[ND.a[i] * M + vo[j]] = (re + ro) * invJ;
            if (i < NO) o[ND.b[i] * M + vo[j]] = (re - ro) * invJ;
          }
        }
      }
    __syncthreads();
  }

  // 5. the stage update and the store, then the group's speed and flags
  ef |= Out::write(a, QS, e0, cnt, tid, buf, rb);
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(lmax, off);
    lmax = o > lmax ? o : lmax;
    ef |= __shfl_xor(ef, off);
  }
  if constexpr (W > 1) {
    if (lane == 0) {
      SPD[wave] = lmax;
      EFW[wave] = ef;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
      for (int w = 1; w < W; ++w) {
        lmax = SPD[w] > lmax ? SPD[w] : lmax;
        ef |= EFW[w];
      }
    }
  }
  if (tid == 0) {
    if (a.speed_part) {
      a.speed_part[2 * grp] = lmax;
      if (cnt > 16) a.speed_part[2 * grp + 1] = lmax;
    }
    if (ef) atomicOr(a.err, ef);
  }
}

}  // namespace apl
