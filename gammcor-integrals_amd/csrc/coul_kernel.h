// Hermite Coulomb potentials of a density on the primitive pairs of a basis
// (coul.hip), the inner kernel of the Coulomb energy and its gradient:
//   J_h(P) = sum_Q sum_k (-1)^{|k|} R_{h+k}(P - Q) D^Q_k,   |h| <= E,
// for every bra primitive pair P of a class against every ket primitive pair Q
// of a class (order F).
//
// One lane owns one P and keeps J in registers; a wave walks a slice of the Q
// list, whose records are the same for all lanes (scalar loads, an SGPR
// operand of the FMAs).  Nothing is shared between lanes, so the work per
// (P, Q) is the integrals and the contraction and nothing else: the row-sum
// mode of md_kernel did the same sums as one-column matrix products, 32 ket
// pairs a tile, with the R table through LDS and 15 of 16 MFMA columns filled
// by queueing.  Energy, then energy and gradient, of 320 AOs (12,880 pairs,
// 1.66e8 pair products): 411 ms there, 3.5 ms here; 225 AOs with f shells:
// 67.8 ms and 2.4 ms.  Bound by FP64 issue (about 100 instructions a pair at
// L = 2) at the low orders, by registers (one wave a SIMD from L = 8 on) and
// launch tails at the high ones.
//
// The R table of order L = E + F has nherm(L) entries (220 at L = 9), too many
// for registers beside J.  It is walked by planes v = t_z: the z recursion
// gives R^(n)_{00v} for n = 0..L - v, and the x, y recursion of the plane
// (at most (L + 1)(L + 2)/2 entries) runs in place from the top level down;
// every (h, k) with h_z + k_z = v is contracted before the next plane.  The
// operation count is that of the full table.
#pragma once
#include "md_kernel.h"

namespace gi {

constexpr int COUL_HC = 8;   // Hermite rows reduced together
constexpr int COUL_EMAX = 7, COUL_FMAX = 6;   // classes with a kernel: E <= 7, F <= 6

struct CoulKet {
  double x, y, z, q, iq;   // centre, exponent and its reciprocal
};
struct CoulArgs {
  const PrimRec *bra;      // nb primitive pairs of the class
  const CoulKet *ket;      // nk primitive pairs
  const double *dk;        // (-1)^{|k|} D^Q_k, nherm(F) per ket primitive
  double *part;            // J of four slices: part[(workgroup y nherm(E) + h) nb + P]
  int nb, nk, per;         // ket primitives per slice
  double kappa;
  const double *boys;
};

// (t, u) entries of a plane, t + u <= M, in order of t + u
__host__ __device__ constexpr int tri2(int M) { return (M + 1) * (M + 2) / 2; }
__host__ __device__ constexpr int idx2(int t, int u) { return (t + u) * (t + u + 1) / 2 + u; }
__host__ __device__ constexpr int u_of2(int i) {
  int n = 0;
  while (tri2(n) <= i) ++n;
  return i - n * (n + 1) / 2;
}
__host__ __device__ constexpr int t_of2(int i) {
  int n = 0;
  while (tri2(n) <= i) ++n;
  return n - (i - n * (n + 1) / 2);
}
template <int M>
struct PlaneRec {   // R_{tu} = X R_{t-1,u} + (t-1) R_{t-2,u}, or along u at t = 0
  int i1[tri2(M)], i2[tri2(M)], y[tri2(M)], c[tri2(M)];
  constexpr PlaneRec() : i1(), i2(), y(), c() {
    for (int i = 1; i < tri2(M); ++i) {
      const int t = t_of2(i), u = u_of2(i);
      y[i] = t == 0;
      c[i] = (t > 0 ? t : u) - 1;
      i1[i] = t > 0 ? idx2(t - 1, u) : idx2(t, u - 1);
      i2[i] = c[i] > 0 ? (t > 0 ? idx2(t - 2, u) : idx2(t, u - 2)) : 0;
    }
  }
};
template <int EH, int FK>   // orders left in the plane for h and k
struct PlaneSum {
  int s[tri2(FK)][tri2(EH)];
  constexpr PlaneSum() : s() {
    for (int k = 0; k < tri2(FK); ++k)
      for (int h = 0; h < tri2(EH); ++h) s[k][h] = idx2(t_of2(h) + t_of2(k), u_of2(h) + u_of2(k));
  }
};
template <int N, int V>
struct PlaneIdx {   // Hermite index of plane entry i at t_z = V
  int v[tri2(N)];
  constexpr PlaneIdx() : v() {
    for (int i = 0; i < tri2(N); ++i) v[i] = hidx(t_of2(i), u_of2(i), V);
  }
};

// plane R2 of order M from the levels c[0..M], in place
template <int M, int N>
__device__ __forceinline__ void coul_plane(double (&R2)[N], const double *c, double X, double Y) {
  constexpr PlaneRec<M> T{};
  R2[0] = c[M];
#pragma unroll
  for (int n = M - 1; n >= 0; --n) {
#pragma unroll
    for (int i = tri2(M - n) - 1; i >= 1; --i) {
      double r = (T.y[i] ? Y : X) * R2[T.i1[i]];
      if (T.c[i] > 0) r += (double)T.c[i] * R2[T.i2[i]];
      R2[i] = r;
    }
    R2[0] = c[n];
  }
}

template <int E, int F, int V, int VK, int N>
__device__ __forceinline__ void coul_contract(double (&J)[nherm(E)], const double (&R2)[N],
                                              const double *__restrict__ dk) {
  constexpr int VH = V - VK;
  if constexpr (VK <= F && VH >= 0) {
    if constexpr (VH <= E) {
      constexpr PlaneSum<E - VH, F - VK> S{};
      constexpr PlaneIdx<F - VK, VK> K{};
      constexpr PlaneIdx<E - VH, VH> H{};
#pragma unroll
      for (int k = 0; k < tri2(F - VK); ++k) {
        const double d = dk[K.v[k]];
#pragma unroll
        for (int h = 0; h < tri2(E - VH); ++h) J[H.v[h]] += d * R2[S.s[k][h]];
      }
    }
    coul_contract<E, F, V, VK + 1>(J, R2, dk);
  }
}

// planes V..L; za holds level values of t_z = V, zb of t_z = V - 1
template <int E, int F, int V>
__device__ __forceinline__ void coul_planes(double (&J)[nherm(E)], double (&za)[E + F + 1], double (&zb)[E + F + 1],
                                            double X, double Y, double Z, const double *__restrict__ dk) {
  constexpr int L = E + F, M = L - V;
  {
    double R2[tri2(M)];
    coul_plane<M>(R2, za, X, Y);
    coul_contract<E, F, V, 0>(J, R2, dk);
  }
  if constexpr (V < L) {
#pragma unroll
    for (int n = 0; n < M; ++n) {
      double r = Z * za[n + 1];
      if (V > 0) r += (double)V * zb[n + 1];
      zb[n] = r;
    }
    coul_planes<E, F, V + 1>(J, zb, za, X, Y, Z, dk);
  }
}

// F_0..F_M at x, the interpolation of boys_fm with the order's coefficients in
// LDS (20 KB: every lane reads its own interval); square roots and quotients
// through one reciprocal square root
template <int M>
__device__ __forceinline__ void coul_boys(double x, const double *s_tab, double (&f)[M + 1]) {
  constexpr double dx = BOYS_XASYM / (double)BOYS_NINT;
  constexpr double inv_dx = (double)BOYS_NINT / BOYS_XASYM;
  const double em = exp(-x);
  if (x < BOYS_XASYM) {
    int k = (int)(x * inv_dx);
    if (k > BOYS_NINT - 1) k = BOYS_NINT - 1;
    const double *c = s_tab + 5 * k;
    const double y = (2.0 * x - (double)(2 * k + 1) * dx) * inv_dx;
    const double twoy = 2.0 * y;
    const double d5 = c[4];
    const double d4v = twoy * d5 + c[3];
    const double d3 = twoy * d4v - d5 + c[2];
    const double d2 = twoy * d3 - d4v + c[1];
    double v = y * d2 - d3 + 0.5 * c[0];
    f[M] = v;
    const double twox = 2.0 * x;
#pragma unroll
    for (int l = M; l >= 1; --l) {
      v = (twox * v + em) * (1.0 / (double)(2 * l - 1));
      f[l - 1] = v;
    }
  } else {
    const double rs = rsqrt(x), beta = 0.5 * rs * rs;
    double v = 0.886226925452758 * rs;   // sqrt(pi) / 2
    f[0] = v;
#pragma unroll
    for (int l = 1; l <= M; ++l) {
      v = beta * ((double)(2 * l - 1) * v - em);
      f[l] = v;
    }
  }
}

// Grid: x = tiles of 64 bra primitive pairs, y = slices of the ket list / 4
// (one slice per wave; a slice past the list's end adds zeros).
template <int E, int F>
__global__ void __launch_bounds__(256) k_coul_j(CoulArgs A, const CoulKet *__restrict__ ket,
                                                const double *__restrict__ dk) {
  constexpr int L = E + F, NHE = nherm(E), NHF = nherm(F);
  __shared__ double s_tab[5 * BOYS_NINT];
  for (int e = threadIdx.x; e < 5 * BOYS_NINT; e += 256) s_tab[e] = A.boys[5 * BOYS_NINT * L + e];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int slice = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * 4 + (threadIdx.x >> 6)));
  const int b = (int)blockIdx.x * 64 + lane;
  const PrimRec B = A.bra[b < A.nb ? b : A.nb - 1];
  const double ip = 1.0 / B.p;
  double J[NHE];
#pragma unroll
  for (int h = 0; h < NHE; ++h) J[h] = 0.0;
  const int q0 = slice * A.per, q1 = q0 + A.per < A.nk ? q0 + A.per : A.nk;
#pragma unroll 1
  for (int q = q0; q < q1; ++q) {
    const CoulKet K = ket[q];
    const double X = B.px - K.x, Y = B.py - K.y, Z = B.pz - K.z;
    const double pq = B.p * K.q;
    const double rd = rsqrt(B.p + K.q + A.kappa * pq);
    const double alpha = pq * rd * rd;
    double za[L + 1], zb[L + 1];
    coul_boys<L>(alpha * (X * X + Y * Y + Z * Z), s_tab, za);
    const double m2a = -2.0 * alpha;
    double pw = 34.986836655249725 * ip * K.iq * rd;   // 2 pi^(5/2)
#pragma unroll
    for (int n = 0; n <= L; ++n) {
      za[n] *= pw;
      pw *= m2a;
    }
    coul_planes<E, F, 0>(J, za, zb, X, Y, Z, dk + (size_t)q * NHF);
  }
  // the four slices' sums through LDS (over the Boys table), COUL_HC rows at a
  // time: a quarter of the slabs to write and add up
  static_assert(4 * COUL_HC * 64 <= 5 * BOYS_NINT, "reduction rows fit the table's LDS");
  double *const o = A.part + (size_t)blockIdx.y * NHE * A.nb;
#pragma unroll
  for (int h0 = 0; h0 < NHE; h0 += COUL_HC) {
    __syncthreads();
#pragma unroll
    for (int h = 0; h < COUL_HC; ++h)
      if (h0 + h < NHE) s_tab[((threadIdx.x >> 6) * COUL_HC + h) * 64 + lane] = J[h0 + h];
    __syncthreads();
    for (int h = (int)threadIdx.x >> 6; h < COUL_HC; h += 4)
      if (h0 + h < NHE && b < A.nb) {
        const double *r = s_tab + h * 64 + lane;
        o[(size_t)(h0 + h) * A.nb + b] =
            (r[0] + r[COUL_HC * 64]) + (r[2 * COUL_HC * 64] + r[3 * COUL_HC * 64]);
      }
  }
}

}  // namespace gi
