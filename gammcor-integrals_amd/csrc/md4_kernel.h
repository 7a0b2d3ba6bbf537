// Hermite-matrix ERI kernel on the 4x4x4 FP64 matrix instruction
// (v_mfma_f64_4x4x4_4b_f64, four independent 4x4x4 blocks per instruction).
//
// Same two products as md_kernel.h,
//   stage 1  X(h, c) = sum_k (-1)^{|k|} R_{h+k} ET_ket(k, c)
//   stage 2  V(r, c) = sum_h ET_bra(h, r) X(h, c),
// (Helgaker, Joergensen, Olsen eqs. 9.9.18-20), organised for thin ket sides:
// one wavefront takes one bra pair and a column tile of four slots, each slot
// four ket columns of one ket pair; block b of every instruction serves
// slot b.  The 4x4x4 instruction's lane layout on gfx950 (measured): lane
// l = 16 q + 4 b + i holds A_b(i, q), B_b(q, i) and D_b(q, i), so the stage-1
// result D = X(h, c) is already the stage-2 B operand and stays in registers.
// Padding is to multiples of four (h, k, rows, columns) instead of sixteen.
//
// R_{tuv} of each quartet is stored densely, R[(t (L+1) + u) (L+1) + v], so
// that the address of R_{h+k} is off(h) + off(k): every stage-1 operand is
// one LDS read at a per-lane offset, no index table.  The R tables of the
// tile's distinct quartets (up to four, fewer for high orders to bound LDS)
// are built together, all lanes over (quartet, entry) per recursion level.
// Contracted pairs: X accumulates over ket primitives in registers; the
// block of a contracted bra accumulates over its primitive pairs in place.
//
// What bounds it: vector instructions (6.2 per matrix instruction over the
// uncontracted (H2O)16 build, 3.6 to 19 by class, and FP64 matrix and vector
// instructions share their units) and the latency of the recursion's levels at
// two to four waves per SIMD; the matrix cores are busy in 15 % of the cycles, 6
// to 22 % by class, and waves wait in 29 % of theirs.  Sum over the
// classes, one after the other: (H2O)12, 900 AOs, uncontracted 35.0 -> 30.2 ms,
// (H2O)5, 375 AOs, contracted 216 -> 135 ms, from the recursion by levels at
// LDS latency (md4_rtable), Boys passes over several primitive steps, and
// stage-1 reads ahead of their instructions.  Tried without gain: records, row
// tables and row groups of all bra pairs of a tile fetched ahead.
#pragma once
#include <type_traits>
#include "md_kernel.h"

namespace gi {

// column tile of a launch: slot s takes columns c0[s] .. c0[s] + 3 of ket
// pair jq[rt[s]] (positions in the launch's ket list); c0 = -1: empty slot
struct ColTile {
  int jq[4];
  int c0[4];
  int rt[4];
  int nq;          // distinct ket pairs jq[0 .. nq-1]
  int pad[3];
};

__host__ __device__ constexpr int m4_dsize(int L) { return (L + 1) * (L + 1) * (L + 1); }
// distinct quartets per tile: their dense R tables within MD4_RBUDGET bytes of LDS
#ifndef MD4_RBUDGET
#define MD4_RBUDGET 9216
#endif
__host__ __device__ constexpr int m4_qmax(int L) {
  return imax(1, imin(4, MD4_RBUDGET / (8 * m4_dsize(L))));
}

#ifndef MD4_ATTR
#define MD4_ATTR
#endif

__device__ __forceinline__ int pick4(const int (&v)[4], int s) {
  return s == 0 ? v[0] : (s == 1 ? v[1] : (s == 2 ? v[2] : v[3]));
}

// a pair record at a uniform address, read into scalar registers
__device__ __forceinline__ QRec load_rec_uniform(const QRec *__restrict__ p) {
  QRec r;
  const int *q = (const int *)p;
  int *o = (int *)&r;
#pragma unroll
  for (int i = 0; i < (int)(sizeof(QRec) / 4); ++i) o[i] = __builtin_amdgcn_readfirstlane(q[i]);
  return r;
}

// 64-bit pointer made provably uniform (scalar registers), so that loads
// through it with a 32-bit lane offset use the scalar-base addressing form
__device__ __forceinline__ const double *uniform_ptr(const double *p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return (const double *)(((unsigned long long)hi << 32) | lo);
}
// raw buffer resource over `bytes` bytes from a uniform base (the gfx9
// descriptor word 3, untyped 32-bit data); loads take a per-lane 32-bit offset
// and a uniform (scalar) offset, and return 0 beyond the range
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const double *ubase, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)ubase, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double buf_ld(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// reads of the R table ahead of the stage-1 instructions
#ifndef MD4_S1D
#define MD4_S1D 8
#endif

// bra pairs per tile (rows of one column tile handled by one wavefront)
#ifndef MD4_NB
#define MD4_NB 4
#endif
constexpr int M4_NB = MD4_NB;

template <int E, int F>
struct Md4 {
  static constexpr int L = E + F, L1 = L + 1;
  static constexpr int NHE = nherm(E), NHF = nherm(F), NHL = nherm(L);
  static constexpr int NHG = (NHE + 3) / 4, KSF = (NHF + 3) / 4;
  static constexpr int DS = m4_dsize(L), QM = m4_qmax(L), NL1 = L >= 1 ? nherm(L - 1) : 1;
  static constexpr int NRMAX = nab_max(E);
};

// Boys function and top recursion level of one quartet (one lane): the
// scaled F_m (2 pi^(5/2) / (p q sqrt(p + q + kappa p q)) (-2 alpha)^m F_m)
// into F[0..L], P - Q into PQ[0..2]
template <int L>
__device__ __forceinline__ void md4_boys(const PrimRec &PB, const PrimRec &PK, double kappa,
                                         const double *__restrict__ boys, double *F, double *PQ) {
  const double PQx = PB.px - PK.px, PQy = PB.py - PK.py, PQz = PB.pz - PK.pz;
  const double pq = PB.p * PK.p;
  const double den = PB.p + PK.p + kappa * pq;
  const double alpha = pq / den;
  const double N = 34.986836655249725 / (pq * sqrt(den));   // 2 pi^(5/2)
  double Fm[L + 1];
  boys_fm<L>(alpha * (PQx * PQx + PQy * PQy + PQz * PQz), boys, Fm);
  const double m2a = -2.0 * alpha;
  double pw = N;
#pragma unroll
  for (int n = 0; n <= L; ++n) {
    F[n] = Fm[n] * pw;
    pw *= m2a;
  }
  PQ[0] = PQx;
  PQ[1] = PQy;
  PQ[2] = PQz;
}

// Orders the LDS accesses of a one-wave workgroup: a wave's LDS instructions
// execute in order, so only the compiler has to keep the order (a workgroup
// barrier would wait for every write to return before the next read).
__device__ __forceinline__ void m4_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

// R table of one quartet by LPQ lanes (sub = 0 .. LPQ - 1), from its scaled
// Boys values F[0..L] and P - Q: the recursion
//   R^(n)_{tuv} = coef R^(n+1)_{i2} + PQ_dir R^(n+1)_{i1},
// levels L-1 .. 1 in the ping-pong tables Ra (odd levels) and Rb (even), level
// 0 into the dense table.  A lane's entries and their codes are the same at
// every level, so they are decoded once, a level's operands are read together,
// and the levels follow each other at LDS latency.  With run-time lane counts,
// codes fetched per entry and a barrier per level the recursion was two thirds
// of the time of the middle orders.  PACKED: level 0 stays packed, in Rb.
template <int L, int LPQ, bool PACKED>
__device__ __forceinline__ void md4_rtable(double *Rd, double *Ra, double *Rb, const double *F, const double *PQ,
                                           const int *s_rrec, const unsigned short *s_dix, int sub, bool act) {
  constexpr int NHL = nherm(L), NJ = (NHL + LPQ - 1) / LPQ;
  m4_fence();   // Boys values written; earlier readers of the tables are ahead in the queue
  if (act) {
    if constexpr (L == 0) {
      if (sub == 0) Rd[0] = F[0];
    } else {
      const double pqx = PQ[0], pqy = PQ[1], pqz = PQ[2];
      // decoded once where few (byte offsets of i1 and i2, coefficient, PQ_dir),
      // at each level from the packed codes where the decoded ones would cost
      // occupancy
      constexpr bool KEEP = NJ <= 8;
      unsigned oo[NJ];
      float cf[NJ];
      double pd[NJ];
      auto decode = [&](int rec, unsigned &o, float &c, double &p) {
        const int dir = (rec >> 22) & 3;
        o = 8u * (rec & 0x7ff) | (8u * ((rec >> 11) & 0x7ff)) << 16;
        c = (float)(rec >> 24);
        p = dir == 0 ? pqx : (dir == 1 ? pqy : pqz);
      };
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int idx = sub + LPQ * j, rec = s_rrec[idx < NHL ? idx : 0];
        if (KEEP) decode(rec, oo[j], cf[j], pd[j]);
        else oo[j] = rec;
      }
      double *const T[2] = {Rb, Ra};   // by level parity
      if (sub == 0) T[L % 2][0] = F[L];
#pragma unroll
      for (int n = L - 1; n >= 0; --n) {
        m4_fence();
        const int cnt = nherm(L - n);
        const double *prv = T[(n + 1) % 2];
        double *cur = T[n % 2];
        const double f = F[n];
        // eight entries of a lane at a time: their reads go out together
#pragma unroll
        for (int j0 = 0; j0 < NJ; j0 += 8) {
          if (LPQ * j0 >= cnt) break;
          double r[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int j = j0 + i;
            if (j < NJ && LPQ * j < cnt) {
              unsigned o = oo[j];
              float c = cf[j];
              double p = pd[j];
              if (!KEEP) {
                int rec = (int)oo[j];
                asm volatile("" : "+v"(rec));   // decoded here, not hoisted
                decode(rec, o, c, p);
              }
              const double p1 = *(const double *)((const char *)prv + (o & 0xffffu));
              const double p2 = *(const double *)((const char *)prv + (o >> 16));
              r[i] = fma((double)c, p2, p * p1);
            }
          }
          if (j0 == 0 && sub == 0) r[0] = f;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int j = j0 + i;
            if (j < NJ && LPQ * j < cnt) {
              if (LPQ * (j + 1) <= cnt || sub + LPQ * j < cnt) {
                if (n == 0 && !PACKED) Rd[s_dix[sub + LPQ * j]] = r[i];
                else cur[sub + LPQ * j] = r[i];
              }
            }
          }
          if (!KEEP) asm volatile("" ::: "memory");
        }
      }
    }
  }
  m4_fence();
}

// PLAIN: every pair of the launch has one primitive pair (uncontracted), so the
// kernel omits the primitive loops
// Waves per SIMD asked of the compiler: two keeps the MFMA accumulators in
// VGPRs (left alone it puts them in AGPRs for most classes, which cost (5,6)
// 21 %, (6,5) and (5,3) 15 %), more where the register count lay a few
// registers above the next step.  Measured per class, (H2O)12 uncontracted and
// (H2O)5 contracted, against the compiler's own choice:
//   uncontracted, three waves: (2,4), (3,3) -15 %, (1,6) -21 %, (2,5), (2,6),
//     (5,2) -6 to -12 %, (4,2..4) -2 to -8 %; four waves for (2,3), (3,2),
//     (3,4), (4,0), (4,1) or three for (0,6), (5,0), (5,1) changed nothing or
//     slowed them;
//   contracted, four waves for (0,3), (1,3), (2,0..2), three for (0,4), (2,3),
//     (2,4), (3,2), (3,4), (4,2), (4,3): 8 to 17 % each; two for (3,1), (4,6),
//     (5,5), (5,6), (6,4), (6,5): 7 to 25 %.  Two slows the others by 2 to 9 %.
// (6,6) spills under either request.
__host__ __device__ constexpr int md4_min_waves(int E, int F, bool plain) {
  if (E == 6 && F == 6) return 1;
  if (plain)
    return ((E == 1 && F == 6) || (E == 2 && F >= 4) || (E == 3 && F == 3) || (E == 4 && F >= 2 && F <= 4) ||
            (E == 5 && F == 2))
               ? 3
               : 2;
  return ((E == 0 && F == 3) || (E == 1 && F == 3) || (E == 2 && F <= 2)) ? 4
         : ((E == 0 && F == 4) || (E == 2 && (F == 3 || F == 4)) || (E == 3 && (F == 2 || F == 4)) ||
            (E == 4 && (F == 2 || F == 3)))
             ? 3
         : ((E == 3 && F == 1) || (E == 4 && F == 6) || (E == 5 && F >= 5) || (E == 6 && F >= 4)) ? 2
                                                                                                  : 1;
}

template <int E, int F, bool PLAIN>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(md4_min_waves(E, F, PLAIN)))) MD4_ATTR
md4_kernel(MdArgs A, const ColTile *__restrict__ ctiles, long long nct, const QRec *__restrict__ rrec) {
  using S = Md4<E, F>;
  constexpr int L = S::L, L1 = S::L1, NHE = S::NHE, NHF = S::NHF, NHL = S::NHL, NHG = S::NHG, KSF = S::KSF;
  constexpr int DS = S::DS, QM = S::QM, NL1 = S::NL1;
  __shared__ double s_Rd[QM][DS];              // level-0 R tables, dense
  __shared__ double s_Rp[2][QM][NL1];          // levels >= 1, packed (ping-pong)
  // quartets whose Boys values are evaluated in one pass, a lane each: the
  // tile's (bra pair, ket pair) quartets, or the primitive quartets of
  // consecutive steps (fewer of them where LDS would cost occupancy)
  constexpr int BL = PLAIN ? M4_NB * QM : (QM == 1 ? 16 : (md4_min_waves(E, F, PLAIN) >= 4 ? 32 : 64));
  __shared__ double s_F[BL][L + 1];            // scaled Boys values per quartet
  __shared__ double s_PQ[BL][4];               // P - Q per quartet
  __shared__ int s_rrec[NHL];
  __shared__ unsigned short s_dix[NHL];        // dense offset of packed index
  __shared__ int s_hoff[NHG * 4];              // dense offset of h (0 for padding)
  __shared__ unsigned s_frow[S::NRMAX + 4];    // byte offset of each bra row's full-block index

  const int lane = threadIdx.x;
  const int lq = lane >> 4, lb = (lane >> 2) & 3, li = lane & 3;
  for (int e = lane; e < NHL; e += 64) {
    s_rrec[e] = c_rrec[e];
    const int th = c_herm[e];
    s_dix[e] = (unsigned short)((px(th) * L1 + py(th)) * L1 + pz(th));
  }
  for (int e = lane; e < NHG * 4; e += 64) {
    int o = 0;
    if (e < NHE) {
      const int th = c_herm[e];
      o = (px(th) * L1 + py(th)) * L1 + pz(th);
    }
    s_hoff[e] = o;
  }
  for (int e = lane; e < QM * DS; e += 64) (&s_Rd[0][0])[e] = 0.0;
  for (int e = lane; e < 2 * QM * NL1; e += 64) (&s_Rp[0][0][0])[e] = 0.0;
  // stage-1 operand offsets of this lane's k = 4 kg + lq and their signs
  int koff[KSF];
  unsigned ksgn = 0;
#pragma unroll
  for (int kg = 0; kg < KSF; ++kg) {
    const int k = 4 * kg + lq;
    koff[kg] = 0;
    if (k < NHF) {
      const int tk = c_herm[k];
      koff[kg] = (px(tk) * L1 + py(tk)) * L1 + pz(tk);
      if ((px(tk) + py(tk) + pz(tk)) & 1) ksgn |= 1u << kg;
    }
  }
  __syncthreads();
  int hoff[NHG];   // dense offset of this lane's h = 4 hg + li
#pragma unroll
  for (int hg = 0; hg < NHG; ++hg) hoff[hg] = s_hoff[4 * hg + li];
  // the last h step pads h beyond NHE (rows h = 4 hg + lq of the stage-2 A operand)
  const bool hlast_ok = 4 * (NHG - 1) + lq < NHE;
  constexpr bool hg_last_mask = (NHE % 4) != 0;

  // XCD-aware order: consecutive tiles (one row block) on one XCD's L2
  const int G = gridDim.x;
  const int w = blockIdx.x;
  const long long v0 = (G % 8 == 0) ? (long long)(w % 8) * (G / 8) + w / 8 : w;
  const long long rs = A.trans ? A.ldo : 1, cs = A.trans ? 1 : A.ldo;
  // row blocks of A.kt (1 .. M4_NB) bra pairs: fewer per tile where a launch
  // has too few tiles to fill the device
  const int nbr = A.kt;
  const long long nrb = (A.nrows + nbr - 1) / nbr;
  const long long ntiles = nrb * nct;

  // R tables of the nq quartets whose Boys values start at f0: 64, 32 or 16
  // lanes per quartet
  auto build_r = [&](int f0, int nq, unsigned actmask) {
    auto build = [&](auto lpq) {
      constexpr int LPQ = decltype(lpq)::value;
      const int ql = lane / LPQ, sub = lane % LPQ, q = ql < QM ? ql : 0;
      md4_rtable<L, LPQ, false>(s_Rd[q], s_Rp[1][q], s_Rp[0][q], s_F[f0 + (ql < nq ? ql : 0)], s_PQ[f0 + (ql < nq ? ql : 0)],
                         s_rrec, s_dix, sub, ql < nq && ((actmask >> ql) & 1u));
    };
    if (QM == 1 || nq == 1) build(std::integral_constant<int, 64>{});
    else if (QM == 2 || nq == 2) build(std::integral_constant<int, 32>{});
    else build(std::integral_constant<int, 16>{});
  };

  for (long long t = v0; t < ntiles; t += G) {
    const long long rb = t / nct, ct = t - rb * nct;
    const long long ir0 = rb * nbr;
    const int nb = (int)((A.nrows - ir0) < nbr ? (A.nrows - ir0) : nbr);
    const ColTile T = ctiles[ct];
    const int nq = T.nq;
    // this lane's slot: ket pair, column (shared by the tile's bra pairs)
    const int myrt = pick4(T.rt, lb);
    const int myc0 = pick4(T.c0, lb);
    const QRec CD = A.crec[pick4(T.jq, myrt)];
    const int c = myc0 + li;
    const bool cval = myc0 >= 0 && c < CD.nrow;
    const int fc = cval ? pair_full(CD, A.sel, c) : 0;
    const int ldk = CD.n0 * CD.n1;

    // stage-1 B operand of ket primitive kp: (-1)^{|k|} ET_ket(k, c).  Every
    // lane loads (index 0 where k or c is outside the table) and scales by
    // +-1 or 0 afterwards: the loads are all in flight together instead of
    // each waiting behind a branch
    double eb[KSF];
    auto load_eb = [&](int kp) {
      // the tables of a pair's primitives follow each other (eri_run), so their
      // addresses need no primitive record
      const bool kval = cval && kp < CD.nprim;
      const int kpc = kp < CD.nprim ? kp : CD.nprim - 1;
      const double *etk = A.et + CD.et + (long long)(kpc * (NHF * ldk));
#pragma unroll
      for (int kg = 0; kg < KSF; ++kg) {
        const int k = 4 * kg + lq;
        const bool ok = kval && k < NHF;
        eb[kg] = etk[ok ? k * ldk + fc : 0];
      }
#pragma unroll
      for (int kg = 0; kg < KSF; ++kg) {
        const bool ok = kval && 4 * kg + lq < NHF;
        eb[kg] *= ok ? (((ksgn >> kg) & 1u) ? -1.0 : 1.0) : 0.0;
      }
    };
    // stage 1: X(h, c) += sum_k R_{h+k} B(k, c) from the dense table of this
    // lane's slot; k step kg updates NHG independent accumulators (the step's
    // offset passes through an empty asm statement so that the NHG addresses
    // are formed in the step instead of all NHG x KSF hoisted into registers).
    // The reads run S1D instructions ahead: left to the compiler every
    // instruction waited for its own read, some 130 cycles in place of 16.
    double X[NHG];
    auto stage1 = [&]() {
      const double *Rq = s_Rd[myrt];
      // (two more places than reads in flight, so that a read does not wait for
      // the instruction that used its place last)
      constexpr int N = KSF * NHG, S1D = imin(MD4_S1D, N), NS = S1D + 2;
      double rv[NS];
      int ko = 0;
      auto rd = [&](int i) {
        if (i % NHG == 0) {
          ko = koff[i / NHG];
          asm volatile("" : "+v"(ko));
        }
        rv[i % NS] = (Rq + ko)[hoff[i % NHG]];
      };
#pragma unroll
      for (int i = 0; i < S1D; ++i) rd(i);
#pragma unroll
      for (int kg = 0; kg < KSF; ++kg)
#pragma unroll
        for (int hg = 0; hg < NHG; ++hg) {
          const int i = kg * NHG + hg;
          __builtin_amdgcn_sched_barrier(0);
          if (i + S1D < N) rd(i + S1D);
          X[hg] = __builtin_amdgcn_mfma_f64_4x4x4f64(rv[i % NS], eb[kg], X[hg], 0, 0, 0);
        }
    };
    // bra rows of RB: byte offset of each row's full-block index
    auto fill_rows = [&](const QRec &RB) {
      for (int r = lane; r < RB.nrow; r += 64) s_frow[r] = 8u * (unsigned)pair_full(RB, A.sel, r);
      if (lane < 4) s_frow[RB.nrow + lane] = 0u;   // padding rows of the last row group
      m4_fence();
    };
    // stage 2 for one bra primitive pair: V(r, c) = sum_h ET_bra(h, r) X(h, c),
    // four bra rows per step (the A operand's row 4 rg + li); the table of h step
    // hg starts at a uniform address, each lane reads at a 32-bit offset.
    // s2_open + load_rows(0) issue the first row group's loads as soon as the
    // bra rows are known, so that they complete under the R recursion and
    // stage 1; each row group then loads the next one while it multiplies.
    __amdgpu_buffer_rsrc_t s2_ub = make_rsrc(uniform_ptr(A.et), 0u);
    unsigned s2_hstep = 0, s2_lrow = 0, s2_lrow_last = 0;
    double ea[NHG];
    auto s2_open = [&](const QRec &RB, const double *etb) {
      const int ldb = RB.n0 * RB.n1;
      s2_ub = make_rsrc(uniform_ptr(etb), 8u * (unsigned)(NHE * ldb));
      s2_hstep = 32u * (unsigned)ldb;   // 4 h rows, bytes
      s2_lrow = 8u * (unsigned)(lq * ldb);
      // the last h step reads row min(h, NHE - 1) (inside the block), masked
      s2_lrow_last = 8u * (unsigned)((imin(4 * (NHG - 1) + lq, NHE - 1) - 4 * (NHG - 1)) * ldb);
    };
    auto load_rows = [&](int rg) {
      const unsigned fro = s_frow[4 * rg + li];
#pragma unroll
      for (int hg = 0; hg < NHG; ++hg) {
        const unsigned o = (hg == NHG - 1 && (NHE % 4) != 0) ? s2_lrow_last + fro : s2_lrow + fro;
        ea[hg] = buf_ld(s2_ub, o, (unsigned)hg * s2_hstep);
      }
    };
    // two accumulator chains (even and odd h steps)
    auto stage2 = [&](const QRec &RB, bool accumulate) {
      const int nr = RB.nrow;
      double *d = A.out + RB.off + CD.off + rs * lq + cs * c;
      const int nrg = (nr + 3) / 4;
      for (int rg = 0; rg < nrg; ++rg) {
        double e[NHG];
#pragma unroll
        for (int hg = 0; hg < NHG; ++hg) e[hg] = ea[hg];
        if (hg_last_mask) e[NHG - 1] = hlast_ok ? e[NHG - 1] : 0.0;
        if (rg + 1 < nrg) load_rows(rg + 1);
        double v0 = 0.0, v1 = 0.0;
#pragma unroll
        for (int hg = 0; hg < NHG; ++hg) {
          if (hg & 1)
            v1 = __builtin_amdgcn_mfma_f64_4x4x4f64(e[hg], X[hg], v1, 0, 0, 0);
          else
            v0 = __builtin_amdgcn_mfma_f64_4x4x4f64(e[hg], X[hg], v0, 0, 0, 0);
        }
        if (cval && 4 * rg + lq < nr) *d = accumulate ? *d + (v0 + v1) : v0 + v1;
        d += 4 * rs;
      }
    };

    if constexpr (PLAIN) {
      // uncontracted tile: one Boys pass for every (bra pair, ket pair)
      // quartet of the tile, then per bra pair the R tables and both stages
      load_eb(0);
      m4_fence();   // earlier readers of s_F / s_PQ are done
      if (lane < nb * nq) {
        const int b = lane / nq, q = lane - b * nq;
        const QRec RB = A.rrec[ir0 + b];
        const QRec CQ = A.crec[pick4(T.jq, q)];
        md4_boys<L>(first_prim(RB), first_prim(CQ), A.kappa, A.boys, s_F[lane], s_PQ[lane]);
      }
      for (int b = 0; b < nb; ++b) {
        const QRec RB = load_rec_uniform(rrec + ir0 + b);
        fill_rows(RB);
        s2_open(RB, A.et + RB.et);
        load_rows(0);
        build_r(b * nq, nq, 0xfu);
#pragma unroll
        for (int hg = 0; hg < NHG; ++hg) X[hg] = 0.0;
        stage1();
        stage2(RB, false);
      }
    } else {
      // contracted pairs: per bra pair and bra primitive pair, X summed over
      // the ket primitive pairs; the block accumulates over bra primitives.
      // Steps (bra pair, bra primitive, ket primitive) are numbered through the
      // tile, and the Boys values of as many steps as there are lanes are
      // evaluated in one pass: it is a chain of some 400 dependent operations,
      // and a pass of at most four steps left most of its lanes idle.
      int npk[4], nprb[M4_NB], maxnp = 1, tot = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        npk[q] = q < nq ? __builtin_amdgcn_readfirstlane(A.crec[T.jq[q]].nprim) : 0;
        maxnp = imax(maxnp, npk[q]);
      }
#pragma unroll
      for (int b = 0; b < M4_NB; ++b) {
        nprb[b] = b < nb ? __builtin_amdgcn_readfirstlane(rrec[ir0 + b].nprim) : 0;
        tot += nprb[b];
      }
      tot *= maxnp;
      const int spc = imin(64, BL) / nq;   // steps per Boys pass
      int step = 0, chunk = -spc;
      for (int b = 0; b < nb; ++b) {
        const QRec RB = load_rec_uniform(rrec + ir0 + b);
        fill_rows(RB);
        for (int bp = 0; bp < RB.nprim; ++bp) {
          s2_open(RB, A.et + RB.et + (long long)(bp * (NHE * RB.n0 * RB.n1)));
          load_rows(0);
#pragma unroll
          for (int hg = 0; hg < NHG; ++hg) X[hg] = 0.0;
          for (int kp = 0; kp < maxnp; ++kp, ++step) {
            if (step >= chunk + spc) {
              chunk = step;
              m4_fence();   // earlier readers of s_F are done
              const int si = lane / nq, q = lane - si * nq;
              int r = step + si;
              if (si < spc && r < tot) {
                int bb = 0;
#pragma unroll
                for (int k = 0; k + 1 < M4_NB; ++k)
                  if (bb == k && r >= nprb[k] * maxnp) {
                    r -= nprb[k] * maxnp;
                    bb = k + 1;
                  }
                const int bpp = r / maxnp, kpp = r - bpp * maxnp;
                const QRec CQ = A.crec[pick4(T.jq, q)];
                if (kpp < CQ.nprim) {
                  const QRec RQ = A.rrec[ir0 + bb];
                  const PrimRec PB = bpp == 0 ? first_prim(RQ) : A.prim[RQ.prim0 + bpp];
                  const PrimRec PK = kpp == 0 ? first_prim(CQ) : A.prim[CQ.prim0 + kpp];
                  md4_boys<L>(PB, PK, A.kappa, A.boys, s_F[lane], s_PQ[lane]);
                }
              }
            }
            unsigned act = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) act |= kp < npk[q] ? 1u << q : 0u;
            load_eb(kp);   // on its way during the recursion
            build_r((step - chunk) * nq, nq, act);
            stage1();
          }
          stage2(RB, bp > 0);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Thin-ket variant: classes whose ket pairs are s-s pairs (F = 0, one Hermite
// function and one column per ket pair).  Stage 1 reduces to
// X(h, c) = R_h(quartet of c) ET_ket(c), a scale instead of a product, so the
// four blocks of an instruction need not share a quartet: a tile is up to
// M4_NB bra pairs x M4S_NK consecutive ket pairs, every column its own quartet, and
// stage 2 (the bra table, shared by all blocks, times X) fills all sixteen
// columns of the instruction.  The R tables are packed (index h, no h + k
// addressing), sixteen per bra pair, four lanes per quartet; even recursion
// levels in one table, odd levels in the other, level 0 last.  The Boys
// values of the tile's quartets stay in the registers of the lane that
// evaluated them and reach the recursion lanes by cross-lane reads.
constexpr int M4S_NK = 16;

// (as the compiler would choose, but without AGPRs and without the decoded
// recursion codes' registers: (6,0) 3.6 -> 2.2 ms and (0,6) 3.2 -> 1.9 ms per
// contracted (H2O)5 build, with four primitive steps per Boys pass)
__host__ __device__ constexpr int md4s_min_waves(int E, bool plain) {
  return E == 6 ? 2 : (E == 5 ? (plain ? 3 : 2) : (E == 4 ? 3 : 4));
}

template <int E, bool PLAIN>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(md4s_min_waves(E, PLAIN)))) MD4_ATTR
md4s_kernel(MdArgs A, const QRec *__restrict__ rrec) {
  constexpr int L = E, NHE = nherm(E), NHG = (NHE + 3) / 4;
  constexpr int NL1 = L >= 1 ? nherm(L - 1) : 1;
  constexpr int SB = NHE | 1, SA = NL1 | 1;   // odd row strides (LDS banks)
  constexpr int NRMAX = nab_max(E);
  __shared__ double s_Rb[M4S_NK * SB];        // even levels, level 0 last
  __shared__ double s_Ra[M4S_NK * SA];        // odd levels
  __shared__ int s_rrec[NHE];
  __shared__ unsigned s_frow[NRMAX + 4];

  const int lane = threadIdx.x;
  const int lq = lane >> 4, li = lane & 3, col = lane & 15;
  for (int e = lane; e < NHE; e += 64) s_rrec[e] = c_rrec[e];
  __syncthreads();
  const bool hlast_ok = 4 * (NHG - 1) + lq < NHE;
  constexpr bool hg_last_mask = (NHE % 4) != 0;

  const int G = gridDim.x;
  const int w = blockIdx.x;
  const long long v0 = (G % 8 == 0) ? (long long)(w % 8) * (G / 8) + w / 8 : w;
  const long long rs = A.trans ? A.ldo : 1;
  const int nbr = A.kt;   // bra pairs per row block, 1 .. M4_NB
  const long long nrb = (A.nrows + nbr - 1) / nbr;
  const long long nct = (A.ncols + M4S_NK - 1) / M4S_NK;
  const long long ntiles = nrb * nct;

  // the Boys values (scaled F_0 .. F_L) and P - Q of this lane's quartet
  double Fq[L + 1], PQq[3];
  auto clear_boys = [&]() {
#pragma unroll
    for (int n = 0; n <= L; ++n) Fq[n] = 0.0;
    PQq[0] = PQq[1] = PQq[2] = 0.0;
  };
  // R tables of the sixteen quartets whose Boys values sit in lanes
  // src0 .. src0 + 15: lanes 4 j .. 4 j + 3 recurse quartet j
  auto build_r = [&](int src0) {
    const int j = lane >> 2, src = src0 + j;
    double F[L + 1], PQ[3];
#pragma unroll
    for (int n = 0; n <= L; ++n) F[n] = __shfl(Fq[n], src);
#pragma unroll
    for (int d = 0; d < 3; ++d) PQ[d] = __shfl(PQq[d], src);
    md4_rtable<L, 4, true>(s_Rb + j * SB, s_Ra + j * SA, s_Rb + j * SB, F, PQ, s_rrec, nullptr, lane & 3, true);
  };
  // stage 1: X(h, c) (+)= R_h ET_ket(c) for this lane's h = 4 hg + lq, c = col
  double X[NHG];
  auto stage1 = [&](double etv, bool add) {
    const double *Rc = s_Rb + col * SB;
#pragma unroll
    for (int hg = 0; hg < NHG; ++hg) {
      const int h = 4 * hg + lq;
      const double v = Rc[h < NHE ? h : NHE - 1] * etv;
      const double xv = (hg == NHG - 1 && hg_last_mask && !hlast_ok) ? 0.0 : v;
      X[hg] = add ? X[hg] + xv : xv;
    }
  };
  auto fill_rows = [&](const QRec &RB) {
    for (int r = lane; r < RB.nrow; r += 64) s_frow[r] = 8u * (unsigned)pair_full(RB, A.sel, r);
    if (lane < 4) s_frow[RB.nrow + lane] = 0u;
    m4_fence();
  };
  // stage 2 as in md4_kernel (first row group loaded ahead): V(r, c) =
  // sum_h ET_bra(h, r) X(h, c), column c of this lane the single column of
  // its ket pair
  __amdgpu_buffer_rsrc_t s2_ub = make_rsrc(uniform_ptr(A.et), 0u);
  unsigned s2_hstep = 0, s2_lrow = 0, s2_lrow_last = 0;
  double ea[NHG];
  auto s2_open = [&](const QRec &RB, const double *etb) {
    const int ldb = RB.n0 * RB.n1;
    s2_ub = make_rsrc(uniform_ptr(etb), 8u * (unsigned)(NHE * ldb));
    s2_hstep = 32u * (unsigned)ldb;
    s2_lrow = 8u * (unsigned)(lq * ldb);
    s2_lrow_last = 8u * (unsigned)((imin(4 * (NHG - 1) + lq, NHE - 1) - 4 * (NHG - 1)) * ldb);
  };
  auto load_rows = [&](int rg) {
    const unsigned fro = s_frow[4 * rg + li];
#pragma unroll
    for (int hg = 0; hg < NHG; ++hg) {
      const unsigned o = (hg == NHG - 1 && (NHE % 4) != 0) ? s2_lrow_last + fro : s2_lrow + fro;
      ea[hg] = buf_ld(s2_ub, o, (unsigned)hg * s2_hstep);
    }
  };
  auto stage2 = [&](const QRec &RB, double *outc, bool cval, bool accumulate) {
    const int nr = RB.nrow;
    double *const out = outc + RB.off;
    const int nrg = (nr + 3) / 4;
    for (int rg = 0; rg < nrg; ++rg) {
      double e[NHG];
#pragma unroll
      for (int hg = 0; hg < NHG; ++hg) e[hg] = ea[hg];
      if (hg_last_mask) e[NHG - 1] = hlast_ok ? e[NHG - 1] : 0.0;
      if (rg + 1 < nrg) load_rows(rg + 1);
      double v0 = 0.0, v1 = 0.0;
#pragma unroll
      for (int hg = 0; hg < NHG; ++hg) {
        if (hg & 1)
          v1 = __builtin_amdgcn_mfma_f64_4x4x4f64(e[hg], X[hg], v1, 0, 0, 0);
        else
          v0 = __builtin_amdgcn_mfma_f64_4x4x4f64(e[hg], X[hg], v0, 0, 0, 0);
      }
      const int ro = 4 * rg + lq;
      if (cval && ro < nr) {
        double *d = out + rs * ro;
        *d = accumulate ? *d + (v0 + v1) : v0 + v1;
      }
    }
  };

  for (long long t = v0; t < ntiles; t += G) {
    const long long rb = t / nct, ct = t - rb * nct;
    const long long ir0 = rb * nbr, jc0 = ct * M4S_NK;
    const int nb = (int)((A.nrows - ir0) < nbr ? (A.nrows - ir0) : nbr);
    const int nk = (int)((A.ncols - jc0) < M4S_NK ? (A.ncols - jc0) : M4S_NK);
    // this lane's column: ket pair jc0 + col, its single orbital pair
    const bool cval = col < nk;
    const QRec CD = A.crec[jc0 + (cval ? col : 0)];
    const int fc = cval ? pair_full(CD, A.sel, 0) : 0;
    double *const outc = A.out + CD.off;

    if constexpr (PLAIN) {
      // one Boys pass for every quartet of the tile: lane 16 b + j takes
      // bra pair b, ket pair j
      {
        const int b = lane >> 4, j = lane & 15;
        clear_boys();
        if (b < nb && j < nk)
          md4_boys<L>(first_prim(A.rrec[ir0 + b]), first_prim(A.crec[jc0 + j]), A.kappa, A.boys, Fq, PQq);
      }
      const double etv = cval ? A.et[CD.et + fc] : 0.0;
      for (int b = 0; b < nb; ++b) {
        const QRec RB = load_rec_uniform(rrec + ir0 + b);
        fill_rows(RB);
        s2_open(RB, A.et + RB.et);
        load_rows(0);
        build_r(16 * b);
        stage1(etv, false);
        stage2(RB, outc, cval, false);
      }
    } else {
      // contracted pairs: per bra pair and bra primitive pair, X summed over
      // the ket primitive pairs.  Steps (bra primitive, ket primitive) of a bra
      // pair are numbered, and one Boys pass serves four of them, lanes
      // 16 s .. 16 s + 15 the sixteen quartets of step s.
      int maxnp = 1;
      for (int j = 0; j < nk; ++j) maxnp = imax(maxnp, A.crec[jc0 + j].nprim);
      maxnp = __builtin_amdgcn_readfirstlane(maxnp);
      for (int b = 0; b < nb; ++b) {
        const QRec RB = load_rec_uniform(rrec + ir0 + b);
        fill_rows(RB);
        int step = 0;
        for (int bp = 0; bp < RB.nprim; ++bp) {
          s2_open(RB, A.et + RB.et + (long long)(bp * (NHE * RB.n0 * RB.n1)));
          load_rows(0);
          for (int kp = 0; kp < maxnp; ++kp, ++step) {
            if ((step & 3) == 0) {
              const int st = step + lq, bpp = st / maxnp, kpp = st - bpp * maxnp;
              clear_boys();
              if (cval && bpp < RB.nprim && kpp < CD.nprim) {
                const PrimRec PB = bpp == 0 ? first_prim(RB) : A.prim[RB.prim0 + bpp];
                const PrimRec PK = kpp == 0 ? first_prim(CD) : A.prim[CD.prim0 + kpp];
                md4_boys<L>(PB, PK, A.kappa, A.boys, Fq, PQq);
              }
            }
            const double etv = cval && kp < CD.nprim ? A.et[CD.et + (long long)(kp * (CD.n0 * CD.n1)) + fc] : 0.0;
            build_r(16 * (step & 3));
            stage1(etv, kp > 0);
          }
          stage2(RB, outc, cval, bp > 0);
        }
      }
    }
  }
}

}  // namespace gi
