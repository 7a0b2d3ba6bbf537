// C = beta C + alpha A B^T for large FP64 operands from int8 matrix products:
// every operand row is scaled to integers, the product of the integer matrices
// is formed modulo CRT_N pairwise coprime numbers of at most eight bits on the
// int8 matrix cores (exact in int32), and the Chinese remainder theorem puts
// the residues together (Ozaki, Uchino, Imamura, "Ozaki Scheme II: A
// GEMM-oriented emulation of floating-point matrix multiplication using an
// integer modular technique", arXiv:2504.08009, 2025).
//
// Scaling.  Row i of A becomes rint(a 2^s_i) with a 2-norm of at most 2^58, the
// rows of B likewise, so by Cauchy-Schwarz every element of the integer product
// is below 2^116 in magnitude, and M/2 = 2^116.78 holds it for the fifteen
// largest such moduli.  Norms are at least 2^57 and an element is off by half a
// unit, so an element of the product is off by at most sqrt(k) 2^-57 |a_i| |b_j|
// (about 2^-59 |a_i| |b_j| in earnest) and one rounding at the end.
//
// That is a bound on the rows' norms, where DGEMM's is on the sum of an
// element's own terms: elements below 2^-5 of their row's norm lose bits, and
// where the large elements of two rows hardly meet, the small result keeps fewer
// digits than DGEMM gives it.  So the route serves only products whose operands
// or whose use have errors of the norms' kind themselves, by far larger ones:
//   vectors Inv_L V^T: Inv_L is an inverse.  Largest error of the product over
//     its largest element, 7809 vectors: 1.8e-12, DGEMM 1.2e-11 (its partial sums
//     cancel by 1e4 and round at every step; fourteen moduli would lose against
//     it).  Against vectors of an extended-precision factorization (1936, the
//     scheme modelled) both are off by the same at every magnitude from 1e-3 (a
//     median of 4.7e-14 of the element, DGEMM 3.1e-14) down to 1e-15 (4.7e-10
//     and 4.1e-10), where neither has a digit left.
//   SubtractR M -= L L^T: |L_i|^2 is at most the diagonal integral, the
//     integrals' own scale; the same pivots.
//   XR, which a solve with the metric S follows: Z of 1296 points against
//     extended precision, the same errors at every magnitude (median 3e-8).
// Products of a caller's own operands (Rkab) stay with DGEMM.
//
// Why it pays: fifteen int8 products cost 30 operations per multiply-add, 12.9 fs
// on the padded tiles of the vectors' product (2.33 POP/s) and 11 on XR (2.7),
// where DGEMM takes 28.6 fs at 70 TFLOP/s.  By the cycle counters the clock goes
// down to 1.6 to 1.77 GHz in those launches (1.44 to 1.76 on XR; 2.4 without such
// load) and the matrix cores are busy in 64 and 77 % of the cycles.  An operand
// element moves 31 bytes (read for the norm, read and written as residues), a
// result element 38 (residues written and read, the result), 46 where it is
// added to, all at memory speed, which takes back a part (crt_pays).  (H2O)16,
// 1200 AOs, 7809 vectors of 316,063 pairs: vectors' product 287 -> 165 ms,
// SubtractR 84 -> 62 ms; XR of 1536 points 115 -> 45 ms.
//
// Layout.  Residues of an operand: [modulus][32-row block][32-k block] fragments
// of 1 KB, lane l of v_mfma_i32_32x32x32_i8 holding row l % 32 and the sixteen k
// from 16 (l / 32), so that tiles go global -> LDS by 16-byte DMA in memory
// order and LDS reads are consecutive.  Residues of the result: bytes,
// [modulus][column][row].
#include <cmath>
#include "crt.h"

namespace gi {

typedef int c_i4 __attribute__((ext_vector_type(4)));
typedef int c_i16 __attribute__((ext_vector_type(16)));

constexpr int CRT_N = 15;
constexpr int CRT_BITS = 58;      // norm of a scaled row
constexpr int CRT_T = 256;        // tile rows and columns
constexpr int CRT_KS = 64;        // k per stage
constexpr int CRT_NST = 4;        // stages in LDS
constexpr long long CRT_KMAX = 65536;   // k per product: 127^2 k stays below 2^31 up to 133,000
__device__ __host__ constexpr int crt_mod(int l) {
  constexpr int m[CRT_N] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197};
  return m[l];
}

struct CrtConst {
  float m[CRT_N], inv[CRT_N], c1[CRT_N], c2[CRT_N], c3[CRT_N];   // modulus, 1/m, 2^15, 2^30, 2^45 mod m
  double hi[CRT_N], lo[CRT_N];   // reconstruction weights, hi a multiple of 2^76
  double mhi, mlo, minv;         // M and 1/M
};

static const CrtConst &crt_const_host() {
  static const CrtConst c = [] {
    CrtConst t{};
    typedef unsigned __int128 u128;
    u128 M = 1;
    for (int l = 0; l < CRT_N; ++l) M *= (u128)crt_mod(l);
    auto top = [](u128 v) { return std::ldexp((double)(unsigned long long)(v >> 76), 76); };
    auto bot = [](u128 v) {
      const u128 r = v & ((((u128)1) << 76) - 1);
      return std::ldexp((double)(unsigned long long)(r >> 38), 38) + (double)(unsigned long long)(r & ((1ull << 38) - 1));
    };
    for (int l = 0; l < CRT_N; ++l) {
      const int m = crt_mod(l);
      auto sym = [m](long long v) {   // residue in [-m/2, m/2]
        const int r = (int)(v % m);
        return (float)(2 * r > m ? r - m : r);
      };
      t.m[l] = (float)m;
      t.inv[l] = 1.0f / (float)m;
      t.c1[l] = sym(1LL << 15);
      t.c2[l] = sym(1LL << 30);
      t.c3[l] = sym(1LL << 45);
      const u128 Ml = M / (u128)m;
      const int r = (int)(Ml % (u128)m);
      int y = 1;
      while ((long long)y * r % m != 1) ++y;
      const u128 w = Ml * (u128)y;   // 1 mod m, 0 modulo the others, below M
      t.hi[l] = top(w);
      t.lo[l] = bot(w);
    }
    t.mhi = top(M);
    t.mlo = bot(M);
    t.minv = 1.0 / (t.mhi + t.mlo);
    return t;
  }();
  return c;
}

// ------------------------------------------------------------------ operands
// element (row, k) of an operand; consecutive rows follow each other in memory
struct CrtMat {
  const double *x;
  long long ld;
  __device__ __forceinline__ double at(long long r, long long k) const { return x[r + ld * k]; }
};
// X(g, p) X(g, q) of column k's orbital pair (p, q), halved for p = q, zero for
// padding columns (p < 0)
struct CrtPairs {
  const double *x;
  long long ld;
  const int *pq;
  __device__ __forceinline__ double at(long long r, long long k) const {
    const int p = pq[2 * k], q = pq[2 * k + 1];
    if (p < 0) return 0.0;
    const double v = x[r + ld * p] * x[r + ld * q];
    return p == q ? 0.5 * v : v;
  }
};

// partial sums of squares of rows over CRT_KSUM columns: part[slice rows + row];
// squares that vanish leave a trace (the smallest denormal) of a nonzero element
constexpr int CRT_KSUM = 256;
template <class Src>
__global__ void __launch_bounds__(256) k_crt_sumsq(Src S, long long rows, long long k0, long long kk, double *part) {
  const long long r = blockIdx.x * 256LL + threadIdx.x;
  if (r >= rows) return;
  const long long a = k0 + blockIdx.y * (long long)CRT_KSUM;
  const long long b = a + CRT_KSUM < k0 + kk ? a + CRT_KSUM : k0 + kk;
  double s = 0.0;
  bool nz = false;
#pragma unroll 8
  for (long long k = a; k < b; ++k) {
    const double v = S.at(r, k);
    s += v * v;
    nz |= v != 0.0;
  }
  part[blockIdx.y * rows + r] = s == 0.0 && nz ? 4.9406564584124654e-324 : s;
}

// scale exponents s of the rows: a norm of at most 2^CRT_BITS after scaling;
// *bad is set by a row that cannot be scaled (NaN, infinities, squares out of range)
__global__ void __launch_bounds__(256) k_crt_exps(const double *__restrict__ part, long long rows, int slices,
                                                  int *__restrict__ e, int *__restrict__ bad) {
  const long long r = blockIdx.x * 256LL + threadIdx.x;
  if (r >= rows) return;
  double s = 0.0;
#pragma unroll 8
  for (int k = 0; k < slices; ++k) s += part[k * rows + r];
  int ex = 0;
  if (!(s < 1e300) || (s > 0.0 && s < 1e-250)) {
    *bad = 1;
  } else if (s > 0.0) {
    (void)frexp(sqrt(s) * 1.000001, &ex);   // norm below 2^ex
    ex = CRT_BITS - ex;
  }
  e[r] = ex;
}

// Residues of 64 rows x 64 k per workgroup: a lane takes one row and sixteen k,
// a scaled element goes into four signed digits of fifteen bits (exact floats),
// and each residue is three multiply-adds and the remainder, all exact in FP32
// (|digits . powers| < 2^23).  Rounding to integers by adding 1.5 2^23 leaves
// the residue's two's complement byte in the low byte.
template <class Src>
__global__ void __launch_bounds__(256) k_crt_residues(Src S, long long r0, long long rows, long long k0, long long kk,
                                                      const int *__restrict__ e, long long rpad, long long nkb,
                                                      const CrtConst *__restrict__ K, c_i4 *__restrict__ out) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // rpad and 32 nkb are multiples of 64: the grid fits exactly
  const long long rl = blockIdx.x * 64LL + lane;             // row in the chunk
  const long long kb = blockIdx.y * 4LL + w;                 // half k block: sixteen k from 16 kb
  float d[4][16];
  const bool rok = rl < rows;
  const int ex = rok ? e[r0 + rl] : 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const long long k = 16 * kb + i;
    double y = rok && k < kk ? S.at(r0 + rl, k0 + k) : 0.0;
    y = rint(ldexp(y, ex));
    const double y3 = rint(y * 0x1p-45);
    y = fma(-y3, 0x1p45, y);
    const double y2 = rint(y * 0x1p-30);
    y = fma(-y2, 0x1p30, y);
    const double y1 = rint(y * 0x1p-15);
    y = fma(-y1, 0x1p15, y);
    d[0][i] = (float)y;
    d[1][i] = (float)y1;
    d[2][i] = (float)y2;
    d[3][i] = (float)y3;
  }
  constexpr float MAGIC = 12582912.0f;   // 1.5 2^23
  c_i4 *o = out + ((rl >> 5) * nkb + (kb >> 1)) * 64 + (rl & 31) + 32 * (kb & 1);
  const size_t plane = (size_t)(rpad / 32) * nkb * 64;
#pragma unroll 1
  for (int l = 0; l < CRT_N; ++l) {
    const float m = K->m[l], inv = K->inv[l], c1 = K->c1[l], c2 = K->c2[l], c3 = K->c3[l];
    unsigned b[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float s = fmaf(d[3][i], c3, fmaf(d[2][i], c2, fmaf(d[1][i], c1, d[0][i])));
      const float q = fmaf(s, inv, MAGIC) - MAGIC;
      b[i] = __float_as_uint(fmaf(-q, m, s) + MAGIC);
    }
    c_i4 v;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const unsigned lo = __builtin_amdgcn_perm(b[4 * g + 1], b[4 * g], 0x0c0c0400);
      const unsigned hi = __builtin_amdgcn_perm(b[4 * g + 3], b[4 * g + 2], 0x04000c0c);
      v[g] = (int)(lo | hi);
    }
    o[l * plane] = v;
  }
}

// ------------------------------------------------------------------ products
struct CrtGemm {
  const c_i4 *A, *B;
  signed char *R;           // [modulus][column][row]
  size_t pa, pb, pr;        // elements of a modulus' plane
  int nkb;                  // 32-k blocks (even)
  int nmt, nnt;             // tiles of rows and columns
  long long ldr;            // rows of a column of R
  int tri;                  // rows of A end with their diagonal: row tile t of the chunk needs k < 256 (t + 1)
  int mt0;                  // the chunk's row tiles before the first one held here
};

// Residue products modulo crt_mod(blockIdx.y): 256 x 256 tiles, four waves of
// 128 x 128 (sixteen 32 x 32 accumulators, all of the AGPRs, one wave per SIMD).
// A stage of 64 k is 32 KB, four of them ring in LDS; per stage a wave issues 32
// MFMAs (1024 cycles), 16 LDS reads and its eighth of the copies.  The second
// half's fragments are read before the first half's products, the next stage's
// before the second half's, and the one barrier of a stage stands between, so
// that reads, copies and the barrier pass under products in flight.
//
// Workgroups go to the eight XCDs in turn; each XCD takes its own eighth of the
// larger tile dimension and walks it in groups of four rows (columns) of
// tiles, the largest k first, so that 32 workgroups share operands in its L2.
__global__ void __launch_bounds__(256, 1) k_crt_gemm(CrtGemm G, const CrtConst *__restrict__ K) {
  __shared__ c_i4 st[CRT_NST][32][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8, mod = blockIdx.y;
  int mt, nt;
  if (G.nnt >= G.nmt) {
    const int n0 = (int)((long long)G.nnt * xcd / 8), cnt = (int)((long long)G.nnt * (xcd + 1) / 8) - n0;
    if (slot >= cnt * G.nmt) return;   // whole workgroup, before any barrier
    const int g = slot / (4 * cnt), in = slot - g * 4 * cnt, rows = G.nmt - 4 * g < 4 ? G.nmt - 4 * g : 4;
    mt = G.nmt - 1 - (4 * g + in % rows);
    nt = n0 + in / rows;
  } else {
    const int m0 = (int)((long long)G.nmt * xcd / 8), cnt = (int)((long long)G.nmt * (xcd + 1) / 8) - m0;
    if (slot >= cnt * G.nnt) return;
    const int g = slot / (4 * cnt), in = slot - g * 4 * cnt, cols = G.nnt - 4 * g < 4 ? G.nnt - 4 * g : 4;
    nt = 4 * g + in % cols;
    mt = m0 + cnt - 1 - in / cols;
  }
  const int wm = w & 1, wn = w >> 1;
  int nks = G.nkb / 2;
  const int diag = (G.mt0 + mt + 1) * (CRT_T / CRT_KS);
  if (G.tri && diag < nks) nks = diag;
  // this wave's copies: 32-row blocks 4 w .. 4 w + 3 of the tile's sixteen (A, then B)
  const c_i4 *src[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int blk = 4 * w + q;
    src[q] = (blk < 8 ? G.A + mod * G.pa + ((size_t)(mt * 8 + blk) * G.nkb) * 64
                      : G.B + mod * G.pb + ((size_t)(nt * 8 + blk - 8) * G.nkb) * 64) + lane;
  }
  // copy q of a stage (eight a wave; past the last stage the last one again,
  // into a buffer that is not read)
  auto copy = [&](int s, int q) {
    const int ss = s < nks ? s : nks - 1;
    const c_i4 *p = src[q / 2] + (size_t)ss * 128;
    auto *d = (void __attribute__((address_space(3))) *)(&st[s % CRT_NST][(4 * w + q / 2) * 2][0]);
    if (q & 1) __builtin_amdgcn_global_load_lds((const void *)p, d, 16, 1024, 0);
    else __builtin_amdgcn_global_load_lds((const void *)p, d, 16, 0, 0);
  };
  c_i16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = c_i16{0};
  c_i4 a0[4], b0[4], a1[4], b1[4];
  // read q of eight: b[0], a[0], b[1], ...
  auto read = [&](c_i4 (&a)[4], c_i4 (&b)[4], int s, int kb, int q) {
    if (q & 1) a[q / 2] = st[s % CRT_NST][(4 * wm + q / 2) * 2 + kb][lane];
    else b[q / 2] = st[s % CRT_NST][16 + (4 * wn + q / 2) * 2 + kb][lane];
  };
  auto multiply = [&](const c_i4 (&a)[4], const c_i4 (&b)[4], int t) {
    acc[t / 4][t % 4] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[t / 4], b[t % 4], acc[t / 4][t % 4], 0, 0, 0);
  };
  // s_waitcnt immediates: vmcnt(n), expcnt free, lgkmcnt free (0xf) or 0
  constexpr int V1 = 8 * (CRT_NST - 1), V2 = 8 * (CRT_NST - 2);
#pragma unroll
  for (int s = 0; s < CRT_NST; ++s)
#pragma unroll
    for (int q = 0; q < 8; ++q) copy(s, q);
  __builtin_amdgcn_s_waitcnt(0x0f70 | (V1 & 15) | ((V1 >> 4) << 14));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int q = 0; q < 8; ++q) read(a0, b0, 0, 0, q);
  // One read or copy behind each product: an MFMA holds the matrix core for 32
  // cycles, in which they issue for free; in a group before the products they
  // left it idle half of the time (1.98 -> 2.38 POP/s when it was made).  Scheduling barriers,
  // since the compiler groups them again.
#pragma unroll 1
  for (int s = 0; s < nks; ++s) {
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      multiply(a0, b0, t);
      if (t < 8) read(a1, b1, s, 1, t);
      __builtin_amdgcn_sched_barrier(0);
    }
    // stage s + 1 has landed (eight copies a stage, two younger stages in
    // flight) and, after the barrier, every wave has read all of stage s
    __builtin_amdgcn_s_waitcnt(0x0070 | (V2 & 15) | ((V2 >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      multiply(a1, b1, t);
      if (t < 8) read(a0, b0, s + 1, 0, t);
      else copy(s + CRT_NST, t - 8);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();   // LDS is free for the result tile
  // residues to bytes through LDS ([column][row], rows padded by four bytes), then whole rows of R
  constexpr int LD = CRT_T / 4 + 1;   // dwords
  int *t = (int *)&st[0][0][0];
  // The quotient's low bits stand in the low bits of x / m + 1.5 2^23, and the
  // byte of x - m q needs no others.  Below 2^22 the float of x is exact and
  // the quotient off from rounding by under 0.001 (the limit is 0.0019: m = 255
  // must leave |x - m q| < 128); larger sums, which need a long k, are first
  // brought below 2 m.  Three operations an element, with two integer
  // multiplications and two roundings in their place the ends of the tiles took
  // as long as 18 stages.
  const unsigned m = (unsigned)(int)K->m[mod], nm = 0x1000000u - m;
  const float inv = K->inv[mod];
  constexpr float MAGIC = 12582912.0f, LIM = 4194304.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float f[16], top = 0.0f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        f[e] = (float)acc[i][j][e];
        top = fmaxf(top, fabsf(f[e]));
      }
      if (__any(top >= LIM)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc[i][j][e] -= (int)m * (int)rintf(f[e] * inv);
          f[e] = (float)acc[i][j][e];
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        // lane (c, h) holds rows 8 g + 4 h .. + 3 of column c
        unsigned b[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
          b[v] = (unsigned)acc[i][j][4 * g + v] + __umul24(__float_as_uint(fmaf(f[4 * g + v], inv, MAGIC)), nm);
        const unsigned lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400);
        const unsigned hi = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0c);
        const int col = wn * 128 + 32 * j + (lane & 31), row = wm * 128 + 32 * i + 8 * g + 4 * (lane >> 5);
        t[col * LD + row / 4] = (int)(lo | hi);
      }
    }
  __syncthreads();
  signed char *R = G.R + mod * G.pr + (size_t)nt * CRT_T * G.ldr + (size_t)mt * CRT_T;
#pragma unroll 4
  for (int c = w; c < CRT_T; c += 4) *(int *)(R + (size_t)c * G.ldr + 4 * lane) = t[c * LD + lane];
}

// C(r, c) = beta C + alpha 2^-(ea + eb) x, x the integer in (-M/2, M/2) with the
// stored residues.  Four rows a lane.  The weights' upper parts add up exactly
// (41 bits, residues of 7 and 15 terms), the quotient by M follows from the
// sum, and what is left of the upper part is exact; the lower part is good to
// 2^34, far below the 2^57 of the operands' own rounding.
__global__ void __launch_bounds__(256) k_crt_result(const signed char *__restrict__ R, size_t pr, long long ldr,
                                                    long long m, long long n, const int *__restrict__ ea,
                                                    const int *__restrict__ eb, double alpha, double beta,
                                                    double *__restrict__ C, long long ldc, CrtConst K) {
  const long long r = (blockIdx.x * 64LL + (threadIdx.x & 63)) * 4;
  const long long c = blockIdx.y * 4LL + (threadIdx.x >> 6);
  if (r >= m || c >= n) return;
  const signed char *p = R + c * ldr + r;
  double hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
#pragma unroll
  for (int l = 0; l < CRT_N; ++l) {
    const int v = *(const int *)(p + l * pr);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double x = (double)(signed char)(v >> (8 * i));
      hi[i] = fma(x, K.hi[l], hi[i]);
      lo[i] = fma(x, K.lo[l], lo[i]);
    }
  }
  const int sc = eb[c];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (r + i >= m) break;
    const double q = rint((hi[i] + lo[i]) * K.minv);
    const double x = fma(-q, K.mhi, hi[i]) + fma(-q, K.mlo, lo[i]);
    const double v = alpha * ldexp(x, -(sc + ea[r + i]));
    double *d = C + (r + i) + ldc * c;
    *d = beta == 0.0 ? v : beta * *d + v;
  }
}

// ------------------------------------------------------------------ driver
static long long crt_up(long long x, long long q) { return (x + q - 1) / q * q; }

// Work arrays, kept in the context and grown only, about int8_work_mb of them
struct CrtWork {
  DBuf<c_i4> keep, pass;   // residues of the operand that stays and of a slice of the other
  DBuf<signed char> R;
  DBuf<double> part;
  DBuf<int> ea, eb, bad;
  DBuf<CrtConst> K;
};
static CrtWork &crt_work(Context &C) {
  if (!C.crtw) {
    C.crtw = new CrtWork();
    C.crtw->K.upload(&crt_const_host(), 1, C.stream);   // from memory that stays
  }
  return *C.crtw;
}
void release_crt_work(Context &C) {
  delete C.crtw;
  C.crtw = nullptr;
}

// The int8 route against DGEMM on one MI355X, in femtoseconds: 28.6 a
// multiply-add by DGEMM (70 TFLOP/s), 14 in the tile kernel on its padded tiles
// (now 11 to 13, see above: the line lies on the safe side), 6500 an operand
// element (norm and conversion: 6.4 ps measured on XR), 5000 a result element,
// and 100 us of launches and the flag's way to the host.  By this a square
// product pays from about 2400 on.  `part`: share of the multiply-adds that a
// triangular A needs.
bool crt_pays(long long m, long long n, long long k, double part) {
  if (m < 512 || n < 512 || k < 512) return false;
  const double mac = (double)m * n * k * part, pad = (double)crt_up(m, CRT_T) * crt_up(n, CRT_T) * crt_up(k, CRT_KS) * part;
  return 28.6 * mac > 14.0 * pad + 6500.0 * (double)(m + n) * k + 5000.0 * (double)m * n + 1e11;
}

static int crt_slices(long long kk) {   // partial sums of a row's squares
  return (int)((kk + CRT_KSUM - 1) / CRT_KSUM);
}

template <class Src>
static void crt_exponents(Context &C, CrtWork &W, const Src &S, long long rows, long long k0, long long kk, int *e) {
  const int slices = crt_slices(kk);
  hipLaunchKernelGGL(k_crt_sumsq<Src>, dim3((unsigned)((rows + 255) / 256), (unsigned)slices), dim3(256), 0, C.stream,
                     S, rows, k0, kk, W.part.p);
  hipLaunchKernelGGL(k_crt_exps, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, C.stream, W.part.p, rows, slices,
                     e, W.bad.p);
  GI_HIP(hipGetLastError());
}

template <class Src>
static void crt_residues(Context &C, CrtWork &W, const Src &S, long long r0, long long rows, long long rpad,
                         long long k0, long long kk, const int *e, c_i4 *out) {
  const long long nkb = crt_up(kk, CRT_KS) / 32;
  hipLaunchKernelGGL(k_crt_residues<Src>, dim3((unsigned)(rpad / 64), (unsigned)(nkb / 2)), dim3(256), 0, C.stream, S,
                     r0, rows, k0, kk, e, rpad, nkb, W.K.p, out);
  GI_HIP(hipGetLastError());
}

// false (and C untouched) when a row cannot be scaled, the work arrays cannot
// be had or the option int8_work_mb is 0
template <class SrcA, class SrcB>
static bool crt_product(Context &C, const SrcA &A, const SrcB &B, long long m, long long n, long long k, double alpha,
                        double beta, double *Cd, long long ldc, bool tri) {
  if (C.int8_work_mb <= 0) return false;
  struct Busy {   // the arrays are in use: not to be given back to an allocation that fails
    Context &C;
    explicit Busy(Context &c) : C(c) { ++C.work_busy; }
    ~Busy() { --C.work_busy; }
  } busy(C);
  // The smaller operand's residues stay for a chunk of k, the larger one passes
  // in slices, whole multiples of eight tiles, at least CRT_ROWS rows (a launch
  // that fills the card).  Of the work arrays' bytes a third is for the operand
  // that stays (what is left of k goes to further chunks, each of which adds a
  // pass over the result), a sixth for the slice, four ninths for the residues
  // of the result.
  constexpr long long CRT_ROWS = 2048, CRT_KMIN = 2048;
  constexpr long long CRT_NMAX = 65535LL * 4 / CRT_ROWS * CRT_ROWS;   // columns of a k_crt_result launch
  const long long mp = crt_up(m, CRT_T), np = crt_up(n, CRT_T);
  const bool keep_a = mp <= np;
  const long long small = std::min(mp, np), large = std::max(mp, np), work = C.int8_work_mb << 20;
  const long long kmax = std::min(CRT_KMAX, std::max(CRT_KMIN, work / 3 / (CRT_N * small) / CRT_T * CRT_T));
  const long long nkc = (k + kmax - 1) / kmax;
  // chunks of a triangular A begin with a row tile: the rows before it end
  // before the chunk, those from it on end at the tiles' diagonal again
  const long long kc = crt_up((k + nkc - 1) / nkc, tri && nkc > 1 ? CRT_T : CRT_KS);
  const long long kp = std::min(kc, crt_up(k, CRT_KS));
  long long step = std::min(work / 6 / (CRT_N * kp), work / 9 * 4 / (CRT_N * small)) / CRT_ROWS * CRT_ROWS;
  step = std::min({large, std::max(step, CRT_ROWS), CRT_NMAX});
  if (!keep_a && np > CRT_NMAX) return false;
  CrtWork *Wp;
  try {
    Wp = &crt_work(C);
    Wp->ea.alloc((size_t)(nkc * mp));
    Wp->eb.alloc((size_t)(nkc * np));
    Wp->bad.alloc(1);
    Wp->part.alloc((size_t)crt_slices(kc) * std::max(m, n));
    Wp->keep.alloc((size_t)(small * kp / 16 * CRT_N));
    Wp->pass.alloc((size_t)(step * kp / 16 * CRT_N));
    Wp->R.alloc((size_t)(small * step * CRT_N));
  } catch (const Error &) {
    (void)hipGetLastError();
    release_crt_work(C);
    return false;
  }
  CrtWork &W = *Wp;
  // the scale exponents of all chunks first
  const int zero = 0;
  C.h2d(W.bad.p, &zero, sizeof(zero));
  for (long long c = 0; c < nkc; ++c) {
    const long long k0 = c * kc, kk = std::min(kc, k - k0);
    if (kk <= 0) break;
    crt_exponents(C, W, A, m, k0, kk, W.ea.p + c * mp);
    crt_exponents(C, W, B, n, k0, kk, W.eb.p + c * np);
  }
  int bad = 0;
  C.read(&bad, W.bad.p, sizeof(bad));
  if (bad) return false;
  c_i4 *const bufa = keep_a ? W.keep.p : W.pass.p, *const bufb = keep_a ? W.pass.p : W.keep.p;
  for (long long c = 0; c < nkc; ++c) {
    const long long k0 = c * kc, kk = std::min(kc, k - k0);
    if (kk <= 0) break;
    const int *ea = W.ea.p + c * mp, *eb = W.eb.p + c * np;
    const long long nkb = crt_up(kk, CRT_KS) / 32;
    const long long m0 = tri ? k0 : 0;   // first row with elements in the chunk
    if (m0 >= m) break;
    if (keep_a) crt_residues(C, W, A, m0, m - m0, crt_up(m - m0, CRT_T), k0, kk, ea, bufa);
    else crt_residues(C, W, B, 0, n, np, k0, kk, eb, bufb);
    const long long end = keep_a ? n : m;
    for (long long s0 = keep_a ? 0 : m0; s0 < end; s0 += step) {
      const long long a0 = keep_a ? m0 : s0, am = keep_a ? m - m0 : std::min(step, end - s0);
      const long long b0 = keep_a ? s0 : 0, bn = keep_a ? std::min(step, end - s0) : n;
      const long long amp = crt_up(am, CRT_T), bnp = crt_up(bn, CRT_T);
      if (keep_a) crt_residues(C, W, B, b0, bn, bnp, k0, kk, eb, bufb);
      else crt_residues(C, W, A, a0, am, amp, k0, kk, ea, bufa);
      CrtGemm G{};
      G.A = bufa;
      G.B = bufb;
      G.R = W.R.p;
      G.pa = (size_t)amp / 32 * nkb * 64;
      G.pb = (size_t)bnp / 32 * nkb * 64;
      G.pr = (size_t)amp * bnp;
      G.nkb = (int)nkb;
      G.nmt = (int)(amp / CRT_T);
      G.nnt = (int)(bnp / CRT_T);
      G.ldr = amp;
      G.tri = tri ? 1 : 0;
      G.mt0 = (int)((a0 - m0) / CRT_T);   // slices are whole tiles
      const long long big = std::max(G.nmt, G.nnt), less = std::min(G.nmt, G.nnt);
      hipLaunchKernelGGL(k_crt_gemm, dim3((unsigned)(8 * ((big + 7) / 8) * less), CRT_N), dim3(256), 0, C.stream, G,
                         W.K.p);
      hipLaunchKernelGGL(k_crt_result, dim3((unsigned)((am + 255) / 256), (unsigned)((bn + 3) / 4)), dim3(256), 0,
                         C.stream, W.R.p, G.pr, G.ldr, am, bn, ea + a0, eb + b0, alpha, c == 0 ? beta : 1.0,
                         Cd + a0 + ldc * b0, ldc, crt_const_host());
      GI_HIP(hipGetLastError());
    }
  }
  return true;
}

bool crt_gemm_nt(Context &C, long long m, long long n, long long k, double alpha, const double *A, long long lda,
                 const double *B, long long ldb, double beta, double *Cd, long long ldc, bool tri) {
  return crt_product(C, CrtMat{A, lda}, CrtMat{B, ldb}, m, n, k, alpha, beta, Cd, ldc, tri);
}

bool crt_pairs_nt(Context &C, long long m, long long n, long long k, double alpha, const double *X, long long ldx,
                  const int *pq, const double *B, long long ldb, double beta, double *Cd, long long ldc) {
  return crt_product(C, CrtPairs{X, ldx, pq}, CrtMat{B, ldb}, m, n, k, alpha, beta, Cd, ldc, false);
}

}  // namespace gi
