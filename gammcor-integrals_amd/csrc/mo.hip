// AO -> MO transform of the Cholesky vectors on the device,
//   Rkab(k, a, b) = sum_{p,q} L^k_{pq} CA(p, a) CB(q, b),
// the operation of chol_gammcor_MOTransf_2 (Cholesky_Gammcor.f90:143-332).
// The reference's first step adds R_k(pq) CA(p,a) into W(:,a,q) and
// R_k(pq) CA(q,a) into W(:,a,p) pair by pair (two dger per orbital pair,
// :215-292).  Here the same sum runs pair-list by pair-list: for every AO q,
// the orbital pairs that contain q (p, column of Rkpq) form a gathered
// product
//   W(k, a, q) = sum_{j in pairs(q)} R(k, col_j) CA(p_j, a)
// on FP64 MFMA (k_mo_half), reading Rkpq in place (no dense L^k), then
//   Rkab(k a, b) = sum_q W(k a, q) CB(q, b)
// is one DGEMM (the reference's second step, dgemv per b, :295-332).
#include <algorithm>
#include <cmath>
#include "gi_context.h"

namespace gi {

#define RB_CHECK(x)                                                                               \
  do {                                                                                           \
    rocblas_status s_ = (x);                                                                     \
    if (s_ != rocblas_status_success)                                                            \
      throw Error{2, std::string("rocBLAS error ") + rocblas_status_to_string(s_) + " at " + __FILE__ + ":" + \
                         std::to_string(__LINE__)};                                              \
  } while (0)

// W(k, a, q) for one AO q (blockIdx.x), 64 vectors from k0 (blockIdx.y) and the
// 4 NAT MO columns from ac (blockIdx.z): one wavefront, FP64 MFMA 4x4x4.  The
// four blocks of an instruction share the A operand (four MO columns of four
// partners p) and take sixteen consecutive vectors of the partners' Rkpq
// columns as B, so a tile pads the MO columns to a multiple of four only (the
// 16x16x4 form padded 40 columns to 64), and 4 NAT independent accumulators per
// wave keep the matrix core busy.  Lane 16 g + 4 b + i holds A_b(i, g),
// B_b(g, i) and D_b(g, i): partner g of the step, MO column i (A) or g (D),
// vector 4 b + i.
//
// Partners come in chunks of MO_JC: while a chunk is multiplied, the Rkpq
// values and MO coefficients of the next one and the list entries of the one
// after it are on their way (32 and 2 NAT registers a lane).  The coefficients
// go through LDS, since the sixteen lanes of a partner need the same ones.
// Consecutive workgroups take all q of one range of vectors: a column is read
// for both of its AOs, and 64 vectors of every column (162 MB at 1200 AOs) stay
// in the last-level cache between the two.
//
// (H2O)16, 7809 vectors, 632,000 list entries: 40 columns 23.2 -> 10.9 ms, 80
// columns 46.5 -> 17.7 ms (16x16x4 tiles without the pipeline before).  At 40
// columns the two reads of Rkpq bound it (39.5 GB, 3.7 TB/s); 32 or 48 vectors
// a wave, which keep more columns cached, took 12.5 and 11.3 ms, and two waves
// of 40 columns for 80 took 20.6 ms.
typedef double mo_d2 __attribute__((ext_vector_type(2)));
constexpr int MO_JC = 16;    // partners per chunk
constexpr int MO_NAT = 20;   // most tiles of four MO columns per wave

template <int NAT>
__global__ void __launch_bounds__(64) k_mo_half(const double *__restrict__ R, long long nvec,
                                                const long long *__restrict__ adj_off,
                                                const long long *__restrict__ adj_col,
                                                const int *__restrict__ adj_p, const double *__restrict__ CT,
                                                int ldct, int nao, long long NA, double *__restrict__ W) {
  constexpr int NC = 4 * NAT;                    // MO columns of the tile
  constexpr int NLD = (MO_JC * NC / 2 + 63) / 64;   // 16-byte coefficient loads per lane and chunk
  __shared__ mo_d2 s_c[2][64 * NLD];
  const int lane = threadIdx.x, v16 = lane & 15, g = lane >> 4, i4 = lane & 3;
  const long long q = blockIdx.x;
  const long long k0 = (long long)blockIdx.y * 64, ac = (long long)blockIdx.z * NC;
  const long long j0 = adj_off[q], j1 = adj_off[q + 1];
  double acc[NAT][4];
#pragma unroll
  for (int at = 0; at < NAT; ++at)
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) acc[at][kt] = 0.0;
  // vectors past the end of a column read the next column (or the 64 doubles
  // behind the last one) and are not stored
  const double *Rk = R + k0 + v16;
  const double *Ca = CT + ac;
  int src[NLD], eo[NLD];   // coefficient load t of a lane: partner and column pair
#pragma unroll
  for (int t = 0; t < NLD; ++t) {
    const int e = lane + 64 * t, j = e / (NC / 2);
    src[t] = j < MO_JC ? j : MO_JC - 1;
    eo[t] = 2 * (e - j * (NC / 2));
  }
  double b[2][MO_JC / 4][4];
  mo_d2 cn[NLD];
  long long col = 0;   // offset of the column of list entry j + v16 (the last entry past the end)
  int po = 0;          // offset of its coefficient row (the zero row past the end)
  auto load_entry = [&](long long j) {
    const long long jj = j + v16;
    const long long je = jj < j1 ? jj : j1 - 1;
    col = nvec * adj_col[je];
    po = ldct * (jj < j1 ? adj_p[je] : nao);
  };
  auto load_values = [&](double (&bn)[MO_JC / 4][4]) {
#pragma unroll
    for (int st = 0; st < MO_JC / 4; ++st) {
      const double *r = Rk + __shfl(col, 4 * st + g);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) bn[st][kt] = r[16 * kt];
    }
#pragma unroll
    for (int t = 0; t < NLD; ++t) cn[t] = *(const mo_d2 *)(Ca + (unsigned)(__shfl(po, src[t]) + eo[t]));
  };
  auto stage = [&](int s) {
#pragma unroll
    for (int t = 0; t < NLD; ++t) s_c[s][lane + 64 * t] = cn[t];
    __syncthreads();
  };
  auto multiply = [&](const double (&bc)[MO_JC / 4][4], int s) {
    const double *sc = (const double *)s_c[s] + g * NC + i4;
#pragma unroll
    for (int st = 0; st < MO_JC / 4; ++st)
#pragma unroll
      for (int at = 0; at < NAT; ++at) {
        const double av = sc[4 * st * NC + 4 * at];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
          acc[at][kt] = __builtin_amdgcn_mfma_f64_4x4x4f64(av, bc[st][kt], acc[at][kt], 0, 0, 0);
      }
    // the next chunk's values are first touched (and waited for) after these
    // products: without the barrier their use moves up between the MFMAs
    __builtin_amdgcn_sched_barrier(0);
  };
  if (j0 < j1) {
    load_entry(j0);
    load_values(b[0]);
    load_entry(j0 + MO_JC);
  }
  // two chunks a turn, on the two halves of the registers and of the LDS; a
  // chunk past the end has zero coefficients
  for (long long j = j0; j < j1; j += 2 * MO_JC) {
    stage(0);
    load_values(b[1]);
    load_entry(j + 2 * MO_JC);
    multiply(b[0], 0);
    stage(1);
    load_values(b[0]);
    load_entry(j + 3 * MO_JC);
    multiply(b[1], 1);
  }
#pragma unroll
  for (int at = 0; at < NAT; ++at) {
    const long long a = ac + 4 * at + g;
    if (a >= NA) continue;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const long long k = k0 + 16 * kt + v16;
      if (k < nvec) W[k + nvec * (a + NA * q)] = acc[at][kt];
    }
  }
}

// tiles of four columns per wave and the number of waves for NA columns: the
// fewest waves (each reads Rkpq), then the smallest instantiated tile
static const int mo_tiles[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 14, 16, 18, MO_NAT};
static int mo_half_tile(long long NA) {
  const long long waves = (NA + 4 * MO_NAT - 1) / (4 * MO_NAT);
  const long long need = ((NA + waves - 1) / waves + 3) / 4;
  for (int t : mo_tiles)
    if (t >= need) return t;
  return MO_NAT;
}

// CT(a, p) = CA(p, a0 + a), zero-padded to ldct rows, and a zero column p = nao
__global__ void k_mo_ct(double *__restrict__ CT, long long ldct, const double *__restrict__ CA, long long lda,
                        long long a0, long long NA, long long nao) {
  const long long a = threadIdx.x + (long long)blockIdx.x * blockDim.x;
  const long long p = blockIdx.y;
  if (a < ldct && p <= nao) CT[a + ldct * p] = a < NA && p < nao ? CA[p + lda * (a0 - 1 + a)] : 0.0;
}

// zero Rkab(:, a, :) for the a columns in `cols`
__global__ void k_zero_acols(double *Rkab, long long nvec, long long na, long long nb, const long long *cols,
                             long long ncols) {
  long long k = threadIdx.x + (long long)blockIdx.x * blockDim.x;
  long long c = blockIdx.y, b = blockIdx.z;
  if (k >= nvec || c >= ncols || b >= nb) return;
  Rkab[k + nvec * (cols[c] + na * b)] = 0.0;
}

void mo_transform(Context &C, const double *dCA, long long lda, long long a0, long long a1, const double *dCB,
                  long long ldb, long long b0, long long b1, long long max_buffer_mb, long long flags,
                  double *dRkab) {
  CholState &S = C.chol;
  if (!S.valid || !S.rkpq.p) throw Error{50, "Cholesky vectors are not available (run gi_chol_build first)"};
  const long long nvec = S.nvecs, nao = C.nao, msd = S.max_subset_dim;
  const long long NA = a1 - a0 + 1, NB = b1 - b0 + 1;
  if (NA <= 0 || NB <= 0 || a0 < 1 || b0 < 1) throw Error{51, "Invalid dimension of Rkab"};
  if (lda < nao || ldb < nao) throw Error{52, "Invalid number of atomic orbitals in CA/CB"};
  // pass structure of the reference (Cholesky_Gammcor.f90:171-185, 190-197)
  long long maxbuf = (max_buffer_mb * 1024 * 1024) / 8;
  long long maxnk = std::min(NA, maxbuf / std::max<long long>(nvec * nao, 1));
  if (!(maxnk > 0)) throw Error{53, "Buffer size too small for Rpq->Rab"};
  std::vector<char> done(NA, 0);
  const long long npasses = NA / maxnk + (NA % maxnk > 0);
  for (long long k = 1; k <= npasses; ++k) {
    long long a0k = (k - 1) * maxnk + a0, a1k = std::min(k * maxnk, a1);
    for (long long a = a0k; a <= a1k; ++a) done[a - a0] = 1;
  }
  // pair lists per AO (cached per Cholesky build): for AO q every BASE
  // orbital pair (p, q) or (q, p) with its Rkpq column (X - 1) msd + position
  if (!S.mo_adj_off.p) {
    std::vector<std::vector<std::pair<int, long long>>> adj(nao);
    for (long long s = 0; s < S.nshell_pairs; ++s) {
      const int A = (int)S.shell_pairs[2 * s] - 1, B = (int)S.shell_pairs[2 * s + 1] - 1;
      const long long X = S.shell_pair_loc[3 * s + 2], pos0 = S.shell_pair_loc[3 * s + 1] - 1;
      const int na = C.shell_nang[A], nb = C.shell_nang[B];
      long long qq = 0;
      for (int b = 0; b < nb; ++b)
        for (int a = (A == B ? b : 0); a < na; ++a) {
          const int p1 = C.shell_loc[A] + a, p2 = C.shell_loc[B] + b;
          const long long col = (X - 1) * msd + pos0 + qq;
          adj[p2].push_back({p1, col});
          if (p1 != p2) adj[p1].push_back({p2, col});
          ++qq;
        }
    }
    std::vector<long long> off(nao + 1, 0), cols;
    std::vector<int> ps;
    for (long long q = 0; q < nao; ++q) {
      off[q + 1] = off[q] + (long long)adj[q].size();
      for (auto &e : adj[q]) {
        ps.push_back(e.first);
        cols.push_back(e.second);
      }
    }
    S.mo_adj_off.upload(off, C.stream);
    S.mo_adj_col.upload(cols, C.stream);
    S.mo_adj_p.upload(ps, C.stream);
  }
  // passes over a-column ranges, W(k, a, q) of at most maxnk columns
  // (the reference's NCholesky*MaxNk*NAO buffer, :186); GI_MO_ALL_COLUMNS
  // takes contiguous ranges covering a0..a1, otherwise the reference's pass
  // bounds (columns they skip stay zero)
  std::vector<std::pair<long long, long long>> passes;
  for (long long k = 1; k <= npasses; ++k) {
    long long a0k, a1k;
    if (flags & 1) {
      a0k = a0 + (k - 1) * maxnk;
      a1k = std::min(a0k + maxnk - 1, a1);
    } else {
      a0k = (k - 1) * maxnk + a0;
      a1k = std::min(k * maxnk, a1);
    }
    if (a1k >= a0k) passes.push_back({a0k, a1k});
  }
  long long nk_max = 0;
  for (auto &pr : passes) nk_max = std::max(nk_max, pr.second - pr.first + 1);
  // leading dimension of CT: whole column tiles of the widest pass
  const long long ldct = (std::max<long long>(nk_max, 1) + 8 * MO_NAT - 1) / (4 * MO_NAT) * (4 * MO_NAT) + 64;
  DBuf<double> dCT, dW;
  dCT.alloc((size_t)ldct * (nao + 1));
  dW.alloc((size_t)nvec * std::max<long long>(nk_max, 1) * nao);
  const double one = 1.0, zero = 0.0;
  for (auto &pr : passes) {
    const long long a0k = pr.first, Nk = pr.second - pr.first + 1;
    hipLaunchKernelGGL(k_mo_ct, dim3((unsigned)((ldct + 63) / 64), (unsigned)(nao + 1)), dim3(64), 0, C.stream, dCT.p, ldct,
                       dCA, lda, a0k, Nk, nao);
    const int nat = mo_half_tile(Nk);
    const dim3 grid((unsigned)nao, (unsigned)((nvec + 63) / 64), (unsigned)((Nk + 4 * nat - 1) / (4 * nat)));
    auto half = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(64), 0, C.stream, S.rkpq.p, nvec, S.mo_adj_off.p, S.mo_adj_col.p,
                         S.mo_adj_p.p, dCT.p, (int)ldct, (int)nao, Nk, dW.p);
    };
    switch (nat) {
      case 1: half(k_mo_half<1>); break;
      case 2: half(k_mo_half<2>); break;
      case 3: half(k_mo_half<3>); break;
      case 4: half(k_mo_half<4>); break;
      case 5: half(k_mo_half<5>); break;
      case 6: half(k_mo_half<6>); break;
      case 8: half(k_mo_half<8>); break;
      case 10: half(k_mo_half<10>); break;
      case 12: half(k_mo_half<12>); break;
      case 14: half(k_mo_half<14>); break;
      case 16: half(k_mo_half<16>); break;
      case 18: half(k_mo_half<18>); break;
      default: half(k_mo_half<MO_NAT>); break;
    }
    GI_HIP(hipGetLastError());
    // Rkab(k, a, b), a in this pass: rows nvec (a0k - a0) .. of each b column
    double *dst = dRkab + nvec * (a0k - a0);
    if (flags & 2)
      split_bf16_gemm(C, rocblas_operation_none, rocblas_operation_none, nvec * Nk, NB, nao, 1.0, dW.p, nvec * Nk,
                      dCB + (b0 - 1) * ldb, ldb, 0.0, dst, nvec * NA);
    else
      RB_CHECK(rocblas_dgemm(C.blas, rocblas_operation_none, rocblas_operation_none, nvec * Nk, NB, nao, &one, dW.p,
                             nvec * Nk, dCB + (b0 - 1) * ldb, ldb, &zero, dst, nvec * NA));
  }
  if (!(flags & 1)) {
    std::vector<long long> skip;
    for (long long a = 0; a < NA; ++a)
      if (!done[a]) skip.push_back(a);
    if (!skip.empty()) {
      DBuf<long long> ds;
      ds.upload(skip, C.stream);
      dim3 g((unsigned)((nvec + 255) / 256), (unsigned)skip.size(), (unsigned)NB);
      hipLaunchKernelGGL(k_zero_acols, g, dim3(256), 0, C.stream, dRkab, nvec, NA, NB, ds.p, (long long)skip.size());
      GI_HIP(hipStreamSynchronize(C.stream));
    }
  }
  GI_HIP(hipStreamSynchronize(C.stream));
}

}  // namespace gi
