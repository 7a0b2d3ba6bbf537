// Coulomb energy of an AO density and its nuclear gradient on the device:
//   E_J = 1/2 sum_{pqrs} D_pq (pq|rs) D_rs,   dE_J/dR_A for every atom A.
// The reference has no gradient code (its ERIs only feed the Cholesky
// decomposition); this is the differentiation form, built on the same
// Hermite-matrix kernels as the ERIs (md_kernel.h).
//
// With the density folded into each primitive pair's Hermite table,
//   D^P_h = sum_{ab in P} w D_ab ET(h, ab)      (w = 2 for two different shells),
// the energy is a sum over ordered pairs of primitive pairs,
//   E_J = 1/2 sum_{P,Q} f(P, Q),   f = sum_{h,k} D^P_h (-1)^{|k|} D^Q_k R_{h+k}(P - Q),
// and, f being symmetric in P and Q, dE_J/dx = sum_{P,Q} d_P f(P, Q): only the
// bra pair is differentiated.  A pair with centres A, B and exponents a, b
// depends on the coordinates through X_AB = A - B (the E coefficients and
// exp(-ab/p AB^2)) and through P = (aA + bB)/p (R, with dR_tuv/dP_x =
// R_{t+1,u,v}):
//   d_A f = df/dX_AB + (a/p) df/dP,    d_B f = -df/dX_AB + (b/p) df/dP.
// Every primitive pair gets a table of GRAD_NCOL columns over the Hermite
// indices of order <= E + 1 (E = la + lb):
//   column 0     D^P_h                        (zero at order E + 1)
//   columns 1-3  dD^P_h / dX_AB,d, d = x, y, z (differentiated E recursion)
//   columns 4-6  D^P_{h - e_d}                (df/dP_d written as a bra of order E + 1)
//   columns 7-9  (a/p) D^P_{h - e_d}
// The kernels of coul_kernel.h give every primitive pair the Hermite potential
// of all ket pairs, J_h = sum_Q sum_k (-1)^{|k|} R_{h+k} D^Q_k, up to order
// E + 1 (E for the energy alone), and the ten sums f(P) = sum_h T(h, column)
// J_h follow once per pair, not once per pair of pairs.  Classes beyond those
// kernels (pairs of g and h shells) run md_kernel's row-sum mode on the same
// tables.  No derivative integral is stored.
#include <algorithm>
#include <cmath>
#include "coul_kernel.h"
#include "gi_context.h"

namespace gi {

// Device arrays of coulomb_energy_grad, kept in the context and grown only up to
// GRAD_KEEP bytes: a program calls it once per geometry, and stream-ordered frees
// of the slabs at the end of every call cost 16 ms of it after some hundred calls
// of 2 ms.  Beyond that (contracted bases from about 350 AOs on, 60 ms a call)
// they are freed when the call ends.
constexpr size_t GRAD_KEEP = 1ull << 30;
struct GradWork {
  DBuf<double> D, et, rows, dk, part, prow, q;
  DBuf<GradJob> jobs;
  DBuf<PrimRec> prim;
  DBuf<int> aoloc, prim0, nprim;
  DBuf<QRec> bra, ket;
  DBuf<CoulKet> kets;
  size_t bytes() const {
    return (D.n + et.n + rows.n + dk.n + part.n + prow.n + q.n) * sizeof(double) + jobs.n * sizeof(GradJob) +
           prim.n * sizeof(PrimRec) + (aoloc.n + prim0.n + nprim.n) * sizeof(int) + (bra.n + ket.n) * sizeof(QRec) +
           kets.n * sizeof(CoulKet);
  }
};
static GradWork &grad_work(Context &C) {
  if (!C.gradw) C.gradw = new GradWork();
  return *C.gradw;
}
void release_grad_work(Context &C) {
  // the frees follow the context stream; a call that ended by an error may have
  // left class launches on the side streams that it has not joined
  if (C.gradw)
    for (hipStream_t s : C.eri_side)
      if (s) (void)hipStreamSynchronize(s);
  delete C.gradw;
  C.gradw = nullptr;
}

// host array into a device array through the context's pinned arena
template <class T>
static void grad_upload(Context &C, DBuf<T> &b, const T *src, size_t count) {
  b.alloc(count);
  C.h2d(b.p, src, count * sizeof(T));
}

// launch records of the shell pairs: first primitive, table, destination rows
__global__ void k_grad_recs(const PrimRec *__restrict__ prims, const int *__restrict__ prim0,
                            const int *__restrict__ nprim, long long n, int nrow, QRec *out) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const PrimRec pr = prims[prim0[i]];
  out[i] = QRec{pr.px, pr.py, pr.pz, pr.p, pr.et, GRAD_NCOL * i, nrow, 0, 0, GRAD_NCOL, 1, nprim[i], prim0[i], 0};
}

// ket records of the primitive pairs lo .. lo + n - 1 (one class, order F):
// centre, exponent, and (-1)^{|k|} times column 0 of the table
__global__ void __launch_bounds__(256) k_coul_kets(const PrimRec *__restrict__ prims, long long lo, long long n, int F,
                                                   const double *__restrict__ et, CoulKet *__restrict__ ket,
                                                   double *__restrict__ dk) {
  const int nh = nherm(F);
  const long long e = blockIdx.x * 256LL + threadIdx.x;
  if (e >= n * nh) return;
  const long long i = e / nh;
  const int k = (int)(e - i * nh);
  const PrimRec p = prims[lo + i];
  int ord = 0;
  while (nherm(ord) <= k) ++ord;
  const double d = et[p.et + (long long)k * GRAD_NCOL];
  dk[e] = (ord & 1) ? -d : d;
  if (k == 0) ket[i] = CoulKet{p.px, p.py, p.pz, p.p, 1.0 / p.p};
}

// The slabs of one class added up into the first: 64 of the n = nherm nb
// elements per workgroup, sixteen waves splitting the slabs (one wave walking
// the slices of all waves took 0.9 ms a class at 320 AOs, bound by the latency
// of its own chain of loads), then a fixed-order sum.
__global__ void __launch_bounds__(1024) k_coul_sum(double *__restrict__ part, long long n, int slabs) {
  __shared__ double s_acc[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long i = blockIdx.x * 64LL + lane;
  double j = 0.0;
  if (i < n) {
#pragma unroll 4
    for (int s = w; s < slabs; s += 16) j += part[(size_t)s * n + i];
  }
  s_acc[w][lane] = j;
  __syncthreads();
  if (w == 0 && i < n) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += s_acc[k][lane];
    part[i] = t;
  }
}

// Potentials of nb primitive pairs (J[h nb + P], nh of them) times the pairs'
// tables: rows[10 P + c] = sum_h T(h, c) J_h for c < ncol.  One lane per pair
// (the potentials are stored pair-fastest), four waves splitting h.
__global__ void __launch_bounds__(256) k_coul_rows(const PrimRec *__restrict__ prims, const double *__restrict__ et,
                                                   const double *__restrict__ pot, int nb, int nh, int ncol,
                                                   double *__restrict__ rows) {
  __shared__ double s_acc[4][GRAD_NCOL][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int b = (int)blockIdx.x * 64 + lane;
  const bool ok = b < nb;
  const long long e0 = prims[ok ? b : nb - 1].et;
  double acc[GRAD_NCOL];
#pragma unroll
  for (int c = 0; c < GRAD_NCOL; ++c) acc[c] = 0.0;
  if (ok)
    for (int h = w; h < nh; h += 4) {
      const double j = pot[(size_t)h * nb + b];
      const double *t = et + e0 + (long long)h * GRAD_NCOL;
#pragma unroll
      for (int c = 0; c < GRAD_NCOL; ++c)
        if (c < ncol) acc[c] += t[c] * j;
    }
#pragma unroll
  for (int c = 0; c < GRAD_NCOL; ++c) s_acc[w][c][lane] = acc[c];
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * GRAD_NCOL; e += 256) {
    const int p = e / GRAD_NCOL, c = e - p * GRAD_NCOL, bb = (int)blockIdx.x * 64 + p;
    if (bb < nb) rows[(size_t)bb * GRAD_NCOL + c] = (s_acc[0][c][p] + s_acc[1][c][p]) + (s_acc[2][c][p] + s_acc[3][c][p]);
  }
}

// rows of a shell pair: the sum over its primitive pairs, added to out
__global__ void k_coul_pair_rows(const double *__restrict__ prow, const int *__restrict__ prim0,
                                 const int *__restrict__ nprim, long long lo, long long n, double *__restrict__ out) {
  const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (e >= n * GRAD_NCOL) return;
  const long long i = lo + e / GRAD_NCOL;
  const int c = (int)(e % GRAD_NCOL);
  double s = 0.0;
  for (int k = 0; k < nprim[i]; ++k) s += prow[(size_t)(prim0[i] + k) * GRAD_NCOL + c];
  out[(size_t)i * GRAD_NCOL + c] += s;
}

// shell pairs (s0 >= s1, s1-major order) kept by the screening of
// coulomb_energy_grad: the Schwarz diagonals (ab|ab) of every pair from one
// diagonal ERI request, the density maxima on the host
static std::vector<char> screened_pairs(Context &C, const double *D, long long ldd, double kappa, double eps) {
  const int nsh = C.nshells;
  std::vector<PairDesc> rd, cd;
  std::vector<int> rows;
  long long loc = 0;
  for (int s1 = 0; s1 < nsh; ++s1)
    for (int s0 = s1; s0 < nsh; ++s0) {
      const int fl = s0 == s1 ? PAIR_SAME : 0;
      rd.push_back(PairDesc{s0, s1, fl, 0, 0, 0, loc});
      cd.push_back(PairDesc{s0, s1, fl, 0, 0, 0, 0});
      rows.push_back((int)rows.size());
      const int n0 = C.shell_nang[s0], n1 = C.shell_nang[s1];
      loc += s0 == s1 ? (long long)n0 * (n0 + 1) / 2 : (long long)n0 * n1;
    }
  DBuf<double> &dq = grad_work(C).q;
  dq.alloc((size_t)loc);
  EriRequest R;
  R.rdesc = &rd;
  R.cdesc = &cd;
  R.rows = &rows;
  R.cols = &rows;
  R.mode = LAUNCH_DIAG;
  R.out = dq.p;
  R.ldo = 0;
  R.kappa = kappa;
  eri_run(C, R);
  std::vector<double> q((size_t)loc);
  C.read(q.data(), dq.p, sizeof(double) * (size_t)loc);
  std::vector<double> w(rows.size());
  double wsum = 0.0;
  for (size_t i = 0; i < rows.size(); ++i) {
    const int s0 = rd[i].s0, s1 = rd[i].s1;
    const int n0 = C.shell_nang[s0], n1 = C.shell_nang[s1];
    const long long o = rd[i].off, nr = s0 == s1 ? (long long)n0 * (n0 + 1) / 2 : (long long)n0 * n1;
    double qm = 0.0, dm = 0.0;
    for (long long r = 0; r < nr; ++r) qm = std::max(qm, q[(size_t)(o + r)]);
    for (int b = 0; b < n1; ++b)
      for (int a = 0; a < n0; ++a) {
        const long long pa = C.shell_loc[s0] + a, pb = C.shell_loc[s1] + b;
        dm = std::max(dm, std::max(std::fabs(D[pa + ldd * pb]), std::fabs(D[pb + ldd * pa])));
      }
    w[i] = std::sqrt(std::max(qm, 0.0)) * dm;
    wsum += w[i];
  }
  std::vector<char> keep(rows.size());
  for (size_t i = 0; i < rows.size(); ++i) keep[i] = w[i] * wsum >= eps ? 1 : 0;
  return keep;
}

constexpr long long COUL_WAVES = 4096, COUL_MIN_KETS = 8;

void coulomb_energy_grad(Context &C, const double *D, long long ldd, double kappa, double *energy,
                         double *grad) {
  if (!C.basis_set) throw Error{4, "basis not set"};
  if (!D || !energy) throw Error{61, "null density or energy pointer"};
  if (ldd < C.nao) throw Error{61, "leading dimension of D smaller than the number of AOs"};
  struct Busy {   // the arrays are in use until the call ends, by an error too
    Context &C;
    explicit Busy(Context &c) : C(c) { ++C.work_busy; }
    ~Busy() {
      --C.work_busy;
      if (C.gradw && C.gradw->bytes() > GRAD_KEEP) release_grad_work(C);
    }
  } busy(C);
  const bool want_grad = grad != nullptr;
  const int nsh = C.nshells;
  // shell pairs s0 >= s1, grouped by E = l0 + l1 so that a class is a contiguous range
  const int nbin = 2 * MAXL + 1;
  std::vector<std::vector<std::pair<int, int>>> bins(nbin);
  // R tables of order (E + 1) + F for the gradient: within the Boys table
  if (want_grad && 4 * C.lmax + 1 > BOYS_MAXM)
    throw Error{62, "the nuclear gradient needs 4 lmax + 1 <= " + std::to_string(BOYS_MAXM) + " (l <= 4)"};
  // density-weighted Schwarz screening (grad_screen = v > 0, eps = 10^-v): with
  // w_s = max_{ab in s} |D_ab| sqrt(max_{ab in s} (ab|ab)) for shell pair s,
  // every term of E_J that involves s is at most w_s sum_t w_t, and the pair
  // is left out when that is below eps (off by default: every pair kept)
  std::vector<char> keep;
  if (C.grad_screen > 0) keep = screened_pairs(C, D, ldd, kappa, std::pow(10.0, -(double)C.grad_screen));
  long long ip = 0;
  for (int s1 = 0; s1 < nsh; ++s1)
    for (int s0 = s1; s0 < nsh; ++s0, ++ip)
      if (keep.empty() || keep[ip]) bins[C.shell_l[s0] + C.shell_l[s1]].push_back({s0, s1});
  std::vector<long long> bin_off(nbin + 1, 0);
  for (int e = 0; e < nbin; ++e) bin_off[e + 1] = bin_off[e] + (long long)bins[e].size();
  const long long npair = bin_off[nbin];
  std::vector<GradJob> jobs;
  std::vector<int> prim0(npair), nprim(npair), pa(npair), pb(npair);
  long long etn = 0;
  for (int e = 0; e < nbin; ++e)
    for (size_t k = 0; k < bins[e].size(); ++k) {
      const long long i = bin_off[e] + (long long)k;
      const int s0 = bins[e][k].first, s1 = bins[e][k].second;
      pa[i] = s0;
      pb[i] = s1;
      prim0[i] = (int)jobs.size();
      nprim[i] = C.shell_np[s0] * C.shell_np[s1];
      for (int ib = 0; ib < C.shell_np[s1]; ++ib)
        for (int ia = 0; ia < C.shell_np[s0]; ++ia) {
          GradJob j{};
          j.s0 = s0;
          j.s1 = s1;
          j.ia = ia;
          j.ib = ib;
          j.prim = (int)jobs.size();
          j.et = etn;
          j.w = s0 != s1 ? 2.0 : 1.0;
          jobs.push_back(j);
          etn += (long long)nherm(e + 1) * GRAD_NCOL;
        }
    }
  const long long nao = C.nao;
  std::vector<int> aoloc(C.shell_loc.begin(), C.shell_loc.end());
  GradWork &W = grad_work(C);
  DBuf<double> &dD = W.D, &det = W.et, &drows = W.rows;
  DBuf<GradJob> &djobs = W.jobs;
  DBuf<PrimRec> &dprim = W.prim;
  DBuf<int> &daoloc = W.aoloc, &dprim0 = W.prim0, &dnprim = W.nprim;
  DBuf<QRec> &dbra = W.bra, &dket = W.ket;
  grad_upload(C, dD, D, (size_t)ldd * (size_t)(nao - 1) + (size_t)nao);
  grad_upload(C, daoloc, aoloc.data(), aoloc.size());
  grad_upload(C, djobs, jobs.data(), jobs.size());
  grad_upload(C, dprim0, prim0.data(), prim0.size());
  grad_upload(C, dnprim, nprim.data(), nprim.size());
  det.alloc((size_t)etn);
  dprim.alloc(jobs.size());
  launch_build_grad_et(C, daoloc.p, dD.p, ldd, djobs.p, (long long)jobs.size(), dprim.p, det.p);
  drows.alloc((size_t)npair * GRAD_NCOL);
  GI_HIP(hipMemsetAsync(drows.p, 0, sizeof(double) * (size_t)npair * GRAD_NCOL, C.stream));
  // primitive pairs of a class are consecutive, like its shell pairs
  std::vector<long long> prim_off(nbin + 1, 0);
  for (int e = 0; e < nbin; ++e) prim_off[e + 1] = bin_off[e + 1] < npair ? prim0[bin_off[e + 1]] : (long long)jobs.size();
  const int up = want_grad ? 1 : 0;
  // potential kernels: every class pair within their orders
  const int ebig = COUL_EMAX - up;   // bra classes e <= ebig, ket classes f <= COUL_FMAX
  DBuf<CoulKet> &dkets = W.kets;
  DBuf<double> &ddk = W.dk, &dpart = W.part, &dprow = W.prow;
  std::vector<long long> dk_off(COUL_FMAX + 2, 0);
  for (int f = 0; f <= std::min(COUL_FMAX, nbin - 1); ++f)
    dk_off[f + 1] = dk_off[f] + (prim_off[f + 1] - prim_off[f]) * nherm(f);
  dkets.alloc(jobs.size());
  ddk.alloc((size_t)dk_off[std::min(COUL_FMAX, nbin - 1) + 1]);
  dprow.alloc(jobs.size() * GRAD_NCOL);
  struct Slab {   // one launch: class pair, slabs and their place in dpart
    int e, f, per, groups;
    long long off;
    double cost;
  };
  std::vector<Slab> slabs;
  std::vector<long long> part_off(nbin + 1, 0);
  std::vector<int> part_groups(nbin, 0);
  long long part_n = 0;
  for (int e = 0; e <= std::min(ebig, nbin - 1); ++e) {
    const long long nb = prim_off[e + 1] - prim_off[e];
    part_off[e] = part_n;
    if (nb == 0) continue;
    if (nb > INT32_MAX / 2) throw Error{63, "too many primitive pairs"};
    for (int f = 0; f <= std::min(COUL_FMAX, nbin - 1); ++f) {
      const long long nk = prim_off[f + 1] - prim_off[f];
      if (nk == 0) continue;
      if (nk > INT32_MAX / 2) throw Error{63, "too many primitive pairs"};
      // slices of the ket list: about COUL_WAVES waves in flight per launch
      // (4 per SIMD), at least COUL_MIN_KETS pairs each where the integrals are
      // cheap (the block first copies 20 KB of Boys coefficients)
      const long long tiles = (nb + 63) / 64;
      const long long least = e + up + f >= 8 ? 1 : COUL_MIN_KETS;
      long long want = std::max<long long>(1, std::min((COUL_WAVES + tiles - 1) / tiles, (nk + least - 1) / least));
      const int per = (int)((nk + want - 1) / want);
      const int groups = (int)(((nk + per - 1) / per + 3) / 4);   // workgroups of four slices, one slab each
      const int nh = nherm(e + up);
      slabs.push_back(Slab{e, f, per, groups, part_n, (double)nb * (double)nk * nh * nherm(f)});
      part_n += (long long)groups * nh * nb;
      part_groups[e] += groups;
    }
  }
  dpart.alloc((size_t)part_n);
  for (int f = 0; f <= std::min(COUL_FMAX, nbin - 1); ++f) {
    const long long nk = prim_off[f + 1] - prim_off[f];
    if (nk == 0) continue;
    hipLaunchKernelGGL(k_coul_kets, dim3((unsigned)((nk * nherm(f) + 255) / 256)), dim3(256), 0, C.stream, dprim.p,
                       prim_off[f], nk, f, det.p, dkets.p + prim_off[f], ddk.p + dk_off[f]);
    GI_HIP(hipGetLastError());
  }
  // the classes write disjoint slabs: spread over the side streams, the
  // largest first, so that small classes fill the tails
  const int nstream = (int)std::min<long long>(C.eri_streams, (long long)slabs.size());
  C.fork_side(nstream);
  std::stable_sort(slabs.begin(), slabs.end(), [](const Slab &x, const Slab &y) { return x.cost > y.cost; });
  std::vector<double> load(std::max(nstream, 1), 0.0);
  for (const Slab &sl : slabs) {
    const int j = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[j] += sl.cost;
    CoulArgs a{};
    a.bra = dprim.p + prim_off[sl.e];
    a.ket = dkets.p + prim_off[sl.f];
    a.dk = ddk.p + dk_off[sl.f];
    a.part = dpart.p + sl.off;
    a.nb = (int)(prim_off[sl.e + 1] - prim_off[sl.e]);
    a.nk = (int)(prim_off[sl.f + 1] - prim_off[sl.f]);
    a.per = sl.per;
    a.kappa = kappa;
    a.boys = C.dboys.p;
    launch_coul_j(sl.e + up, sl.f, a, sl.groups, j == 0 ? C.stream : C.eri_side[j - 1]);
    GI_HIP(hipGetLastError());
  }
  C.join_side(nstream);
  for (int e = 0; e <= std::min(ebig, nbin - 1); ++e) {
    const long long nb = prim_off[e + 1] - prim_off[e], ns = bin_off[e + 1] - bin_off[e];
    if (nb == 0 || part_groups[e] == 0) continue;
    const long long n = nb * nherm(e + up);
    hipLaunchKernelGGL(k_coul_sum, dim3((unsigned)((n + 63) / 64)), dim3(1024), 0, C.stream, dpart.p + part_off[e], n,
                       part_groups[e]);
    hipLaunchKernelGGL(k_coul_rows, dim3((unsigned)((nb + 63) / 64)), dim3(256), 0, C.stream, dprim.p + prim_off[e],
                       det.p, dpart.p + part_off[e], (int)nb, nherm(e + up), want_grad ? GRAD_NCOL : 1,
                       dprow.p + (size_t)prim_off[e] * GRAD_NCOL);
    hipLaunchKernelGGL(k_coul_pair_rows, dim3((unsigned)((ns * GRAD_NCOL + 255) / 256)), dim3(256), 0, C.stream,
                       dprow.p, dprim0.p, dnprim.p, bin_off[e], ns, drows.p);
    GI_HIP(hipGetLastError());
  }
  // the others: md_kernel in row-sum mode (each row's sum over the ket pairs
  // added to the pair's rows)
  bool recs = false;
  for (int eb = 0; eb < nbin; ++eb) {
    const long long nr = bin_off[eb + 1] - bin_off[eb];
    if (nr == 0) continue;
    for (int fk = 0; fk < nbin; ++fk) {
      const long long nc = bin_off[fk + 1] - bin_off[fk];
      if (nc == 0 || (eb <= ebig && fk <= COUL_FMAX)) continue;
      if (!recs) {
        recs = true;
        dbra.alloc(npair);
        dket.alloc(npair);
        const unsigned gb = (unsigned)((npair + 255) / 256);
        hipLaunchKernelGGL(k_grad_recs, dim3(gb), dim3(256), 0, C.stream, dprim.p, dprim0.p, dnprim.p, npair,
                           want_grad ? GRAD_NCOL : 1, dbra.p);
        hipLaunchKernelGGL(k_grad_recs, dim3(gb), dim3(256), 0, C.stream, dprim.p, dprim0.p, dnprim.p, npair, 1,
                           dket.p);
      }
      MdArgs a{};
      a.prim = dprim.p;
      a.et = det.p;
      a.rrec = dbra.p + bin_off[eb];
      a.crec = dket.p + bin_off[fk];
      a.nrows = nr;
      a.ncols = nc;
      a.mode = LAUNCH_PRODUCT;
      a.trans = 0;
      a.rowsum = 1;
      a.kappa = kappa;
      a.out = drows.p;
      a.ldo = 0;
      a.sel = nullptr;
      a.boys = C.dboys.p;
      // one-column ket pairs: 32 of them fill the stacked stage-2 columns
      long long kt = std::max<long long>(1, std::min<long long>(32, C.eri_max_kt));
      while (kt > 1 && nr * ((nc + kt - 1) / kt) < C.eri_min_tiles) kt = (kt + 1) / 2;
      a.kt = (int)kt;
      a.ntiles = nr * ((nc + kt - 1) / kt);
      long long grid = std::min<long long>(a.ntiles, 4096);
      if (grid >= 8) grid = (grid + 7) / 8 * 8;
      launch_md_class(want_grad ? eb + 1 : eb, fk, a, (int)grid, C.stream);
      GI_HIP(hipGetLastError());
    }
  }
  std::vector<double> rows((size_t)npair * GRAD_NCOL);
  C.read(rows.data(), drows.p, sizeof(double) * rows.size());
  double e = 0.0;
  for (long long i = 0; i < npair; ++i) e += rows[GRAD_NCOL * i];
  *energy = 0.5 * e;
  if (want_grad) {
    std::fill(grad, grad + 3 * (size_t)C.natoms, 0.0);
    for (long long i = 0; i < npair; ++i) {
      const int A = C.shell_atom[pa[i]], B = C.shell_atom[pb[i]];
      const double *r = rows.data() + GRAD_NCOL * i;
      for (int d = 0; d < 3; ++d) {
        const double gE = r[1 + d], gR = r[4 + d], gRa = r[7 + d];
        grad[3 * A + d] += gE + gRa;
        grad[3 * B + d] += -gE + (gR - gRa);
      }
    }
  }
}

}  // namespace gi
