// Symmetric tridiagonal divide and conquer on the GPU, FP64 throughout.
// Replaces the host LAPACKE_dstedc('I') call of the reference driver
// (src/EVD/myEVD.cu:529).  The mathematics is Cuppen's method as published
// (Cuppen 1981; Gu & Eisenstat 1995) in the form LAPACK's dlaed0/1/2/3/4 use:
//
//  * tearing: T = diag(T1 - |e| e_k e_k^T, T2 - |e| e_1 e_1^T) + |e| v v^T,
//    v = [e_k; sign(e) e_1], applied at every split up front;
//  * merge: d = [lambda(T1); lambda(T2)], z = [last row of Q1; sign(e) first
//    row of Q2] / sqrt(2), rho = 2|e|; sort d; deflate small |rho z_j| and
//    close pairs (Givens rotation of the two columns, tol = 8 eps max(|d|,|z|));
//  * secular equation 1 + rho sum z_j^2/(d_j - lambda) = 0 per root, solved
//    relative to the nearer pole with a two-pole rational model step inside a
//    bisection bracket;
//  * Loewner recomputation of z (Gu-Eisenstat) for orthogonal vectors;
//  * Q_new = Q' [U 0; 0 I] by grouped FP64 MFMA GEMMs over the top and bottom
//    row blocks (column types 1/2/3 as in dlaed2/dlaed3).
//
// GPU layout: the binary split tree goes down to single rows.  The merges of the
// subtrees of at most kDcLeaf rows (the leaves of the host's tree) run in one launch, a
// workgroup per leaf; above them all merges of one
// tree height run in the same launches (grid.y = merge), every merge working
// in the index range [start, start+N) of n-long scratch arrays and in the
// diagonal block of the n x n Q / scratch matrices.  The deflation scan is
// parallel except for the chain of Givens rotations (processed 64 pairs at a
// time by one wave).
#include <algorithm>
#include <cfloat>

#include <rocblas/rocblas.h>

#include "common.hpp"

namespace evd {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// order of a wave's LDS accesses
static __device__ __attribute__((always_inline)) inline void lds_order() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

struct MergeDesc {
  int start, n1, n2, pad;
  double rho;  // |e| at the split
  double sgn;  // sign(e)
};
// a leaf of the tree: rows start .. start + size - 1 of problem `problem`
struct LeafDesc {
  int start, size, problem;
};
// Rows of a leaf: a row of 16 lanes holds the poles of its largest merge.  A small
// merge level costs 35 to 60 us of dependent launches whatever its size; one
// launch does the four below 16 rows in 40 us (n = 256 and 2500; 50 us for 32
// problems of order 256).
constexpr int kDcLeaf = 16;
struct MergeOut {
  int K, K1, K2, K3, ndefl, nrot;
  double rho2;  // 2|e|
  double zsum;  // sum of squares of non-deflated z
};

struct DCScratch {
  double *ds, *zs;     // sorted d, z
  int *cs;             // sorted -> local column
  double *nd_d, *nd_z; // non-deflated
  int *nd_col, *qpos;
  double *df_d;
  int *df_col;
  int *rot_p, *rot_n;
  double *rot_c, *rot_s;
  int *types;
  int *orig;
  double *tau, *lam, *zhat;
  int *colmap, *dmap;
  double *Qc = nullptr, *Uc = nullptr;  // n x n, ld n (with vectors)
  // Same-size batches run as one concatenated index space: merge starts (and
  // every vector above) are global, problem q = MergeDesc::pad owns indices
  // [q n, q n + n).  Its matrices sit at their own offsets; adding
  // q * zmul (Z) or q * qmul (Qc, Uc) to an index formed from global starts
  // lands in problem q's matrix (0 for a single problem).
  long zmul = 0, qmul = 0;
};

// Eigenvalues only: a merge needs just the last row of its first child's
// vectors and the first row of its second's, so the vectors are never formed.
// first / last hold those two rows of every node's vectors (by column, in the
// place of D); rot_first / rot_last a merge's rows after its deflation
// rotations.  Null when vectors are wanted.
struct DCRows {
  double *first = nullptr, *last = nullptr, *rot_first = nullptr, *rot_last = nullptr;
};

// Tearing of every split at once, one thread per diagonal entry: the tree's
// splits are all the boundaries between rows of a problem, and an entry between two of
// them is adjusted by both.
__global__ void dc_tear_kernel(long n, long total, const double *__restrict__ E, double *__restrict__ D) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    double d = D[i];
    const long r = i % n;
    if (r > 0) d -= fabs(E[i - 1]);
    if (r + 1 < n) d -= fabs(E[i]);
    D[i] = d;
  }
}

// Normalisation of each problem's tridiagonal to max(|d_i|, |e_i|) = 1
// before the merges and back afterwards (the scaling step of LAPACK dstedc,
// which the reference's MKL call performs): the deflation tolerance
// 8 eps max(|d|max, |z|max) mixes the matrix scale with the unit-vector
// scale of z, so it is only relative to the matrix on a normalised problem.
// One workgroup per problem (blockIdx.x); nrm[q] keeps the factor.
__global__ __launch_bounds__(256) void dc_normalize_kernel(long n, double *__restrict__ D, double *__restrict__ E,
                                                           double *__restrict__ nrm) {
  __shared__ double red[256];
  const int q = blockIdx.x;
  double *d = D + q * n, *e = E + q * n;
  double mx = 0.0;
  for (long i = threadIdx.x; i < n; i += 256) {
    mx = fmax(mx, fabs(d[i]));
    if (i < n - 1) mx = fmax(mx, fabs(e[i]));
  }
  red[threadIdx.x] = mx;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  const double s = red[0];
  if (threadIdx.x == 0) nrm[q] = s;
  if (s == 0.0 || s == 1.0) return;
  for (long i = threadIdx.x; i < n; i += 256) {
    d[i] /= s;
    if (i < n - 1) e[i] /= s;
  }
}

__global__ void dc_denormalize_kernel(long n, double *__restrict__ D, const double *__restrict__ nrm) {
  const int q = blockIdx.y;
  const double s = nrm[q];
  if (s == 0.0 || s == 1.0) return;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    D[q * n + i] *= s;
}

// |e| and sign(e) at every split, read on the device so no host round trip
// sits between the tridiagonal stage's producer and the merges.
__global__ void dc_rho_kernel(int nmerge, MergeDesc *__restrict__ md, const double *__restrict__ E) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nmerge; i += gridDim.x * blockDim.x) {
    const double e = E[md[i].start + md[i].n1 - 1];
    md[i].rho = fabs(e);
    md[i].sgn = (e >= 0.0) ? 1.0 : -1.0;
  }
}

// d and z of one merge in ascending order of d, elements first, first + step, ...
__device__ inline void merge_sorted(const MergeDesc &m, const double *__restrict__ D, const double *__restrict__ Z,
                                    long ldz, const DCScratch &sc, const DCRows &rows, int first, int step) {
  const int N = m.n1 + m.n2, st = m.start;
  for (int t = first; t < N; t += step) {
    double d = D[st + t], z;
    int pos;
    if (t < m.n1) {
      z = rows.last ? rows.last[st + t] : Z[(long)m.pad * sc.zmul + (st + m.n1 - 1) + (long)(st + t) * ldz];
      int lo = 0, hi = m.n2;
      while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (D[st + m.n1 + mid] < d)
          lo = mid + 1;
        else
          hi = mid;
      }
      pos = t + lo;
    } else {
      z = m.sgn * (rows.first ? rows.first[st + t] : Z[(long)m.pad * sc.zmul + (st + m.n1) + (long)(st + t) * ldz]);
      int lo = 0, hi = m.n1;
      while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (D[st + mid] <= d)
          lo = mid + 1;
        else
          hi = mid;
      }
      pos = (t - m.n1) + lo;
    }
    sc.ds[st + pos] = d;
    sc.zs[st + pos] = z * 0.70710678118654752440;
    sc.cs[st + pos] = t;
  }
}
__global__ void dc_sort_kernel(const MergeDesc *__restrict__ md, const double *__restrict__ D,
                               const double *__restrict__ Z, long ldz, DCScratch sc, DCRows rows) {
  merge_sorted(md[blockIdx.y], D, Z, ldz, sc, rows, (int)(blockIdx.x * blockDim.x + threadIdx.x), (int)(gridDim.x * blockDim.x));
}
// merges up to this order are sorted by their deflation workgroup
constexpr int kDcSortInline = 512;

// One thread per merge: deflation scan in sorted order (dlaed2 logic).
// Block-wide helpers for one 256-thread workgroup.
__device__ inline double block_max256(double v, double *red) {
  v = fmax(v, __shfl_xor(v, 32, 64));
  for (int o = 16; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
// exclusive prefix of per-thread counts (thread order); returns the total.
// Three counts of up to 2^21 may share the word.
__device__ inline unsigned long long block_scan256(unsigned long long v, unsigned long long *sh,
                                                   unsigned long long &excl) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned long long x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  __syncthreads();
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  unsigned long long before = 0;
  for (int w = 0; w < wave; w++) before += sh[w];
  excl = before + x - v;
  return sh[0] + sh[1] + sh[2] + sh[3];
}

// Deflation of one merge (LAPACK dlaed2), one 256-thread workgroup per merge.
// z-deflation (rho |z_j| <= tol) is decided in parallel and compacted in
// order.  The Givens deflation scan over the remaining entries is sequential
// only through its rotations (pair (p, j) depends on the previous pair only if
// that pair rotated), so wave 0 tests 64 consecutive pairs at once on the
// current values, accepts every pair before the first rotation, applies that
// rotation and continues after it.  The deflated list is the in-order
// z-deflated run merged with the (few) rotated entries; type counts and the
// type-stable positions come from block scans (shuffles within a wave; a scan
// by one thread had made this kernel 16-23 us long, four times per merge level).
__global__ __launch_bounds__(256) void dc_deflate_kernel(const MergeDesc *__restrict__ md, MergeOut *__restrict__ mo,
                                                         const double *__restrict__ D, const double *__restrict__ Z,
                                                         long ldz, int sort, DCScratch sc, DCRows rows) {
  __shared__ double red[4], zpart[256];
  __shared__ unsigned long long sh[4];
  __shared__ int s_nc, s_K, s_nrot;
  const MergeDesc m = md[blockIdx.x];
  const int N = m.n1 + m.n2, st = m.start, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double rho = 2.0 * m.rho;
  if (sort) {
    merge_sorted(m, D, Z, ldz, sc, rows, tid, 256);
    __syncthreads();
  }
  double *ds = sc.ds + st, *zs = sc.zs + st;
  // sorted -> local column; a NaN among d leaves places of the order unwritten, so
  // what is read there is kept within the merge
  const int *order = sc.cs + st;
  auto cs = [&](int i) { return (int)min((unsigned)order[i], (unsigned)(N - 1)); };
  int *types = sc.types + st;
  double *nd_d = sc.nd_d + st, *nd_z = sc.nd_z + st;
  int *nd_col = sc.nd_col + st, *qpos = sc.qpos + st;
  double *df_d = sc.df_d + st;
  int *df_col = sc.df_col + st;
  int *rot_p = sc.rot_p + st, *rot_n = sc.rot_n + st;
  double *rot_c = sc.rot_c + st, *rot_s = sc.rot_s + st;
  int *cand = sc.orig + st;     // candidate list (orig is written later by the secular solve)
  double *tmp_d = sc.tau + st;  // merge buffer (tau likewise)
  int *tmp_c = sc.dmap + st;    // (dmap is written after the deflation)
  // chunk of N owned by this thread, in order
  const int per = (N + 255) / 256, i0 = min(N, tid * per), i1 = min(N, i0 + per);

  double dmax = 0.0, zmax = 0.0;
  for (int i = i0; i < i1; i++) {
    types[i] = (i < m.n1) ? 1 : 3;
    dmax = fmax(dmax, fabs(ds[i]));
    zmax = fmax(zmax, fabs(zs[i]));
  }
  dmax = block_max256(dmax, red);
  zmax = block_max256(zmax, red);
  const double eps = DBL_EPSILON * 0.5;
  const double tol = 8.0 * eps * fmax(dmax, zmax);
  const bool all_defl = (rho * zmax <= tol);

  // z-deflated run (in order) and the candidate list, by compaction
  int nz_loc = 0;
  for (int i = i0; i < i1; i++) nz_loc += (all_defl || rho * fabs(zs[i]) <= tol) ? 1 : 0;
  unsigned long long before;
  const int nzd = (int)block_scan256((unsigned long long)nz_loc, sh, before);
  int zoff = (int)before, coff = i0 - zoff;  // candidates before my chunk = i0 - (z-deflated before it)
  for (int i = i0; i < i1; i++) {
    if (all_defl || rho * fabs(zs[i]) <= tol) {
      df_d[zoff] = ds[i];
      df_col[zoff] = cs(i);
      zoff++;
    } else {
      cand[coff++] = i;
    }
  }
  if (tid == 0) s_nc = N - nzd;
  __syncthreads();
  const int nc = s_nc;

  // Givens scan (wave 0)
  if (wave == 0) {
    int K = 0, nrot = 0;
    int pj = nc > 0 ? cand[0] : -1;
    int k = 1;
    while (k < nc) {
      const int nvalid = min(64, nc - k);
      const bool valid = lane < nvalid;
      const int j = valid ? cand[k + lane] : 0;
      const int prv = (lane == 0) ? pj : (valid ? cand[k + lane - 1] : 0);
      bool rot = false;
      double c = 0.0, sn = 0.0, tau = 0.0;
      if (valid) {
        sn = zs[prv];
        c = zs[j];
        tau = hypot(c, sn);
        const double t = ds[j] - ds[prv];
        c /= tau;
        sn = -sn / tau;
        rot = fabs(t * c * sn) <= tol;
      }
      const unsigned long long mask = __ballot(rot);
      const int first = mask ? __ffsll((long long)mask) - 1 : nvalid;
      if (lane < first) {
        nd_d[K + lane] = ds[prv];
        nd_z[K + lane] = zs[prv];
        nd_col[K + lane] = cs(prv);
      }
      K += first;
      if (first < nvalid) {
        if (lane == first) {
          zs[j] = tau;
          zs[prv] = 0.0;
          const int cp = cs(prv), cn = cs(j);
          if (types[cp] != types[cn]) types[cn] = 2;
          types[cp] = 4;
          rot_p[nrot] = cp;
          rot_n[nrot] = cn;
          rot_c[nrot] = c;
          rot_s[nrot] = sn;
          const double tt = ds[prv] * c * c + ds[j] * sn * sn;
          ds[j] = ds[prv] * sn * sn + ds[j] * c * c;
          ds[prv] = tt;
          df_d[nzd + nrot] = tt;
          df_col[nzd + nrot] = cp;
        }
        nrot++;
        pj = __shfl(j, first, 64);
        k += first + 1;
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      } else {
        pj = __shfl(j, nvalid - 1, 64);
        k += nvalid;
      }
    }
    if (pj >= 0) {
      if (lane == 0) {
        nd_d[K] = ds[pj];
        nd_z[K] = zs[pj];
        nd_col[K] = cs(pj);
      }
      K++;
    }
    if (lane == 0) {
      s_K = K;
      s_nrot = nrot;
    }
  }
  __syncthreads();
  const int K = s_K, nrot = s_nrot, nd = nzd + nrot;

  // deflated list ascending: the rotated entries (few) sorted in place, then
  // merged with the z-deflated run (already ascending; ties keep the run first)
  if (tid == 0) {
    for (int i = nzd + 1; i < nd; i++) {
      const double v = df_d[i];
      const int cc = df_col[i];
      int j = i - 1;
      while (j >= nzd && df_d[j] > v) {
        df_d[j + 1] = df_d[j];
        df_col[j + 1] = df_col[j];
        j--;
      }
      df_d[j + 1] = v;
      df_col[j + 1] = cc;
    }
  }
  __syncthreads();
  if (nrot > 0) {
    for (int e = tid; e < nd; e += 256) {
      const double v = df_d[e];
      int pos;
      if (e < nzd) {  // rank among rotated entries with value < v
        int lo = nzd, hi = nd;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (df_d[mid] < v) lo = mid + 1; else hi = mid;
        }
        pos = e + (lo - nzd);
      } else {  // rank among z-deflated entries with value <= v
        int lo = 0, hi = nzd;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (df_d[mid] <= v) lo = mid + 1; else hi = mid;
        }
        pos = (e - nzd) + lo;
      }
      tmp_d[pos] = v;
      tmp_c[pos] = df_col[e];
    }
    __syncthreads();
    for (int e = tid; e < nd; e += 256) {
      df_d[e] = tmp_d[e];
      df_col[e] = (int)min((unsigned)tmp_c[e], (unsigned)(N - 1));
    }
  }

  // type counts, z sum and type-stable positions of the non-deflated entries
  const int kp = (K + 255) / 256, k0 = min(K, tid * kp), k1 = min(K, k0 + kp);
  int c1 = 0, c2 = 0, c3 = 0;
  double zs2 = 0.0;
  for (int kk = k0; kk < k1; kk++) {
    const int ty = types[nd_col[kk]];
    c1 += (ty == 1);
    c2 += (ty == 2);
    c3 += (ty == 3);
    zs2 += nd_z[kk] * nd_z[kk];
  }
  const unsigned long long counts =
      block_scan256((unsigned long long)c1 | (unsigned long long)c2 << 21 | (unsigned long long)c3 << 42, sh, before);
  const int mask21 = (1 << 21) - 1;
  const int K1 = (int)(counts & mask21), K2 = (int)(counts >> 21 & mask21), K3 = (int)(counts >> 42);
  int e1 = (int)(before & mask21), e2 = (int)(before >> 21 & mask21), e3 = (int)(before >> 42);
  for (int kk = k0; kk < k1; kk++) {
    const int ty = types[nd_col[kk]];
    qpos[kk] = (ty == 1) ? e1++ : (ty == 2) ? K1 + e2++ : K1 + K2 + e3++;
  }
  // z sum in a fixed order (deterministic): per-thread chunks, then thread order
  __syncthreads();
  zpart[tid] = zs2;
  __syncthreads();
  if (tid == 0) {
    const int np = kp > 0 ? (K + kp - 1) / kp : 0;  // threads that had a chunk
    double zsum = 0.0;
#pragma unroll 8
    for (int t = 0; t < np; t++) zsum += zpart[t];
    MergeOut o;
    o.K = K;
    o.K1 = K1;
    o.K2 = K2;
    o.K3 = K3;
    o.ndefl = nd;
    o.nrot = nrot;
    o.rho2 = rho;
    o.zsum = zsum;
    mo[blockIdx.x] = o;
  }
}

// Row-parallel: apply the deflation rotations to Q's columns.
__global__ void dc_rotate_kernel(const MergeDesc *__restrict__ md, const MergeOut *__restrict__ mo,
                                 double *__restrict__ Z, long ldz, DCScratch sc) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  if (o.nrot == 0) return;
  const int N = m.n1 + m.n2, st = m.start;
  double *Zb = Z + ((long)m.pad * sc.zmul + st + (long)st * ldz);
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < N; r += gridDim.x * blockDim.x) {
    for (int t = 0; t < o.nrot; t++) {
      const int p = sc.rot_p[st + t], q = sc.rot_n[st + t];
      const double c = sc.rot_c[st + t], s = sc.rot_s[st + t];
      const double x = Zb[r + (long)p * ldz], y = Zb[r + (long)q * ldz];
      Zb[r + (long)p * ldz] = c * x + s * y;
      Zb[r + (long)q * ldz] = c * y - s * x;
    }
  }
}

// Gather the permuted copy Qc = [non-deflated by type | deflated]: blocks of
// 64 rows x 16 destination columns, four independent copies per thread (grid z
// over merges; a thread that copied 64 columns one by one took 12-16 us).
__global__ __launch_bounds__(256) void dc_gather_kernel(const MergeDesc *__restrict__ md,
                                                        const MergeOut *__restrict__ mo, const double *__restrict__ Z,
                                                        long ldz, DCScratch sc, long ldq) {
  const MergeDesc m = md[blockIdx.z];
  const int N = m.n1 + m.n2, st = m.start;
  const int r = blockIdx.x * 64 + (threadIdx.x & 63);
  const int c0 = blockIdx.y * 16 + (threadIdx.x >> 6);
  if (r >= N || c0 >= N) return;
  const int K = mo[blockIdx.z].K;
  const double *Zb = Z + ((long)m.pad * sc.zmul + st + (long)st * ldz);
  double *Qc = sc.Qc + ((long)m.pad * sc.qmul + st + (long)st * ldq);
  int src[4], dst[4];
  double v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int k = min(c0 + 4 * i, N - 1);
    src[i] = k < K ? sc.nd_col[st + k] : sc.df_col[st + (k - K)];
    dst[i] = k < K ? sc.qpos[st + k] : k;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = Zb[r + (long)src[i] * ldz];
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (c0 + 4 * i < N) Qc[r + (long)dst[i] * ldq] = v[i];
}

// f(tau) pieces relative to pole `org`: psi over poles <= lower, phi over the rest.
// The secular function and its split derivatives at d[org] + tau, summed by W
// lanes: lane l takes poles l, l + W, ...; a butterfly allreduce leaves the same
// sums in every lane, so the root iteration stays uniform.  For K <= 16 both forms
// give the same bits: the butterfly's steps over lanes without a pole add zeros.
template <int W>
__device__ inline void secular_eval(const double *__restrict__ d, const double *__restrict__ z, int K, int org,
                                    int lower, double tau, double rho, double &f, double &psi, double &dpsi,
                                    double &phi, double &dphi, int lane) {
  static_assert(W == 64 || W == 16, "a wave or a row of lanes");
  const double dorg = d[org];
  psi = dpsi = phi = dphi = 0.0;
  for (int k = lane; k < K; k += W) {
    const double del = (d[k] - dorg) - tau;
    const double zk = z[k];
    const double t = zk / del;
    const double term = zk * t;
    const double dterm = t * t;
    if (k <= lower) {
      psi += term;
      dpsi += dterm;
    } else {
      phi += term;
      dphi += dterm;
    }
  }
  psi = W == 64 ? wave_sum(psi) : row_sum16(psi);
  dpsi = W == 64 ? wave_sum(dpsi) : row_sum16(dpsi);
  phi = W == 64 ? wave_sum(phi) : row_sum16(phi);
  dphi = W == 64 ? wave_sum(dphi) : row_sum16(dphi);
  psi *= rho;
  dpsi *= rho;
  phi *= rho;
  dphi *= rho;
  f = 1.0 + psi + phi;
}

// Root i of the secular equation by W lanes: lambda = d[org] + tau.  Returns
// whether the iteration converged.
template <int W>
__device__ inline bool secular_root(const double *__restrict__ d, const double *__restrict__ z, int K, int i,
                                    double rho, double zsum, int lane, int &org, double &tau) {
  const double eps = DBL_EPSILON * 0.5;
  double lo, hi;
  if (i < K - 1) {
    const double gap = d[i + 1] - d[i];
    const double mid = 0.5 * gap;
    double f, psi, dpsi, phi, dphi;
    secular_eval<W>(d, z, K, i, i, mid, rho, f, psi, dpsi, phi, dphi, lane);
    if (f >= 0.0) {
      org = i;
      lo = 0.0;
      hi = mid;
    } else {
      org = i + 1;
      lo = mid - gap;  // relative to d[i+1]
      hi = 0.0;
    }
  } else {
    org = K - 1;
    lo = 0.0;
    hi = rho * zsum;
    if (hi <= 0.0) hi = rho;
  }
  const int lower = i;  // poles d[0..i] lie below the root
  tau = 0.5 * (lo + hi);
  bool conv = false;
  for (int it = 0; it < 200; it++) {
    double f, psi, dpsi, phi, dphi;
    secular_eval<W>(d, z, K, org, lower, tau, rho, f, psi, dpsi, phi, dphi, lane);
    if (f < 0.0)
      lo = tau;
    else
      hi = tau;
    const double erretm = 10.0 * (fabs(psi) + fabs(phi)) + 4.0;
    if (fabs(f) <= eps * erretm || (hi - lo) <= 4.0 * eps * fmax(fabs(lo), fabs(hi))) {
      conv = true;
      break;
    }
    // two-pole rational model around the current point
    const double dl = (d[i] - d[org]) - tau;  // < 0
    double tn;
    bool ok = false;
    if (i < K - 1) {
      const double du = (d[i + 1] - d[org]) - tau;  // > 0
      const double q = dl * dl * dpsi, s = du * du * dphi;
      const double C = f - dl * dpsi - du * dphi;
      const double a2 = C, a1 = -(C * (dl + du) + q + s), a0 = C * dl * du + q * du + s * dl;
      double eta = 0.0;
      if (fabs(a2) < 1e-300) {
        if (a1 != 0.0) {
          eta = -a0 / a1;
          ok = true;
        }
      } else {
        const double disc = a1 * a1 - 4.0 * a2 * a0;
        if (disc >= 0.0) {
          const double sq = sqrt(disc);
          const double qq = -0.5 * (a1 + (a1 >= 0.0 ? sq : -sq));
          const double r1 = qq / a2;
          const double r2 = (qq != 0.0) ? a0 / qq : r1;
          const bool in1 = (r1 > dl && r1 < du), in2 = (r2 > dl && r2 < du);
          if (in1 && (!in2 || fabs(r1) <= fabs(r2))) {
            eta = r1;
            ok = true;
          } else if (in2) {
            eta = r2;
            ok = true;
          }
        }
      }
      tn = tau + eta;
    } else {
      // single pole below: C + q/(dl - eta) = 0
      const double q = dl * dl * dpsi;
      const double C = f - dl * dpsi;
      if (C > 0.0) {
        tn = tau + dl + q / C;
        ok = true;
      } else {
        tn = tau;
      }
    }
    if (!ok || !(tn > lo && tn < hi)) tn = 0.5 * (lo + hi);
    if (tn == tau || tn <= lo || tn >= hi) {
      // the bracket cannot be split further in FP64: tau is as good as it gets
      conv = true;
      break;
    }
    tau = tn;
  }
  return conv;
}

__global__ void dc_secular_kernel(const MergeDesc *__restrict__ md, const MergeOut *__restrict__ mo, DCScratch sc,
                                  unsigned *err) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  const int st = m.start, K = o.K;
  const double *d = sc.nd_d + st, *z = sc.nd_z + st;
  // one wave per root
  const int waves = blockDim.x >> 6, lane = threadIdx.x & 63;
  for (int i = blockIdx.x * waves + (threadIdx.x >> 6); i < K; i += gridDim.x * waves) {
    int org;
    double tau;
    const bool conv = secular_root<64>(d, z, K, i, o.rho2, o.zsum, lane, org, tau);
    if (lane == 0) {
      if (!conv) atomicOr(err, kErrNoconverge);
      sc.orig[st + i] = org;
      sc.tau[st + i] = tau;
      sc.lam[st + i] = d[org] + tau;
    }
  }
}

// zhat_j^2 = prod_i (lambda_i - d_j) / (rho prod_{k != j} (d_k - d_j)), the factor
// of j first, then those of k = 0, 1, ... in order: one wave per four j.  Lane l
// divides for k = k0 + l, then the wave multiplies the 64 quotients of each j in
// order (j by lane & 3).  The divisions are what takes the time, the products
// only K dependent multiplications; the order of the products decides the last
// bits of zhat, and with them what the next merge deflates.  n = 2500: 124 us over
// eight levels (a thread per j, which also divided: 73 us at the top one alone;
// products of every 64th quotient, in another order: 74 us over all).
constexpr int kLoewnerJ = 4;
__global__ __launch_bounds__(256) void dc_loewner_kernel(const MergeDesc *__restrict__ md,
                                                         const MergeOut *__restrict__ mo, DCScratch sc) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  const int st = m.start, K = o.K, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double *d = sc.nd_d + st, *z = sc.nd_z + st;
  const int *orig = sc.orig + st;
  const double *tau = sc.tau + st;
  __shared__ double quot[4][kLoewnerJ][65];
  for (int j0 = (blockIdx.x * 4 + wave) * kLoewnerJ; j0 < K; j0 += gridDim.x * 4 * kLoewnerJ) {
    const int jl = min(j0 + (lane & (kLoewnerJ - 1)), K - 1);
    double prod = ((d[orig[jl]] - d[jl]) + tau[jl]) / o.rho2;  // (lambda_j - d_j) / rho
    for (int k0 = 0; k0 < K; k0 += 64) {
      const int k = min(k0 + lane, K - 1);
      const double dk = d[k], ok = d[orig[k]], tk = tau[k];
#pragma unroll
      for (int u = 0; u < kLoewnerJ; u++) {
        const int j = min(j0 + u, K - 1);
        const double dj = d[j];
        quot[wave][u][lane] = (k == j || k0 + lane >= K) ? 1.0 : ((ok - dj) + tk) / (dk - dj);
      }
      lds_order();
#pragma unroll 16
      for (int t = 0; t < 64; t++) prod *= quot[wave][lane & (kLoewnerJ - 1)][t];
      lds_order();
    }
    const double zh = sqrt(fabs(prod));
    if (lane < kLoewnerJ && j0 + lane < K) sc.zhat[st + jl] = (z[jl] >= 0.0) ? zh : -zh;
  }
}

// Ascending position of element t of [lambda (K) ; deflated (nd)]: the new D
// and the column maps.
__device__ inline void merged_position(int t, int st, int K, int nd, const DCScratch &sc, double *__restrict__ D) {
  const double *lam = sc.lam + st, *df = sc.df_d + st;
  if (t < K) {
    const double v = lam[t];
    int lo = 0, hi = nd;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (df[mid] < v)
        lo = mid + 1;
      else
        hi = mid;
    }
    const int pos = t + lo;
    D[st + pos] = v;
    sc.colmap[st + t] = st + pos;
  } else {
    const int u = t - K;
    const double v = df[u];
    int lo = 0, hi = K;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (lam[mid] <= v)
        lo = mid + 1;
      else
        hi = mid;
    }
    const int pos = u + lo;
    D[st + pos] = v;
    sc.dmap[st + u] = st + pos;
  }
}

// Grouped-GEMM problems of one merge, from its deflation results: problem 2i
// is the top rows (Qc[:, 0:K1+K2]), 2i+1 the bottom rows (Qc[:, K1:K]).  Tile
// offsets are fixed per level from the bound K <= N; tiles past a problem's
// actual K columns exit at once, and a merge with K = 0 gets m = 0.
__device__ inline void merge_problems(int i, const MergeDesc &m, const MergeOut &o, const int *__restrict__ tile_begin,
                                      const DCScratch &sc, long ldq, double *Z, long ldz,
                                      DGemmProblem *__restrict__ probs) {
  const int st = m.start;
  const long zsh = (long)m.pad * sc.zmul, qsh = (long)m.pad * sc.qmul;
  DGemmProblem top;
  top.m = o.K > 0 ? m.n1 : 0;
  top.n = o.K;
  top.k = o.K1 + o.K2;
  top.tile_begin = tile_begin[2 * i];
  top.A = sc.Qc + (qsh + st + (long)st * ldq);
  top.lda = ldq;
  top.B = sc.Uc + (qsh + st + (long)st * ldq);
  top.ldb = ldq;
  top.C = Z + (zsh + st);
  top.ldc = ldz;
  top.colmap = sc.colmap + st;
  probs[2 * i] = top;
  DGemmProblem bot;
  bot.m = o.K > 0 ? m.n2 : 0;
  bot.n = o.K;
  bot.k = o.K2 + o.K3;
  bot.tile_begin = tile_begin[2 * i + 1];
  bot.A = sc.Qc + (qsh + (st + m.n1) + (long)(st + o.K1) * ldq);
  bot.lda = ldq;
  bot.B = sc.Uc + (qsh + (st + o.K1) + (long)st * ldq);
  bot.ldb = ldq;
  bot.C = Z + (zsh + st + m.n1);
  bot.ldc = ldz;
  bot.colmap = sc.colmap + st;
  probs[2 * i + 1] = bot;
}

// One workgroup per index i < N of one merge: eigenvector column i (Uc[qpos[j],
// i], i < K), the position of element i in the merged order, and once per merge
// its two product problems.
__global__ __launch_bounds__(256) void dc_vectors_kernel(const MergeDesc *__restrict__ md,
                                                         const MergeOut *__restrict__ mo, DCScratch sc, long ldu,
                                                         double *__restrict__ D, const int *__restrict__ tile_begin,
                                                         double *Z, long ldz, DGemmProblem *__restrict__ probs) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  const int st = m.start, K = o.K;
  const int i = blockIdx.x;
  if (threadIdx.x == 0 && i < K + o.ndefl) merged_position(i, st, K, o.ndefl, sc, D);
  if (threadIdx.x == 64 && i == 0) merge_problems(blockIdx.y, m, o, tile_begin, sc, ldu, Z, ldz, probs);
  if (i >= K) return;
  const double *d = sc.nd_d + st;
  const double dorg = d[sc.orig[st + i]];
  const double ti = sc.tau[st + i];
  double *Uc = sc.Uc + ((long)m.pad * sc.qmul + st + (long)st * ldu);
  __shared__ double red[4];
  double ss = 0.0;
  for (int j = threadIdx.x; j < K; j += 256) {
    const double v = sc.zhat[st + j] / ((d[j] - dorg) - ti);
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const double inv = 1.0 / sqrt(red[0] + red[1] + red[2] + red[3]);
  for (int j = threadIdx.x; j < K; j += 256) {
    const double v = sc.zhat[st + j] / ((d[j] - dorg) - ti);
    Uc[sc.qpos[st + j] + (long)i * ldu] = v * inv;
  }
}

// Values only: the merge's two rows before the rotations (zero in the columns
// of the other child) and the rotations on them.  Rotation t acts on columns
// (p, n); its p is the n of rotation t - 1 or a column no rotation has touched,
// so wave 0 takes 64 rotations' data at once and passes one pair of values on
// from rotation to rotation.
__global__ __launch_bounds__(256) void dc_rows_rotate_kernel(const MergeDesc *__restrict__ md,
                                                             const MergeOut *__restrict__ mo, DCScratch sc,
                                                             DCRows rows) {
  const MergeDesc m = md[blockIdx.x];
  const int N = m.n1 + m.n2, st = m.start, nrot = mo[blockIdx.x].nrot, tid = threadIdx.x;
  double *rf = rows.rot_first + st, *rl = rows.rot_last + st;
  for (int c = tid; c < N; c += 256) {
    rf[c] = c < m.n1 ? rows.first[st + c] : 0.0;
    rl[c] = c < m.n1 ? 0.0 : rows.last[st + c];
  }
  __syncthreads();
  if (tid >= 64) return;
  const int lane = tid;
  double cf = 0.0, cl = 0.0;  // the rotated n column of the previous rotation
  int cn = -1;
  auto of_lane = [](double v, int i) {
    const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)x, i);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(x >> 32), i);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
  };
  for (int t0 = 0; t0 < nrot; t0 += 64) {
    const int cnt = min(64, nrot - t0);
    const bool on = lane < cnt;
    const int p = on ? sc.rot_p[st + t0 + lane] : -1, n = on ? sc.rot_n[st + t0 + lane] : -1;
    const double c = on ? sc.rot_c[st + t0 + lane] : 1.0, s = on ? sc.rot_s[st + t0 + lane] : 0.0;
    const double pf = on ? rf[p] : 0.0, pl = on ? rl[p] : 0.0, nf = on ? rf[n] : 0.0, nl = on ? rl[n] : 0.0;
    double of = 0.0, ol = 0.0, qf = 0.0, ql = 0.0;
    for (int i = 0; i < cnt; i++) {
      const bool chained = __builtin_amdgcn_readlane(p, i) == cn;
      const double ci = of_lane(c, i), si = of_lane(s, i);
      const double xf = chained ? cf : of_lane(pf, i), xl = chained ? cl : of_lane(pl, i);
      const double yf = of_lane(nf, i), yl = of_lane(nl, i);
      cf = ci * yf - si * xf;
      cl = ci * yl - si * xl;
      cn = __builtin_amdgcn_readlane(n, i);
      if (lane == i) {
        of = ci * xf + si * yf;
        ol = ci * xl + si * yl;
        qf = cf;
        ql = cl;
      }
    }
    // column n's value first: where the next rotation takes it on as its p,
    // that rotation's store comes later (the next lane's below, or the next
    // round's)
    if (on) {
      const int pnext = __shfl_down(p, 1, 64);
      if (lane == cnt - 1 || pnext != n) {
        rf[n] = qf;
        rl[n] = ql;
      }
      rf[p] = of;
      rl[p] = ol;
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  }
}

// Values only: the merged node's two rows and the positions of its values, one
// wave per index i < N.  Vector i has the entries zhat_j / (d_j - lambda_i) over
// the non-deflated columns, so its first and last entries are two sums beside
// its norm's; a deflated column keeps its entries.
__global__ __launch_bounds__(256) void dc_rows_kernel(const MergeDesc *__restrict__ md, const MergeOut *__restrict__ mo,
                                                      DCScratch sc, DCRows rows, int sums, double *__restrict__ D) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  const int st = m.start, K = o.K, lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= K + o.ndefl) return;
  int pos = 0;
  if (lane == 0) {
    merged_position(i, st, K, o.ndefl, sc, D);
    pos = i < K ? sc.colmap[st + i] : sc.dmap[st + i - K];
  }
  if (!sums) return;
  const double *rf = rows.rot_first + st, *rl = rows.rot_last + st;
  if (i >= K) {
    if (lane == 0) {
      const int c = sc.df_col[st + i - K];
      rows.first[pos] = rf[c];
      rows.last[pos] = rl[c];
    }
    return;
  }
  const double *d = sc.nd_d + st;
  const double dorg = d[sc.orig[st + i]], ti = sc.tau[st + i];
  double ss = 0.0, a = 0.0, b = 0.0;
  for (int j = lane; j < K; j += 64) {
    const double v = sc.zhat[st + j] / ((d[j] - dorg) - ti);
    const int c = sc.nd_col[st + j];
    ss += v * v;
    a += v * rf[c];
    b += v * rl[c];
  }
  ss = wave_sum(ss);
  a = wave_sum(a);
  b = wave_sum(b);
  if (lane == 0) {
    const double inv = 1.0 / sqrt(ss);
    rows.first[pos] = a * inv;
    rows.last[pos] = b * inv;
  }
}

__global__ void dc_copy_deflated_kernel(const MergeDesc *__restrict__ md, const MergeOut *__restrict__ mo,
                                        DCScratch sc, long ldq, double *__restrict__ Z, long ldz) {
  const MergeDesc m = md[blockIdx.y];
  const MergeOut o = mo[blockIdx.y];
  const int st = m.start, N = m.n1 + m.n2;
  const long total = (long)N * o.ndefl;
  const double *Qc = sc.Qc + ((long)m.pad * sc.qmul + st + (long)st * ldq);
  const long zsh = (long)m.pad * sc.zmul;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int r = (int)(e % N);
    const int u = (int)(e / N);
    Z[zsh + (st + r) + (long)sc.dmap[st + u] * ldz] = Qc[r + (long)(o.K + u) * ldq];
  }
}

// One merge of a leaf's subtree.
struct LeafMerge {
  int off, n1, n2;  // rows off .. off + n1 - 1 and the n2 after them
  int K, K1, K2, ndefl;
  double rho2, zsum;
};

// The subtrees of the leaves: one workgroup per leaf of m <= kDcLeaf rows, the
// four tree levels below it one after the other in LDS, each step of a merge as the
// kernels of the levels above do it, operation for operation.  With it the tree ends
// at single rows, and the sign of every vector follows from the merges alone: a
// non-deflated one has v^T x < 0, a deflated one its child's sign, a single row is 1.
// (Leaves by the QR algorithm gave other signs to the vectors that deflate all
// the way up, and other last bits to the rest, which decide whether an entry at
// the edge of the deflation tolerance is deflated: 8 of 4.1 million vectors of order
// 256 changed sign.)
// A row of 16 lanes serves one merge in the sort and the deflation, and one
// root, one column and one position of the leaf in the other steps (16 rows of lanes,
// 16 positions): no step loops over more than the 16 poles of a merge.  As one
// launch instead of 4 x 8, which are bound by their launch gaps at these sizes.
// Bound by the chain of the roots' iterations.
__global__ __launch_bounds__(256) void dc_leaf_kernel(const LeafDesc *__restrict__ lf, const double *__restrict__ E,
                                                      double *__restrict__ D, double *__restrict__ Z, long ldz,
                                                      long zmul, DCRows rows, unsigned *__restrict__ err) {
  constexpr int L = kDcLeaf;
  __shared__ double e[L], d[L], ds[L], zs[L], sq[L], nd_d[L], nd_z[L], df_d[L], tmp_d[L], tau[L], lam[L], zhat[L];
  __shared__ double rot_c[L], rot_s[L], quot[L][L + 1];
  __shared__ double V[L][L + 1], Q[L][L + 1], U[L][L + 1];  // by column
  __shared__ int cs[L], types[L], nd_col[L], qpos[L], df_col[L], tmp_c[L], cand[L], rot_p[L], rot_n[L], org[L], pos[L];
  __shared__ LeafMerge mg[L / 2];
  const LeafDesc leaf = lf[blockIdx.x];
  const int m = leaf.size, st = leaf.start, tid = threadIdx.x, g = tid >> 4, l = tid & 15;
  const int lane = tid & 63, wave = tid >> 6;
  // the votes of this row of lanes
  auto votes = [&](bool p) { return (unsigned)(__ballot(p) >> (16 * (g & 3))) & 0xffffu; };
  const unsigned below = (1u << l) - 1u;
  if (tid < m) {
    d[tid] = D[st + tid];
    e[tid] = tid < m - 1 ? E[st + tid] : 0.0;
  }
  if (g < m) V[g][l] = (g == l) ? 1.0 : 0.0;
  __syncthreads();
  for (int depth = 3; depth >= 0; depth--) {
    if ((m + (1 << depth) - 1) >> depth < 2) continue;  // no node of this depth has two rows
    // ---- node g of this depth: sort and deflation
    if (g < (1 << depth)) {
      int off = 0, N = m;
      for (int b = depth - 1; b >= 0; b--) {
        const int n1 = N / 2;
        if ((g >> b) & 1) {
          off += n1;
          N -= n1;
        } else {
          N = n1;
        }
      }
      LeafMerge o;
      o.off = off;
      o.n1 = N / 2;
      o.n2 = N - o.n1;
      o.K = o.K1 = o.K2 = o.ndefl = 0;
      o.rho2 = o.zsum = 0.0;
      if (N >= 2) {
        const double es = e[off + o.n1 - 1];
        const double rho = 2.0 * fabs(es);
        o.rho2 = rho;
        if (l < N) {
          // every place holds a column also where a NaN leaves one out below
          ds[off + l] = d[off + l];
          zs[off + l] = 0.0;
          cs[off + l] = l;
          lds_order();
          const double dv = d[off + l];
          double z;
          int at = 0;
          if (l < o.n1) {
            z = V[off + l][off + o.n1 - 1];
            for (int i = 0; i < o.n2; i++) at += d[off + o.n1 + i] < dv ? 1 : 0;
            at += l;
          } else {
            z = ((es >= 0.0) ? 1.0 : -1.0) * V[off + l][off + o.n1];
            for (int i = 0; i < o.n1; i++) at += d[off + i] <= dv ? 1 : 0;
            at += l - o.n1;
          }
          ds[off + at] = dv;
          zs[off + at] = z * 0.70710678118654752440;
          cs[off + at] = l;
          types[off + l] = (l < o.n1) ? 1 : 3;
        }
        lds_order();
        const double dl = l < N ? ds[off + l] : 0.0, zl = l < N ? zs[off + l] : 0.0;
        const double dmax = row_max16(fabs(dl)), zmax = row_max16(fabs(zl));
        const double eps = DBL_EPSILON * 0.5;
        const double tol = 8.0 * eps * fmax(dmax, zmax);
        const bool zd = l < N && (rho * zmax <= tol || rho * fabs(zl) <= tol), cd = l < N && !zd;
        const unsigned mz = votes(zd), mc = votes(cd);
        const int nzd = __popc(mz), nc = __popc(mc);
        if (zd) {
          df_d[off + __popc(mz & below)] = dl;
          df_col[off + __popc(mz & below)] = cs[off + l];
        }
        if (cd) cand[off + __popc(mc & below)] = l;
        lds_order();
        // pairs of neighbours in order: all before the first rotation, the
        // rotation, the rest after it
        int K = 0, nrot = 0, pj = nc > 0 ? cand[off] : -1, k = 1;
        while (k < nc) {
          const int nvalid = nc - k;
          const bool valid = l < nvalid;
          const int j = valid ? cand[off + k + l] : 0;
          const int prv = (l == 0) ? pj : (valid ? cand[off + k + l - 1] : 0);
          bool rot = false;
          double c = 0.0, sn = 0.0, ta = 0.0;
          if (valid) {
            sn = zs[off + prv];
            c = zs[off + j];
            ta = hypot(c, sn);
            const double t = ds[off + j] - ds[off + prv];
            c /= ta;
            sn = -sn / ta;
            rot = fabs(t * c * sn) <= tol;
          }
          const unsigned mask = votes(rot);
          const int first = mask ? __ffs((int)mask) - 1 : nvalid;
          if (l < first) {
            nd_d[off + K + l] = ds[off + prv];
            nd_z[off + K + l] = zs[off + prv];
            nd_col[off + K + l] = cs[off + prv];
          }
          K += first;
          if (first < nvalid) {
            if (l == first) {
              zs[off + j] = ta;
              zs[off + prv] = 0.0;
              const int cp = cs[off + prv], cn = cs[off + j];
              if (types[off + cp] != types[off + cn]) types[off + cn] = 2;
              types[off + cp] = 4;
              rot_p[off + nrot] = cp;
              rot_n[off + nrot] = cn;
              rot_c[off + nrot] = c;
              rot_s[off + nrot] = sn;
              const double tt = ds[off + prv] * c * c + ds[off + j] * sn * sn;
              ds[off + j] = ds[off + prv] * sn * sn + ds[off + j] * c * c;
              ds[off + prv] = tt;
              df_d[off + nzd + nrot] = tt;
              df_col[off + nzd + nrot] = cp;
            }
            nrot++;
            pj = __shfl(j, first, 16);
            k += first + 1;
            lds_order();
          } else {
            pj = __shfl(j, nvalid - 1, 16);
            k = nc;
          }
        }
        if (pj >= 0) {
          if (l == 0) {
            nd_d[off + K] = ds[off + pj];
            nd_z[off + K] = zs[off + pj];
            nd_col[off + K] = cs[off + pj];
          }
          K++;
        }
        lds_order();
        const int nd = nzd + nrot;
        if (nrot > 0) {
          // the rotations on the vectors' columns, one row per lane
          if (l < N)
            for (int t = 0; t < nrot; t++) {
              const double x = V[off + rot_p[off + t]][off + l], y = V[off + rot_n[off + t]][off + l];
              const double c = rot_c[off + t], s = rot_s[off + t];
              V[off + rot_p[off + t]][off + l] = c * x + s * y;
              V[off + rot_n[off + t]][off + l] = c * y - s * x;
            }
          // deflated list ascending: the rotated entries among themselves, then
          // merged with the z-deflated run (ties keep the run first)
          if (l < nd) {
            const double v = df_d[off + l];
            int at = 0;
            tmp_d[off + l] = v;
            tmp_c[off + l] = df_col[off + l];
            lds_order();
            if (l < nzd) {
              at = l;
              for (int i = nzd; i < nd; i++) at += df_d[off + i] < v ? 1 : 0;
            } else {
              for (int i = 0; i < nzd; i++) at += df_d[off + i] <= v ? 1 : 0;
              for (int i = nzd; i < nd; i++)
                at += (df_d[off + i] < v || (df_d[off + i] == v && i < l)) ? 1 : 0;
            }
            tmp_d[off + at] = v;
            tmp_c[off + at] = df_col[off + l];
          }
          lds_order();
          if (l < nd) {
            df_d[off + l] = tmp_d[off + l];
            df_col[off + l] = tmp_c[off + l];
          }
        }
        // types, positions by type, sum of the squares in order
        const int ty = l < K ? types[off + nd_col[off + l]] : 0;
        const unsigned m1 = votes(ty == 1), m2 = votes(ty == 2), m3 = votes(ty == 3);
        o.K = K;
        o.K1 = __popc(m1);
        o.K2 = __popc(m2);
        o.ndefl = nd;
        if (l < K) {
          qpos[off + l] = (ty == 1)   ? __popc(m1 & below)
                          : (ty == 2) ? o.K1 + __popc(m2 & below)
                                      : o.K1 + o.K2 + __popc(m3 & below);
          sq[off + l] = nd_z[off + l] * nd_z[off + l];
        }
        lds_order();
        for (int i = 0; i < K; i++) o.zsum += sq[off + i];
      }
      if (l == 0) mg[g] = o;
    }
    __syncthreads();
    // ---- position g: its node, its column, its root
    int node = 0, off = 0, N = m;
    for (int b = 0; b < depth; b++) {
      const int n1 = N / 2, right = g - off >= n1 ? 1 : 0;
      node = 2 * node + right;
      off += right ? n1 : 0;
      N = right ? N - n1 : n1;
    }
    const bool on = g < m && N >= 2;
    const LeafMerge o = mg[node];
    const int i = g - off, K = o.K;
    if (on) {
      const int src = i < K ? nd_col[off + i] : df_col[off + i - K], dst = i < K ? qpos[off + i] : i;
      if (l < N) Q[off + dst][off + l] = V[off + src][off + l];
      if (i < K) {
        int og;
        double t;
        const bool conv = secular_root<16>(nd_d + off, nd_z + off, K, i, o.rho2, o.zsum, l, og, t);
        if (l == 0) {
          if (!conv) atomicOr(err, kErrNoconverge);
          org[g] = og;
          tau[g] = t;
          lam[g] = nd_d[off + og] + t;
        }
      }
    }
    __syncthreads();
    if (on && i < K) {
      const double dj = nd_d[off + i];
      if (l < K) {
        const double lk = (nd_d[off + org[off + l]] - dj) + tau[off + l];
        quot[g][l] = lk / (l == i ? o.rho2 : nd_d[off + l] - dj);
      }
      lds_order();
      double prod = quot[g][i];
      for (int k = 0; k < K; k++)
        if (k != i) prod *= quot[g][k];
      const double zh = sqrt(fabs(prod));
      if (l == 0) zhat[g] = (nd_z[g] >= 0.0) ? zh : -zh;
    }
    __syncthreads();
    if (on) {
      int at = i < K ? i : i - K;
      if (i < K) {
        const double dorg = nd_d[off + org[g]], ti = tau[g];
        const double v = l < K ? zhat[off + l] / ((nd_d[off + l] - dorg) - ti) : 0.0;
        // the square rounded by itself, as where it is added to a sum of zero
        const double inv = 1.0 / sqrt(row_sum16(__builtin_fma(v, v, 0.0)));
        if (l < K) U[g][qpos[off + l]] = v * inv;
        for (int u = 0; u < o.ndefl; u++) at += df_d[off + u] < lam[g] ? 1 : 0;
      } else {
        for (int u = 0; u < K; u++) at += lam[off + u] <= df_d[g - K] ? 1 : 0;
      }
      if (l == 0) {
        pos[g] = off + at;
        d[off + at] = i < K ? lam[g] : df_d[g - K];
      }
    }
    __syncthreads();
    // ---- vectors: columns that deflated keep theirs, the others are products
    // with the rows of each child
    if (on && i >= K && l < N) V[pos[g]][off + l] = Q[g][off + l];
    for (int t = wave; t < (2 << depth); t += 4) {
      const LeafMerge p = mg[t >> 1];
      if (p.K == 0) continue;
      const int r0 = p.off + ((t & 1) ? p.n1 : 0), nr = (t & 1) ? p.n2 : p.n1;
      const int k0 = (t & 1) ? p.K1 : 0, nk = (t & 1) ? p.K - p.K1 : p.K1 + p.K2;
      const int r = lane & 15;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
      for (int ks = 0; ks < nk; ks += 4) {
        const int k = ks + (lane >> 4);
        const double a = (k < nk && r < nr) ? Q[p.off + k0 + k][r0 + r] : 0.0;
        const double b = (k < nk && r < p.K) ? U[p.off + r][k0 + k] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, acc, 0, 0, 0);
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int col = (lane >> 4) + 4 * c;
        if (r < nr && col < p.K) V[pos[p.off + col]][r0 + r] = acc[c];
      }
    }
    __syncthreads();
  }
  if (tid < m) D[st + tid] = d[tid];
  if (rows.first) {
    if (tid < m) {
      rows.first[st + tid] = V[tid][0];
      rows.last[st + tid] = V[tid][m - 1];
    }
    return;
  }
  double *Zb = Z + ((long)leaf.problem * zmul + st + (long)st * ldz);
  if (g < m && l < m) Zb[l + (long)g * ldz] = V[g][l];
}

struct TreeNode {
  int start, size, left, right, height;
};

static int build_tree(std::vector<TreeNode> &nodes, int start, int size) {
  int id = (int)nodes.size();
  nodes.push_back({start, size, -1, -1, 0});
  if (size > kDcLeaf) {
    int n1 = size / 2;
    int l = build_tree(nodes, start, n1);
    int r = build_tree(nodes, start + n1, size - n1);
    nodes[id].left = l;
    nodes[id].right = r;
    nodes[id].height = 1 + std::max(nodes[l].height, nodes[r].height);
  }
  return id;
}

// Merges of order >= kDcLibMinN form their FP64 products with rocBLAS (the
// library's dgemm runs these shapes at 71-75 TFLOP/s on MI355X, the grouped
// tile kernel here at about 48) when the host may read the level's
// deflation counts, i.e. outside graph capture; the product goes through a
// temporary of (n/2 + 1) x n doubles and is scattered to its columns.
constexpr long kDcLibMinN = 4096;
static size_t dc_lib_temp_words(long n) { return n >= kDcLibMinN ? (size_t)(n / 2 + 1) * n : 0; }

static size_t dc_per_problem(long n) {
  size_t b = 0;
  b += align256((size_t)n * n * sizeof(double)) * 2;  // Qc, Uc
  b += align256((size_t)n * sizeof(double)) * 12;
  b += align256((size_t)n * sizeof(int)) * 12;
  b += align256((size_t)n * sizeof(MergeOut));
  b += align256((size_t)2 * n * sizeof(DGemmProblem));
  return b;
}

// arena bytes of the values-only form (no matrices), count problems at a time
size_t stedc_values_workspace(int count, long n) {
  const int per = (int)std::max<long>(1, 65535 / ((n + 1) / 2));
  return (dc_per_problem(n) - align256((size_t)n * n * sizeof(double)) * 2 + align256((size_t)n * sizeof(double)) * 4) *
             (size_t)std::min(count, per) +
         (1 << 16);
}

size_t stedc_workspace(long n) { return dc_per_problem(n) + align256(dc_lib_temp_words(n) * sizeof(double)) + (1 << 16); }

// Merge plan of order n, built once per context: the tree (halving splits
// down to leaves), merges grouped by height, the leaves and the
// per-level tile offsets of the grouped GEMMs, copied to device memory that
// lives as long as the context.  Only the split values (rho, sign) change per
// solve; dc_rho_kernel writes them into the device descriptors.
int dc_plan(evd_ctx *ctx, long n, int count, const DcPlan **out) {
  const long key = n | ((long)count << 32);
  auto it = ctx->dc_plans.find(key);
  if (it != ctx->dc_plans.end()) {
    *out = &it->second;
    return 0;
  }
  if (ctx->capturing)
    return set_error(ctx, EVD_E_UNSUPPORTED, "D&C plan for %d x n = %ld missing during capture", count, n);
  std::vector<TreeNode> nodes;
  nodes.reserve(2 * n);
  build_tree(nodes, 0, (int)n);
  DcPlan plan;
  plan.H = nodes[0].height;
  const int H = plan.H;
  std::vector<std::vector<int>> by_height(H + 1);
  for (int i = 0; i < (int)nodes.size(); i++)
    by_height[nodes[i].height].push_back(i);
  std::vector<MergeDesc> all;
  std::vector<int> tiles;
  std::vector<LeafDesc> leaves;
  for (int q = 0; q < count; q++)
    for (int id : by_height[0]) leaves.push_back({(int)(q * n) + nodes[id].start, nodes[id].size, q});
  plan.nleaf = (int)leaves.size();
  plan.level_off.assign(H + 2, 0);
  plan.level_maxN.assign(H + 1, 0);
  plan.level_tiles.assign(H + 1, 0);
  auto ceil_div = [](int a, int b) { return (a + b - 1) / b; };
  for (int h = 1; h <= H; h++) {
    plan.level_off[h] = (int)all.size();
    int t = 0;
    for (int q = 0; q < count; q++)
    for (int id : by_height[h]) {
      const TreeNode &nd = nodes[id];
      MergeDesc m;
      m.start = (int)(q * n) + nd.start;
      m.n1 = nodes[nd.left].size;
      m.n2 = nodes[nd.right].size;
      m.pad = q;
      m.rho = 0.0;
      m.sgn = 1.0;
      all.push_back(m);
      const int N = m.n1 + m.n2, tn = ceil_div(N, kDGroupTile);
      plan.level_maxN[h] = std::max(plan.level_maxN[h], N);
      tiles.push_back(t);
      t += ceil_div(m.n1, kDGroupTile) * tn;
      tiles.push_back(t);
      t += ceil_div(m.n2, kDGroupTile) * tn;
    }
    plan.level_tiles[h] = t;
  }
  plan.level_off[H + 1] = (int)all.size();
  plan.nmerge = (int)all.size();
  const size_t b_md = align256(sizeof(MergeDesc) * all.size()), b_tiles = align256(sizeof(int) * tiles.size());
  std::vector<char> &host = plan.host;
  host.assign(b_md + b_tiles + sizeof(LeafDesc) * leaves.size(), 0);
  if (!all.empty()) memcpy(host.data(), all.data(), sizeof(MergeDesc) * all.size());
  if (!tiles.empty()) memcpy(host.data() + b_md, tiles.data(), sizeof(int) * tiles.size());
  memcpy(host.data() + b_md + b_tiles, leaves.data(), sizeof(LeafDesc) * leaves.size());
  // device copy: carved from the context's plan pool (one allocation for all
  // plans), else an allocation of its own; the upload is stream-ordered and
  // its source stays alive with the plan
  EVD_TRY(plan_pool_reserve(ctx, kPlanPoolBytes));
  const size_t need = align256(host.size());
  if (ctx->plan_pool_used + need <= ctx->plan_pool_bytes) {
    plan.dev = ctx->plan_pool + ctx->plan_pool_used;
    ctx->plan_pool_used += need;
  } else {
    EVD_HIP(ctx, hipMalloc(&plan.dev, host.size()));
    plan.own = true;
  }
  const hipError_t e = hipMemcpyAsync(plan.dev, host.data(), host.size(), hipMemcpyHostToDevice, ctx->stream);
  if (e != hipSuccess) {
    if (plan.own) hipFree(plan.dev);
    return set_error(ctx, EVD_E_HIP, "D&C plan upload failed: %s", hipGetErrorString(e));
  }
  auto ins = ctx->dc_plans.emplace(key, std::move(plan));
  *out = &ins.first->second;
  return 0;
}

int stedc_batched(evd_ctx *ctx, int count, long n, double *D, double *E, double *Z, long ldz, long zs);

int stedc(evd_ctx *ctx, long n, double *D, double *E, double *Z, long ldz) {
  return stedc_batched(ctx, 1, n, D, E, Z, ldz, 0);
}

size_t stedc_batched_workspace(int count, long n) {
  const int per = (int)std::max<long>(1, 65535 / ((n + 1) / 2));
  return dc_per_problem(n) * (size_t)std::min(count, per) + align256(dc_lib_temp_words(n) * sizeof(double)) +
         (1 << 16);
}

// C[:, colmap[j]] = T[:, j] (j < n, rows < m) of one merge product
__global__ void dc_scatter_cols_kernel(int m, int n, const double *__restrict__ T, double *__restrict__ C, long ldc,
                                       const int *__restrict__ colmap) {
  const long total = (long)m * n;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int r = (int)(e % m), j = (int)(e / m);
    const int oc = colmap ? colmap[j] : j;
    C[r + (long)oc * ldc] = T[e];
  }
}

// One merge level's products on rocBLAS: the problem list the device built
// (sizes from the deflation results) is read back, each product goes to the
// temporary T and is scattered to its output columns.  Per problem, so the
// problems of a batch get the arithmetic of their single solves.
static int dc_level_library(evd_ctx *ctx, const DGemmProblem *dprob, int nprob, double *T, size_t t_words) {
  std::vector<DGemmProblem> hp((size_t)nprob);
  EVD_HIP(ctx, hipMemcpyAsync(hp.data(), dprob, sizeof(DGemmProblem) * nprob, hipMemcpyDeviceToHost, ctx->stream));
  EVD_HIP(ctx, hipStreamSynchronize(ctx->stream));
  const double one = 1.0, zero = 0.0;
  if (rocblas_set_stream(ctx->blas, ctx->stream) != rocblas_status_success)
    return set_error(ctx, EVD_E_HIP, "rocblas_set_stream failed");
  for (const DGemmProblem &p : hp) {
    if (p.m <= 0 || p.n <= 0) continue;
    if ((size_t)p.m * p.n > t_words)
      return set_error(ctx, EVD_E_UNSUPPORTED, "D&C product %d x %d exceeds its temporary", p.m, p.n);
    if (p.k > 0) {
      const rocblas_status st = rocblas_dgemm(ctx->blas, rocblas_operation_none, rocblas_operation_none, p.m, p.n,
                                              p.k, &one, p.A, (rocblas_int)p.lda, p.B, (rocblas_int)p.ldb, &zero, T,
                                              p.m);
      if (st != rocblas_status_success)
        return set_error(ctx, EVD_E_HIP, "rocblas_dgemm(%d x %d x %d) failed: status %d", p.m, p.n, p.k, (int)st);
    } else {
      EVD_HIP(ctx, hipMemsetAsync(T, 0, sizeof(double) * p.m * p.n, ctx->stream));
    }
    const long total = (long)p.m * p.n;
    dc_scatter_cols_kernel<<<(unsigned)std::min<long>((total + 255) / 256, 8192), 256, 0, ctx->stream>>>(
        p.m, p.n, T, p.C, p.ldc, p.colmap);
    EVD_LAUNCHED(ctx);
  }
  return 0;
}

// `count` same-size tridiagonals (D, E of problem q at q n, Z at q zs): every
// merge level of all problems is one set of launches.  Each problem's merges
// and their arithmetic are those of its single solve.  Z = nullptr: eigenvalues
// only, by the two rows of each node's vectors that the merges read (O(n^2) work
// instead of O(n^3): n = 3001 1.74 -> 0.70 ms, n = 16384 70 -> 5.4 ms).
int stedc_batched(evd_ctx *ctx, int count, long n, double *D, double *E, double *Z, long ldz, long zs) {
  if (n <= 0 || count <= 0) return 0;
  if (n == 1) {
    for (int q = 0; Z && q < count; q++) EVD_TRY(set_identity_f64(ctx, Z + q * zs, 1, ldz));
    return 0;
  }
  // the merges of one level are a launch dimension (at most 65535)
  const int per = (int)std::max<long>(1, 65535 / ((n + 1) / 2));
  if (count > per) {
    for (int q0 = 0; q0 < count; q0 += per) {
      const int c = std::min(per, count - q0);
      EVD_TRY(stedc_batched(ctx, c, n, D + q0 * n, E + q0 * n, Z ? Z + q0 * zs : nullptr, ldz, zs));
    }
    return 0;
  }
  ArenaFrame frame(ctx);
  DCScratch sc;
  const long ldq = n, nt = n * count;
  const bool vec = Z != nullptr;
  DCRows rows;
  if (vec) {
    sc.Qc = arena_alloc_n<double>(ctx, (size_t)n * n * count);
    sc.Uc = arena_alloc_n<double>(ctx, (size_t)n * n * count);
    if (!sc.Qc || !sc.Uc) return EVD_E_NOMEM;
  } else {
    double **rbufs[] = {&rows.first, &rows.last, &rows.rot_first, &rows.rot_last};
    for (auto p : rbufs) *p = arena_alloc_n<double>(ctx, (size_t)nt);
    if (!rows.rot_last) return EVD_E_NOMEM;
  }
  double **dbufs[] = {&sc.ds, &sc.zs, &sc.nd_d, &sc.nd_z, &sc.df_d, &sc.rot_c, &sc.rot_s, &sc.tau, &sc.lam, &sc.zhat};
  for (auto p : dbufs) *p = arena_alloc_n<double>(ctx, (size_t)nt);
  int **ibufs[] = {&sc.cs, &sc.nd_col, &sc.qpos, &sc.df_col, &sc.rot_p, &sc.rot_n, &sc.types, &sc.orig, &sc.colmap, &sc.dmap};
  for (auto p : ibufs) *p = arena_alloc_n<int>(ctx, (size_t)nt);
  if (!sc.zhat || !sc.dmap) return EVD_E_NOMEM;
  sc.zmul = zs - n * (1 + ldz);
  sc.qmul = -n;

  const DcPlan *plan = nullptr;
  EVD_TRY(dc_plan(ctx, n, count, &plan));
  const int nmerge = plan->nmerge, H = plan->H;
  char *pdev = static_cast<char *>(plan->dev);
  MergeDesc *dmd = reinterpret_cast<MergeDesc *>(pdev);
  const int *dtiles = reinterpret_cast<const int *>(pdev + align256(sizeof(MergeDesc) * nmerge));
  const LeafDesc *dleaf = reinterpret_cast<const LeafDesc *>(reinterpret_cast<const char *>(dtiles) +
                                                             align256(sizeof(int) * 2 * nmerge));
  MergeOut *dmo = static_cast<MergeOut *>(arena_alloc(ctx, sizeof(MergeOut) * std::max(1, nmerge)));
  // temporary of the library products (large merges, eager solves)
  double *libT = nullptr;
  if (vec && ctx->blas && !ctx->tune.own_gemm && !ctx->capturing && dc_lib_temp_words(n) > 0) {
    libT = arena_alloc_n<double>(ctx, dc_lib_temp_words(n));
    if (!libT) return EVD_E_NOMEM;
  }
  DGemmProblem *dprob = static_cast<DGemmProblem *>(arena_alloc(ctx, sizeof(DGemmProblem) * 2 * std::max(1, nmerge)));
  double *nrm = arena_alloc_n<double>(ctx, (size_t)count);
  if (!dmo || !dprob || !nrm) return EVD_E_NOMEM;
  unsigned *err = ctx->ctrl + kCtrlError;

  // split values and signs, tearing of every split, then the leaves
  dc_normalize_kernel<<<(unsigned)count, 256, 0, ctx->stream>>>(n, D, E, nrm);
  EVD_LAUNCHED(ctx);
  dc_tear_kernel<<<(unsigned)std::min<long>((nt + 255) / 256, 1024), 256, 0, ctx->stream>>>(n, nt, E, D);
  EVD_LAUNCHED(ctx);
  if (nmerge > 0) {
    dc_rho_kernel<<<(unsigned)std::min((nmerge + 255) / 256, 1024), 256, 0, ctx->stream>>>(nmerge, dmd, E);
    EVD_LAUNCHED(ctx);
    // outside the leaves' diagonal blocks Z starts as zeros
    if (vec && zs == n * ldz)
      EVD_TRY(fill_f64(ctx, Z, n, n * count, ldz, 0.0));
    else
      for (int q = 0; vec && q < count; q++) EVD_TRY(fill_f64(ctx, Z + q * zs, n, n, ldz, 0.0));
  }
  dc_leaf_kernel<<<(unsigned)plan->nleaf, 256, 0, ctx->stream>>>(dleaf, E, D, Z, ldz, sc.zmul, rows, err);
  EVD_LAUNCHED(ctx);

  // Merges level by level (by height).  Launch shapes come from the largest
  // merge of the level; every kernel bounds its work by the deflation
  // results it reads on the device, so no level waits for the host.
  for (int h = 1; h <= H; h++) {
    const int off = plan->level_off[h], nm = plan->level_off[h + 1] - off;
    if (nm == 0) continue;
    const MergeDesc *lmd = dmd + off;
    MergeOut *lmo = dmo + off;
    const int maxN = plan->level_maxN[h];
    const unsigned gx = (unsigned)std::min(64, (maxN + 255) / 256);
    const bool sort_inline = maxN <= kDcSortInline;
    if (!sort_inline) {
      dc_sort_kernel<<<dim3(gx, nm), 256, 0, ctx->stream>>>(lmd, D, Z, ldz, sc, rows);
      EVD_LAUNCHED(ctx);
    }
    dc_deflate_kernel<<<nm, 256, 0, ctx->stream>>>(lmd, lmo, D, Z, ldz, sort_inline ? 1 : 0, sc, rows);
    EVD_LAUNCHED(ctx);
    if (vec) {
      dc_rotate_kernel<<<dim3(gx, nm), 256, 0, ctx->stream>>>(lmd, lmo, Z, ldz, sc);
      EVD_LAUNCHED(ctx);
      dc_gather_kernel<<<dim3((unsigned)((maxN + 63) / 64), (unsigned)((maxN + 15) / 16), nm), 256, 0, ctx->stream>>>(
          lmd, lmo, Z, ldz, sc, ldq);
      EVD_LAUNCHED(ctx);
    } else if (h < H) {
      dc_rows_rotate_kernel<<<nm, 256, 0, ctx->stream>>>(lmd, lmo, sc, rows);
      EVD_LAUNCHED(ctx);
    }
    const unsigned gw = (unsigned)std::min(16384, (maxN + 3) / 4);  // 4 roots (waves) per workgroup
    dc_secular_kernel<<<dim3(gw, nm), 256, 0, ctx->stream>>>(lmd, lmo, sc, err);
    EVD_LAUNCHED(ctx);
    if (vec || h < H) {  // the last merge's vectors are not needed for the values
      const unsigned gl = (unsigned)std::min(16384, (maxN + 4 * kLoewnerJ - 1) / (4 * kLoewnerJ));
      dc_loewner_kernel<<<dim3(gl, nm), 256, 0, ctx->stream>>>(lmd, lmo, sc);
      EVD_LAUNCHED(ctx);
    }
    if (!vec) {
      dc_rows_kernel<<<dim3((unsigned)((maxN + 3) / 4), nm), 256, 0, ctx->stream>>>(lmd, lmo, sc, rows, h < H ? 1 : 0, D);
      EVD_LAUNCHED(ctx);
      continue;
    }
    dc_vectors_kernel<<<dim3(maxN, nm), 256, 0, ctx->stream>>>(lmd, lmo, sc, ldq, D, dtiles + 2 * off, Z, ldz, dprob);
    EVD_LAUNCHED(ctx);
    if (libT && maxN >= kDcLibMinN && !ctx->capturing)
      EVD_TRY(dc_level_library(ctx, dprob, 2 * nm, libT, dc_lib_temp_words(n)));
    else
      EVD_TRY(dgemm_grouped(ctx, dprob, 2 * nm, plan->level_tiles[h]));
    const unsigned gd = (unsigned)std::min<long>(((long)maxN * maxN + 255) / 256, 1024);
    dc_copy_deflated_kernel<<<dim3(gd, nm), 256, 0, ctx->stream>>>(lmd, lmo, sc, ldq, Z, ldz);
    EVD_LAUNCHED(ctx);
  }
  dc_denormalize_kernel<<<dim3((unsigned)std::min<long>((n + 255) / 256, 64), (unsigned)count), 256, 0,
                          ctx->stream>>>(n, D, nrm);
  EVD_LAUNCHED(ctx);
  return 0;
}

}  // namespace evd

using namespace evd;

extern "C" int evd_stedc_f64(evd_ctx *ctx, long n, double *D, double *E, double *Z, long ldz) {
  if (!ctx) return -1;
  EVD_ARG(ctx, n >= 0, 2);
  EVD_ARG(ctx, D != nullptr || n == 0, 3);
  EVD_ARG(ctx, E != nullptr || n <= 1, 4);
  EVD_ARG(ctx, Z != nullptr || n == 0, 5);
  EVD_ARG(ctx, ldz >= std::max<long>(1, n), 6);
  if (ctx->arena_top == 0) EVD_TRY(arena_ensure(ctx, stedc_workspace(n)));
  EVD_TRY(stedc(ctx, n, D, E, Z, ldz));
  return check_device_error(ctx, "evd_stedc_f64");
}
