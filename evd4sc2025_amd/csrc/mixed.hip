// Mixed-size batches: problems of different orders solved as a few same-size
// batches.  The reference solves one matrix per process run
// (src/EVD/myEVD.cu:251-706); here each problem of order n is embedded in the
// next bucket order N of a ladder (64, 96, 128, 192, ..., 2^k, 3 * 2^(k-1))
//
//   P = [ A  0 ]      S = diag(s_1 .. s_{N-n}),  s_j > ||A||_inf >= lambda_max(A)
//       [ 0  S ]
//
// so the n smallest eigenvalues of P are those of A and their eigenvectors
// are [v; 0]: w(A) = w(P)[0:n] and Z(A) = Z(P)[0:n, 0:n].  Every bucket (and
// eigenvector flag) is one evd_syevd_batched_f32 solve, i.e. one launch per
// stage for all of its problems.  Orders above the largest bucket are solved
// one at a time, unpadded.  With b = 0 each bucket of order N runs at
// bandwidth min(32, N / 4) (16 and 24 for the two smallest buckets).
#include "common.hpp"

namespace evd {


namespace {

constexpr long kMaxBucket = 4096;

long bucket_order(long n) {
  long p = 64;
  while (true) {
    if (n <= p) return p;
    if (n <= p + p / 2) return p + p / 2;
    p *= 2;
  }
}

// norm[q] = max(norm[q], ||A_q||_inf) of the symmetric matrices held in the
// lower triangles: row i sums |A[i, 0:i]| + |A[i:n, i]|.  A workgroup takes 64
// rows of one problem (grid (ceil(N / 64), count)): lanes along the rows left of
// the diagonal block, a wave per column below.  The lower triangle is read
// twice, at unit stride both times; one workgroup a matrix with a thread per row
// (strided in the second part) took 909 us a group over the 17 groups of 40
// matrices of order 64 to 2048, this 76 us.
__global__ __launch_bounds__(256) void inf_norm_kernel(const long *__restrict__ n_of, float *const *__restrict__ A_of,
                                                       const long *__restrict__ lda_of, double *__restrict__ norm) {
  const int q = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long n = n_of[q], lda = lda_of[q], i0 = 64L * blockIdx.x;
  if (i0 >= n) return;
  const float *A = A_of[q];
  __shared__ double sum[4][64], below[64];
  const long i = i0 + lane;
  double s = 0.0;
  if (i < n)
    for (long j = w; j < i; j += 4) s += fabs((double)A[i + j * lda]);
  sum[w][lane] = s;
  for (int c = w; c < 64; c += 4) {
    double t = 0.0;
    if (i0 + c < n)
      for (long r = i0 + c + lane; r < n; r += 64) t += fabs((double)A[r + (i0 + c) * lda]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) below[c] = t;
  }
  __syncthreads();
  if (w > 0) return;
  s = ((sum[0][lane] + sum[1][lane]) + (sum[2][lane] + sum[3][lane])) + below[lane];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s = fmax(s, __shfl_xor(s, o, 64));
  // sums of magnitudes: their bits order as the values do (a NaN, which the
  // solve reports, counts as 0)
  if (lane == 0 && s > 0.0)
    atomicMax(reinterpret_cast<unsigned long long *>(norm + q), (unsigned long long)__double_as_longlong(s));
}

// P_q (N x N, column major, stride N^2): A_q's lower triangle in the
// top-left block, zeros elsewhere, s_j = (1.5 + j / (N - n)) (||A_q|| + tiny)
// on the padded diagonal.  grid (ceil(N / 256), N, count).
__global__ void pad_kernel(long N, const long *__restrict__ n_of, float *const *__restrict__ A_of,
                           const long *__restrict__ lda_of, const double *__restrict__ norm, float *__restrict__ P) {
  const int q = blockIdx.z;
  const long c = blockIdx.y, n = n_of[q], lda = lda_of[q];
  const float *A = A_of[q];
  float *Pq = P + (long)q * N * N;
  const double base = norm[q] + 1e-30;
  for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < N; r += (long)gridDim.x * blockDim.x) {
    float v = 0.f;
    if (r < n && c < n) {
      if (r >= c) v = A[r + c * lda];
    } else if (r == c) {
      v = (float)(base * (1.5 + (double)(r - n) / (double)(N - n)));
    }
    Pq[r + c * N] = v;
  }
}

// w_q[0:n] = wP_q[0:n]; Z_q = ZP_q[0:n, 0:n] (Z_q may be null).  grid
// (ceil(N / 256), N, count).
__global__ void unpad_kernel(long N, const long *__restrict__ n_of, const double *__restrict__ wP,
                             const float *__restrict__ ZP, double *const *__restrict__ w_of,
                             float *const *__restrict__ Z_of, const long *__restrict__ ldz_of) {
  const int q = blockIdx.z;
  const long c = blockIdx.y, n = n_of[q];
  if (c >= n) return;
  const long r0 = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (c == 0)
    for (long i = r0; i < n; i += (long)gridDim.x * blockDim.x) w_of[q][i] = wP[(long)q * N + i];
  float *Z = Z_of[q];
  if (!Z) return;
  const long ldz = ldz_of[q];
  for (long r = r0; r < n; r += (long)gridDim.x * blockDim.x) Z[r + c * ldz] = ZP[(long)q * N * N + r + c * N];
}

struct Group {
  long N;
  char jobz;
  std::vector<int> members;
};

// Groups of (bucket order, eigenvector flag) in first-appearance order, and
// the problems of orders above the largest bucket (solved alone, unpadded).
void plan_groups(const MixedArgs &a, std::vector<Group> &groups, std::vector<int> &alone) {
  for (int q = 0; q < a.count; q++) {
    const char jz = (a.jobz[q] == 'V' || a.jobz[q] == 'v') ? 'V' : 'N';
    if (a.n[q] > kMaxBucket) {
      alone.push_back(q);
      continue;
    }
    const long N = bucket_order(std::max<long>(a.n[q], a.b > 0 ? 2 * a.b : 64));
    auto it = std::find_if(groups.begin(), groups.end(), [&](const Group &g) { return g.N == N && g.jobz == jz; });
    if (it == groups.end()) {
      groups.push_back(Group{N, jz, {}});
      it = groups.end() - 1;
    }
    it->members.push_back(q);
  }
}

long group_band(const MixedArgs &a, const Group &g) { return a.b > 0 ? a.b : std::min<long>(32, g.N / 4); }
long group_nb(long bg) { return bg * std::max<long>(1, 1024 / bg); }

// Device descriptors of one group: six arrays of c 8-byte entries (n, lda,
// ldz, A, Z, w), each 256-byte aligned, back to back.
size_t group_desc_bytes(int c) { return 6 * align256((size_t)c * 8); }

// Arena bytes one group's solve takes beyond the descriptors.
size_t group_stage_bytes(const evd_ctx *ctx, const MixedArgs &a, const Group &g) {
  const int c = (int)g.members.size();
  const long N = g.N, bg = group_band(a, g);
  return align256((size_t)c * sizeof(double)) + align256((size_t)c * N * N * sizeof(float)) * (g.jobz == 'V' ? 2 : 1) +
         align256((size_t)c * N * sizeof(double)) + syevd_batched_call_workspace(ctx, c, N, bg, group_nb(bg), g.jobz);
}

// One group: row-sum norms, padded copies, one batched solve, the leading
// blocks back into the callers' buffers.  `desc` is the group's descriptor
// block on the device.  Enqueues only (no host round trip).
int solve_group(evd_ctx *ctx, const MixedArgs &a, const Group &g, const char *desc) {
  const int c = (int)g.members.size();
  const long N = g.N, bg = group_band(a, g);
  const bool vec = g.jobz == 'V';
  const size_t s = align256((size_t)c * 8);
  const long *dn = reinterpret_cast<const long *>(desc), *dlda = reinterpret_cast<const long *>(desc + s),
             *dldz = reinterpret_cast<const long *>(desc + 2 * s);
  float *const *dA = reinterpret_cast<float *const *>(desc + 3 * s);
  float *const *dZ = reinterpret_cast<float *const *>(desc + 4 * s);
  double *const *dw = reinterpret_cast<double *const *>(desc + 5 * s);
  EVD_TRY(arena_ensure(ctx, group_stage_bytes(ctx, a, g)));
  ArenaFrame frame(ctx);
  double *norm = arena_alloc_n<double>(ctx, c);
  float *P = arena_alloc_n<float>(ctx, (size_t)c * N * N);
  float *ZP = vec ? arena_alloc_n<float>(ctx, (size_t)c * N * N) : nullptr;
  double *wP = arena_alloc_n<double>(ctx, (size_t)c * N);
  if (!norm || !P || (vec && !ZP) || !wP) return EVD_E_NOMEM;
  EVD_TRY(fill_f64(ctx, norm, c, 1, c, 0.0));
  inf_norm_kernel<<<dim3((unsigned)((N + 63) / 64), (unsigned)c), 256, 0, ctx->stream>>>(dn, dA, dlda, norm);
  EVD_LAUNCHED(ctx);
  const dim3 grid((unsigned)((N + 255) / 256), (unsigned)N, (unsigned)c);
  pad_kernel<<<grid, 256, 0, ctx->stream>>>(N, dn, dA, dlda, norm, P);
  EVD_LAUNCHED(ctx);
  // the scaling of the input screen follows A's entries, not the pads: the
  // split-FP16 form scales each problem to max |a_ij| in [0.5, 1), and a
  // pad-driven scale would push A's entries toward FP16 subnormals (pads
  // <= 2.5 ||A||_inf <= 2.5 n max |a_ij| stay inside the FP16 range, and
  // the reduction never multiplies them with anything but exact zeros)
  std::vector<long> rows(c);
  for (int i = 0; i < c; i++) rows[i] = a.n[g.members[i]];
  struct AmaxRows {
    evd_ctx *c;
    AmaxRows(evd_ctx *c_, const long *r) : c(c_) { c->amax_rows = r; }
    ~AmaxRows() { c->amax_rows = nullptr; }
  } amax_rows(ctx, rows.data());
  EVD_TRY(syevd_batched_call(ctx, g.jobz, c, N, bg, group_nb(bg), P, N, N * N, wP, N, ZP, N, N * N));
  unpad_kernel<<<grid, 256, 0, ctx->stream>>>(N, dn, wP, ZP, dw, dZ, dldz);
  EVD_LAUNCHED(ctx);
  return 0;
}

}  // namespace

size_t mixed_desc_bytes(const MixedArgs &a) {
  std::vector<Group> groups;
  std::vector<int> alone;
  plan_groups(a, groups, alone);
  size_t bytes = 0;
  for (const Group &g : groups) bytes += group_desc_bytes((int)g.members.size());
  return bytes;
}

int mixed_upload(evd_ctx *ctx, const MixedArgs &a, char *dev) {
  std::vector<Group> groups;
  std::vector<int> alone;
  plan_groups(a, groups, alone);
  std::vector<char> host(mixed_desc_bytes(a));
  if (host.empty()) return 0;
  size_t off = 0;
  for (const Group &g : groups) {
    const int c = (int)g.members.size();
    const size_t s = align256((size_t)c * 8);
    const bool vec = g.jobz == 'V';
    for (int i = 0; i < c; i++) {
      const int q = g.members[i];
      const long ldz = vec ? a.ldz[q] : 1;
      float *Zq = vec ? a.Z[q] : nullptr;
      std::memcpy(&host[off + i * 8], &a.n[q], 8);
      std::memcpy(&host[off + s + i * 8], &a.lda[q], 8);
      std::memcpy(&host[off + 2 * s + i * 8], &ldz, 8);
      std::memcpy(&host[off + 3 * s + i * 8], &a.A[q], 8);
      std::memcpy(&host[off + 4 * s + i * 8], &Zq, 8);
      std::memcpy(&host[off + 5 * s + i * 8], &a.w[q], 8);
    }
    off += group_desc_bytes(c);
  }
  EVD_HIP(ctx, hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, ctx->stream));
  EVD_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the host block is released on return
  return 0;
}

size_t mixed_stage_bytes(const evd_ctx *ctx, const MixedArgs &a) {
  std::vector<Group> groups;
  std::vector<int> alone;
  plan_groups(a, groups, alone);
  size_t need = 0;
  for (const Group &g : groups) need = std::max(need, group_stage_bytes(ctx, a, g));
  for (int q : alone) need = std::max(need, syevd_call_workspace(ctx, a.n[q], a.b > 0 ? a.b : 32, 0, a.jobz[q]));
  return need;
}

int mixed_enqueue(evd_ctx *ctx, const MixedArgs &a, const char *dev) {
  std::vector<Group> groups;
  std::vector<int> alone;
  plan_groups(a, groups, alone);
  size_t off = 0;
  for (const Group &g : groups) {
    EVD_TRY(solve_group(ctx, a, g, dev + off));
    off += group_desc_bytes((int)g.members.size());
  }
  for (int q : alone)
    EVD_TRY(syevd_call(ctx, a.jobz[q], a.n[q], a.b > 0 ? a.b : 32, 0, a.A[q], a.lda[q], a.w[q], a.Z[q], a.ldz[q]));
  return 0;
}

int mixed_check(evd_ctx *ctx, const MixedArgs &a) {
  EVD_ARG(ctx, a.count >= 0, 2);
  EVD_ARG(ctx, a.count == 0 || (a.n && a.A && a.lda && a.w && a.Z && a.ldz && a.jobz), 3);
  EVD_ARG(ctx, a.b == 0 || a.b == 32 || a.b == 64, 10);  // 0: b = min(32, N / 4) for each bucket order N
  for (int q = 0; q < a.count; q++) {
    const bool vec = (a.jobz[q] == 'V' || a.jobz[q] == 'v');
    if (!(vec || a.jobz[q] == 'N' || a.jobz[q] == 'n')) return set_error(ctx, -9, "jobz[%d] invalid", q);
    if (a.n[q] < 1 || a.lda[q] < a.n[q] || !a.A[q] || !a.w[q] || (vec && (!a.Z[q] || a.ldz[q] < a.n[q])))
      return set_error(ctx, -3, "problem %d: invalid order, buffer or leading dimension", q);
  }
  return 0;
}

}  // namespace evd

using namespace evd;

extern "C" int evd_syevd_mixed_f32(evd_ctx *ctx, int count, const long *n, float *const *A, const long *lda,
                                   double *const *w, float *const *Z, const long *ldz, const char *jobz, long b) {
  if (!ctx) return -1;
  const MixedArgs a{count, n, A, lda, w, Z, ldz, jobz, b};
  EVD_TRY(mixed_check(ctx, a));
  if (ctx->arena_top != 0) return set_error(ctx, EVD_E_UNSUPPORTED, "evd_syevd_mixed_f32 cannot nest");
  const size_t desc = mixed_desc_bytes(a);
  EVD_TRY(arena_ensure(ctx, align256(desc) + mixed_stage_bytes(ctx, a)));
  ArenaFrame frame(ctx);
  char *dev = arena_alloc_n<char>(ctx, desc);
  if (desc && !dev) return EVD_E_NOMEM;
  EVD_TRY(mixed_upload(ctx, a, dev));
  EVD_TRY(mixed_enqueue(ctx, a, dev));
  return check_device_error(ctx, "evd_syevd_mixed_f32");
}
