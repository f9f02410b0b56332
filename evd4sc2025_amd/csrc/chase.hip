// Band -> tridiagonal bulge chasing (the role of chasing_kernel_one_timeV10
// in util/inc/bugle_chasingV10.h:21-392 and its driver src/EVD/myEVD.cu:365-451).
//
// Algorithm (same arithmetic as the reference): sweep s annihilates column s
// below the subdiagonal with a reflector of length <= b on rows s+1..s+b and
// chases the bulge down in steps of b rows.  One step at row p:
//   x = first column of B1 (the block left of the diagonal block), H = I - u u^T
//   with u = (x/||x|| + sign(x0) e1)/sqrt(|.|) so that ||u||^2 = 2 and
//   Hx = -sign(x0)||x|| e1;  B1 <- H B1;  S <- H S H (diagonal block);
//   N <- N H (block below S, which becomes the next B1 - the bulge).
// u is stored in U[p .. p+len-1, s] ("noBandU" layout, FP32).
//
// MI355X design: sweeps are handed out by atomic tickets, runs of consecutive
// ones to one XCD, in an order that leaves every sweep's predecessor finished
// or owned by a running workgroup, so no co-residency (cooperative launch) is
// needed.  A sweep does not update a band in memory: it receives the window of
// each of its steps from its predecessor as a message and sends the next
// sweep's windows on (chase_kernel below).  A message within an XCD goes
// through its L2 (plain stores, loads that pass the CU's cache by); one that
// crosses XCDs is device-coherent on both sides (sc1).
// Every wait is bounded by a watchdog so the grid always drains.
#include <climits>
#include <map>
#include <mutex>
#include <type_traits>

#include "common.hpp"

namespace evd {

// one progress word per 128-byte line: the word a sweep publishes is polled by
// its successor only, and words sharing a line would serialise unrelated
// sweeps' polls and stores on that line
constexpr long kComStride = 32;
constexpr unsigned kBufferWord3 = 0x00020000u;  // raw buffer descriptor: 32-bit data format

constexpr int kSc1 = 16;  // buffer-op cache policy: sc1, device-coherent

// byte offset past every band (< 2 GiB): the buffer range check drops the
// store or returns 0 for the load, so every lane issues every access
constexpr unsigned kOutOfRange = 0x80000000u;

__device__ __attribute__((always_inline)) inline double ld_band_at(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, byte_off, 0, kSc1));
}
template <int POLICY>
__device__ __attribute__((always_inline)) inline void st_band_at(__amdgpu_buffer_rsrc_t r, unsigned byte_off, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned, v),
                                        r, byte_off, 0, POLICY);
}

__device__ __attribute__((always_inline)) inline void grp_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __attribute__((always_inline)) inline void wave_lds_order() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// s_waitcnt with only the vector-memory count: vmcnt(N), N <= 63
template <int N>
__device__ __attribute__((always_inline)) inline void wait_vm() {
  static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// 64-bit DPP move of v (rows outside RM read 0)
template <int CTRL, int RM>
__device__ __attribute__((always_inline)) inline double dpp_f64(double v) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)x, CTRL, RM, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(x >> 32), CTRL, RM, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// v of lane ^ 32.  v_permlane32_swap exchanges one half of its destination
// with the other half of its source; with both operands v, one result holds
// this lane's own value and the other the partner's, so xor-ing out the own
// value leaves the partner's whichever half was exchanged.
__device__ __attribute__((always_inline)) inline double half_swap(double v) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
  const auto rl = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto rh = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  const unsigned plo = rl[0] ^ rl[1] ^ lo, phi = rh[0] ^ rh[1] ^ hi;
  return __builtin_bit_cast(double, ((unsigned long long)phi << 32) | plo);
}
// v of lane ^ 16 (v_permlane16_swap: the same, rows of 16 lanes)
__device__ __attribute__((always_inline)) inline double row_swap(double v) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
  const auto rl = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto rh = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  const unsigned plo = rl[0] ^ rl[1] ^ lo, phi = rh[0] ^ rh[1] ^ hi;
  return __builtin_bit_cast(double, ((unsigned long long)phi << 32) | plo);
}

// sum over aligned groups of W lanes (8 .. 64), returned in every lane of the
// group: each step adds the other half of a group whose halves already agree,
// so mirrors serve as exchanges
template <int W>
__device__ __attribute__((always_inline)) inline double group_sum(double v) {
  v += dpp_f64<0xb1, 0xf>(v);                  // quad_perm [1, 0, 3, 2]
  v += dpp_f64<0x4e, 0xf>(v);                  // quad_perm [2, 3, 0, 1]
  v += dpp_f64<0x141, 0xf>(v);                 // row_half_mirror
  if (W >= 16) v += dpp_f64<0x140, 0xf>(v);    // row_mirror
  if (W >= 32) v += row_swap(v);
  if (W >= 64) v += half_swap(v);
  return v;
}

// a b + c d with both products rounded, so that exchanging (a, d) and (b, c)
// gives the same bits: the two halves of a symmetric block stay equal
__device__ __attribute__((always_inline)) inline double sym_pair(double a, double b, double c, double d) {
#pragma clang fp contract(off)
  const double x = a * b, y = c * d;
  return x + y;
}

// Reflector of the chase (reference sign convention) from the column whose
// entry i is x in lane i (W entries, zeros past its length, repeated every W
// lanes): u = (x/||x|| + sign(x0) e1) / sqrt(|x0/||x|| + sign(x0)|), so that
// ||u||^2 = 2 and H x = beta e1.  Returns lane i's u_i; u0 = u_0.
template <int W>
__device__ __attribute__((always_inline)) inline double chase_reflector(double x, int lane, double &u0, double &beta) {
  const double nn = group_sum<W>(x * x);
  const unsigned long long xb = __builtin_bit_cast(unsigned long long, x);
  const double x0 = __builtin_bit_cast(double, ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(
                                                    (int)(unsigned)(xb >> 32), 0)
                                                << 32) |
                                                   (unsigned)__builtin_amdgcn_readlane((int)(unsigned)xb, 0));
  u0 = 0.0;
  beta = x0;
  if (!(nn > 0.0)) return 0.0;
  double inv, nrm, scl, root;
  rsqrt_sqrt(nn, inv, nrm);
  const double a = x0 * inv + (x0 >= 0.0 ? 1.0 : -1.0);
  rsqrt_sqrt(fabs(a), scl, root);
  beta = x0 >= 0.0 ? -nrm : nrm;
  u0 = a * scl;
  return (lane & (W - 1)) == 0 ? u0 : x * inv * scl;
}

// ---------------------------------------------------------------------------
// One workgroup per sweep in flight, 8 threads per row of a BW x BW block:
// thread (ri, kc) holds row ri, columns kc + 8 r.
//
// The chase is a chain of dependent steps and nothing else bounds it, so the
// kernel is built for the latency of that chain: the steps of a sweep, and the
// hand-off from a sweep to the next.
//
// Step.  The window -> q = N u (FMAs, a DPP sum over the row's 8 lanes) ->
// barrier -> the next column x = N[:, 0] - q u_0, its norm and the next u,
// which every wave forms for itself.  Everything else fills the waits: B1 <-
// H B1 and its part of a message need no window and come before it, the slot is
// emptied in the shadow of the reflector, and the rest of the message goes out
// with S(:, 0) and beta first, which complete what the next sweep waits for.
// b = 32, n = 6000: 21.1 -> 16.3 ms, n = 1000: 3.33 -> 2.46 ms; b = 64, n = 8192:
// 86.5 -> 67.7 ms.  B1 is the previous N, passed
// through LDS transposed, so that its column sums u^T B1 are row sums of a
// wave's own lanes as well.
//
// Hand-off.  Step (s + 1, j) works on the window of step (s, j) shifted by one
// row and column: S'(i, k) = S(i+1, k+1) of step (s, j), its last row and
// column from B1 and S(0, 0) of step (s, j+1); N'(i, k) = B1(i+1, k+1) of step
// (s, j+1), its last column from S(:, 0) and the next beta of that step, its
// last row zero otherwise.  Sweep s sends these elements as message j, in the
// order in which the receiver's threads load them (plane r of a block is
// element (i, 8 r + kc) at 8 i + kc), so every access of either side covers
// whole runs of lines; X is the same for column s + 1 below the diagonal, from
// which sweep s + 1 starts.  An empty slot holds kEmpty, a signalling NaN that
// no arithmetic returns: the receiver loads its window until no element is
// empty, so data and its arrival are one access and nobody waits for a store
// to complete, then a flag, then a load (n = 16384, b = 32: store 0.33-0.48 us,
// flag 0.5-0.66 us, loads behind it).  Having read a slot, the receiver empties it again.
// Slots are doubled by the sweep's parity, and reuse is safe by the order of
// the chain alone: a step's sends but those of B1 follow a barrier before which
// every wave has waited for loads issued after the previous step's empties
// (memory operations complete in order), so message j of sweep s, which S(:, 0)
// and beta complete at step (s, j + 1), proves that s has emptied slot j of the
// other parity; B1 goes to slot j - 1, which the step before proved empty.  In
// the last step, whose message nothing follows, a wave completes its empties
// before it sends (every wave that empties elements there sends some).  Only a
// sweep's first slots have no such message before them: the receiver waits for
// the predecessor's start word, set once it holds its own first window.
// What a sweep sends is exactly what the next one loads (both bounded by row
// < n), so no stale element stays behind.
//
// Measured against one workgroup per sweep on a band in HBM with progress
// words (window loads, stores and a flag in every step's chain): b = 32,
// n = 6000: 49.2 -> 25.6 ms, n = 16384: 137 -> 85 ms; b = 64, n = 8192:
// 156 -> 92 ms (with every message between XCDs, see below).
//
// Where the messages go decides the hand-off: from one XCD to another a store
// reaches a poll after 820 ns, through the XCD's own L2 after 340 ns (a message
// of 64 doubles sent to and fro).  So consecutive sweeps run on one XCD, each
// of which has a box of slots of its own: a slot of a box is only ever
// accessed through one L2.  All messages between
// XCDs -> this: b = 32: n = 1000 3.88 -> 3.33 ms, n = 6000 25.6 -> 21.1 ms,
// n = 16384 85.7 -> 59.6 ms; b = 64, n = 8192: 93.5 -> 86.5 ms.
//
// A batch of `count` same-size problems shares one launch, its units mixed.
template <int BW>
struct ChaseShape {
  static constexpr int EPT = BW / 8;    // window columns per thread
  static constexpr int NT = BW * 8;     // threads
  static constexpr int NW = NT / 64;    // waves
  // stride of the transposed N in LDS: 8 mod 32 doubles, so that a wave's
  // 8 x 8 elements fall on distinct banks in the write and in the read
  static constexpr int LD = BW + 8;
};

constexpr unsigned kEmptyHi = 0x7FF7A5C3u;  // high word of an empty slot element
constexpr int kXWords = 64;                 // doubles of an X slot

// message slots of one problem: [parity][slot][S planes, N planes], each
// parity followed by its X slot
__host__ __device__ inline long mail_plane(long b) { return 8 * b; }
__host__ __device__ inline long mail_slot(long b) { return 2 * ((b + 7) / 8) * mail_plane(b); }
__host__ __device__ inline long mail_slots(long n, long b) { return (n + b - 1) / b; }
__host__ __device__ inline long mail_half(long n, long b) { return mail_slots(n, b) * mail_slot(b) + kXWords; }

// Messages of parity 1 for sweep 0, from the band, into the box between XCDs
// (grid z = 0); everything else, the other boxes included, empty.
__global__ __launch_bounds__(256) void mail_fill_kernel(int n, int b, const double *__restrict__ band_all, long ldb,
                                                        long band_stride, double *__restrict__ mail_all,
                                                        double *__restrict__ boxes, double *__restrict__ D_all,
                                                        long d_stride) {
  const long q = blockIdx.y;
  const double *band = band_all + q * band_stride;
  const long half = mail_half(n, b), slot = mail_slot(b), plane = mail_plane(b), nslots = mail_slots(n, b);
  const double empty = __builtin_bit_cast(double, (unsigned long long)kEmptyHi << 32);
  if (blockIdx.z > 0) {
    double *box = boxes + ((blockIdx.z - 1L) * gridDim.y + q) * 2 * half;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < 2 * half; e += gridDim.x * 256L) box[e] = empty;
    return;
  }
  double *mail = mail_all + q * 2 * half;
  if (blockIdx.x == 0 && threadIdx.x == 0) D_all[q * d_stride] = band[0];
  for (long e = blockIdx.x * 256L + threadIdx.x; e < 2 * half; e += gridDim.x * 256L) {
    double v = empty;
    if (e >= half) {
      const long f = e - half;
      long row = -1, col = 0;  // element of the band, row < 0: none
      if (f >= nslots * slot) {
        const long i = f - nslots * slot;
        if (i < b) row = 1 + i;
      } else {
        const long j = f / slot, w = f % slot;
        const bool isn = w >= slot / 2;
        const long v2 = isn ? w - slot / 2 : w;
        const long i = (v2 % plane) / 8, k = (v2 / plane) * 8 + (v2 & 7);
        const long p = 1 + j * b, len = min((long)b, n - p), len2 = max(0L, min((long)b, n - p - len));
        if (k < len && i < (isn ? len2 : len) && !(isn && i == b - 1 && k < b - 1)) {
          row = isn ? p + len + i : p + max(i, k);
          col = isn ? p + k : p + min(i, k);
        }
      }
      if (row >= 0 && row < n) {
        v = band[(row - col) + col * ldb];
        // a caller's NaN must not read as an empty slot
        if (!(v == v)) v = __builtin_nan("");
      }
    }
    mail[e] = v;
  }
}

// Handing out sweeps.  A unit is a run of `len` consecutive sweeps of one
// problem; units are numbered run by run over the problems (run u / count of
// problem u % count) and an XCD takes the next one when all sweeps of its last
// are handed out.  So the first sweep that is not finished is running or next
// in its XCD's unit, whose workgroups have only finished ones behind them:
// the chain always moves.  Units go to the first `members` XCDs that ask; the
// workgroups of the others leave.
// Words at `ticket`: the next unit, the members so far, and at
// kXcdWords (x + 1) the 64-bit state of XCD x: member number << 61 | unit + 1
// << 30 | sweeps handed out (0: no unit yet).
constexpr int kXcds = 8, kXcdWords = 32;
constexpr long kTicketWords = (long)kXcdWords * (kXcds + 1);
constexpr unsigned kNoUnit = 0x7fffffffu;

struct ChaseUnits {
  int len, total, members;
};

// sweep (s of problem q) for this workgroup, whose XCD is member m; false: no
// more.  One thread calls.
__device__ inline bool next_sweep(unsigned *ticket, int x, const ChaseUnits &units, int count, int nsweeps,
                                  unsigned *err, int &s, int &q, int &m) {
  unsigned long long *state = reinterpret_cast<unsigned long long *>(ticket + kXcdWords * (x + 1));
  auto field = [](unsigned long long v) -> unsigned { return (unsigned)(v >> 30) & kNoUnit; };
  while (true) {
    const unsigned long long v = __hip_atomic_fetch_add(state, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned unit = field(v), idx = (unsigned)v & 0x3fffffffu;
    m = (int)(v >> 61);
    if (unit == kNoUnit) return false;
    if (unit != 0 && idx < (unsigned)units.len) {
      s = (int)((unit - 1) / count) * units.len + (int)idx;
      q = (int)((unit - 1) % count);
      if (s < nsweeps) return true;
      continue;
    }
    if (idx == (unit == 0 ? 0u : (unsigned)units.len)) {  // fetch the XCD's next unit, and take its first sweep
      if (unit == 0) m = (int)__hip_atomic_fetch_add(ticket + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      unsigned u = kNoUnit - 1;
      if (m < units.members) {
        const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (t < (unsigned)units.total) u = t;
      }
      const bool none = u == kNoUnit - 1;
      __hip_atomic_store(state, (none ? 0ull : (unsigned long long)m << 61) | (unsigned long long)(u + 1) << 30 | 1ull,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (none) return false;
      s = (int)(u / count) * units.len;
      q = (int)(u % count);
      return true;
    }
    // another workgroup fetches it
    const unsigned long long t0 = clock100();
    while (field(__hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == unit) {
      __builtin_amdgcn_s_sleep(2);
      if (clock100() - t0 > kWatchdogTicks) {
        atomicOr(err, (unsigned)EVD_E_TIMEOUT);
        return false;
      }
    }
  }
}

// LOCAL: messages between sweeps of one unit go through box m of the XCD's
// member number (boxes; one per member and problem) and stay in its L2; the
// first sweep of a unit receives, and the last one sends, through mail_all.
// Otherwise every message goes through mail_all.
template <int BW, bool LOCAL>
__global__ __launch_bounds__(ChaseShape<BW>::NT) void chase_kernel(
    int n, int b, double *__restrict__ mail_all, double *__restrict__ boxes, ChaseUnits units,
    float *__restrict__ U_all, long ldu, long u_stride, int *__restrict__ com_all, unsigned *__restrict__ ticket,
    unsigned *__restrict__ err, int count, double *__restrict__ D_all, long d_stride, double *__restrict__ E_all,
    long e_stride) {
  using Sh = ChaseShape<BW>;
  constexpr int EPT = Sh::EPT, NT = Sh::NT, NW = Sh::NW, LD = Sh::LD;
  __shared__ double sB[BW * LD];      // N^T of the last step: the next B1
  __shared__ double sU[NW][BW];       // each wave's copy of u
  __shared__ double sY[BW], sQ[BW], sN0[BW], sX[BW];
  __shared__ int s_sweep, s_problem, s_member, s_abort;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ri = tid >> 3, kc = tid & 7, xi = lane & (BW - 1);
  const int nsweeps = n - 2;
  const long half = mail_half(n, b), slot = mail_slot(b);
  const int slot_bytes = (int)(slot * 8);
  const unsigned pb = (unsigned)(mail_plane(b) * 8), nb0 = (unsigned)slot_bytes / 2;  // bytes of a plane, start of N
  typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u2;

  // byte offset of S'(i, k) in a slot (N' at + nb0)
  auto at = [&](int i, int k) -> unsigned { return (unsigned)(k >> 3) * pb + (unsigned)(i * 8 + (k & 7)) * 8u; };

  const int xcd = LOCAL ? (int)__builtin_amdgcn_s_getreg((3 << 11) | 20) & (kXcds - 1) : 0;  // HW_REG_XCC_ID

  // one sweep, messages in and out with these store policies (0: within the
  // XCD, kSc1: device-coherent); true: aborted
  auto sweep = [&](auto in_policy, auto out_policy, const int s, const int q, double *mail_in, double *mail_out)
                   __attribute__((always_inline)) -> bool {
    constexpr int IN = decltype(in_policy)::value, OUT = decltype(out_policy)::value;
    // slot 0 of this sweep's messages in, out
    double *rd = mail_in + ((s + 1) & 1) * half, *wr = mail_out + (s & 1) * half;
    const __amdgpu_buffer_rsrc_t rxi =
        __builtin_amdgcn_make_buffer_rsrc(rd + half - kXWords, 0, kXWords * 8, kBufferWord3);
    const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(
        U_all + (long)q * u_stride + (long)s * ldu, 0, (int)((n + b) * 4), kBufferWord3);
    int *com = com_all + (long)q * n * kComStride;
    double *Dq = D_all + q * d_stride, *Eq = E_all + q * e_stride;

    int p = s + 1, len = min(b, n - p), len2 = max(0, min(b, n - p - len));

    // watchdog of a wait; true = give up
    auto expired = [&](unsigned long long t0) -> bool {
      if (clock100() - t0 <= kWatchdogTicks) return false;
      if (lane == 0) {
        atomicOr(err, (unsigned)EVD_E_TIMEOUT);
        s_abort = 1;
      }
      return true;
    };
    // offsets of a window's elements (kOutOfRange: not part of it)
    unsigned oS[EPT], oN[EPT];
    auto window_offsets = [&](int wlen, int wlen2) {
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        const int kk = kc + 8 * r;
        oS[r] = (ri < wlen && kk < wlen) ? at(ri, kk) : kOutOfRange;
        oN[r] = (ri < wlen2 && kk < wlen && !(ri == b - 1 && kk < b - 1)) ? nb0 + at(ri, kk) : kOutOfRange;
      }
    };
    // offsets of a step's sends: S to slot j, B1 (thread = column ri, rows
    // kk) to slot j - 1, row 0 of B1 mirrored, and thread kc = 0's S(ri, 0)
    // (X in the first step)
    unsigned oA[EPT], oB[EPT], oM, oC, oX;
    auto send_offsets = [&](int wlen) {
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        const int kk = kc + 8 * r;
        oA[r] = (ri >= 1 && kk >= 1 && ri < wlen && kk < wlen) ? at(ri - 1, kk - 1) : kOutOfRange;
        oB[r] = (ri >= 1 && ri < b && kk < wlen) ? (kk == 0 ? at(b - 1, ri - 1) : nb0 + at(kk - 1, ri - 1)) : kOutOfRange;
      }
      oM = (kc == 0 && ri >= 1 && ri < b) ? at(ri - 1, b - 1) : kOutOfRange;
      oC = (kc == 0 && ri < wlen) ? (ri == 0 ? at(b - 1, b - 1) : nb0 + at(ri - 1, b - 1)) : kOutOfRange;
      oX = (kc == 0 && ri >= 1 && ri < wlen) ? (unsigned)(ri - 1) * 8u : kOutOfRange;
    };
    window_offsets(len, len2);
    send_offsets(len);

    // the predecessor's first slots are this sweep's to poll once it has started
    if (s > 0) {
      const unsigned long long t0 = clock100();
      while (ld_dev(&com[(long)(s - 1) * kComStride]) == 0) {
        if (expired(t0)) break;
        __builtin_amdgcn_s_sleep(1);
      }
    }
    // column s below the diagonal: wave 0 receives it for all
    if (wave == 0) {
      const unsigned ox = lane < min(b, n - p) ? (unsigned)lane * 8u : kOutOfRange;
      const unsigned long long t0 = clock100();
      double x;
      while (true) {
        x = ld_band_at(rxi, ox);
        const bool ready = (unsigned)(__builtin_bit_cast(unsigned long long, x) >> 32) != kEmptyHi;
        if (__all(ready) || expired(t0)) break;
      }
      __builtin_amdgcn_raw_buffer_store_b64(u2{0u, kEmptyHi}, rxi, ox, 0, IN);
      if (lane < BW) sX[lane] = x;
    }
    grp_barrier();
    double u0, beta;
    {
      const double uu = chase_reflector<BW>(sX[xi], lane, u0, beta);
      if (lane < BW) sU[wave][lane] = uu;
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)uu), ru,
                                            (wave == 0 && lane < len) ? (unsigned)(p + lane) * 4u : kOutOfRange, 0, 0);
      if (tid == 0) Eq[s] = beta;
    }

    auto load_window = [&](const double *base, double(&S)[EPT], double(&N)[EPT]) {
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(base), 0, slot_bytes, kBufferWord3);
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        S[r] = ld_band_at(rs, oS[r]);
        N[r] = ld_band_at(rs, oN[r]);
      }
    };
    auto arrived = [&](const double(&S)[EPT], const double(&N)[EPT]) -> bool {
      unsigned m = ~0u;
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        m = min(m, (unsigned)(__builtin_bit_cast(unsigned long long, S[r]) >> 32) ^ kEmptyHi);
        m = min(m, (unsigned)(__builtin_bit_cast(unsigned long long, N[r]) >> 32) ^ kEmptyHi);
      }
      return __all(m != 0u);
    };

    // one step on the window in (S, N); the next one's is loaded into
    // (Sn, Nn).  0: go on, 1: last step, 2: aborted
    auto step = [&](auto is_first, double(&S)[EPT], double(&N)[EPT], double(&Sn)[EPT], double(&Nn)[EPT])
                    __attribute__((always_inline)) -> int {
      constexpr bool first = decltype(is_first)::value;
      const bool last = (len2 == 0);
      // ---- B1 <- H B1 (B1 transposed), for which u is all it takes: done and
      // sent while the window is on its way
      double uk[EPT];
      const double ui = sU[wave][ri];
#pragma unroll
      for (int r = 0; r < EPT; r++) uk[r] = sU[wave][kc + 8 * r];
      if constexpr (!first) {
        double bt[EPT], t = 0.0;
#pragma unroll
        for (int r = 0; r < EPT; r++) bt[r] = sB[ri * LD + kc + 8 * r];
#pragma unroll
        for (int r = 0; r < EPT; r++) t += bt[r] * uk[r];
        t = group_sum<8>(t);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(wr - slot, 0, slot_bytes, kBufferWord3);
#pragma unroll
        for (int r = 0; r < EPT; r++) {
          bt[r] -= uk[r] * t;
          st_band_at<OUT>(rv, oB[r], bt[r]);
        }
        st_band_at<OUT>(rv, oM, bt[0]);
      }
      if (!arrived(S, N)) {
        const unsigned long long t0 = clock100();
        do {
          load_window(rd, S, N);
        } while (!arrived(S, N) && !expired(t0));
      }
      // ---- row sums q = N u, y = S u
      double y = 0.0, qq = 0.0;
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        qq += N[r] * uk[r];
        y += S[r] * uk[r];
      }
      qq = group_sum<8>(qq);
      y = group_sum<8>(y);
      if (kc == 0) {
        sQ[ri] = qq;
        sN0[ri] = N[0];
        sY[ri] = y;
      }
      grp_barrier();
      // ---- the next column and its reflector (every wave for itself), the
      // slot emptied in its shadow
      const double x = sN0[xi] - sQ[xi] * u0;
      double yk[EPT];
#pragma unroll
      for (int r = 0; r < EPT; r++) yk[r] = sY[kc + 8 * r];
      const int aborted = s_abort;
      {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(rd, 0, slot_bytes, kBufferWord3);
#pragma unroll
        for (int r = 0; r < EPT; r++) {
          __builtin_amdgcn_raw_buffer_store_b64(u2{0u, kEmptyHi}, rs, oS[r], 0, IN);
          __builtin_amdgcn_raw_buffer_store_b64(u2{0u, kEmptyHi}, rs, oN[r], 0, IN);
        }
      }
      double un0 = 0.0, betan = 0.0, uu = 0.0;
      uu = chase_reflector<BW>(x, lane, un0, betan);
      if (len2 <= 1) {  // a single row is left as it is
        uu = un0 = 0.0;
        betan = __shfl(x, 0, 64);
      }
      if (lane < BW) sU[wave][lane] = uu;
      // ---- S <- H S H (rank-2 with w = y - (u^T y / 2) u), N <- N H
      double psi = 0.0;
#pragma unroll
      for (int r = 0; r < EPT; r++) psi += uk[r] * yk[r];
      psi = 0.5 * group_sum<8>(psi);
      const double wi = y - psi * ui;
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        const double wk = yk[r] - psi * uk[r];
        S[r] -= sym_pair(ui, wk, wi, uk[r]);
      }
      // S(:, 0) and the next beta complete message j - 1 (X in the first step)
      {
        const unsigned ob = first ? (unsigned)(b - 1) * 8u : nb0 + at(b - 1, b - 1);
        const unsigned oc = tid == 1 ? (len2 > 0 ? ob : kOutOfRange) : (first ? oX : oC);
        const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
            first ? mail_out + (s & 1) * half + (half - kXWords) : wr - slot, 0, first ? kXWords * 8 : slot_bytes,
            kBufferWord3);
        st_band_at<OUT>(rc, oc, tid == 1 ? betan : S[0]);
      }
#pragma unroll
      for (int r = 0; r < EPT; r++) {
        N[r] -= qq * uk[r];
        sB[(kc + 8 * r) * LD + ri] = N[r];
      }
      // the last message has no step behind it to show that the slot is empty
      if (last) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(wr, 0, slot_bytes, kBufferWord3);
#pragma unroll
        for (int r = 0; r < EPT; r++) st_band_at<OUT>(rw, oA[r], S[r]);
      }
      const int pn = p + len, len3 = max(0, min(b, n - pn - len2));
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)uu), ru,
                                            (wave == 0 && lane < len2) ? (unsigned)(pn + lane) * 4u : kOutOfRange, 0, 0);
      if constexpr (first) {
        if (tid == 0) {
          Dq[s + 1] = S[0];
          st_dev(&com[(long)s * kComStride], 1);
        }
        if (s == nsweeps - 1) {  // the last 2 x 2 block is final
          if (tid == 8) Eq[n - 2] = S[0];
          if (tid == 9) Dq[n - 1] = S[0];
        }
      }
      // look for the next window (loads behind this step's empties: see above)
      asm volatile("" ::: "memory");
      rd += slot;
      if (len3 != b) window_offsets(len2, len3);
      load_window(rd, Sn, Nn);
      grp_barrier();
      if (aborted) return 2;
      if (last) return 1;
      wr += slot;
      u0 = un0;
      beta = betan;
      p = pn;
      len = len2;
      len2 = len3;
      if (len != b) send_offsets(len);
      return 0;
    };

    double Sa[EPT], Na[EPT], Sb[EPT], Nb[EPT];
    load_window(rd, Sa, Na);
    int end = step(std::true_type{}, Sa, Na, Sb, Nb);
    while (!end) {
      end = step(std::false_type{}, Sb, Nb, Sa, Na);
      if (end) break;
      end = step(std::false_type{}, Sa, Na, Sb, Nb);
    }
    return end == 2;
  };

  const std::integral_constant<int, 0> local{};
  const std::integral_constant<int, kSc1> coherent{};
  while (true) {
    if (tid == 0) {
      int s, q, m;
      if (LOCAL) {
        s_sweep = next_sweep(ticket, xcd, units, count, nsweeps, err, s, q, m) ? s : -1;
      } else {  // sweep by sweep over the problems
        const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s = (int)(t / count);
        q = (int)(t % count);
        m = 0;
        s_sweep = s < nsweeps ? s : -1;
      }
      s_problem = q;
      s_member = m;
      s_abort = 0;
    }
    grp_barrier();
    const int s = __builtin_amdgcn_readfirstlane(s_sweep), q = __builtin_amdgcn_readfirstlane(s_problem);
    const int m = __builtin_amdgcn_readfirstlane(s_member);
    grp_barrier();
    if (s < 0) return;
    double *mail = mail_all + (long)q * 2 * half, *box = boxes + ((long)m * count + q) * 2 * half;
    bool aborted;
    if (!LOCAL)
      aborted = sweep(coherent, coherent, s, q, mail, mail);
    else if (s % units.len == 0)
      aborted = sweep(coherent, local, s, q, mail, box);
    else if ((s + 1) % units.len == 0)
      aborted = sweep(local, coherent, s, q, box, mail);
    else
      aborted = sweep(local, local, s, q, box, box);
    if (aborted) return;
  }
}

// ---------------------------------------------------------------------------
// Grouped chase (b <= 32): a workgroup owns a group of D consecutive sweeps,
// s0 .. s0 + D - 1, one wave per sweep.  The waves step in lockstep: at time
// step t, sweep s0 + i does its step t - 2i (the two-step lag of the sweep
// order), all on a window of band columns held in LDS (column c in slot
// c mod kGW, offsets 0 .. 2b-1), so the hand-off between the group's sweeps
// never leaves the CU.  One more wave moves the window (I/O wave):
//  * it brings in the columns the front sweep s0 first needs at
//    step j (columns s0 .. p_0 + len_0 at j = 0, p_j .. p_j + len_j later, up
//    to n at the front's last step) from HBM: the loads are issued at time
//    j - 3, once the previous group's progress word is >= p_j + 2b - 1, into
//    one of two register buffers, and written to LDS at time j - 1.  The
//    last column of a chunk, p_j + b - 1, is a step row of the previous
//    group's last sweep, which writes it back down to its early-published
//    beta only (offset b): the fill below is zeroed by that sweep's next
//    step, so the I/O wave writes those zeros;
//  * it writes back, at time t, the columns the group's last sweep finished
//    at t - 1 (all columns up to its step row P; column P down to offset b)
//    and publishes that sweep's next row P + len at t + 1, once those stores
//    have completed; the last write-back covers every remaining column and
//    publishes INT_MAX.
// Every step issues the same number of memory operations in the same order
// (kGChunk stores, one poll of the predecessor's progress word, kGChunk
// loads; unused lanes address past the end of the band, which the buffer
// range check drops), so the wait before the publish is a fixed count - the
// newest kGChunk loads stay in flight - and the loads have two steps to land.
// Within a time step the waves' LDS accesses are disjoint and every slot is
// rewritten only after its previous column was written back, provided
// kGW >= (2D + 2) b - D + 1; a CPU model of this schedule (random
// interleavings of groups, access-set and slot checks) reproduces the
// sequential chase.  Groups are handed out by ticket in increasing order, so
// a group's predecessor is always running; every wait is bounded.
constexpr int kGW = 256;  // window columns
// doubles per window column (2b <= 64 offsets).  Element (row R, column C)
// sits at C * kGLD + R - C, so a band row runs through the window with stride
// kGLD - 1 = 63 doubles (odd: the 32 lanes of a row access hit 32 distinct
// banks) and a band column with stride 1.
constexpr int kGLD = 64;
// most columns the front brings in at one step: b + 2 at b = 32 (the first
// chunk s0 .. n of a sweep whose first step is also its last)
constexpr int kGChunk = 34;

__device__ inline int sweep_nsteps(int n, int b, int s) {
  int p = s + 1, len = min(b, n - p), k = 1;
  while (true) {
    const int len2 = max(0, min(b, n - p - len));
    if (len2 <= 1) return k;
    p += len;
    len = len2;
    k++;
  }
}

// sum over the 64 lanes, returned in every lane: quad, half-row and row
// reductions by DPP, then row 15 -> rows 1 and 3 and lane 31 -> rows 2 and 3
// broadcasts; lane 63 holds the total
__device__ __attribute__((always_inline)) inline double wave_total(double v) {
  v += dpp_f64<0xb1, 0xf>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_f64<0x4e, 0xf>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_f64<0x141, 0xf>(v);  // row_half_mirror
  v += dpp_f64<0x140, 0xf>(v);  // row_mirror
  v += dpp_f64<0x142, 0xa>(v);  // row_bcast:15
  v += dpp_f64<0x143, 0xc>(v);  // row_bcast:31
  const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)x, 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(x >> 32), 63);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// reflector of the chase's convention from x (lane < lenx, zero elsewhere),
// wave-wide; uu is zero for lanes >= lenx
__device__ __attribute__((always_inline)) inline void grp_reflector(double x, int lane, int lenx, double &uu,
                                                                   double &beta) {
  const double nrm = sqrt(wave_total(x * x));
  const unsigned long long xb = __builtin_bit_cast(unsigned long long, x);
  const double x0 = __builtin_bit_cast(double, ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(
                                                    (int)(unsigned)(xb >> 32), 0)
                                                << 32) |
                                                   (unsigned)__builtin_amdgcn_readlane((int)(unsigned)xb, 0));
  uu = 0.0;
  if (nrm > 0.0) {
    const double inv = 1.0 / nrm;
    const double u0 = x0 * inv + (x0 >= 0.0 ? 1.0 : -1.0);
    const double scl = 1.0 / sqrt(fabs(u0));
    uu = (lane == 0 ? u0 : x * inv) * scl;
  }
  if (lane >= lenx) uu = 0.0;
  beta = (nrm > 0.0) ? (x0 >= 0.0 ? -nrm : nrm) : x0;
}

// one chunk of the front's columns in flight: registers + where they go
// (columns lo .. hi-1; hi == lo when the step loads nothing)
struct GrpChunk {
  double v[kGChunk];
  int lo, hi, syn;
};

template <int D>
__global__ __launch_bounds__((D + 1) * 64, 1) void chase_group_kernel(
    int n, int b, double *__restrict__ band_all, long ldb, unsigned band_bytes, float *__restrict__ U_all, long ldu,
    int *__restrict__ com_all, unsigned *__restrict__ ticket, unsigned *__restrict__ err, int count, long band_stride,
    long u_stride, long com_stride) {
  // the window, then one column-sized slot that takes the chunk writes of
  // unused registers (every loaded register is written somewhere, so no load
  // is dropped on some paths and the memory-operation count per step stays
  // fixed)
  __shared__ double win[kGW * kGLD + 64];
  __shared__ double uS[D][32], yS[D][32];
  __shared__ int s_ticket, s_abort;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nsweeps = n - 2;
  const int ngroups = (nsweeps + D - 1) / D;
  const unsigned ld = (unsigned)ldb;
  const int b2 = 2 * b;

  while (true) {
    if (tid == 0) {
      s_ticket = (int)__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_abort = 0;
    }
    grp_barrier();
    const int tk = s_ticket;
    grp_barrier();
    if (tk >= ngroups * count) return;
    const int q = tk % count, g = tk / count;
    const int s0 = g * D, nsw = min(D, nsweeps - s0);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(band_all + (long)q * band_stride, 0, (int)band_bytes, kBufferWord3);
    float *U = U_all + (long)q * u_stride;
    int *com = com_all + (long)q * com_stride;
    const int tail_steps = sweep_nsteps(n, b, s0 + nsw - 1);
    const int front_steps = sweep_nsteps(n, b, s0);
    const int te = tail_steps - 1 + 2 * (nsw - 1);  // time step of the last sweep's last step
    // the time loop runs t = -3 .. t_last, an even number of steps (the I/O
    // wave's loop body is two steps, one per register buffer, with no exit
    // between them: an exit there costs the loads their overlap)
    const int t_last = te + 2 + ((te + 6) & 1);

    // Each role runs its own copy of the time loop (one barrier per time
    // step in every copy), so the roles' registers do not add up.
    if (wave < D) {
      // ---- worker: sweep ws of this group.  Lane (c, h) = (lane & 31,
      // lane >> 5) holds rows 2r + h of B1 column c; lane (ri, kc) = the same
      // pair holds row ri, columns kc + 2r of the S and N blocks.  LDS reads
      // are gathered into registers before any write of the same phase.
      const int ws = s0 + wave;
      const int w_steps = (wave < nsw) ? sweep_nsteps(n, b, ws) : 0;
      const int c = lane & 31, h = lane >> 5;
      int wp = ws + 1, wlen = min(b, n - wp), cB1 = ws, colB1 = 1;
      bool wfirst = true;
      double wbeta = 0.0;
      double *u = uS[wave], *yv = yS[wave];
      for (int t = -3; t <= t_last; ++t) {
        const int js = t - 2 * wave;
        if (js >= 0 && js < w_steps) {
          const int p = wp, len = wlen;
          const int len2 = max(0, min(b, n - p - len));
          const bool last = (len2 <= 1);
          if (wfirst) {
            // the sweep's first reflector, from column ws below the diagonal
            const double x = (lane < len) ? win[(ws & (kGW - 1)) * kGLD + 1 + lane] : 0.0;
            double uu, beta;
            grp_reflector(x, lane, len, uu, beta);
            if (lane < 32) u[lane] = uu;
            if (lane < len) U[(p + lane) + (long)ws * ldu] = (float)uu;
            wbeta = beta;
          }
          double u16[16];
#pragma unroll
          for (int r = 0; r < 16; r++) u16[r] = u[2 * r + h];
          const double uc = u[c];
          // ---- B1 <- H B1 (columns 1 .. colB1-1); column 0 becomes beta e1
          {
            const bool act = (c >= 1 && c < colB1);
            // row p of column cB1 + c (lanes past the block read slot 0, unused)
            const int base = (c < colB1) ? ((cB1 + c) & (kGW - 1)) * kGLD + (p - cB1 - c) : 0;
            double bv[16];
#pragma unroll
            for (int r = 0; r < 16; r++) bv[r] = win[base + 2 * r + h];
            double tsum = 0.0;
#pragma unroll
            for (int r = 0; r < 16; r++) {
              const int i = 2 * r + h;
              if (!(act && i < len)) bv[r] = 0.0;
              tsum += u16[r] * bv[r];
            }
            tsum += half_swap(tsum);
#pragma unroll
            for (int r = 0; r < 16; r++) {
              const int i = 2 * r + h;
              if (act && i < len) win[base + i] = bv[r] - u16[r] * tsum;
              if (c == 0 && i < len && !(i == 0 && !wfirst)) win[base + i] = (i == 0) ? wbeta : 0.0;
            }
          }
          // ---- S <- H S H, N <- N H (S from the lower band)
          const int ri = c, kc = h;
          double Sr[16], Nr[16];
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int kk = kc + 2 * r;
            const int lo = min(ri, kk), hi = max(ri, kk);
            Sr[r] = win[((p + lo) & (kGW - 1)) * kGLD + (hi - lo)];
            Nr[r] = win[((p + kk) & (kGW - 1)) * kGLD + ((len + ri - kk) & 63)];
          }
          double yp = 0.0, qp = 0.0;
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int kk = kc + 2 * r;
            if (!(ri < len && kk < len)) Sr[r] = 0.0;
            if (!(ri < len2 && kk < len)) Nr[r] = 0.0;
            yp += Sr[r] * u16[r];
            qp += Nr[r] * u16[r];
          }
          yp += half_swap(yp);  // y = S u, row ri (both halves)
          qp += half_swap(qp);  // q = N u, row ri
          if (kc == 0) yv[ri] = yp;
          double yk[16];
#pragma unroll
          for (int r = 0; r < 16; r++) yk[r] = yv[kc + 2 * r];
          // u^T y over the 64 lanes counts every row twice
          const double hpsi = 0.5 * (0.5 * wave_total(uc * yp));
          const double wi = yp - hpsi * uc;
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const double wk = yk[r] - hpsi * u16[r];
            Sr[r] -= uc * wk + wi * u16[r];
            Nr[r] -= qp * u16[r];
          }
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int kk = kc + 2 * r;
            if (ri >= kk && ri < len && kk < len) win[((p + kk) & (kGW - 1)) * kGLD + (ri - kk)] = Sr[r];
            if (ri < len2 && kk < len) win[((p + kk) & (kGW - 1)) * kGLD + (len + ri - kk)] = Nr[r];
          }
          // ---- next reflector from N[:, 0] (column p, held by lanes kc = 0);
          // its beta goes in now
          if (!last) {
            const double x = (kc == 0 && ri < len2) ? Nr[0] : 0.0;
            double uu, beta;
            grp_reflector(x, lane, len2, uu, beta);
            if (lane < 32) u[lane] = uu;
            if (lane < len2) U[(p + len + lane) + (long)ws * ldu] = (float)uu;
            if (lane == 0) win[(p & (kGW - 1)) * kGLD + len] = beta;
            wbeta = beta;
            wfirst = false;
            cB1 = p;
            colB1 = len;
            wp = p + len;
            wlen = len2;
          }
        }
        grp_barrier();
        if (((t + 3) & 1) && s_abort) break;
      }
    } else {
      // ---- I/O wave (see the schedule above); chunk j lives in buffer j & 1
      int fp = s0 + 1, flen = min(b, n - s0 - 1), lj = 0;  // next front step to load
      int known = (g == 0) ? INT_MAX : -1, pv = -1;
      const int *pcom = com + (long)max(g - 1, 0) * kComStride;
      int tp = s0 + nsw, tlen = min(b, n - s0 - nsw), wb = s0, pval = 0;
      bool pend = false;
      GrpChunk ca, cb;
#pragma unroll
      for (int k = 0; k < kGChunk; k++) ca.v[k] = cb.v[k] = 0.0;
      ca.lo = ca.hi = cb.lo = cb.hi = 0;
      ca.syn = cb.syn = -1;
      auto io_step = [&](int t, GrpChunk &ch) {
        // all but the newest kGChunk loads (the other buffer's chunk) are done:
        // this buffer's chunk, last step's stores and poll
        wait_vm<kGChunk>();
        if (pend) {
          if (pval == INT_MAX) wait_mem();
          if (lane == 0) st_dev(&com[(long)g * kComStride], pval);
          pend = false;
        }
        known = max(known, pv);  // group 0: known is INT_MAX already
        // chunk t + 1 -> LDS
#pragma unroll
        for (int k = 0; k < kGChunk; k++) {
          const int cc = ch.lo + k;
          const int at = (cc < ch.hi && lane < b2) ? (cc & (kGW - 1)) * kGLD + lane : kGW * kGLD + lane;
          win[at] = (cc == ch.syn && lane > b) ? 0.0 : ch.v[k];
        }
        // write-back of the columns the last sweep finished at t - 1
        const int k = t - 1 - 2 * (nsw - 1);
        const bool wbk = (k >= 0 && k < tail_steps);
        const bool wlast = wbk && (k == tail_steps - 1);
        const int P = tp;
        const int whi = wbk ? (wlast ? n : P + 1) : wb;
        int c0 = wb;
        do {
          // kGChunk stores (two halves of reads then stores); lanes past the
          // columns or past a column's valid offsets store out of range
#pragma unroll
          for (int half = 0; half < 2; half++) {
            double sv[kGChunk / 2];
#pragma unroll
            for (int k2 = 0; k2 < kGChunk / 2; k2++) {
              const int cc = min(c0 + half * (kGChunk / 2) + k2, n - 1);
              sv[k2] = win[(cc & (kGW - 1)) * kGLD + lane];
            }
#pragma unroll
            for (int k2 = 0; k2 < kGChunk / 2; k2++) {
              const int cc = c0 + half * (kGChunk / 2) + k2;
              const int dmax = (wlast || cc < P) ? b2 : b + 1;
              const unsigned off = (cc < whi && lane < dmax) ? ((unsigned)lane + (unsigned)cc * ld) * 8u : kOutOfRange;
              __builtin_amdgcn_raw_buffer_store_b64(
                  __builtin_bit_cast(__attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned, sv[k2]), rb, off,
                  0, kSc1);
            }
          }
          c0 += kGChunk;
        } while (c0 < whi);
        if (wbk) {
          wb = whi;
          pend = true;
          pval = wlast ? INT_MAX : P + tlen;
          const int nl = max(0, min(b, n - P - tlen));
          tp = P + tlen;
          tlen = nl;
        }
        // poll of the predecessor's progress word (its own word for group 0)
        pv = ld_dev(pcom);
        // loads of front step t + 3
        const bool ld_now = (lj < front_steps);
        if (ld_now && known < fp + 2 * b - 1 && !s_abort) {
          const int need = fp + 2 * b - 1;
          const unsigned long long t0 = clock100();
          while (true) {
            known = max(known, ld_dev(pcom));
            if (known >= need) break;
            if (clock100() - t0 > kWatchdogTicks) {
              if (lane == 0) {
                atomicOr(err, (unsigned)EVD_E_TIMEOUT);
                s_abort = 1;
              }
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        const int lo = (lj == 0) ? s0 : fp;
        const int hi = ld_now ? ((lj == front_steps - 1) ? n : fp + flen) : lo;
#pragma unroll
        for (int k2 = 0; k2 < kGChunk; k2++) {
          const int cc = lo + k2;
          const unsigned off = (cc < hi && lane < b2) ? ((unsigned)lane + (unsigned)cc * ld) * 8u : kOutOfRange;
          ch.v[k2] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, off, 0, kSc1));
        }
        ch.lo = lo;
        ch.hi = hi;
        ch.syn = fp + b - 1;
        if (ld_now) {
          fp += flen;
          flen = min(b, n - fp);
          lj++;
        }
        grp_barrier();
      };
      for (int t = -3; t <= t_last; t += 2) {
        io_step(t, ca);
        io_step(t + 1, cb);
        if (s_abort) break;
      }
      wait_mem();
    }
    if (s_abort) {
      if (wave == D && lane == 0) st_dev(&com[(long)g * kComStride], INT_MAX);
      return;
    }
  }
}

__global__ void band_pack_kernel(int n, int b, const float *__restrict__ A, long lda, long a_stride,
                                 double *__restrict__ band, long ldb, long band_stride) {
  A += blockIdx.z * a_stride;
  band += blockIdx.z * band_stride;
  long c = blockIdx.y * (long)blockDim.y + threadIdx.y;
  for (; c < n; c += (long)gridDim.y * blockDim.y)
    for (int i = threadIdx.x; i < 2 * b; i += blockDim.x) {
      double v = 0.0;
      if (i <= b && c + i < n) v = (double)A[(c + i) + c * lda];
      band[i + c * ldb] = v;
    }
}

int band_pack_batched(evd_ctx *ctx, int count, long n, long b, const float *A, long lda, long a_stride, double *band,
                      long ldband, long band_stride) {
  if (n <= 0) return 0;
  dim3 blk(64, 4);
  unsigned gy = (unsigned)std::min<long>((n + 3) / 4, 65535);
  band_pack_kernel<<<dim3(1, gy, (unsigned)count), blk, 0, ctx->stream>>>((int)n, (int)b, A, lda, a_stride, band, ldband,
                                                                          band_stride);
  EVD_LAUNCHED(ctx);
  return 0;
}
int band_pack(evd_ctx *ctx, long n, long b, const float *A, long lda, double *band, long ldband) {
  return band_pack_batched(ctx, 1, n, b, A, lda, 0, band, ldband, 0);
}

// largest sweeps-per-group whose window fits kGW columns: (2D + 2) b - D + 1 <= kGW
static int group_depth_max(long b) { return (int)std::max<long>(0, (kGW - 1 - 2 * b) / (2 * b - 1)); }

template <int D>
static int launch_chase_group(evd_ctx *ctx, int count, long n, long b, double *band, long ldb, long band_stride,
                              float *U, long ldu, long u_stride, int *com, long com_stride, unsigned *ticket) {
  const long bytes = ldb * n * (long)sizeof(double);
  if (bytes >= (1L << 31))
    return set_error(ctx, EVD_E_UNSUPPORTED, "band of %ld bytes exceeds the 2 GiB buffer range of the chase", bytes);
  // groups in flight: a group lags its predecessor by about 2D + 4 steps and
  // lives about n / b steps
  int resident = 0;
  EVD_TRY(max_coresident_blocks(ctx, (const void *)chase_group_kernel<D>, (D + 1) * 64, 0, &resident));
  const long ngroups = (n - 2 + D - 1) / D;
  const long inflight = (((n + b - 1) / b + 2 * D + 3) / (2 * D + 4) + 2) * count;
  long G = ctx->tune.chase_groups > 0 ? ctx->tune.chase_groups : inflight;
  G = std::max<long>(1, std::min<long>(std::min<long>(G, resident), ngroups * count));
  unsigned *err = ctx->ctrl + kCtrlError;
  if (ctx->timing && !ctx->capturing) hipEventRecord(ctx->cev[0], ctx->stream);
  chase_group_kernel<D><<<(unsigned)G, (D + 1) * 64, 0, ctx->stream>>>((int)n, (int)b, band, ldb, (unsigned)bytes, U,
                                                                        ldu, com, ticket, err, count, band_stride,
                                                                        u_stride, com_stride);
  EVD_LAUNCHED(ctx);
  if (ctx->timing && !ctx->capturing) hipEventRecord(ctx->cev[1], ctx->stream);
  return 0;
}

// Sweeps in flight of one problem (a sweep trails its predecessor by two to
// three steps of b rows) and the XCDs that run the chase: 32 sweeps an XCD, one
// per CU, keep a chain of up to 32 on one XCD; at b = 64, 16, whose slots (64
// KiB, two steps apart, both parities) fit the 4 MiB of its L2.  Where the eight
// XCDs do not hold all that are in flight, the slots would not stay in the L2s: a
// large batch runs as several launches, and single chases beyond that (n >
// 20000 at b = 32) do without boxes.
static long chase_inflight(long n, long b) { return (2 * n + 5 * b - 1) / (5 * b) + 4; }
static int chase_members(int count, long n, long b) {
  const long per = b <= 32 ? 32 : 16;
  return (int)((chase_inflight(n, b) * count + per - 1) / per);
}
// problems of a batch per launch: as many as the XCDs hold in flight
static int chase_batch(int count, long n, long b) {
  return (int)std::max<long>(1, std::min<long>(count, kXcds * (b <= 32 ? 32 : 16) / chase_inflight(n, b)));
}

template <int BW>
static int launch_chase(evd_ctx *ctx, int count, long n, long b, const double *band, long ldb, long band_stride,
                        double *mail, double *boxes, float *U, long ldu, long u_stride, int *com, unsigned *ticket,
                        double *D, long d_stride, double *E, long e_stride) {
  // workgroups: as many as sweeps are in flight (a workgroup takes its next
  // sweep as soon as it finishes one), at most one per CU.  Those beyond that
  // only poll and crowd out concurrent solves.  With boxes that many on each
  // member XCD: workgroups are dealt to the XCDs in turn, so eight times as many
  // are launched, of which those on other XCDs leave at once.
  int resident = 0;
  const void *kernel = boxes ? (const void *)chase_kernel<BW, true> : (const void *)chase_kernel<BW, false>;
  EVD_TRY(max_coresident_blocks(ctx, kernel, ChaseShape<BW>::NT, 0, &resident));
  const long nsweeps = n - 2, inflight = chase_inflight(n, b);
  const int members = boxes ? chase_members(count, n, b) : 1;
  // units: everything on one XCD where that holds a problem's sweeps in
  // flight; else as many sweeps as an XCD holds; batches mix the problems
  long per = std::min<long>(inflight * count, ctx->num_cus), len = 1;
  if (boxes) {
    per = std::min<long>((inflight * count + members - 1) / members + 2, resident / kXcds);
    len = count > 1 ? std::min(inflight, per) : members == 1 ? nsweeps : per;
    len = std::max<long>(2, std::min(len, nsweeps));
    per *= kXcds;
  }
  long G = ctx->tune.chase_groups > 0 ? ctx->tune.chase_groups : per;
  G = std::min<long>(G, std::max<long>(1, nsweeps * count * (boxes ? kXcds : 1)));
  const ChaseUnits units{(int)len, (int)(((nsweeps + len - 1) / len) * count), members};
  unsigned *err = ctx->ctrl + kCtrlError;
  const long words = 2 * mail_half(n, b);
  mail_fill_kernel<<<dim3((unsigned)std::min<long>((words + 255) / 256, 4096), (unsigned)count,
                          boxes ? members + 1u : 1u),
                     256, 0, ctx->stream>>>((int)n, (int)b, band, ldb, band_stride, mail, boxes, D, d_stride);
  EVD_LAUNCHED(ctx);
  if (ctx->timing && !ctx->capturing) hipEventRecord(ctx->cev[0], ctx->stream);
  if (boxes)
    chase_kernel<BW, true><<<(unsigned)G, ChaseShape<BW>::NT, 0, ctx->stream>>>(
        (int)n, (int)b, mail, boxes, units, U, ldu, u_stride, com, ticket, err, count, D, d_stride, E, e_stride);
  else
    chase_kernel<BW, false><<<(unsigned)G, ChaseShape<BW>::NT, 0, ctx->stream>>>(
        (int)n, (int)b, mail, boxes, units, U, ldu, u_stride, com, ticket, err, count, D, d_stride, E, e_stride);
  EVD_LAUNCHED(ctx);
  if (ctx->timing && !ctx->capturing) hipEventRecord(ctx->cev[1], ctx->stream);
  return 0;
}

__global__ void band_extract_batched_kernel(int n, const double *__restrict__ band, long ldb, long band_stride,
                                            double *__restrict__ D, long d_stride, double *__restrict__ E,
                                            long e_stride) {
  const long q = blockIdx.y;
  band += q * band_stride;
  D += q * d_stride;
  E += q * e_stride;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    D[i] = band[i * ldb];
    if (i < n - 1) E[i] = band[1 + i * ldb];
  }
}

// A band of width 1 is tridiagonal already; the sweeps' reflectors have length
// 1 and flip signs (H = -1 where the entry below the diagonal is not zero).
__global__ void chase_signs_kernel(int n, const double *__restrict__ band, long ldb, long band_stride,
                                   float *__restrict__ U, long ldu, long u_stride, double *__restrict__ D,
                                   long d_stride, double *__restrict__ E, long e_stride) {
  const long q = blockIdx.y;
  band += q * band_stride;
  for (long s = blockIdx.x * (long)blockDim.x + threadIdx.x; s < n; s += (long)gridDim.x * blockDim.x) {
    D[q * d_stride + s] = band[s * ldb];
    if (s >= n - 1) continue;
    double x = band[1 + s * ldb];
    if (s > 0 && band[1 + (s - 1) * ldb] != 0.0) x = -x;
    if (s < n - 2 && x != 0.0) {
      U[q * u_stride + s + 1 + s * ldu] = (float)(x >= 0.0 ? 1.41421356237309504880 : -1.41421356237309504880);
      x = -x;
    }
    E[q * e_stride + s] = x;
  }
}

size_t sb2st_batched_workspace(int count, long n, long b) {
  return align256((size_t)count * 2 * mail_half(n, b) * sizeof(double) +
                  ((size_t)count * n * kComStride + kTicketWords) * sizeof(int));
}

// The XCDs' boxes are scratch on top of that, used where the arena has room
// (a call never fails for want of them; the results are the same).
static size_t chase_boxes_bytes(int count, long n, long b) {
  count = chase_batch(count, n, b);
  return (size_t)chase_members(count, n, b) * count * 2 * mail_half(n, b) * sizeof(double);
}

// Bulge chasing of `count` same-size bands in one persistent launch (problem q
// at band + q band_stride, U + q u_stride, D + q d_stride, E + q e_stride).
// The progress words and the ticket come from the arena, or from ext_com
// (at least sb2st_batched_workspace(count, n, b) bytes) when it is given.
int sb2st_batched(evd_ctx *ctx, int count, long n, long b, double *band, long ldband, long band_stride, float *U,
                  long ldu, long u_stride, double *D, long d_stride, double *E, long e_stride, int *ext_com) {
  if (n <= 0 || count <= 0) return 0;
  if (u_stride == ldu * n)
    EVD_TRY(fill_f32(ctx, U, ldu, n * count, ldu, 0.f));
  else
    for (int q = 0; q < count; q++) EVD_TRY(fill_f32(ctx, U + (long)q * u_stride, ldu, n, ldu, 0.f));
  if (n > 2) {
    ArenaFrame frame(ctx);
    // messages, then progress words com[q * n * kComStride + s * kComStride]
    // and the ticket
    const long com_stride = n * kComStride;
    const size_t words = (size_t)count * com_stride + kTicketWords;
    double *mail = ext_com ? reinterpret_cast<double *>(ext_com)
                           : arena_alloc_n<double>(ctx, sb2st_batched_workspace(count, n, b) / sizeof(double));
    if (!mail) return EVD_E_NOMEM;
    int *com = reinterpret_cast<int *>(mail + 2 * mail_half(n, b) * count);
    unsigned *ticket = reinterpret_cast<unsigned *>(com + (size_t)count * com_stride);
    EVD_TRY(fill_u32(ctx, reinterpret_cast<unsigned *>(com), words, 0u));
    // sweeps per workgroup: the knob (0 = 1, one sweep per workgroup), at most
    // what the LDS window holds and at most 3 (with more than four waves a
    // workgroup's waves share SIMDs and the grouped kernel's registers spill)
    const int depth = std::min({ctx->tune.chase_depth > 0 ? ctx->tune.chase_depth : 1, group_depth_max(b), 3});
    if (b > 64) return set_error(ctx, EVD_E_UNSUPPORTED, "bandwidth %ld > 64", b);
    auto boxes = [&]() -> double * {
      if (chase_members(chase_batch(count, n, b), n, b) > kXcds) return nullptr;
      const size_t bytes = chase_boxes_bytes(count, n, b);
      const size_t room = ctx->arena_bytes - std::min(ctx->arena_bytes, align256(ctx->arena_top));
      return ext_com || bytes > room ? nullptr : static_cast<double *>(arena_alloc(ctx, bytes));
    };
    if (b <= 32 && depth > 1) {
      if (depth == 3)
        EVD_TRY(launch_chase_group<3>(ctx, count, n, b, band, ldband, band_stride, U, ldu, u_stride, com, com_stride,
                                      ticket));
      else
        EVD_TRY(launch_chase_group<2>(ctx, count, n, b, band, ldband, band_stride, U, ldu, u_stride, com, com_stride,
                                      ticket));
    } else if (b == 1) {
      chase_signs_kernel<<<dim3((unsigned)std::min<long>((n + 255) / 256, 1024), (unsigned)count), 256, 0,
                           ctx->stream>>>((int)n, band, ldband, band_stride, U, ldu, u_stride, D, d_stride, E, e_stride);
      EVD_LAUNCHED(ctx);
      return 0;
    } else {
      double *bx = boxes();
      const int batch = bx ? chase_batch(count, n, b) : count;
      for (int q0 = 0; q0 < count; q0 += batch) {
        const int c = std::min(batch, count - q0);
        if (q0 > 0) EVD_TRY(fill_u32(ctx, ticket, kTicketWords, 0u));
        const double *bq = band + (long)q0 * band_stride;
        double *mq = mail + (long)q0 * 2 * mail_half(n, b);
        float *Uq = U + (long)q0 * u_stride;
        int *cq = com + (long)q0 * com_stride;
        double *Dq = D + (long)q0 * d_stride, *Eq = E + (long)q0 * e_stride;
        if (b <= 32)
          EVD_TRY(launch_chase<32>(ctx, c, n, b, bq, ldband, band_stride, mq, bx, Uq, ldu, u_stride, cq, ticket, Dq,
                                   d_stride, Eq, e_stride));
        else
          EVD_TRY(launch_chase<64>(ctx, c, n, b, bq, ldband, band_stride, mq, bx, Uq, ldu, u_stride, cq, ticket, Dq,
                                   d_stride, Eq, e_stride));
      }
      return 0;
    }
  }
  band_extract_batched_kernel<<<dim3((unsigned)std::min<long>((n + 255) / 256, 1024), (unsigned)count), 256, 0,
                                ctx->stream>>>((int)n, band, ldband, band_stride, D, d_stride, E, e_stride);
  EVD_LAUNCHED(ctx);
  return 0;
}


int sb2st(evd_ctx *ctx, long n, long b, double *band, long ldband, float *U, long ldu, double *D, double *E) {
  return sb2st_batched(ctx, 1, n, b, band, ldband, 0, U, ldu, 0, D, 0, E, 0, nullptr);
}

// arena of a chase called by itself: with the XCDs' boxes where it may grow to
// that (no captured graph, lent arena or budget against it), else without
static int chase_arena(evd_ctx *ctx, int count, long n, long b) {
  const size_t need = sb2st_batched_workspace(count, n, b) + 4096, all = need + chase_boxes_bytes(count, n, b);
  if (chase_members(chase_batch(count, n, b), n, b) <= kXcds && all > ctx->arena_bytes && ctx->graphs == 0 && !ctx->arena_external && !(ctx->budget && all > ctx->budget) &&
      arena_ensure(ctx, all) == 0)
    return 0;
  return arena_ensure(ctx, need);
}

// ---- the chase without allocation: scratch in a file-scope device array.
// Messages, progress words (one per sweep, kComStride apart) and the sweep
// ticket of one problem of order <= kNoAllocMaxN: 69 MiB per device, held
// until the process ends.  Host code never passes the array's name to a kernel (it is a
// host-side stand-in); it uses the device address that hipGetSymbolAddress
// returns, looked up once per device with that device current.
constexpr long kNoAllocMaxN = 32768;
constexpr size_t kNoAllocWords = (size_t)kNoAllocMaxN * (kComStride + 4 * 2 * 64) + 131072;
static __device__ __align__(256) int scratch[kNoAllocWords];

static int noalloc_scratch(evd_ctx *ctx, int **out) {
  static std::mutex mu;
  static std::map<int, int *> ptrs;
  std::lock_guard<std::mutex> lk(mu);
  auto it = ptrs.find(ctx->device);
  if (it != ptrs.end()) {
    *out = it->second;
    return 0;
  }
  int cur = -1;
  EVD_HIP(ctx, hipGetDevice(&cur));
  if (cur != ctx->device) EVD_HIP(ctx, hipSetDevice(ctx->device));
  int *p = nullptr;
  const hipError_t e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
  if (cur != ctx->device) EVD_HIP(ctx, hipSetDevice(cur));
  if (e != hipSuccess || !p)
    return set_error(ctx, EVD_E_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
  ptrs[ctx->device] = p;
  *out = p;
  return 0;
}

}  // namespace evd

using namespace evd;

extern "C" int evd_band_pack_f32(evd_ctx *ctx, long n, long b, const float *A, long lda, double *band, long ldband) {
  if (!ctx) return -1;
  EVD_ARG(ctx, n >= 0, 2);
  EVD_ARG(ctx, b >= 1 && b <= 64, 3);
  EVD_ARG(ctx, lda >= std::max<long>(1, n), 5);
  EVD_ARG(ctx, ldband >= 2 * b, 7);
  return band_pack(ctx, n, b, A, lda, band, ldband);
}

extern "C" int evd_sb2st_f64(evd_ctx *ctx, long n, long b, double *band, long ldband, float *U, long ldu, double *D,
                             double *E) {
  if (!ctx) return -1;
  EVD_ARG(ctx, n >= 0, 2);
  EVD_ARG(ctx, b >= 1 && b <= 64, 3);
  EVD_ARG(ctx, ldband >= 2 * b, 5);
  EVD_ARG(ctx, ldu >= n + b, 7);
  if (ctx->arena_top == 0) EVD_TRY(chase_arena(ctx, 1, n, b));
  EVD_TRY(sb2st(ctx, n, b, band, ldband, U, ldu, D, E));
  return check_device_error(ctx, "evd_sb2st_f64");
}

extern "C" int evd_sb2st_f64_noalloc(evd_ctx *ctx, long n, long b, double *band, long ldband, float *U, long ldu,
                                     double *D, double *E) {
  if (!ctx) return -1;
  EVD_ARG(ctx, n >= 0, 2);
  EVD_ARG(ctx, b >= 1 && b <= 64, 3);
  EVD_ARG(ctx, ldband >= 2 * b, 5);
  EVD_ARG(ctx, ldu >= n + b, 7);
  if (n > kNoAllocMaxN)
    return set_error(ctx, EVD_E_UNSUPPORTED, "evd_sb2st_f64_noalloc: n = %ld exceeds the scratch limit n <= %ld", n,
                     kNoAllocMaxN);
  if (sb2st_batched_workspace(1, n, b) > kNoAllocWords * sizeof(int))
    return set_error(ctx, EVD_E_UNSUPPORTED, "evd_sb2st_f64_noalloc: n = %ld, b = %ld exceed the scratch", n, b);
  int *com = nullptr;
  EVD_TRY(noalloc_scratch(ctx, &com));
  EVD_TRY(sb2st_batched(ctx, 1, n, b, band, ldband, 0, U, ldu, 0, D, 0, E, 0, com));
  return check_device_error(ctx, "evd_sb2st_f64_noalloc");
}

extern "C" int evd_sb2st_batched_f64(evd_ctx *ctx, int count, long n, long b, double *band, long ldband,
                                     long band_stride, float *U, long ldu, long u_stride, double *D, long d_stride,
                                     double *E, long e_stride) {
  if (!ctx) return -1;
  EVD_ARG(ctx, count >= 0 && count <= 65535, 2);  // the band extraction carries the problem in grid y
  EVD_ARG(ctx, n >= 0, 3);
  EVD_ARG(ctx, b >= 1 && b <= 64, 4);
  EVD_ARG(ctx, ldband >= 2 * b, 6);
  EVD_ARG(ctx, count <= 1 || band_stride >= ldband * n, 7);
  EVD_ARG(ctx, ldu >= n + b, 9);
  EVD_ARG(ctx, count <= 1 || u_stride >= ldu * n, 10);
  EVD_ARG(ctx, count <= 1 || d_stride >= n, 12);
  EVD_ARG(ctx, count <= 1 || e_stride >= std::max<long>(1, n - 1), 14);
  EVD_ARG(ctx, (long)count * std::max<long>(n, 1) < (1L << 30), 2);
  if (ctx->arena_top == 0) EVD_TRY(chase_arena(ctx, count, n, b));
  EVD_TRY(sb2st_batched(ctx, count, n, b, band, ldband, band_stride, U, ldu, u_stride, D, d_stride, E, e_stride,
                        nullptr));
  return check_device_error(ctx, "evd_sb2st_batched_f64");
}
