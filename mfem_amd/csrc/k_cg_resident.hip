// Jacobi-preconditioned CG with the whole system resident in registers: one
// cooperative launch runs every iteration of a solve (k_solver.hip holds the
// one-kernel-per-iteration CG, whose algorithm, scalars and stopping test this
// kernel follows).
//
// What bounds the CG of a system that fits the chip is not its bytes but the
// chain of one iteration: launch, stop flag, partial sums, row pointers,
// columns, gathers, block reduction, and K read again. Here every lane keeps
// its blocks of K in registers (some in LDS, the last ones of a large system in
// the L2) for the whole solve, and a workgroup keeps r, p and D^-1 of every
// column that its rows touch, its own and its neighbours', so that an iteration
// exchanges only q = K p (one word per scalar row) and five partial sums per
// workgroup:
//
//   wait for all partial sums of iteration it-1   -> alpha, beta
//   wait for q_{it-1} at the neighbours' columns
//   r -= alpha q, p = D^-1 r + beta p at every column (the same arithmetic as
//     in the row's own workgroup, so the copies equal it bit for bit); p in LDS
//   q_it = K p; publish q_it and the workgroup's partial sums
//
// Measured on MI355X, us per iteration against the one-kernel-per-iteration CG:
// 468 rows FP64 2.9 (8.1), 4840 rows FP64 3.5 (9.2), 37.5k rows FP64 4.9 (16),
// 54.8k rows FP32 6.3 (13.2), 168k rows FP32 14.3 (26). What is left of a small
// system's 2.9 us is the exchange (0.6 us on one XCD, 1-2 us over all), three
// workgroup barriers, two chains of wave sums, the two divisions and the loads
// of q.
//
// Exchange. Every published word is its own flag: buffers hold a signalling
// NaN (no arithmetic produces one) until the value is stored, and a reader
// polls the word itself. Words are relaxed agent-scope atomics, which are
// coherent between the XCDs without any cache being written back or invalidated
// (while one XCD alone touches a word its L2 serves it in 0.1 us; store to load
// across XCDs takes 1-2 us); no ordering between different words is needed except
// for the reset below. Three slots rotate with the iteration:
//   - a workgroup publishes its sums of `it` only after all its lanes have read
//     every word of it-1 that they need, so once all sums of it-1 have arrived,
//     nobody reads slot it-2 any more, and its owner resets it;
//   - the owner's reset has completed (vmcnt) before it publishes the sums of
//     `it`, and a reader polls the slot's next value (q_{it+1}) only after
//     those sums have arrived: it never sees a value of it-2.
// Every wait ends: the launch is cooperative (all workgroups are resident), and
// a wait that lasts longer than `wait_ticks` of the wall clock raises a flag
// that every other wait polls; all workgroups then leave, the control block
// says so, and the host solves with the one-kernel-per-iteration CG instead.
//
// Verdict. A solve has one verdict word, which leaves 0 once, by compare-exchange:
// workgroup 0 makes it `done` when it has the sums that stop the solve, and a
// workgroup that gives up a wait makes it `expired`. Whoever loses follows the
// winner, so all workgroups leave a solve with the same answer:
//   - a workgroup whose wait runs out behind `done` keeps polling. Workgroup 0 has
//     seen the sums of every workgroup, so each of them is past every other wait
//     of this solve, and the sums that it still polls are all there;
//   - a workgroup that has the stopping sums itself waits for the verdict before
//     it writes its rows of x. The sums are published, so workgroup 0 gets them
//     too, or leaves by a wait that ran out, and gives the verdict either way.
// x is therefore written whole, or not at all.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include "kernels.h"
#include "reduce.h"

namespace mfemhip {

namespace {

template <typename T>
struct Word;
template <>
struct Word<double> {
  using U = unsigned long long;
  static constexpr U kEmpty = 0x7FF45A5AC3C39696ull;
};
template <>
struct Word<float> {
  using U = unsigned int;
  static constexpr U kEmpty = 0x7FA5C396u;
};
using U64 = unsigned long long;
constexpr U64 kEmpty64 = Word<double>::kEmpty;

template <typename U>
__device__ __forceinline__ U word_load(const U* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void word_store(U* p, U v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// base[i] with a 32-bit byte offset (one register next to a uniform base)
template <typename U>
__device__ __forceinline__ U* word_at(U* base, unsigned i) {
  using C = typename std::conditional<std::is_const<U>::value, const char, char>::type;
  return reinterpret_cast<U*>(reinterpret_cast<C*>(base) + i * (unsigned)sizeof(U));
}
// v, recomputed where it is used instead of being kept in registers over an
// iteration
__device__ __forceinline__ unsigned opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

// whether a word has not been published (its upper half tells: no number and
// no NaN of the arithmetic has it)
__device__ __forceinline__ bool is_empty(U64 w) {
  return (unsigned)(w >> 32) == (unsigned)(kEmpty64 >> 32);
}
__device__ __forceinline__ bool is_empty(unsigned w) { return w == Word<float>::kEmpty; }

// v of the lane that the DPP control names (0 where there is none)
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const U64 b = __builtin_bit_cast(U64, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((U64)(unsigned)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

// Sum over 8 or 16 consecutive lanes of three values at once: lane l of a
// group gets the sum of value l & 3 (value 3 is 0). Lanes exchange the value
// that the other one keeps (xor 1, then xor 2 by quad_perm); the mirrors of
// half rows and rows stand for xor 4 and xor 8 between equal lanes l & 3.
template <int G, typename T>
__device__ __forceinline__ T group_sum3(T y0, T y1, T y2, int lane) {
  static_assert(G == 8 || G == 16, "lane group");
  const bool b0 = lane & 1, b1 = lane & 2;
  const T lo = (b0 ? y1 : y0) + dpp_mov<0xB1>(b0 ? y0 : y1);
  const T hi = (b0 ? (T)0 : y2) + dpp_mov<0xB1>(b0 ? y2 : (T)0);
  T v = (b1 ? hi : lo) + dpp_mov<0x4E>(b1 ? lo : hi);
  // half_mirror maps lane l to 7 - l: quad order reversed, undone by [3,2,1,0]
  v += dpp_mov<0x1B>(dpp_mov<0x141>(v));
  if constexpr (G == 16) v += dpp_mov<0x1B>(dpp_mov<0x140>(v));
  return v;
}
// Sum over the wave, valid in lane 63.
__device__ __forceinline__ double wave_sum_63(double v) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  v += dpp_mov<0x140>(v);
  const int row = (threadIdx.x & 63) >> 4;
  const double a = dpp_mov<0x142>(v);  // lane 15 of the previous row
  if (row & 1) v += a;
  const double b = dpp_mov<0x143>(v);  // lane 31 to the upper half
  if (row & 2) v += b;
  return v;
}

// The control block to the device copy and, every field before done, to the
// host's mapped one.
__device__ __forceinline__ void publish_stop(const PcgCtrl& c, PcgCtrl* ctrl, PcgCtrl* mirror) {
  *ctrl = c;
  if (!mirror) return;
  PcgCtrl m = c;
  m.done = 0;
  *mirror = m;
  __threadfence_system();
  __hip_atomic_store(&mirror->done, c.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// v, the same in every lane, as one scalar
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Makes the verdict v if there is none yet; returns the verdict.
__device__ __forceinline__ int decide(int* verdict, int v) {
  int is = 0;
  return __hip_atomic_compare_exchange_strong(verdict, &is, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT)
             ? v
             : is;
}

// Bounded wait. The flag is 0 until a workgroup of the launch gives up. It is looked
// at, and the clock, every 16th poll: from 0, or from 15 where there is no time at
// all (as a test of `ticks` in every poll it cost 0.3 ms of a 34 ms step of 48 beams).
struct Waiter {
  int* flag;
  int* verdict;
  long long ticks;
  int polls;
  long long start = 0;
  // true when the wait has to be given up
  __device__ __forceinline__ bool expired() {
    if (__builtin_expect(++polls & 15, 1)) return false;
    const int left = word_load(flag);
    if (!left) {
      const long long now = (long long)wall_clock64();
      if (polls == 16) start = now;
      if (now - start < ticks) return false;
    }
    if (decide(verdict, kCgExpired) == kCgDone) return false;
    if (!left) word_store(flag, kCgExpired);
    return true;
  }
};

// Inclusive scan of one value per thread over the workgroup.
template <int BS>
__device__ __forceinline__ unsigned block_scan(unsigned v, unsigned* sm) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned t = __shfl_up(v, off, kWave);
    if (lane >= off) v += t;
  }
  if (lane == kWave - 1) sm[wid] = v;
  __syncthreads();
  for (int i = 0; i < wid; ++i) v += sm[i];
  return v;
}

// LDS of a workgroup: the list of its columns, then either the bit set that
// numbers them (start) or the block values beyond NREG, x, z, D^-1 and q of its
// own rows and p of its columns (solve; p takes what is left).
template <int R, int NLDS, int EPT, int BS, int G, typename T>
struct ResidentLds {
  static constexpr int kRows = R * (BS / G);  // most rows of a workgroup
  static constexpr int kList = EPT * BS / 3;  // most columns of a workgroup
  static constexpr int list = 0;
  static constexpr int start = (4 * kList + 15) / 16 * 16;
  static constexpr int x = start;
  static constexpr int v = x + 8 * 3 * kRows;
  static constexpr int z = v + NLDS * 9 * BS * (int)sizeof(T);
  static constexpr int d = z + 3 * kRows * (int)sizeof(T);
  static constexpr int q = d + 3 * kRows * (int)sizeof(T);
  static constexpr int p = (q + 3 * kRows * (int)sizeof(T) + 15) / 16 * 16;
};

// G lanes per block row, U blocks of the row per lane, R rows per lane group:
// a workgroup holds up to R BS / G rows of up to U G blocks each. The values of
// a lane's first NREG blocks stay in registers, of the next NLDS in LDS; those
// of any further ones are copied once, lane by lane, to global memory
// (A.spill) and read back every iteration, from the XCD's L2 or the Infinity
// Cache, in coalesced loads. The columns
// that the workgroup's rows touch are numbered locally (ascending); their p
// lives in LDS, their r and D^-1 with the thread that updates them, EPT scalar
// columns ("entries") per thread.
//
// One system takes all workgroups. Of many independent ones (A.sys) each is
// solved by a team on one XCD, 32 workgroups for the large systems (phase 0)
// and then 8 for the small ones (phase 1); a team takes its list of systems
// one after the other, its slots rotating on.
template <int G, int U, int R, int NREG, int NLDS, int EPT, int BS, typename T>
__global__ __launch_bounds__(BS) void k_cg_resident(CgResidentArgs<T> A) {
  using W = typename Word<T>::U;
  constexpr W kEmpty = Word<T>::kEmpty;
  constexpr int NB = R * U;
  constexpr int NSTR = NB - NREG - NLDS;
  constexpr bool kLean = (NREG * 9 + 3 * EPT) * sizeof(T) > 100 * 4;  // registers are short
  constexpr int NP = kCgParts + 1;  // five sums, and |b|^2 with the first
  constexpr int kAcc = 3 * (BS / G);
  constexpr int kPolls = kCgResidentMaxWg / kWave;
  using L = ResidentLds<R, NLDS, EPT, BS, G, T>;
  constexpr int NW = BS / kWave;
  extern __shared__ __align__(16) unsigned char dyn[];
  __shared__ double s_acc[NP][BS / 4 > kAcc ? BS / 4 : kAcc];
  __shared__ double s_tot[NP];
  __shared__ unsigned s_scan[BS / kWave];
  __shared__ int s_dead, s_verdict;
  if (blockIdx.x % A.stride) return;
  const unsigned n = 3u * (unsigned)A.nrows;
  const int first_look = A.wait_ticks > 0 ? 0 : 15;
  for (int phase = 0; phase < (A.sys ? 2 : 1); ++phase) {
  int nw = gridDim.x / A.stride;  // workgroups of the team
  int wg;                         // this one's number in it
  int g0 = 0;                     // the team's first place in A.parts
  int s0 = 0, s1 = 1;             // its systems
  if (A.sys) {
    nw = phase ? kCgTeamSmall : kCgTeamLarge;
    const int g = (blockIdx.x & 7) * kCgTeamLarge + (blockIdx.x >> 3);
    wg = g % nw;
    g0 = g - wg;
    const int* t = A.team + (phase ? 9 : 0) + g / nw;
    s0 = uniform(t[0]);
    s1 = uniform(t[1]);
  } else {
    // workgroups go round-robin over the 8 XCDs: neighbouring rows on one XCD
    wg = blockIdx.x / A.stride;
    if (A.stride == 1 && (nw & 7) == 0) wg = (blockIdx.x & 7) * (nw >> 3) + (blockIdx.x >> 3);
  }
  U64* const parts = A.parts + (size_t)phase * 3 * kCgResidentMaxWg * 8;
  int slot = 0, prev = 2, prev2 = 1;  // iterations it, it-1 and it-2 of the team, modulo 3
  bool used = false;                  // slot prev2 holds sums
  for (int si = s0; si < s1; ++si) {
  // (nothing of a lane is kept in registers from one system to the next)
  const int tid = opaque(threadIdx.x), lane = tid & (G - 1), wid = tid / kWave;
  CgResidentSys sys{0, A.nrows, A.max_iters, 0, A.tol};
  if (A.sys) {
    const CgResidentSys q = A.sys[si];
    sys = CgResidentSys{uniform(q.row0), uniform(q.row1), uniform(q.max_iters), uniform(q.id),
                        q.tol};
  }
  int* const verdict = A.flag + 1 + sys.id;
  PcgCtrl* const ctrl = A.ctrl + sys.id;
  PcgCtrl* const mirror = A.mirror ? A.mirror + sys.id : nullptr;
  const int nrows = sys.row1 - sys.row0;
  const int c0 = sys.row0 + (int)((long long)nrows * wg / nw);
  const int c1 = sys.row0 + (int)((long long)nrows * (wg + 1) / nw);
  const int rows = c1 - c0;
  __syncthreads();  // the LDS of the previous system
  if (tid == 0) s_dead = 0;

  // local numbering of the columns: a bit per block row, ranks by popcount
  unsigned* const list = reinterpret_cast<unsigned*>(dyn + L::list);
  const int nword = (nrows + 31) / 32;
  unsigned* const bits = reinterpret_cast<unsigned*>(dyn + L::start);
  unsigned* const pre = bits + nword;
  for (int i = tid; i < nword; i += BS) bits[i] = 0;
  __syncthreads();
  const int b0 = A.rowptr[c0], b1 = A.rowptr[c1];
  for (int q = b0 + tid; q < b1; q += BS) {
    const unsigned j = A.col[q] - sys.row0;
    atomicOr(&bits[j >> 5], 1u << (j & 31));
  }
  for (int i = c0 - sys.row0 + tid; i < c1 - sys.row0; i += BS)
    atomicOr(&bits[i >> 5], 1u << (i & 31));
  __syncthreads();
  const int per = (nword + BS - 1) / BS;
  const int i0 = min(nword, tid * per), i1 = min(nword, i0 + per);
  unsigned cnt = 0;
  for (int i = i0; i < i1; ++i) cnt += __popc(bits[i]);
  unsigned at = block_scan<BS>(cnt, s_scan) - cnt;
  for (int i = i0; i < i1; ++i) {
    pre[i] = at;
    for (unsigned m = bits[i]; m; m &= m - 1) {
      if (at < (unsigned)L::kList) list[at] = sys.row0 + 32u * i + (__ffs(m) - 1);
      ++at;
    }
  }
  __syncthreads();
  auto rank = [&](unsigned j) {
    j -= sys.row0;
    return pre[j >> 5] + __popc(bits[j >> 5] & ((1u << (j & 31)) - 1u));
  };
  const unsigned H = uniform(pre[nword - 1] + __popc(bits[nword - 1]));
  const unsigned nent = 3 * H, own0 = 3 * uniform(rank(c0)), nown = 3 * (c1 - c0);
  // p has one more row, of zeros, for the lanes without a block
  const size_t pbytes = (size_t)(nent + 3) * sizeof(T);
  if (H > (unsigned)L::kList || L::p + pbytes > (size_t)A.lds || pbytes > 65536) {
    // the same for every thread of the workgroup; the others leave by the flag
    if (tid == 0) word_store(A.flag, kCgNoFit);
    if (tid == 0 && wg == 0) {
      PcgCtrl o{};
      o.done = kCgNoFit;
      publish_stop(o, ctrl, mirror);
    }
    return;
  }
  // the lane's blocks: byte offset of p at their columns, 16 bits each
  unsigned off[(NB + 1) / 2];
#pragma unroll
  for (int i = 0; i < (NB + 1) / 2; ++i) off[i] = 0;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int row = c0 + (i / U) * (BS / G) + tid / G;
    const int q = row < c1 ? A.rowptr[row] + lane + (i % U) * G : 0;
    const bool on = row < c1 && q < A.rowptr[row + 1];
    off[i / 2] |= (3 * (on ? rank(A.col[q]) : H) * (unsigned)sizeof(T)) << (16 * (i & 1));
  }
  __syncthreads();  // the bit set is read; its LDS takes the solve's arrays
  double* const xl = reinterpret_cast<double*>(dyn + L::x);
  T* const vl = reinterpret_cast<T*>(dyn + L::v);
  T* const zl = reinterpret_cast<T*>(dyn + L::z);
  T* const dl = reinterpret_cast<T*>(dyn + L::d);
  T* const ql = reinterpret_cast<T*>(dyn + L::q);
  T* const pl = reinterpret_cast<T*>(dyn + L::p);
  T* const vs = A.spill + (size_t)(g0 + wg) * NSTR * 9 * BS;  // [NSTR][9][BS]
  T V[NREG][9];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int row = c0 + (i / U) * (BS / G) + tid / G;
    const int q = row < c1 ? A.rowptr[row] + lane + (i % U) * G : 0;
    const bool on = row < c1 && q < A.rowptr[row + 1];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const T v = on ? A.K[(size_t)9 * q + k] : (T)0;
      if (i < NREG) V[i][k] = v;
      else if (i < NREG + NLDS) vl[((i - NREG) * 9 + k) * BS + tid] = v;
      else vs[((i - NREG - NLDS) * 9 + k) * BS + tid] = v;
    }
  }
  // entries: r = b, D^-1 and p = 0
  T r[EPT], d[EPT];
  double bb = 0.0;
#pragma unroll
  for (int m = 0; m < EPT; ++m) {
    const unsigned e = tid + m * BS, o = e - own0;
    r[m] = d[m] = (T)0;
    if (e < nent + 3) pl[e] = (T)0;
    if (e < nent) {
      const unsigned g = 3 * list[e / 3] + e % 3;
      const double b = A.b[g];
      r[m] = (T)b;
      d[m] = A.invdiag[g];
      if (o < nown) {
        bb += b * b;
        xl[o] = 0.0;
        dl[o] = d[m];
        ql[o] = (T)0;
      }
    }
  }
  for (unsigned e = EPT * BS + tid; e < nent + 3; e += BS) pl[e] = (T)0;  // the zero row
  double threshold = 0.0, b2 = 0.0, alpha = 0.0, beta = 0.0;
  int done = kCgExpired;
  for (int it = 0;; ++it) {
    Waiter wait{A.flag, verdict, A.wait_ticks, first_look};
    bool dead = false;
    W w[EPT];
#pragma unroll
    for (int m = 0; m < EPT; ++m) w[m] = 0;
    const W* qv = A.q + (size_t)prev * n;
    if (it > 0) {
      // q_{it-1} of the other workgroups' columns, in flight while the sums
      // are awaited
      const unsigned t = (kLean ? opaque(tid) : (unsigned)tid);
#pragma unroll
      for (int m = 0; m < EPT; ++m) {
        const unsigned e = t + m * BS;
        if (m * BS < nent && e < nent && e - own0 >= nown)
          w[m] = word_load(word_at(qv, 3 * list[e / 3] + e % 3));
      }
      // sums of iteration it-1 over the workgroups, one per wave at a time
      for (int k = wid; k < (it == 1 ? NP : kCgParts); k += NW) {
        const U64* src = parts + ((size_t)prev * kCgResidentMaxWg + g0) * 8 + k;
        U64 s[kPolls];
#pragma unroll
        for (int h = 0; h < kPolls; ++h) {
          const int o = h * kWave + (tid & (kWave - 1));
          s[h] = o < nw ? word_load(src + 8 * o) : 0;
        }
        double v = 0.0;
#pragma unroll
        for (int h = 0; h < kPolls; ++h) {
          const int o = h * kWave + (tid & (kWave - 1));
          while (s[h] == kEmpty64 && !dead) {
            dead = wait.expired();
            s[h] = word_load(src + 8 * o);
          }
          v += __builtin_bit_cast(double, s[h]);
        }
        v = wave_sum_63(v);
        if ((tid & (kWave - 1)) == kWave - 1) s_tot[k] = v;
      }
      if (dead) s_dead = 1;
      __syncthreads();
      if (s_dead) break;
      // slot it-2 has been read everywhere: empty it for it+1
      if (used && tid < NP)
        word_store(parts + ((size_t)prev2 * kCgResidentMaxWg + g0 + wg) * 8 + tid, kEmpty64);
      const double pq = s_tot[0], zq = s_tot[1], qdq = s_tot[2], rr = s_tot[3], rz = s_tot[4];
      if (it == 1) {
        b2 = s_tot[kCgParts];
        threshold = fmax(sys.tol * sys.tol * b2, DBL_MIN);
      }
      const int jt = it - 1;  // iteration of the sums
      const bool converged = rr < threshold || b2 == 0.0;
      if (converged || jt >= sys.max_iters) {
        if (tid == 0) {
          int v;
          if (wg == 0) {
            v = decide(verdict, kCgDone);
            if (v == kCgDone) {
              PcgCtrl o{};
              o.rr = rr;
              o.b2 = b2;
              o.threshold = threshold;
              o.iter = converged ? (jt > 0 ? jt - 1 : 0) : jt;
              o.done = kCgDone;
              o.max_iters = sys.max_iters;
              o.stop_it = it;
              o.started = it;
              publish_stop(o, ctrl, mirror);
            }
          } else {
            while (!(v = word_load(verdict))) __builtin_amdgcn_s_sleep(1);
          }
          s_verdict = v;
        }
        __syncthreads();
        done = s_verdict;
        break;
      }
      // (the two divisions side by side)
      const double irz = 1.0 / rz;
      alpha = rz / pq;
      beta = (rz - 2.0 * alpha * zq + alpha * alpha * qdq) * irz;
    }
    const T a = (T)alpha, bt = (T)beta;
    double acc[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) acc[k] = 0.0;
    acc[kCgParts] = bb;
    W* old = A.q + (size_t)prev2 * n;
    {
      const unsigned t = (kLean ? opaque(tid) : (unsigned)tid);
#pragma unroll
      for (int m = 0; m < EPT; ++m) {
        const unsigned e = t + m * BS, o = e - own0;
        if (m * BS < nent && e < nent) {
          const bool own = o < nown;
          T q;
          if (own) {
            q = ql[o];
            if (it > 1) word_store(word_at(old, 3 * (unsigned)c0 + o), kEmpty);
          } else {
            while (is_empty(w[m]) && !dead) {
              dead = wait.expired();
              w[m] = word_load(word_at(qv, 3 * list[e / 3] + e % 3));
            }
            q = __builtin_bit_cast(T, w[m]);
          }
          const T p = pl[e];
          r[m] = fma(-a, q, r[m]);
          const T z = d[m] * r[m];
          pl[e] = fma(bt, p, z);
          if (own) {
            xl[o] += alpha * (double)p;
            zl[o] = z;
            acc[3] += (double)r[m] * (double)r[m];
            acc[4] += (double)r[m] * (double)z;
          }
        }
      }
    }
    if (dead) s_dead = 1;  // seen behind the barriers below
    __syncthreads();
    // q = K p, published pass by pass
    W* now = A.q + (size_t)slot * n;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      T y0 = 0, y1 = 0, y2 = 0;
      if (R == 1 || j * (BS / G) < rows) {  // the pass has rows
        // one pass's loads at a time where registers are short
        if constexpr (NSTR > 0 || NLDS > 0) asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = j * U + u;
          const T* p = reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(pl) +
                                                  ((off[i / 2] >> (16 * (i & 1))) & 0xffff));
          T v[9];
          unsigned ks = i < NREG + NLDS ? 0 : opaque((i - NREG - NLDS) * 9 * BS + tid);
#pragma unroll
          for (int k = 0; k < 9; ++k) {
            v[k] = i < NREG ? V[i < NREG ? i : 0][k]
                   : i < NREG + NLDS ? vl[((i - NREG) * 9 + k) * BS + tid]
                                     : *word_at(vs, ks);
            ks += BS;
          }
          const T p0 = p[0], p1 = p[1], p2 = p[2];
          y0 += v[0] * p0 + v[1] * p1 + v[2] * p2;
          y1 += v[3] * p0 + v[4] * p1 + v[5] * p2;
          y2 += v[6] * p0 + v[7] * p1 + v[8] * p2;
        }
      }
      const T q = group_sum3<G>(y0, y1, y2, lane);
      // the resets of this iteration are complete before anything of it is
      // published
      if (j == 0) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      const unsigned o = 3 * (j * (BS / G) + tid / G) + lane;
      if (lane < 3 && o < nown) {
        word_store(word_at(now, 3 * (unsigned)c0 + o), __builtin_bit_cast(W, q));
        ql[o] = q;
        const double dq = (double)q;
        acc[0] += (double)pl[own0 + o] * dq;
        acc[1] += (double)zl[o] * dq;
        acc[2] += dq * ((double)dl[o] * dq);
      }
    }
    // sums of the workgroup: r.r, r.z and |b|^2 from any lane (by quads), the
    // others from lanes 0-2 of the groups
#pragma unroll
    for (int k = 3; k < NP; ++k) {
      acc[k] += dpp_mov<0xB1>(acc[k]);
      acc[k] += dpp_mov<0x4E>(acc[k]);
      if ((tid & 3) == 0) s_acc[k][tid / 4] = acc[k];
    }
    if (lane < 3) {
#pragma unroll
      for (int k = 0; k < 3; ++k) s_acc[k][(tid / G) * 3 + lane] = acc[k];
    }
    __syncthreads();
    if (s_dead) break;
    for (int k = wid; k < (it == 0 ? NP : kCgParts); k += NW) {
      double t = 0.0;
      const int m = k < 3 ? kAcc : BS / 4;
#pragma unroll
      for (int o = 0; o < (kAcc > BS / 4 ? kAcc : BS / 4); o += kWave) {
        const int i = o + (tid & (kWave - 1));
        t += i < m ? s_acc[k][i] : 0.0;
      }
      t = wave_sum_63(t);
      if ((tid & (kWave - 1)) == kWave - 1)
        word_store(parts + ((size_t)slot * kCgResidentMaxWg + g0 + wg) * 8 + k,
                   __builtin_bit_cast(U64, t));
    }
    used = used || it > 0 || si > s0;
    prev2 = prev;
    prev = slot;
    slot = slot == 2 ? 0 : slot + 1;
  }
  if (done != kCgDone) {  // x is not a solution
    if (wg == 0 && tid == 0) {
      PcgCtrl o{};
      o.done = word_load(A.flag) == kCgNoFit ? kCgNoFit : kCgExpired;
      publish_stop(o, ctrl, mirror);
    }
    return;
  }
  // the solution (the iterate of the last completed update)
  for (unsigned o = tid; o < nown; o += BS) A.x[3 * (unsigned)c0 + o] = xl[o];
  }
  }
}

// Empties the exchange buffers and the flag ahead of a solve.
template <typename W>
__global__ __launch_bounds__(256) void k_cg_resident_clear(W* q, long nq, W empty, U64* parts,
                                                           long np, int* flag, int nflag,
                                                           double* x, long nx) {
  const long i0 = blockIdx.x * 256L + threadIdx.x, step = gridDim.x * 256L;
  for (long i = i0; i < nq; i += step) q[i] = empty;
  for (long i = i0; i < nx; i += step) x[i] = 0.0;  // systems that are not solved
  for (long i = i0; i < np; i += step) parts[i] = kEmpty64;
  for (long i = i0; i < nflag; i += step) flag[i] = 0;
}

constexpr int kBS = 512;  // threads of a workgroup
constexpr int kLdsBytes = 150 * 1024;  // dynamic LDS of a workgroup (one per CU)

template <int G, int U, int R, int NREG, int NLDS, int EPT, int BS = kBS, typename T>
bool launch_shape(const CgResidentArgs<T>& A, int nwg, hipStream_t st) {
  static_assert(NREG + NLDS + kCgResidentSpill >= R * U, "spill area");
  using L = ResidentLds<R, NLDS, EPT, BS, G, T>;
  static_assert(L::p < kLdsBytes, "LDS");
  if (NREG + NLDS < R * U && !A.spill) return false;
  // the bit set that numbers one system's columns, and its ranks
  const long rows = A.sys ? A.sys_rows : A.nrows;
  if (L::start + 8L * ((rows + 31) / 32) > kLdsBytes) return false;
  const void* f = reinterpret_cast<const void*>(
      &k_cg_resident<G, U, R, NREG, NLDS, EPT, BS, T>);
  if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess)
    return false;
  CgResidentArgs<T> a = A;
  a.lds = kLdsBytes;
  void* args[] = {&a};
  return hipLaunchCooperativeKernel(f, dim3(nwg * A.stride), dim3(BS), args, kLdsBytes, st) ==
         hipSuccess;
}

// Rows per lane group (R) that each row length and value size has a kernel for,
// and the blocks of a lane that these keep in registers or LDS.
int max_passes(int max_row, int value_bytes) {
  const bool f32 = value_bytes == 4;
  return max_row <= 8 ? (f32 ? 16 : 8) : max_row <= 16 ? (f32 ? 11 : 5) : f32 ? 4 : 2;
}
int lane_group(int max_row) { return max_row > 32 ? 16 : 8; }
// more passes than the kernels without blocks in A.spill have
bool needs_spill(int R, int max_row, int value_bytes) {
  const bool f32 = value_bytes == 4;
  return R > (max_row <= 8 ? (f32 ? 8 : 4) : max_row <= 16 ? (f32 ? 6 : 3) : (f32 ? 2 : 1));
}

}  // namespace

// Workgroups: the exchange costs about the same from 8 to 256 of them, a pass
// of rows about 0.7 us, so a system gets one pass (64 rows) per workgroup while
// there are CUs left. Up to 32 workgroups stay on one XCD (every eighth
// workgroup of the launch), whose L2 they share: 468 rows in FP64 take 2.9 us
// an iteration on 16 workgroups of one XCD, 3.9 us on 64 over all of them; 4840
// rows 4.5 us on the 32 of one XCD, 3.5 us on three times as many over all.
// Over all XCDs 31 CUs of each at most: kernels of other streams still find one
// while a solve spins (256 instead of 248 workgroups gained nothing: 15.0 us an
// iteration at 168k rows either way). A small system may take a whole XCD, a batch
// takes every CU.
CgResidentPlan cg_resident_plan(int nrows, int max_row, int value_bytes) {
  constexpr int kMaxWg = kCgResidentMaxWg / 32 * 31;
  CgResidentPlan P;
  if (nrows <= 0 || max_row <= 0 || max_row > 64) return P;
  const long per_pass = kBS / lane_group(max_row);
  const long most = kMaxWg * per_pass * max_passes(max_row, value_bytes);
  if (nrows > most) return P;
  if (nrows <= 32 * per_pass) {
    P.stride = 8;
    P.nwg = (int)std::min<long>(32, (nrows + 31) / 32);
  } else {
    P.nwg = (int)std::min<long>(kMaxWg, (nrows + 8 * 50 - 1) / (8 * 50) * 8);
  }
  const int rows = (nrows + P.nwg - 1) / P.nwg;
  const int passes = (int)((rows + per_pass - 1) / per_pass);
  if (needs_spill(passes, max_row, value_bytes))
    P.spill = 9L * kCgResidentSpill * kBS * P.nwg;
  return P;
}

namespace {

template <typename T>
void clear(const CgResidentArgs<T>& A, hipStream_t st) {
  using W = typename std::remove_pointer<decltype(A.q)>::type;
  const long nq = 9L * A.nrows, np = (A.sys ? 2L : 1L) * 3 * 8 * kCgResidentMaxWg;
  const int gc = (int)std::min<long>(1024, (std::max(nq, np) + 255) / 256);
  hipLaunchKernelGGL(k_cg_resident_clear<W>, dim3(gc), dim3(256), 0, st, A.q, nq, Word<T>::kEmpty,
                     A.parts, np, A.flag, 1 + A.nsys, A.x, A.sys ? 3L * A.nrows : 0L);
}

// The kernel for R passes of rows of at most max_row blocks on nwg workgroups.
template <typename T>
bool launch_passes(const CgResidentArgs<T>& A, int nwg, int R, int max_row, hipStream_t st) {
  constexpr bool f32 = sizeof(T) == 4;
  // <lanes per row, blocks per lane, passes, blocks in registers, in LDS, columns
  // per thread / 3>. A register spilled to scratch costs an iteration as much as
  // a block value in A.spill and more latency, so the counts are the largest
  // that spill none or next to none: for 11 passes in FP32, 8 blocks in
  // registers take 15.0 us an iteration at 168k rows, 10 take 16.7, 11 took 18.4.
  if (max_row <= 8) {
    if (R <= 1) return launch_shape<8, 1, 1, 1, 0, 8>(A, nwg, st);
    if (R <= 2) return launch_shape<8, 1, 2, 2, 0, 8>(A, nwg, st);
    if (R <= 4) return launch_shape<8, 1, 4, 4, 0, 8>(A, nwg, st);
    if constexpr (f32) {
      if (R <= 8) return launch_shape<8, 1, 8, 8, 0, 12>(A, nwg, st);
      if (R <= 16) return launch_shape<8, 1, 16, 7, 3, 14>(A, nwg, st);
    } else {
      if (R <= 8) return launch_shape<8, 1, 8, 4, 2, 8>(A, nwg, st);
    }
  } else if (max_row <= 16) {
    if (R <= 1) return launch_shape<8, 2, 1, 2, 0, 8>(A, nwg, st);
    if (R <= 2) return launch_shape<8, 2, 2, 4, 0, 8>(A, nwg, st);
    if constexpr (f32) {
      if (R <= 4) return launch_shape<8, 2, 4, 8, 0, 8>(A, nwg, st);
      if (R <= 6) return launch_shape<8, 2, 6, 9, 3, 12>(A, nwg, st);
      if (R <= 11) return launch_shape<8, 2, 11, 8, 3, 14>(A, nwg, st);
    } else {
      if (R <= 3) return launch_shape<8, 2, 3, 4, 2, 8>(A, nwg, st);
      if (R <= 5) return launch_shape<8, 2, 5, 4, 2, 8>(A, nwg, st);
    }
  } else if (max_row <= 32) {
    if (R <= 1) return launch_shape<8, 4, 1, 4, 0, 8>(A, nwg, st);
    if constexpr (f32) {
      if (R <= 2) return launch_shape<8, 4, 2, 8, 0, 8>(A, nwg, st);
      if (R <= 4) return launch_shape<8, 4, 4, 10, 3, 12>(A, nwg, st);
    } else {
      if (R <= 2) return launch_shape<8, 4, 2, 4, 2, 8>(A, nwg, st);
    }
  } else if (max_row <= 64) {
    if (R <= 1) return launch_shape<16, 4, 1, 4, 0, 8>(A, nwg, st);
    if constexpr (f32) {
      if (R <= 2) return launch_shape<16, 4, 2, 8, 0, 8>(A, nwg, st);
      if (R <= 4) return launch_shape<16, 4, 4, 10, 3, 12>(A, nwg, st);
    } else {
      if (R <= 2) return launch_shape<16, 4, 2, 4, 2, 8>(A, nwg, st);
    }
  }
  return false;
}

}  // namespace

template <typename T>
bool launch_cg_resident(const CgResidentArgs<T>& A, int nwg, int max_row, hipStream_t st) {
  clear(A, st);
  const int rows = (A.nrows + nwg - 1) / nwg;  // the most rows a workgroup gets
  const int per_pass = kBS / lane_group(max_row);
  return launch_passes(A, nwg, (rows + per_pass - 1) / per_pass, max_row, st);
}

// Teams: a system of up to 8 * 128 rows takes a team of 8 workgroups, a larger
// one the 32 of an XCD. (An iteration costs 3-5 us in either, so small systems
// run four to an XCD; with few systems every one takes 32, as there is room.)
int cg_team_of(int rows, int nsys) {
  return rows <= kCgTeamSmall * 128 && nsys > 8 ? kCgTeamSmall : kCgTeamLarge;
}

int cg_resident_batch_passes(const int* row0, int nsys, int max_row, int value_bytes, long* spill) {
  *spill = 0;
  if (max_row <= 0 || max_row > 64) return 0;
  const int per_pass = kBS / lane_group(max_row);
  int R = 0;
  for (int b = 0; b < nsys; ++b) {
    const int rows = row0[b + 1] - row0[b], w = cg_team_of(rows, nsys);
    R = std::max(R, ((rows + w - 1) / w + per_pass - 1) / per_pass);
  }
  if (R > max_passes(max_row, value_bytes)) return 0;
  if (needs_spill(R, max_row, value_bytes))
    *spill = 9L * kCgResidentSpill * kBS * kCgResidentMaxWg;
  return R;
}

template <typename T>
bool launch_cg_resident_batch(const CgResidentArgs<T>& A, int passes, int max_row,
                              hipStream_t st) {
  clear(A, st);
  return launch_passes(A, kCgResidentMaxWg, passes, max_row, st);
}
template bool launch_cg_resident_batch<double>(const CgResidentArgs<double>&, int, int,
                                               hipStream_t);
template bool launch_cg_resident_batch<float>(const CgResidentArgs<float>&, int, int, hipStream_t);
template bool launch_cg_resident<double>(const CgResidentArgs<double>&, int, int, hipStream_t);
template bool launch_cg_resident<float>(const CgResidentArgs<float>&, int, int, hipStream_t);

}  // namespace mfemhip
