// fx_resident.hpp -- solver loops that stay on the chip: one launch (of more
// than one workgroup: a cooperative one) runs many iterations, each workgroup owning a contiguous range of
// rows whose vectors live in registers and LDS between the iterations.
//
// Kernel by kernel an iteration pays, for every kernel, a launch gap, the
// re-summing of the previous kernel's partials and a trip of every vector
// through memory: 17 us per CG iteration at 1024 unknowns, 19.6 us at 512^2.
// Here only the vector that neighbouring workgroups gather from (CG: p)
// passes through memory, and a reduction is an exchange of one 64-byte slot
// per workgroup.
//
// What workgroups exchange is written and read with relaxed agent-scope
// atomics, which bypass the XCDs' own L2s, so no cache is flushed or
// invalidated (an agent-scope fence writes back a whole L2).  A writer waits
// for its stores (vmcnt) before it stores the flag or slot that announces
// them; a reader looks at the data only after it has seen that.
//
// A launch that waits is cooperative: every workgroup is on the chip, so each
// wait ends.  Waits are bounded all the same; one that runs out raises *fail and
// every workgroup leaves.  The host then starts over kernel by kernel, from
// the caller's x (the refinement: from its last outer iterate).  A launch that
// is refused goes on kernel by kernel from where the last one ended.
//
// Environment, for tests: FASPXX_FX_NORESIDENT=1 none of this;
// FASPXX_FX_RESIDENT_FAIL=1 launches of one iteration that find *fail raised,
// as by a wait that gave up; FASPXX_FX_RESIDENT_LAUNCHES=N launches of one loop before they are refused.
#pragma once

#include <cstdlib>
#include <utility>

#include "fx_internal.hpp"

namespace fx {

constexpr int kResThreads = 1024;
constexpr int kResWaves = kResThreads / 64;
constexpr uint32_t kResMaxWgs = 256;  // 8 groups of 32 slots
constexpr int kResBufs = 8;           // slot buffers in rotation
constexpr int kResSlot = 8;           // doubles per slot: one 64-byte line
constexpr unsigned long long kResEmpty = ~0ull;  // a NaN that is never published
constexpr int kResSpins = 1 << 21;    // polls before a wait gives up (seconds)

struct ResComm {
  unsigned long long* slots;  // [kResBufs][kResMaxWgs][kResSlot]
  unsigned long long* gsum;   // [kResBufs][8][kResSlot]
  unsigned long long* flags;  // [kResMaxWgs]: iterations whose export is visible
  unsigned long long* fail;
};
constexpr size_t kResSlotWords = (size_t)kResBufs * kResMaxWgs * kResSlot;
constexpr size_t kResGsumWords = (size_t)kResBufs * 8 * kResSlot;
constexpr size_t kResCommWords = kResSlotWords + kResGsumWords + kResMaxWgs + 8;
inline ResComm res_comm(void* mem) {
  unsigned long long* w = (unsigned long long*)mem;
  return {w, w + kResSlotWords, w + kResSlotWords + kResGsumWords,
          w + kResSlotWords + kResGsumWords + kResMaxWgs};
}

// Empty slots and zero flags, before each launch; *fail as given.
static __global__ __launch_bounds__(kThreads) void k_res_clear(unsigned long long* w,
                                                               unsigned long long fail) {
  for (size_t i = blockIdx.x * kThreads + threadIdx.x; i < kResCommWords;
       i += (size_t)gridDim.x * kThreads)
    w[i] = i < kResSlotWords + kResGsumWords                ? kResEmpty
           : i == kResSlotWords + kResGsumWords + kResMaxWgs ? fail
                                                             : 0ull;
}

__device__ __forceinline__ void res_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long res_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_store(double* p, double v) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p),
                     (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double res_load(const double* p) {
  return __longlong_as_double((long long)__hip_atomic_load(
      reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void res_store(float* p, float v) {
  __hip_atomic_store(reinterpret_cast<unsigned int*>(p), __float_as_uint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float res_load(const float* p) {
  return __uint_as_float(__hip_atomic_load(reinterpret_cast<const unsigned int*>(p),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
// Every store of this wave has reached the point where all XCDs see it.
__device__ __forceinline__ void res_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sums and maxima over 16, 8 or 64 lanes by DPP row permutations (a lane
// shuffle through LDS costs several times as much latency per step).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <bool MAX>
__device__ __forceinline__ double res_join(double a, double b) {
  return MAX ? fmax(a, b) : a + b;
}
template <bool MAX>
__device__ __forceinline__ double res_lanes8(double v) {  // in each aligned group of 8 lanes
  v = res_join<MAX>(v, dpp_move<0xB1>(v));   // quad_perm [1,0,3,2]
  v = res_join<MAX>(v, dpp_move<0x4E>(v));   // quad_perm [2,3,0,1]
  return res_join<MAX>(v, dpp_move<0x141>(v));  // row_half_mirror
}
template <bool MAX>
__device__ __forceinline__ double res_lanes16(double v) {  // in each row of 16 lanes
  v = res_lanes8<MAX>(v);
  return res_join<MAX>(v, dpp_move<0x140>(v));  // row_mirror
}
__device__ __forceinline__ double res_lane(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <bool MAX>
__device__ __forceinline__ double res_wave(double v) {
  v = res_lanes16<MAX>(v);
  return res_join<MAX>(res_join<MAX>(res_lane(v, 0), res_lane(v, 16)),
                       res_join<MAX>(res_lane(v, 32), res_lane(v, 48)));
}

// f(0), f(1), .. f(N - 1) with the index a constant expression, so that arrays
// indexed by it are registers from the first optimisation on (indexed in a
// loop they were turned into addresses, and those into LDS or scratch).
template <int... I, class F>
__device__ __forceinline__ void res_each(std::integer_sequence<int, I...>, const F& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void res_for(const F& f) {
  res_each(std::make_integer_sequence<int, N>{}, f);
}

// v as a value of its own: a choice between two array elements that pass
// through here stays a choice of registers, not of addresses.
__device__ __forceinline__ double res_value(double v) {
  asm("" : "+v"(v));
  return v;
}

// LDS of the exchanges.
struct ResShared {
  double red[kResSlot][kResWaves];
  double tot[kResSlot];
  int bad;
};

// The K per-thread values v summed (slot k: maximum when bit k of MaxMask is
// set) over every thread of every workgroup; every thread gets the same
// bits, in v.  post(tot) is run by the first wave (all its lanes hold the
// same sums) before the others go on: scalars formed there and left in LDS
// cost one wave's latency and no further barrier.  Call t of a launch uses slot buffer t mod 8 and empties the
// one that call t + 4 will use: by then every workgroup has left call t - 4,
// which used it last.  Up to 32 workgroups each reads all slots; more go in
// groups of 32, the group's first workgroup publishing its sum (one more
// hop, but 256 workgroups polling 256 lines took longer).  False when a wait
// gave up.
// DRAIN: what this workgroup exported before the call is visible to every
// workgroup that has left it.
template <int K, unsigned MaxMask, bool DRAIN = false, class Post>
__device__ __forceinline__ bool res_allreduce(double (&v)[K], const ResComm& cm, uint32_t t,
                                              ResShared& sh, const Post& post) {
  static_assert(K <= kResSlot, "one line per slot");
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const uint32_t G = gridDim.x, g = blockIdx.x;
  res_for<K>([&](auto k) {
    const double s = res_wave<((MaxMask >> k) & 1u) != 0>(v[k]);
    if (lane == 0) sh.red[k][wid] = s;
  });
  if constexpr (DRAIN) res_drain();
  __syncthreads();
  if (wid == 0) {
    double tot[K];
    res_for<K>([&](auto k) {
      tot[k] = res_lanes16<((MaxMask >> k) & 1u) != 0>(sh.red[k][lane & 15]);
    });
    bool ok = true;
    if (G > 1) {
      unsigned long long* cur = cm.slots + (size_t)(t % kResBufs) * kResMaxWgs * kResSlot;
      unsigned long long* old = cm.slots + (size_t)((t + 4) % kResBufs) * kResMaxWgs * kResSlot;
      unsigned long long* gcur = cm.gsum + (size_t)(t % kResBufs) * 8 * kResSlot;
      unsigned long long* gold = cm.gsum + (size_t)((t + 4) % kResBufs) * 8 * kResSlot;
      auto publish = [&](unsigned long long* at, unsigned long long* stale, const double (&val)[K]) {
        double mine = val[0];
        res_for<K>([&](auto k) {
          const double vk = res_value(val[k]);
          if (lane == k) mine = vk;
        });
        if (lane < K) {
          const unsigned long long bits =
              mine != mine ? 0x7FF8000000000000ull : (unsigned long long)__double_as_longlong(mine);
          res_store(at + lane, bits);
          res_store(stale + lane, kResEmpty);
        }
      };
      // waits until the word this lane reads is there (in every active lane)
      auto poll = [&](const unsigned long long* p, bool active) -> double {
        unsigned long long x = kResEmpty;
        for (int spin = 0;; ++spin) {
          if (active) x = res_load(p);
          if (__all(!active || x != kResEmpty)) break;
          if (spin > kResSpins || ((spin & 1023) == 1023 && res_load(cm.fail) != 0)) {
            ok = false;
            break;
          }
        }
        return __longlong_as_double((long long)x);
      };
      // slot words of 32 workgroups from w0: slots 2 i (lanes 0..31) and
      // 2 i + 1 (lanes 32..63) per step
      auto gather32 = [&](uint32_t w0) {
        const uint32_t w = w0 + (lane & 31);
        constexpr int I = (K + 1) / 2;
        unsigned long long x[I];
        bool act[I];
        res_for<I>([&](auto i) { act[i] = w < G && 2 * i + (lane >> 5) < K; });
        for (int spin = 0;; ++spin) {
          bool have = true;
          res_for<I>([&](auto i) {
            x[i] = act[i] ? res_load(cur + (size_t)w * kResSlot + 2 * i + (lane >> 5)) : 0ull;
          });
          res_for<I>([&](auto i) { have = have && (!act[i] || x[i] != kResEmpty); });
          if (__all(have)) break;
          if (spin > kResSpins || ((spin & 1023) == 1023 && res_load(cm.fail) != 0)) {
            ok = false;
            break;
          }
        }
        res_for<K>([&](auto k) {
          constexpr bool mx = ((MaxMask >> k) & 1u) != 0;
          const bool on = act[k / 2] && (lane >> 5) == (k & 1);
          const double d = on ? __longlong_as_double((long long)x[k / 2]) : mx ? -INFINITY : 0.0;
          const double s = res_lanes16<mx>(d);
          tot[k] = res_join<mx>(res_lane(s, 32 * (k & 1)), res_lane(s, 32 * (k & 1) + 16));
        });
      };
      res_drain();  // the emptied slots of earlier calls are empty for everyone
      publish(cur + (size_t)g * kResSlot, old + (size_t)g * kResSlot, tot);
      if (G <= 32) {
        gather32(0);
      } else {
        const uint32_t ng = (G + 31) / 32;
        if ((g & 31u) == 0) {
          gather32(g);
          if (ok) publish(gcur + (g >> 5) * kResSlot, gold + (g >> 5) * kResSlot, tot);
        }
        const uint32_t gg = lane & 7;
        const int k = lane >> 3;
        const bool act = gg < ng && k < K;
        const double d0 = poll(gcur + gg * kResSlot + k, act);
        const bool mx = (MaxMask >> k) & 1u;
        const double s0 = res_lanes8<false>(act && !mx ? d0 : 0.0);
        const double s1 = MaxMask ? res_lanes8<true>(act && mx ? d0 : -INFINITY) : 0.0;
        res_for<K>([&](auto kk) {
          tot[kk] = ((MaxMask >> kk) & 1u) ? res_lane(s1, 8 * kk) : res_lane(s0, 8 * kk);
        });
      }
    }
    if (ok) post(tot);
    if (lane == 0) {
      res_for<K>([&](auto k) { sh.tot[k] = tot[k]; });
      sh.bad = ok ? 0 : 1;
      if (!ok) res_store(cm.fail, 1ull);
    }
  }
  __syncthreads();
  res_for<K>([&](auto k) { v[k] = sh.tot[k]; });
  return sh.bad == 0;
}

// Announce this workgroup's exported entries of step `epoch` and wait for
// those of the workgroups lo .. hi (its gathers' range).  Every thread
// calls it after its stores.
__device__ __forceinline__ bool res_exchange(const ResComm& cm, unsigned long long epoch,
                                             uint32_t lo, uint32_t hi, ResShared& sh) {
  if (gridDim.x == 1) {
    __syncthreads();
    return true;
  }
  res_drain();
  __syncthreads();
  if (threadIdx.x == 0) {
    sh.bad = 0;
    res_store(cm.flags + blockIdx.x, epoch);
  }
  __syncthreads();
  const uint32_t w = lo + threadIdx.x;
  if (w <= hi && w != blockIdx.x) {
    for (int spin = 0; res_load(cm.flags + w) < epoch; ++spin) {
      if (spin > kResSpins || ((spin & 1023) == 1023 && res_load(cm.fail) != 0)) {
        sh.bad = 1;
        res_store(cm.fail, 1ull);
        break;
      }
    }
  }
  asm volatile("" ::: "memory");  // the gathers stay behind the waits
  __syncthreads();
  return sh.bad == 0;
}

// ---- the matrix -----------------------------------------------------------
struct ResMat {
  const uint32_t* __restrict__ rp;
  const uint32_t* __restrict__ ci;   // columns, when pid is null
  const uint8_t* __restrict__ pid;   // row patterns
  const int32_t* __restrict__ pdict; // offsets, plen per pattern
  const void* __restrict__ va;       // values in CSR order
  const int32_t* __restrict__ vdict; // row values: offsets, vstride per pattern
  const void* __restrict__ vval;     // row values
  uint32_t n, plen, npat, vstride;
};

// How a workgroup holds its rows: RM_REG entries and their places in
// registers (rows of at most 8 entries, at most 2 rows per thread); RM_MEM
// values re-read from memory each time (they stay in L2 or the Infinity
// Cache); RM_VAL row values (at most 8 per row), from a dictionary in LDS.
enum { RM_REG = 0, RM_MEM = 1, RM_VAL = 2 };

template <class MT, int R, int MM>
struct ResRows {
  static constexpr uint32_t kRows = R * kResThreads;  // rows of a workgroup
  static constexpr int kPack = (R + 3) / 4;           // bytes of R rows, four to a word
  struct Lds {
    alignas(16) int32_t dict[kPatDict];
    alignas(16) MT val[MM == RM_VAL ? kPatDict : 1];
    uint32_t lo, hi;
  };
  MT a[MM == RM_REG ? R : 1][8];
  int32_t at[MM == RM_REG ? R : 1][8];  // LDS place, or ~column outside the workgroup's rows
  uint32_t start[MM == RM_MEM ? R : 1];
  uint32_t len4[kPack], pid4[kPack];  // row lengths and patterns

  __device__ __forceinline__ uint32_t len(int q) const { return (len4[q / 4] >> (8 * (q % 4))) & 255u; }
  __device__ __forceinline__ uint32_t pid(int q) const { return (pid4[q / 4] >> (8 * (q % 4))) & 255u; }

  // The places of the entries as values of this moment: addresses formed from
  // them are not kept from one product to the next (two products per
  // iteration kept more of them than there are registers).
  __device__ __forceinline__ void fresh() {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if constexpr (MM == RM_REG) {
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(at[q][j]));
      }
      if constexpr (MM == RM_MEM) asm volatile("" : "+v"(start[q]));
    }
#pragma unroll
    for (int w = 0; w < kPack; ++w) asm volatile("" : "+v"(len4[w]), "+v"(pid4[w]));
  }

  // lo .. hi: the workgroups whose rows this one's rows gather from.
  __device__ __forceinline__ void load(const ResMat& A, Lds& l, uint32_t& lo, uint32_t& hi) {
    const uint32_t tid = threadIdx.x, base = blockIdx.x * kRows;
    if (A.pid) {
      const uint32_t nd = MM == RM_VAL ? A.npat * A.vstride : A.npat * A.plen;
      const int32_t* d = MM == RM_VAL ? A.vdict : A.pdict;
      for (uint32_t i = tid; i < nd; i += kResThreads) {
        l.dict[i] = d[i];
        if constexpr (MM == RM_VAL) l.val[i] = ((const MT*)A.vval)[i];
      }
    }
    if (tid == 0) {
      l.lo = 0xffffffffu;
      l.hi = 0;
    }
    __syncthreads();
    uint32_t cmin = 0xffffffffu, cmax = 0;
#pragma unroll
    for (int w = 0; w < kPack; ++w) len4[w] = pid4[w] = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t i = base + q * kResThreads + tid;
      const bool has = i < A.n;
      uint32_t s = 0, n = 0, p = 0;
      if (has) {
        s = A.rp[i];
        n = A.rp[i + 1] - s;
        if (A.pid) p = A.pid[i];
      }
      len4[q / 4] |= n << (8 * (q % 4));
      pid4[q / 4] |= p << (8 * (q % 4));
      if constexpr (MM == RM_MEM) start[q] = s;
      const uint32_t stride = MM == RM_VAL ? A.vstride : A.plen;
      auto col = [&](uint32_t j) -> uint32_t {
        return A.pid ? i + (uint32_t)l.dict[p * stride + j] : A.ci[s + j];
      };
      if constexpr (MM == RM_REG) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a[q][j] = (MT)0;
          at[q][j] = 0;
          if ((uint32_t)j < n) {
            const uint32_t c = col(j);
            a[q][j] = ((const MT*)A.va)[s + j];
            at[q][j] = c - base < kRows ? (int32_t)(c - base) : ~(int32_t)c;
            cmin = min(cmin, c);
            cmax = max(cmax, c);
          }
        }
      } else {
        for (uint32_t j = 0; j < n; ++j) {
          const uint32_t c = col(j);
          cmin = min(cmin, c);
          cmax = max(cmax, c);
        }
      }
    }
    if (cmin <= cmax) {
      atomicMin(&l.lo, cmin);
      atomicMax(&l.hi, cmax);
    }
    __syncthreads();
    lo = min(l.lo, base) / kRows;
    hi = max(l.hi, base) / kRows;
  }

  // RM_REG: f(place, column) for each of the thread's entries outside the
  // workgroup's rows.
  template <class F>
  __device__ __forceinline__ void outside(const F& f) const {
    static_assert(MM == RM_REG, "places are in registers");
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (at[q][j] < 0) f(8 * q + j, (uint32_t)~at[q][j]);
  }

  // RM_REG: the product below with the outside entries given in vo, or with
  // none (one workgroup).
  template <class VT, class At>
  __device__ __forceinline__ void product_at(double (&out)[R], const At& entry) const {
    static_assert(MM == RM_REG, "places are in registers");
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t n = len(q);
      VT x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = entry(8 * q + j, at[q][j]);
      double t = 0.0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if ((uint32_t)j < n)
          t = j == 0 ? (double)a[q][j] * (double)x[j] : fma((double)a[q][j], (double)x[j], t);
      out[q] = t;
    }
  }
  template <class VT>
  __device__ __forceinline__ void product_of(const VT* vl, const VT (&vo)[8 * R],
                                             double (&out)[R]) const {
    product_at<VT>(out, [&](int e, int32_t d) {
      const VT in = vl[d < 0 ? 0 : d];
      return d < 0 ? vo[e] : in;
    });
  }
  template <class VT>
  __device__ __forceinline__ void product_within(const VT* vl, double (&out)[R]) const {
    product_at<VT>(out, [&](int, int32_t d) { return vl[d]; });
  }

  // (A v)_i of the thread's q-th row, left to right as in the SpMV kernels
  // (w = v0 * x0, then fma).  vl: the workgroup's own entries in LDS; vg: the
  // exported vector.  Two rows at a time: their outside entries are all asked
  // for before the first sum, and no more than two rows' are held in registers.
  template <class VT>
  __device__ __forceinline__ void product(const ResMat& A, const Lds& l, const VT* vl,
                                          const VT* vg, double (&out)[R]) const {
    constexpr int PQ = R < 2 ? 1 : 2;
    const uint32_t tid = threadIdx.x, base = blockIdx.x * kRows;
    auto term = [&](double& t, bool first, MT av, VT xv) {
      t = first ? (double)av * (double)xv : fma((double)av, (double)xv, t);
    };
    auto fetch = [&](uint32_t c) -> VT {
      const uint32_t d = c - base;
      return d < kRows ? vl[d] : res_load(vg + c);
    };
#pragma unroll
    for (int q0 = 0; q0 < R; q0 += PQ) {
      VT x[PQ][8];
      if constexpr (MM == RM_MEM) {
        // the rows' first 8 entries
#pragma unroll
        for (int u = 0; u < PQ; ++u) {
          const int q = q0 + u;
          const uint32_t i = base + q * kResThreads + tid, n = len(q);
          const uint32_t* cj = A.ci + start[q];
          const int32_t* pd = l.dict + pid(q) * A.plen;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if ((uint32_t)j < n) x[u][j] = fetch(A.pid ? i + (uint32_t)pd[j] : cj[j]);
        }
      } else {
#pragma unroll
        for (int u = 0; u < PQ; ++u) {
          const int q = q0 + u;
          if constexpr (MM == RM_REG) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const int32_t d = at[q][j];
              x[u][j] = d >= 0 ? vl[d] : res_load(vg + ~d);
            }
          } else {
            const uint32_t i = base + q * kResThreads + tid, n = len(q);
            const int4* pd = reinterpret_cast<const int4*>(l.dict + pid(q) * 8);
            const int4 o0 = pd[0], o1 = pd[1];
            const int off[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if ((uint32_t)j < A.plen) x[u][j] = fetch(n ? i + (uint32_t)off[j] : base);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < PQ; ++u) {
        const int q = q0 + u;
        const uint32_t n = len(q);
        double t = 0.0;
        if constexpr (MM == RM_MEM) {
          const uint32_t i = base + q * kResThreads + tid;
          const MT* va = (const MT*)A.va + start[q];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if ((uint32_t)j < n) term(t, j == 0, va[j], x[u][j]);
          for (uint32_t j = 8; j < n; ++j)
            term(t, false, va[j],
                 fetch(A.pid ? i + (uint32_t)l.dict[pid(q) * A.plen + j] : A.ci[start[q] + j]));
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if ((uint32_t)j < n)
              term(t, j == 0, MM == RM_REG ? a[MM == RM_REG ? q : 0][j] : l.val[pid(q) * 8 + j], x[u][j]);
        }
        out[q] = t;
      }
      if constexpr (R > PQ) __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// ---- host side --------------------------------------------------------------
// Rows per thread and workgroups for n rows, or rows = 0 when the loop does
// not fit the chip.  One workgroup up to 2048 rows: it needs no exchange at
// all (a CG iteration at 2025 unknowns 5.9 us; at 4096 in one workgroup
// 10.6 us, in four 6.6).  Beyond, 1024 rows per workgroup while there are
// CUs for it: an exchange among 256 workgroups costs about 3 us whatever
// they hold, so fewer, longer ones gain nothing.
#ifndef FX_RES_ALONE
#define FX_RES_ALONE 2048
#endif
constexpr uint32_t kResAlone = FX_RES_ALONE;
struct ResShape {
  uint32_t rows = 0, wgs = 0;
};
inline ResShape res_shape(uint32_t n, int cus) {
  if (n == 0) return {};
  const uint32_t t = kResThreads;
  if (n <= kResAlone) return {n <= t ? 1u : 2u, 1u};
  const uint32_t most = (uint32_t)cus < kResMaxWgs ? (uint32_t)cus : kResMaxWgs;
  for (uint32_t r : {1u, 2u, 4u, 8u}) {
    const uint32_t g = (n + r * kResThreads - 1) / (r * kResThreads);
    if (g <= most) return {r, g};
  }
  return {};
}

template <class MT>
inline ResMat res_mat(const fx_csr_s* A) {
  const void* va = sizeof(MT) == 8 ? (const void*)A->va : (const void*)A->va32;
  const void* vv = sizeof(MT) == 8 ? (const void*)A->vd64 : (const void*)A->vd32;
  return {A->rp, A->ci, A->pid, A->pdict, va, A->vdict, vv, A->nrow, A->plen, A->npat, A->vstride};
}
template <class MT>
inline int res_mode(const fx_csr_s* A, uint32_t rows) {
  if (rows == 1 && A->max_row <= 8) return RM_REG;
  if (rows > 1 && has_row_values<MT>(A) && A->vstride == 8) return RM_VAL;
  if (rows == 2 && A->max_row <= 8) return RM_REG;
  return RM_MEM;
}

// Whether a matrix suits a resident loop: banded forms (row patterns or
// 16-bit column deltas; scattered columns would all be gathered past L2), and
// rows that are faster there than kernel by kernel.  Rows held in registers
// or as row values (at most 8 entries) always are.  Where values are re-read
// from memory, a row's entries past the eighth are one dependent gather each,
// and every entry outside the workgroup's rows is one past the L2; so the
// lines lie by length and by how far the row reaches (near: no offset leaves
// a workgroup's rows altogether).  us per iteration, resident against kernel
// by kernel; k: entries of a row:
//   one workgroup, 900 rows: CG k 17 13.1 / 17.2, k 25 20.9 / 17.4
//   one row per thread: CG k 11 13.9 .. 26.8 / 18.2 .. 26.6,
//     k 13 14.8 .. 36.8 / 18.2 .. 28.1, k 27 (64^3) 182 / 35
//   two: CG k 11 near 24.5 / 26.6, far 33.3 / 28.5; k 9 no patterns 24.9 / 27.1
//   four: CG k 5 22.8 / 35.6, k 7 far 30.0 / 31.2, k 9 near 39.0 / 41.0, far
//     38.0 / 35.1; k 9 with row values for the kernels 34.4 / 31.8; k 7 no
//     patterns 35.2 / 32.2 at 551368 rows and 38.9 / 41.3 at 1000000
//     (BiCGStab 61.5 / 61.4, 70.8 / 81.9)
//   four, refinement: k 5 10.9 / 17.9, k 9 near 18.8 / 20.6, k 7 far 18.1 / 15.5
//   eight (this form spills 165 registers): CG k 5 near 41.1 / 40.5 at 1210000
//     rows, 42.1 / 43.5 at 1345600, 46.8 / 59.1 at 2096704; no patterns 51.2 /
//     39.1 .. 53.9 / 53.7 to 1690000; k 7 far 58.8 / 43.0 .. 67.6 / 64.7;
//     k 9 66.7 / 39.1
// The refinement's loop is left out with eight rows per thread: with row
// values 19.1 / 17.7 at 102^3, 20.9 / 20.2 at 115^3, 24.1 / 24.1 at 128^3; with
// values from memory 41 / 28.
enum ResLoop { RES_CG, RES_BICGSTAB, RES_IR };
template <class MT>
inline bool res_suits(const fx_csr_s* A, ResLoop loop, int cus) {
  if (!A || !A->has_values || !(A->pid || A->cd) || A->nrow != A->mcol) return false;
  const ResShape rs = res_shape(A->nrow, cus);
  if (rs.rows == 0 || (rs.rows == 8 && loop == RES_IR)) return false;
  if (res_mode<MT>(A, rs.rows) != RM_MEM) return true;
  const uint32_t k = A->max_row;
  const bool near = rs.wgs == 1 || (A->pid && A->reach <= rs.rows * kResThreads);
  const uint32_t near9 = near && !A->vconst ? 9 : 8;
  if (rs.rows == 1) return k <= (rs.wgs == 1 ? 17u : 11u);
  if (rs.rows == 2) return k <= (near ? 11u : 9u);
  if (rs.rows == 4) {
    if (k <= 5) return true;
    if (loop == RES_IR) return near && k <= near9;
    if (A->pid) return k <= near9;
    return k <= 8 && (loop == RES_BICGSTAB || A->nrow > 3u << 18);
  }
  return near && k <= 5 && A->nrow > 5u << 18;
}

// make(rows, mode) for the instantiations that res_shape and res_mode give.
template <class F>
inline const void* res_pick(uint32_t rows, int mode, const F& make) {
  using std::integral_constant;
  const void* k = nullptr;
  auto pick = [&](auto r) {
    constexpr int R = decltype(r)::value;
    if constexpr (R <= 2)
      if (mode == RM_REG) k = make(r, integral_constant<int, RM_REG>{});
    if constexpr (R >= 2)
      if (mode == RM_VAL) k = make(r, integral_constant<int, RM_VAL>{});
    if (mode == RM_MEM) k = make(r, integral_constant<int, RM_MEM>{});
  };
  if (rows == 1) pick(integral_constant<int, 1>{});
  if (rows == 2) pick(integral_constant<int, 2>{});
  if (rows == 4) pick(integral_constant<int, 4>{});
  if (rows == 8) pick(integral_constant<int, 8>{});
  return k;
}

inline bool res_fail_forced() {
  const char* e = std::getenv("FASPXX_FX_RESIDENT_FAIL");
  return e && e[0] == '1';
}

// Iterations of one launch (the host looks at the state in between).
constexpr uint32_t kResLaunchIters = 2048;
inline uint32_t res_launch_iters(uint32_t wgs) {
  return wgs > 1 && res_fail_forced() ? 1 : kResLaunchIters;
}

// One cooperative launch of `kernel` on a comm block that is cleared first
// (one workgroup waits for nobody: an ordinary launch, which those of other
// streams may overlap, and nothing to clear; the runtime takes cooperative
// launches one after the other);
// 1 when it cannot be had (the device cannot hold all its workgroups at
// once, or another process on the card holds its cooperative queue: the
// caller then goes kernel by kernel), else 0 or an error.  before: the
// launches of this loop so far.
inline int res_launch(fx_ctx ctx, const void* kernel, uint32_t wgs, void* comm, void** args,
                      uint64_t before) {
  const char* e = std::getenv("FASPXX_FX_RESIDENT_LAUNCHES");
  if (e && before >= (uint64_t)std::atoll(e)) return 1;
  if (wgs == 1) {
    FX_HIP(hipLaunchKernel(kernel, dim3(1), dim3(kResThreads), args, 0, ctx->stream));
    return 0;
  }
  int per_cu = 0, coop = 0;
  FX_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device));
  FX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kResThreads, 0));
  if (!coop || (uint64_t)per_cu * (uint64_t)ctx->sms < wgs) return 1;
  hipLaunchKernelGGL(k_res_clear, dim3(16), dim3(kThreads), 0, ctx->stream,
                     (unsigned long long*)comm, res_fail_forced() ? 1ull : 0ull);
  FX_HIP(hipGetLastError());
  if (hipLaunchCooperativeKernel(kernel, dim3(wgs), dim3(kResThreads), args, 0, ctx->stream) !=
      hipSuccess) {
    (void)hipGetLastError();  // not an error of the solve
    return 1;
  }
  return 0;
}

// What became of a launch.  A loop that stopped is whole even where a wait
// gave up: workgroup 0 stops on a reduction that every workgroup entered, so
// the one that gave up waiting for its result had done all the work before it.
enum ResOutcome {
  RES_RAN,      // the state tells whether the loop goes on
  RES_REFUSED,  // no launch: vectors and state are as they were
  RES_LOST      // a wait gave up on the way: start over
};
inline ResOutcome res_outcome(bool running, unsigned long long fail) {
  return running && fail != 0 ? RES_LOST : RES_RAN;
}

inline bool resident_disabled() {
  const char* e = std::getenv("FASPXX_FX_NORESIDENT");
  return e && e[0] == '1';
}

}  // namespace fx
