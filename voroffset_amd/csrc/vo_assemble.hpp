// vo_assemble.hpp -- columns to CSR in one launch.
//
// Every kernel that makes a volume knows, per column, how many endpoints the
// column gets and where they come from.  The CSR needs the exclusive sum of
// the lengths first; here it is taken and used in the same launch, by
// workgroups that pass their sums on to the next one (a chained scan: a
// workgroup publishes its own sum, adds up what the ones before it have
// published, and publishes the total so far).
#pragma once

#include "vo_sweeps.hpp"

namespace vo {

constexpr int kAssembleThreads = 512;
// Columns per thread: one while that gives at most 256 workgroups, else four.
// A hop of the chained scan over 64 workgroups costs microseconds (the sums
// travel between XCDs), so the chain has to stay short, and the copy wants
// many workgroups: 1, 2, 4 and 8 columns take 55, 36, 22 and 19 us for 1024^2
// columns, 21, 17, 20 and 32 us for 544^2, 174, 98, 69 and 73 us for 1896^2
// (scan, report and copy as launches of their own: 32, 23 and 75 us).
constexpr int kAssembleMany = 4;
inline int assemble_items(int64_t n) { return n <= 256 * int64_t(kAssembleThreads) ? 1 : kAssembleMany; }

// What the chained scan keeps between launches: all zero, which the last
// workgroup to finish restores.  The state of a workgroup is its flag in the
// top two bits (1: its own sum, 2: the sum up to and including it) and the sum.
struct AssembleState {
  unsigned* ticket;  // [0] workgroups started, [1] workgroups done
  unsigned long long* sum;
};

// What the last workgroup tells the host (pinned words, null: nothing): the
// total, the status, the tiles given back, and the input check's two words.
struct AssembleReport {
  int64_t* host = nullptr;
  const int* status = nullptr;
  const int* tiles = nullptr;
  const int* check_word = nullptr;
};

constexpr unsigned long long kSumFlag = 1ull << 62;

// Columns [0, n): length(c) endpoints each, written by fill(c, out index) at
// offsets off[0 .. n] where they end at or below `cap`.
template <int kItems, class Length, class Fill>
__device__ void assemble(int64_t n, int64_t* off, int64_t cap, const AssembleState& st, const AssembleReport& rep,
                         Length&& length, Fill&& fill) {
  constexpr int kWaves = kAssembleThreads / kWave;
  __shared__ unsigned s_block;
  __shared__ int64_t s_wave[kWaves];
  __shared__ int64_t s_before;
  const int L = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  // workgroups take their columns in the order they start, so that those
  // before one are running or done and its wait ends
  if (threadIdx.x == 0) s_block = atomicAdd(&st.ticket[0], 1u);
  __syncthreads();
  const unsigned b = s_block;
  // a wavefront's columns are consecutive, 64 at a time
  const int64_t c0 = int64_t(b) * (kAssembleThreads * kItems) + w * (kWave * kItems) + L;
  int64_t len[kItems], at[kItems], carry = 0;
#pragma unroll
  for (int i = 0; i < kItems; ++i) len[i] = c0 + i * kWave < n ? length(c0 + i * kWave) : 0;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    int64_t v = len[i];
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int64_t o = __shfl_up(v, d);
      if (L >= d) v += o;
    }
    at[i] = carry + v - len[i];
    carry += __shfl(v, kWave - 1);
  }
  if (L == 0) s_wave[w] = carry;
  __syncthreads();
  int64_t mine = 0, all = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    mine += i < w ? s_wave[i] : 0;
    all += s_wave[i];
  }
  if (w == 0) {
    auto publish = [&](unsigned long long flag, int64_t sum) {
      if (L == 0)
        __hip_atomic_store(&st.sum[b], flag * kSumFlag | (unsigned long long)sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    int64_t before = 0;
    if (b > 0) {
      publish(1, all);
      // (a word says all there is to know: relaxed, or every look would flush
      // or drop caches.)  64 predecessors at a time, nearest first, up to one that has the
      // whole sum before it
      for (int64_t top = int64_t(b) - 1; top >= 0; top -= kWave) {
        const int64_t p = top - L;
        unsigned long long s = 2 * kSumFlag;
        uint64_t whole;
        for (;;) {
          if (p >= 0) s = __hip_atomic_load(&st.sum[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          whole = ballot(s >= 2 * kSumFlag);
          const uint64_t none = ballot(s < kSumFlag);
          const int first = whole ? __builtin_ctzll(whole) : kWave;
          // all of those up to it have something
          if ((none & (first < kWave ? (uint64_t(2) << first) - 1 : ~uint64_t(0))) == 0) break;
          __builtin_amdgcn_s_sleep(1);
        }
        const int first = whole ? __builtin_ctzll(whole) : kWave;
        int64_t part = L <= first ? int64_t(s & (kSumFlag - 1)) : 0;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) part += __shfl_xor(part, d);
        before += part;
        if (whole) break;
      }
    }
    publish(2, before + all);
    if (L == 0) s_before = before;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t c = c0 + i * kWave, o = s_before + mine + at[i];
    if (c < n) {
      off[c] = o;
      if (o + len[i] <= cap) fill(c, o);
    }
  }
  const int64_t total = s_before + all;
  if (b == gridDim.x - 1 && threadIdx.x == 0) {
    off[n] = total;
    if (rep.host) {
      rep.host[0] = total;
      rep.host[1] = rep.status ? int64_t(uint32_t(*rep.status)) : 0;
      rep.host[2] = rep.tiles ? int64_t(uint32_t(*rep.tiles)) : 0;
      if (rep.check_word)
        rep.host[3] = int64_t(uint64_t(uint32_t(rep.check_word[0])) | uint64_t(uint32_t(rep.check_word[1])) << 32);
      __threadfence_system();
    }
  }
  // the last workgroup to come here leaves everything zero: nobody looks at
  // the sums any more, and none is still on its way: the wavefront that
  // published this workgroup's waits for the store's completion (an agent-scope
  // store completes where every XCD sees it) before it counts itself done.
  // Without the wait the two words are not ordered, and a late sum would stay
  // for the next launch to take for its own.
  if (threadIdx.x == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    s_block = atomicAdd(&st.ticket[1], 1u);
  }
  __syncthreads();
  if (s_block == gridDim.x - 1) {
    for (unsigned i = threadIdx.x; i < gridDim.x; i += kAssembleThreads) st.sum[i] = 0;
    if (threadIdx.x < 2) st.ticket[threadIdx.x] = 0;
  }
}

// The output of a dilation: column c's intervals at start[c], `interleaved`
// (see gather_kernel), to CSR.
template <class T, int kItems>
__global__ __launch_bounds__(kAssembleThreads) void assemble_dilation_kernel(int64_t n, const T* src, const int64_t* start,
                                                                             const int64_t* cnt, int64_t* off, T* dst,
                                                                             int64_t cap, AssembleState st, AssembleReport rep) {
  assemble<kItems>(n, off, cap, st, rep, [&](int64_t c) { return cnt[c]; },
           [&](int64_t c, int64_t o) {
             const int64_t s = start[c], m = cnt[c];
             for (int64_t i = 0; i < m; i += 2) {
               dst[o + i] = src[s + (i >> 1) * kOutStride];
               dst[o + i + 1] = src[s + (i >> 1) * kOutStride + 1];
             }
           });
}

// The complements (ring_column, crop_column): lengths and data in one launch.
template <class T, bool kRing, int kItems>
__global__ __launch_bounds__(kAssembleThreads) void assemble_complement_kernel(ColumnJob<T> g, int64_t n, int64_t* off,
                                                                               int64_t cap, AssembleState st,
                                                                               AssembleReport rep) {
  assemble<kItems>(n, off, cap, st, rep, [&](int64_t c) { return complement_column<T, kRing>(g, c, nullptr); },
           [&](int64_t c, int64_t o) { complement_column<T, kRing>(g, c, g.out + o); });
}

}  // namespace vo
