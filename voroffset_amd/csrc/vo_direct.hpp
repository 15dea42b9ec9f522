// vo_direct.hpp -- dilation in one pass over the input.
//
// The result at column (x, y) is the union, over the source columns at offset
// (dx, dy) with dx^2 + dy^2 <= R^2, of their segments grown by
// H = sqrt(R^2 - dx^2 - dy^2).  The two sweeps (vo_sweeps.hpp) reach it through
// an intermediate of nearest-line pieces; here it is evaluated as it stands,
// and nearly all of the disk is left out because it lies inside what the
// nearer columns already gave: a segment whose growth stays inside the union
// of every output column it reaches changes nothing.
//
// Both forms unite the same closed intervals up to pieces that another of
// their pieces contains, and an interval's ends are the same a - H and b + H
// of the same table, rounded monotonically, so the results are equal bit for
// bit.
#pragma once

#include <cfloat>
#include <type_traits>

#include "vo_sweeps.hpp"

namespace vo {

constexpr int kSide = 8;               // an output tile, and a block of source columns, is kSide x kSide
// Largest radius whose H table is staged in LDS (2.3 KB): one wavefront per
// workgroup lets the tiles of a launch end one by one, and a larger table of
// its own costs waves.  Against four wavefronts sharing tables up to R = 31:
// 1024^2 R = 16 402 -> 392 us (FP64 510 -> 404), R = 64 390 -> 354, 1896^2
// closing at R = 48 1577 -> 1455, 1000^2 at R = 4 1640 -> 1523.
constexpr int kDirectLdsTableMax = 9;
constexpr int kDirectMaxR = 255;       // largest radius this form takes
constexpr int kDirectMaxList = 512;    // longest list it grows to; the sweeps take volumes that need more
// Sizes that go with the LDS entries of a lane's list: segments and columns
// that may wait, and the segments worth a drain between blocks.  With a short
// list (large radii) the waves that fit count, and early drains keep the cover
// fresh; with a long one (small radii) fewer drains do.
template <int kList>
struct DirectShape {
  static constexpr bool kSmallR = kList > 4;
  static constexpr int kRecs = kSmallR ? 192 : 160, kPend = kSmallR ? 128 : 96, kDrainAt = kSmallR ? 64 : 24;
  static_assert(kDrainAt + 2 * kWave <= kRecs, "a block's first and last segments fit beside what waits");
};
constexpr int kHeld = 2;               // runs a lane may hold back before they meet its list
constexpr int kAhead = 4;              // segments whose growths are read together
constexpr int kCommon = 6;             // intervals of the tile's common cover the segment test looks at

// The H table of this form: entry [adx * W + ady] for column offsets up to
// rint + kSide - 1 (what a block partly in reach asks for), NaN out of reach.
__host__ __device__ constexpr int direct_htab_width(int rint) { return rint + kSide; }

// First and last segment of a column (or their envelopes over a block), empty
// as (+inf, -inf).
template <class T>
struct alignas(4 * sizeof(T)) Ends {
  T lo0, hi0, lo1, hi1;
};

// A column's start and segment count in one word; counts past 65534 read
// 65535 (the offsets have them).
constexpr int kCountMany = 65535;
__host__ __device__ inline uint64_t column_at(int64_t start, int64_t count) {
  return uint64_t(start) | uint64_t(count < kCountMany ? count : kCountMany) << 48;
}

template <class T>
struct SummaryArgs {
  int nx, ny, nbx, nby;  // grid, and its blocks
  const int64_t* off;
  const T* z;
  Ends<T>* col;  // per column, block by block: block * 64 + (y % 8) * 8 + x % 8
  uint64_t* at;  // where the column's endpoints start (low 48 bits) and its segments (column_at), same order
  Ends<T>* blk;  // per block: min lo0, max hi0, min lo1, max hi1
  int* bcnt;     // per block: most segments in a column
  // the input check of the operation (null: none), with the rules and words
  // of check_input_kernel
  int* check_word;
  int check_range;
  double check_lo, check_hi;
};

// Eight wavefronts take 64 x 8 columns (a row of 64 each): every lane notes
// its column's first and last segment, and the workgroup the envelopes of its
// eight blocks.  The endpoints in between are read only to be checked.
template <class T>
__device__ void summary_rows(const SummaryArgs<T>& g, int gx, int gy, Ends<T>* s_row, int* s_cnt) {
  const int L = threadIdx.x & (kWave - 1), row = threadIdx.x / kWave;
  const int x = gx * kWave + L, y = gy * kSide + row;
  const bool has = x < g.nx && y < g.ny;
  const int64_t c = int64_t(y) * g.nx + x;
  const int64_t s = has ? g.off[c] : 0, e = has ? g.off[c + 1] : 0;
  const int64_t pairs = e > s ? (e - s) / 2 : 0;
  const int n = int(pairs < INT32_MAX ? pairs : INT32_MAX);
  Ends<T> r{T(INFINITY), T(-INFINITY), T(INFINITY), T(-INFINITY)};
  if (n > 0) {
    r.lo0 = g.z[s];
    r.hi0 = g.z[s + 1];
    r.lo1 = g.z[s + 2 * int64_t(n) - 2];
    r.hi1 = g.z[s + 2 * int64_t(n) - 1];
  }
  if (g.check_word) {
    int bad = (has && (e < s || ((e - s) & 1))) ? kInputMalformed : 0;
    const int last = min(g.nx - gx * kWave, kWave) - 1;
    const int64_t S = __shfl(s, 0), E = __shfl(e, last < 0 ? 0 : last);
    if (y < g.ny && ballot(bad != 0) == 0 && E > S)
      bad |= check_range(g.z, S, E, s, e, has, g.check_range, g.check_lo, g.check_hi);
    if (bad) {
      atomicOr(g.check_word, bad);
      atomicMin(g.check_word + 1, 0);
    }
  }
  const int b = gx * kSide + L / kSide;  // block column
  const bool inb = b < g.nbx && gy < g.nby;
  if (inb) {
    const int64_t at = (int64_t(gy) * g.nbx + b) * kWave + row * kSide + L % kSide;
    g.col[at] = r;
    g.at[at] = column_at(s, n);
  }
  // envelopes: over the 8 lanes of a block's row, then over the 8 rows
  int m = n;
#pragma unroll
  for (int d = 1; d < kSide; d <<= 1) {
    r.lo0 = min(r.lo0, __shfl_xor(r.lo0, d));
    r.hi0 = max(r.hi0, __shfl_xor(r.hi0, d));
    r.lo1 = min(r.lo1, __shfl_xor(r.lo1, d));
    r.hi1 = max(r.hi1, __shfl_xor(r.hi1, d));
    m = max(m, __shfl_xor(m, d));
  }
  if (L % kSide == 0) {
    s_row[row * kSide + L / kSide] = r;
    s_cnt[row * kSide + L / kSide] = m;
  }
  __syncthreads();
  if (threadIdx.x < kSide) {
    const int k = threadIdx.x, bx = gx * kSide + k;
    Ends<T> v = s_row[k];
    int mm = s_cnt[k];
    for (int i = 1; i < kSide; ++i) {
      const Ends<T> o = s_row[i * kSide + k];
      v.lo0 = min(v.lo0, o.lo0);
      v.hi0 = max(v.hi0, o.hi0);
      v.lo1 = min(v.lo1, o.lo1);
      v.hi1 = max(v.hi1, o.hi1);
      mm = max(mm, s_cnt[i * kSide + k]);
    }
    if (bx < g.nbx && gy < g.nby) {
      g.blk[int64_t(gy) * g.nbx + bx] = v;
      g.bcnt[int64_t(gy) * g.nbx + bx] = mm;
    }
  }
}

template <class T>
__global__ __launch_bounds__(kWave* kSide) void summary_kernel(SummaryArgs<T> g) {
  __shared__ Ends<T> s_row[kSide * kSide];
  __shared__ int s_cnt[kSide * kSide];
  const int ngx = (g.nbx + kSide - 1) / kSide;
  summary_rows(g, int(blockIdx.x) % ngx, int(blockIdx.x) / ngx, s_row, s_cnt);
}

// Batched: job j owns the workgroups [base[j], base[j + 1]).
template <class T>
__global__ __launch_bounds__(kWave* kSide) void summary_batch_kernel(const SummaryArgs<T>* jobs, const int64_t* base,
                                                                     int njobs) {
  __shared__ Ends<T> s_row[kSide * kSide];
  __shared__ int s_cnt[kSide * kSide];
  const int j = find_job(base, njobs, blockIdx.x);
  const SummaryArgs<T> g = jobs[j];
  const int i = int(blockIdx.x - base[j]), ngx = (g.nbx + kSide - 1) / kSide;
  summary_rows(g, i % ngx, i / ngx, s_row, s_cnt);
}

template <class T>
struct DirectArgs {
  int nx, ny, nbx, nby;
  int rint;
  const int64_t* off;
  const T* z;
  const Ends<T>* col;
  const uint64_t* at;
  const Ends<T>* blk;
  const int* bcnt;
  const double* htab;    // direct_htab_width(rint)^2 entries
  const int2* order;     // block offsets within reach, nearest first (the first is (0, 0))
  int norder;
  T* o_z;                // output arena, garena endpoints per tile, interval i of lane L at i * 128 + 2 L
  int64_t garena, o_base;
  int64_t* o_start;
  int64_t* o_cnt;
  int cap;               // intervals a lane's list may hold
  double* spill;         // per tile 2 * (cap - kList) * 64 doubles: the lists' entries past the LDS ones
  int* tile_list;        // [0] = count, then the tiles whose lists overflowed (null: raise the status)
  int* status;
  const int* only;       // tiles to do (null: all)
  int64_t least = INT64_MIN, most = INT64_MAX;  // endpoints in the volume for which this launch works
};

// Lane values combined over the wavefront (result in every lane, scalar).
template <bool kMax>
__device__ __forceinline__ float wave_extreme(float v) {
  const float none = kMax ? -INFINITY : INFINITY;
  auto step = [&](auto ctrl) {
    const int o = __builtin_amdgcn_update_dpp(__float_as_int(none), __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, false);
    v = kMax ? fmaxf(v, __int_as_float(o)) : fminf(v, __int_as_float(o));
  };
  step(std::integral_constant<int, 0x111>{});  // row_shr 1, 2, 4, 8
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});  // row_bcast 15, 31
  step(std::integral_constant<int, 0x143>{});
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), kWave - 1));
}
// A double as a float at or above / at or below it.  Past the largest float
// that is the largest one on the side towards zero and infinity on the other;
// the last term is what floats too small to have a rounding step are off by.
__device__ __forceinline__ float float_up(double v) {
  const float f = fmaxf(float(v), -FLT_MAX);
  return f + fmaf(fabsf(f), 2.4e-7f, 1e-37f);
}
__device__ __forceinline__ float float_down(double v) {
  const float f = fminf(float(v), FLT_MAX);
  return f - fmaf(fabsf(f), 2.4e-7f, 1e-37f);
}
// The smaller / larger of this lane's value and the one of lane L ^ D, in
// registers (no LDS round trip).
template <int D>
__device__ __forceinline__ void pair_minmax(uint32_t v, uint32_t& lo, uint32_t& hi) {
  if constexpr (D == 16 || D == 32) {
    // the swap leaves one of the pair in each of the two results
    const auto r = D == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                           : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    lo = min(uint32_t(r[0]), uint32_t(r[1]));
    hi = max(uint32_t(r[0]), uint32_t(r[1]));
  } else {
    int o;
    if constexpr (D == 1) o = __builtin_amdgcn_update_dpp(0, int(v), 0xb1, 0xf, 0xf, true);        // quad_perm 1 0 3 2
    else if constexpr (D == 2) o = __builtin_amdgcn_update_dpp(0, int(v), 0x4e, 0xf, 0xf, true);   // quad_perm 2 3 0 1
    else if constexpr (D == 4) {
      o = __builtin_amdgcn_update_dpp(0, int(v), 0x141, 0xf, 0xf, true);                           // row_half_mirror: ^ 7
      o = __builtin_amdgcn_update_dpp(0, o, 0x1b, 0xf, 0xf, true);                                 // quad_perm 3 2 1 0: ^ 3
    } else {
      o = __builtin_amdgcn_update_dpp(0, int(v), 0x128, 0xf, 0xf, true);                           // row_ror 8
    }
    lo = min(v, uint32_t(o));
    hi = max(v, uint32_t(o));
  }
}
// |a - b| + c
__device__ __forceinline__ uint32_t abs_diff_add(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_sad_u32 %0, %1, %2, %3" : "=v"(r) : "s"(a), "v"(b), "v"(c));
  return r;
}
// One compare-exchange step of a bitonic network: pairs at distance D,
// ascending where `up`.
template <int D>
__device__ __forceinline__ uint32_t exchange(uint32_t v, bool up) {
  const int L = threadIdx.x & (kWave - 1);
  uint32_t lo, hi;
  pair_minmax<D>(v, lo, hi);
  return ((L & D) == 0) == up ? lo : hi;
}
template <int D>
__device__ __forceinline__ uint32_t merge_keys(uint32_t v, bool up) {
  v = exchange<D>(v, up);
  if constexpr (D > 1) v = merge_keys<D / 2>(v, up);
  return v;
}
// 64 keys sorted over the lanes.
__device__ __forceinline__ uint32_t sort64(uint32_t v, bool up) {
  const int L = threadIdx.x & (kWave - 1);
  v = merge_keys<1>(v, (L & 2) == 0);
  v = merge_keys<2>(v, (L & 4) == 0);
  v = merge_keys<4>(v, (L & 8) == 0);
  v = merge_keys<8>(v, (L & 16) == 0);
  v = merge_keys<16>(v, (L & 32) == 0);
  return merge_keys<32>(v, up);
}
// 64 or 128 keys sorted ascending over (key[0] of the lanes, key[1] of the lanes).
__device__ __forceinline__ void sort_keys(uint32_t (&key)[2], bool two) {
  key[0] = sort64(key[0], true);
  if (!two) return;
  key[1] = sort64(key[1], false);
  const uint32_t lo = min(key[0], key[1]), hi = max(key[0], key[1]);
  key[0] = merge_keys<32>(lo, true);
  key[1] = merge_keys<32>(hi, true);
}
// orders a wavefront's LDS accesses for the compiler (the hardware keeps
// them in order)
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T, int kList>
struct DirectSmem {
  static constexpr int kRecs = DirectShape<kList>::kRecs, kPend = DirectShape<kList>::kPend;
  double list[2][kList][kWave];  // the lanes' lists, first kList entries ([lower, upper][entry][lane])
  double held[2][kHeld][kWave];  // runs on their way to the lists
  T rz[kRecs][2];           // waiting segments
  int rc[kRecs];            // and their column: (x - tile x + 1024) | 8 (y - tile y + 1024) << 16
  double cm[kCommon][2];    // common cover of the tile
  uint64_t pw[kPend];       // columns whose inner segments are still to be looked at: start and count
  int pc[kPend];            // and their place, as in rc
};

// One tile of 8 x 8 output columns, one lane each.  With kSplit > 1 as many
// wavefronts share the tile: each unites its part of the source columns, and
// the first one unites the parts (`sm` is the first one's memory, the others'
// follow it).
template <class T, int kList, int kSplit>
__device__ void direct_tile(const DirectArgs<T>& g, int tile, int64_t slot, DirectSmem<T, kList>* sms, int part,
                            const double* htab) {
  DirectSmem<T, kList>& sm = sms[part];
  constexpr int kRecs = DirectShape<kList>::kRecs, kPend = DirectShape<kList>::kPend, kDrainAt = DirectShape<kList>::kDrainAt;
  const int L = threadIdx.x & (kWave - 1);
  const int lx = L % kSide, ly = L / kSide;
  const int tx = tile % g.nbx, ty = tile / g.nbx;
  const int x = tx * kSide + lx, y = ty * kSide + ly;
  const bool active = x < g.nx && y < g.ny;
  const int64_t colidx = int64_t(y) * g.nx + x;
  const int rint = g.rint, W = direct_htab_width(rint);
  const int cap = g.cap;
  // --- the lane's union: a sorted list of n intervals ------------------------
  // Its first and its last interval are in registers: F = [flo, fhi] and, with
  // n > 1, E = [elo, ehi] (else empty), with the bounds next to them: `lo1`
  // above F and `hi1` below E.  The entries past kList are in global memory
  // (the two address spaces are kept apart by type, or the compiler reads
  // both through flat instructions).
  int n = 0, ok = 1, dirty = 0, at = 0;
  double flo = INFINITY, fhi = -INFINITY, elo = INFINITY, ehi = -INFINITY, lo1 = INFINITY, hi1 = -INFINITY;
  using LdsDouble = __attribute__((address_space(3))) double;
  using GlobalDouble = __attribute__((address_space(1))) double;
  LdsDouble* const lds = (LdsDouble*)&sm.list[0][0][L];
  GlobalDouble* const far = (GlobalDouble*)(g.spill + (slot * kSplit + part) * (2 * int64_t(cap - kList) * kWave) + L);
  auto get = [&](int end, int i) -> double {
    if (i < kList) return lds[(end * kList + i) * kWave];
    return far[(end * (cap - kList) + (i - kList)) * kWave];
  };
  auto put = [&](int i, double a, double b) {
    if (i < kList) {
      lds[i * kWave] = a;
      lds[(kList + i) * kWave] = b;
    } else {
      far[(i - kList) * kWave] = a;
      far[(cap - kList + i - kList) * kWave] = b;
    }
  };
  auto settle = [&]() {  // the list in memory as in registers
    if (dirty) {
      put(0, flo, fhi);
      if (n > 1) put(n - 1, elo, ehi);
      dirty = 0;
    }
  };
  // [s, e] into the list, wherever it belongs.  Reads that do not depend on
  // each other go together: the lists' latency is what this costs.
  auto unite_slow = [&](double s, double e) {
    settle();
    // the intervals it meets: [k, j)
    int k = 0, j = 0;
    if (n <= kList) {
#pragma unroll
      for (int i = 0; i < kList; ++i) {
        const double a = lds[i * kWave], b = lds[(kList + i) * kWave];
        k += i < n && b < s ? 1 : 0;
        j += i < n && a <= e ? 1 : 0;
      }
      // (an unsorted column's run, of a call that will be refused, may have
      // s > e: it meets nothing, and the list stays within its room)
      j = max(j, k);
    } else {
      // long lists: from where the last one went (runs come nearly in order)
      k = min(at, n);
      while (k > 0 && get(1, k - 1) >= s) --k;
      while (k < n && get(1, k) < s) ++k;
      j = k;
      while (j < n && get(0, j) <= e) ++j;
    }
    at = k;
    if (k == j) {
      if (n >= cap) {
        ok = 0;
        return;
      }
      for (int i = n; i > k; --i) put(i, get(0, i - 1), get(1, i - 1));
    } else {
      s = fmin(get(0, k), s);
      e = fmax(get(1, j - 1), e);
      if (j > k + 1)
        for (int i = j; i < n; ++i) put(i - (j - k - 1), get(0, i), get(1, i));
    }
    n += 1 - (j - k);
    put(k, s, e);
    flo = get(0, 0);
    fhi = get(1, 0);
    elo = n > 1 ? get(0, n - 1) : INFINITY;
    ehi = n > 1 ? get(1, n - 1) : -INFINITY;
    lo1 = n > 1 ? get(0, 1) : INFINITY;
    hi1 = n > 1 ? get(1, n - 2) : -INFINITY;
  };
  // A run that does not simply extend F or E is held back, and the lanes'
  // held runs go through the lists together: at different segments a run ends
  // in different lanes, and one by one nearly every segment would take the
  // wavefront through the list code.
  int held = 0;
  auto flush = [&]() {
    for (int i = 0; ballot(i < held) != 0; ++i) {
      if (i < held && ok) {
        const double s = sm.held[0][i][L], e = sm.held[1][i][L];
        if ((s < flo || e > fhi) && (s < elo || e > ehi)) unite_slow(s, e);
      }
    }
    held = 0;
  };
  auto unite = [&](bool run, double s, double e) {
    const bool want = run && active && (s < flo || e > fhi) && (s < elo || e > ehi);
    if (ballot(want) == 0) return;
    const bool first = want && s <= fhi && e >= flo && e < lo1;
    const bool last = want && !first && s <= ehi && e >= elo && s > hi1;
    flo = first && s < flo ? s : flo;
    fhi = first && e > fhi ? e : fhi;
    elo = last && s < elo ? s : elo;
    ehi = last && e > ehi ? e : ehi;
    // (with two intervals each is the other's neighbour)
    hi1 = n == 2 ? fhi : hi1;
    lo1 = n == 2 ? elo : lo1;
    dirty = first || last ? 1 : dirty;
    if (want && !first && !last) {
      sm.held[0][held][L] = s;
      sm.held[1][held][L] = e;
      ++held;
    }
    if (ballot(held == kHeld) != 0) flush();
  };

  const uint32_t mx = uint32_t(lx + 1024), my = uint32_t(ly + 1024) * 8u;
  // --- waiting segments ------------------------------------------------------
  // They are taken nearly in the order of their lower ends, so that a lane's
  // grown segments follow each other and fuse into runs in registers; a run
  // meets the list when a gap ends it.
  int nrec = 0;
  bool old = true;  // the lists changed since the common cover was taken
  auto drain = [&]() {
    lds_order();
    const double qnan = __builtin_nan("");
    double rs = qnan, re = qnan;
    // the last 128 of them, sorted
    const int first = max(nrec - 2 * kWave, 0), cnt2 = nrec - first;
    float lo[2];
    uint32_t key[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int r = t * kWave + L;
      lo[t] = r < cnt2 ? float(sm.rz[first + r][0]) : NAN;
    }
    const float zmin = wave_extreme<false>(fminf(lo[0], lo[1])), zmax = wave_extreme<true>(fmaxf(lo[0], lo[1]));
    constexpr float kKeyMax = 33000000.f;  // below 2^25
    const float scale = kKeyMax / fmaxf(zmax - zmin, 1e-20f);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      // (every waiting segment's key holds its place, also that of a lower end
      // that is not finite, in a call that will be refused; fmaxf drops a NaN)
      key[t] = t * kWave + L < cnt2 ? uint32_t(fminf(fmaxf((lo[t] - zmin) * scale, 0.f), kKeyMax)) << 7 | uint32_t(t * kWave + L) : ~0u;
    sort_keys(key, cnt2 > kWave);
    for (int base = 0; base < cnt2; base += kWave) {
      const int cnt = min(cnt2 - base, kWave);
      const int from = L < cnt ? first + int(key[0] & 127u) : 0;
      key[0] = key[1];
      // (past the last one: NaN, which changes nothing)
      const double va = L < cnt ? double(sm.rz[from][0]) : qnan, vb = L < cnt ? double(sm.rz[from][1]) : qnan;
      const int vc = sm.rc[from];
      for (int r = 0; r < cnt; r += kAhead) {
        // the growths of several segments are read together
        double h[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          // H's byte offset in the table is |dx| * 8 W + |8 dy|
          const uint32_t code = uint32_t(__builtin_amdgcn_readlane(vc, r + u));
          const uint32_t dx = abs_diff_add(code & 0xffffu, mx, 0u);
          h[u] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(htab) +
                                                  abs_diff_add(code >> 16, my, __umul24(dx, 8u * uint32_t(W))));
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const double s = lane_bcast(va, r + u) - h[u], e = lane_bcast(vb, r + u) + h[u];
          // out of reach: NaN, no comparison holds and the run stays
          const bool apart = s > re || e < rs;
          if (ballot(apart) != 0) {
            unite(apart, rs, re);
            rs = apart ? qnan : rs;
            re = apart ? qnan : re;
          }
          rs = qmin(rs, s);
          re = qmax(re, e);
        }
      }
    }
    unite(rs == rs, rs, re);
    flush();
    nrec = first;
    old = true;
    lds_order();
  };

  // distance of v to [a, b]
  auto gap = [](int v, int a, int b) { return max(max(a - v, v - b), 0); };

  int ncm = 0;       // intervals in sm.cm
  // The cover common to the lanes that have a list: what lies inside it is
  // inside every such lane's union.
  auto common = [&]() {
    const bool has = active && n > 0;
    old = false;
    if (ballot(has && n > 2) == 0) {
      // F and E of every lane (with one interval, that one)
      const bool two = ballot(has && n > 1) != 0;
      const float P0 = wave_extreme<true>(has ? float_up(flo) : -INFINITY);
      const float Q0 = wave_extreme<false>(has ? float_down(fhi) : INFINITY);
      ncm = P0 < Q0 && Q0 < INFINITY ? 1 : 0;
      if (L == 0) {
        sm.cm[0][0] = double(P0);
        sm.cm[0][1] = double(Q0);
      }
      if (two) {
        const float P1 = wave_extreme<true>(has ? float_up(n > 1 ? elo : flo) : -INFINITY);
        const float Q1 = wave_extreme<false>(has ? float_down(n > 1 ? ehi : fhi) : INFINITY);
        if (P1 < Q1 && Q1 < INFINITY) {
          if (L == 0) {
            sm.cm[ncm][0] = double(P1);
            sm.cm[ncm][1] = double(Q1);
          }
          ++ncm;
        }
      }
      lds_order();
      return;
    }
    settle();
    lds_order();
    int p = 0;
    ncm = 0;
    float z = -INFINITY;
    for (int it = 0; it < 2 * kCommon && ncm < kCommon; ++it) {
      float a = -INFINITY, b = INFINITY;
      if (has) {
        // (the first and the last interval are in registers)
        auto bound = [&](int end) { return p == 0 ? (end ? fhi : flo) : p == n - 1 ? (end ? ehi : elo) : get(end, p); };
        while (p < n && float_down(bound(1)) <= z) ++p;
        a = p < n ? float_up(bound(0)) : INFINITY;
        b = p < n ? float_down(bound(1)) : INFINITY;
      }
      if (ballot(has && p >= n) != 0) break;
      const float P = wave_extreme<true>(a), Q = wave_extreme<false>(b);
      if (P < Q) {
        if (L == 0) {
          sm.cm[ncm][0] = double(P);
          sm.cm[ncm][1] = double(Q);
        }
        ++ncm;
        z = Q;
      } else {
        z = P;
      }
    }
    lds_order();
  };
  int npend = 0;
  // which of the first nc common intervals holds [s, e] (-1: none)
  auto covered = [&](int nc, double s, double e) {
    int m = -1;
    for (int i = 0; i < nc; ++i) {
      const double P = sm.cm[i][0], Q = sm.cm[i][1];
      m = (s >= P && e <= Q) ? i : m;
    }
    return m;
  };
  auto keep = [&](bool add, T a, T b, int code) {
    const uint64_t mask = ballot(add);
    if (add) {
      const int q = nrec + count_below(mask);
      sm.rz[q][0] = a;
      sm.rz[q][1] = b;
      sm.rc[q] = code;
    }
    nrec += popc(mask);
  };
  // Source block (bx, by): one lane per source column (those with `take`).  A
  // column's first and last segment wait for the next drain where they are
  // not inside one of the first `nc` common intervals; if it has more, and
  // they may not all be inside, the column waits to be looked at.
  auto block = [&](int bx, int by, bool take, int nc) {
    const int cx = bx * kSide + lx, cy = by * kSide + ly;
    const int64_t slot = (int64_t(by) * g.nbx + bx) * kWave + L;
    const Ends<T> r = g.col[slot];
    const uint64_t word = g.at[slot];
    // the column's largest growth on any output column of the tile
    const int gx = gap(cx, tx * kSide, tx * kSide + kSide - 1), gy = gap(cy, ty * kSide, ty * kSide + kSide - 1);
    const double h = htab[min(gx, W - 1) * W + min(gy, W - 1)];
    const int count = int(word >> 48);
    const bool live = take && count > 0 && h == h;
    const int m0 = live ? covered(nc, double(r.lo0) - h, double(r.hi0) + h) : 0;
    const int m1 = live ? covered(nc, double(r.lo1) - h, double(r.hi1) + h) : 0;
    const int code = (cx - tx * kSide + 1024) | (cy - ty * kSide + 1024) << 19;
    keep(m0 < 0, r.lo0, r.hi0, code);
    keep(m1 < 0 && count > 1, r.lo1, r.hi1, code);
    const bool inner = live && count > 2 && !(m0 >= 0 && m0 == m1);
    const uint64_t mask = ballot(inner);
    if (inner) {
      const int q = npend + count_below(mask);
      sm.pw[q] = word;
      sm.pc[q] = code;
    }
    npend += popc(mask);
  };
  // The last `m` waiting columns, one per lane: their segments between the
  // first and the last that may change some lane wait for a drain, which
  // follows where `drain_at` or more do.
  auto columns = [&](int m, int drain_at, int nc) {
    lds_order();
    const bool mine = L < m;
    const int q = npend - m + L;
    const uint64_t word = mine ? sm.pw[q] : 0;
    const int code = mine ? sm.pc[q] : 1024 | 1024 << 19;
    npend -= m;
    int64_t s = int64_t(word & ((uint64_t(1) << 48) - 1));
    int count = int(word >> 48);
    const int px = (code & 0xffff) - 1024, py = (code >> 19) - 1024;  // place relative to the tile
    if (ballot(count == kCountMany) != 0) {
      if (count == kCountMany) {
        const int64_t c = int64_t(ty * kSide + py) * g.nx + tx * kSide + px;
        count = int(min<int64_t>((g.off[c + 1] - s) / 2, INT32_MAX));
      }
    }
    double h = 0;
    int left = 0, stop_at = 0;
    bool back = false;
    if (m > 0) {
      h = htab[gap(px, 0, kSide - 1) * W + gap(py, 0, kSide - 1)];
      T r[4] = {T(0), T(0), T(0), T(0)};
      if (mine) {
        r[0] = g.z[s];
        r[1] = g.z[s + 1];
        r[2] = g.z[s + 2 * int64_t(count) - 2];
        r[3] = g.z[s + 2 * int64_t(count) - 1];
      }
      const int m0 = covered(nc, double(r[0]) - h, double(r[1]) + h), m1 = covered(nc, double(r[2]) - h, double(r[3]) + h);
      // From the end that is not covered towards the other one, until a
      // segment is inside the common interval that holds the other end
      // (sorted columns: so is the rest).
      left = mine && !(m0 >= 0 && m0 == m1) ? count - 2 : 0;
      back = m0 >= 0 && m1 < 0;
      stop_at = back ? m0 : m1;
    }
    // U segments of a column per round trip, the next ones loaded while these
    // are looked at
    constexpr int U = 2;
    T a[U], b[U];
    auto load = [&](int j0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = back ? count - 2 - (j0 + u) : j0 + u + 1;
        a[u] = b[u] = T(0);
        if (j0 + u < left) {
          a[u] = g.z[s + 2 * int64_t(j)];
          b[u] = g.z[s + 2 * int64_t(j) + 1];
        }
      }
    };
    load(0);
    for (int j0 = 0;; j0 += U) {
      const bool last = ballot(j0 < left) == 0;
      while (nrec > kRecs - U * kWave || (last && nrec >= drain_at)) drain();
      if (last) break;
      T ta[U], tb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ta[u] = a[u];
        tb[u] = b[u];
      }
      load(j0 + U);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool here = j0 + u < left;
        const int m = here ? covered(nc, double(ta[u]) - h, double(tb[u]) + h) : 0;
        keep(m < 0, ta[u], tb[u], code);
        left = here && m >= 0 && m == stop_at ? 0 : left;
      }
    }
  };

  // With kSplit > 1 a wavefront takes its share of the own block's columns
  // (the first stage's are everyone's: without that cover the others' segments
  // would all stay) and of the other blocks.
  const bool mine = kSplit == 1 || ((lx >> 1) + (ly >> 1)) % kSplit == part;
  const int first_mask = rint >= 12 ? 3 : (rint >= 4 ? 1 : 0), first_at = rint >= 12 ? 2 : 0;
  for (int g0 = 0; g0 < g.norder; g0 += kWave) {
    // 64 blocks at a time, one lane each: their summaries
    int2 o = make_int2(0, 0);
    if (g0 + L < g.norder) o = g.order[g0 + L];
    const int bx = tx + o.x, by = ty + o.y;
    Ends<T> bs{T(INFINITY), T(-INFINITY), T(INFINITY), T(-INFINITY)};
    int bc = 0;
    if (g0 + L < g.norder && bx >= 0 && by >= 0 && bx < g.nbx && by < g.nby) {
      bs = g.blk[int64_t(by) * g.nbx + bx];
      bc = g.bcnt[int64_t(by) * g.nbx + bx];
    }
    uint64_t todo = ballot(bc > 0);
    // the tile's own block goes first, and of it first a sixteenth or a
    // quarter of its columns, which cover most of what the others have
    uint64_t share = ~uint64_t(0);
    if constexpr (kSplit > 1) {
      share = 0;
      for (int i = 0; i < kWave; i += kSplit) share |= uint64_t(1) << i;
      share <<= part;
    }
    int own = g0 == 0 && (todo & 1) ? 2 : 0;
    bool sharing = own > 0;
    todo &= g0 == 0 ? share & ~uint64_t(1) : share;
    bool fresh = true;
    const bool end = g0 + kWave >= g.norder;  // what is left waiting goes with the last group
    while (own > 0 || todo != 0 || (end && nrec + npend > 0)) {
      bool take = true, reached = active, now = false, visit = own > 0;
      int ux = tx, uy = ty;
      if (own > 0) {
        take = (((lx - first_at) | (ly - first_at)) & first_mask) == 0;
        take = take == (own == 2);
        if constexpr (kSplit > 1) take = take && ((own == 2 && first_mask != 0) || mine);
        --own;
        now = true;
      } else if (todo == 0) {
        now = true;
      } else {
        if (fresh) {
          // blocks inside the first and last intervals of every lane, 64 at once
          fresh = false;
          const double A0 = wave_extreme<true>(active ? float_up(flo) : -INFINITY);
          const double B0 = wave_extreme<false>(active ? float_down(fhi) : INFINITY);
          const double A1 = wave_extreme<true>(active ? float_up(n > 1 ? elo : flo) : -INFINITY);
          const double B1 = wave_extreme<false>(active ? float_down(n > 1 ? ehi : fhi) : INFINITY);
          const int gx = o.x == 0 ? 0 : kSide * (abs(o.x) - 1) + 1, gy = o.y == 0 ? 0 : kSide * (abs(o.y) - 1) + 1;
          const double h = bc > 0 ? htab[gx * W + gy] : 0.0;
          const bool low = double(bs.lo0) - h >= A0;
          const bool in =
              (low && double(bs.hi1) + h <= B0) ||
              (bc <= 2 && low && double(bs.hi0) + h <= B0 && double(bs.lo1) - h >= A1 && double(bs.hi1) + h <= B1);
          todo &= ~ballot(in);
          if (todo == 0) continue;
        }
        const int i = __builtin_ctzll(todo);
        todo &= todo - 1;
        ux = __builtin_amdgcn_readlane(bx, i);
        uy = __builtin_amdgcn_readlane(by, i);
        const int uc = __builtin_amdgcn_readlane(bc, i);
        const Ends<double> u{double(lane_bcast(bs.lo0, i)), double(lane_bcast(bs.hi0, i)),
                             double(lane_bcast(bs.lo1, i)), double(lane_bcast(bs.hi1, i))};
        // the block against each lane it reaches, at the lane's own distance
        const int gx = gap(x, ux * kSide, ux * kSide + kSide - 1), gy = gap(y, uy * kSide, uy * kSide + kSide - 1);
        const double h = htab[min(gx, W - 1) * W + min(gy, W - 1)];
        visit = true;
        reached = active && h == h;
        const bool low = u.lo0 - h >= flo;
        const bool in = (low && u.hi1 + h <= fhi) || (u.lo0 - h >= elo && u.hi1 + h <= ehi) ||
                        (uc <= 2 && low && u.hi0 + h <= fhi && u.lo1 - h >= elo && u.hi1 + h <= ehi);
        if (ballot(reached && !in) == 0) continue;
      }
      if (old) common();
      // (a lane that has no list yet is covered by nothing)
      const int nc = ballot(reached && n == 0) != 0 ? 0 : ncm;
      if (visit) block(ux, uy, take, nc);

      const int m = now || npend > kPend - kWave ? min(npend, kWave) : 0;
      // (the waiting columns are of several blocks: any lane without a list counts)
      columns(m, now ? 1 : kDrainAt, ballot(active && n == 0) != 0 ? 0 : ncm);
      if constexpr (kSplit > 1) {
        // the own block done, the wavefronts' first and last intervals go to
        // all of them: with a part of the cover each, the blocks to come
        // would cost every wavefront what they cost one alone
        if (sharing && own == 0) {
          sharing = false;
          sm.held[0][0][L] = flo;
          sm.held[0][1][L] = elo;
          sm.held[1][0][L] = fhi;
          sm.held[1][1][L] = ehi;
          __syncthreads();
          for (int w = 1; w < kSplit; ++w) {
            const DirectSmem<T, kList>& o = sms[(part + w) % kSplit];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const double s = o.held[0][i][L], e = o.held[1][i][L];
              if (active && ok && s <= e && (s < flo || e > fhi) && (s < elo || e > ehi)) unite_slow(s, e);
            }
          }
          old = true;
          __syncthreads();
        }
      }
    }
  }
  if constexpr (kSplit > 1) {
    settle();
    sm.rc[L] = ok ? n : -1;  // the list's length, where nothing waits any more
    __syncthreads();
    if (part != 0) return;
    for (int w = 1; w < kSplit; ++w) {
      const int nw = sms[w].rc[L];
      ok = nw < 0 ? 0 : ok;
      const GlobalDouble* const fw = (const GlobalDouble*)(g.spill + (slot * kSplit + w) * (2 * int64_t(cap - kList) * kWave) + L);
      for (int i = 0; ballot(ok && i < nw) != 0; ++i) {
        if (!ok || i >= nw) continue;
        const double s = i < kList ? sms[w].list[0][i][L] : double(fw[(i - kList) * kWave]);
        const double e = i < kList ? sms[w].list[1][i][L] : double(fw[(cap - kList + i - kList) * kWave]);
        if ((s < flo || e > fhi) && (s < elo || e > ehi)) unite_slow(s, e);
      }
    }
  }
  if (ballot(active && ok == 0) != 0) {
    // the scan and the CSR copy that follow before the host looks at the
    // list read nothing for this tile
    if (active) {
      g.o_start[colidx] = 0;
      g.o_cnt[colidx] = 0;
    }
    if (L == 0) {
      if (g.tile_list)
        g.tile_list[1 + atomicAdd(g.tile_list, 1)] = tile;
      else
        atomicOr(g.status, kStatusGatherOverflow);  // batched: the host redoes this volume alone
    }
    return;
  }
  if (!active) return;
  settle();
  const int64_t ob = g.o_base + slot * g.garena + 2 * int64_t(L);
  for (int i = 0; i < n; ++i) {
    g.o_z[ob + int64_t(i) * (2 * kWave)] = T(get(0, i));
    g.o_z[ob + int64_t(i) * (2 * kWave) + 1] = T(get(1, i));
  }
  g.o_start[colidx] = ob;
  g.o_cnt[colidx] = 2 * n;
}

extern __shared__ double vo_direct_htab[];

// The H table of radius rint, staged in the workgroup's LDS or where it is.
template <bool kLdsTable>
__device__ __forceinline__ const double* stage_htab(const double* htab, int rint) {
  if constexpr (kLdsTable) {
    const int W = direct_htab_width(rint);
    for (int i = threadIdx.x; i < W * W; i += blockDim.x) vo_direct_htab[i] = htab[i];
    __syncthreads();
    return vo_direct_htab;
  } else {
    return htab;
  }
}

// Registers: four waves per SIMD, where the short lists' LDS allows them.
template <int kList, int kSplit>
constexpr int direct_waves() {
  return kSplit > 1 || kList > 4 ? 2 : 4;
}

// One tile per workgroup of kSplit wavefronts.  Where only the device knows
// how many endpoints the volume has, and nothing else depends on them, two
// launches of different splits go out and the one whose range does not hold
// them returns at once (its 4,600 empty workgroups cost 4-7 us at 544^2; a
// first call that waits for the answer instead 60).
template <class T, int kList, bool kLdsTable, int kSplit>
__global__ __launch_bounds__(kWave* kSplit, (direct_waves<kList, kSplit>())) void direct_kernel(DirectArgs<T> g) {
  __shared__ DirectSmem<T, kList> sm[kSplit];
  const int64_t ncols = int64_t(g.nx) * g.ny, endpoints = g.off[ncols] - g.off[0];
  if (endpoints < g.least || endpoints > g.most) return;
  const double* htab = stage_htab<kLdsTable>(g.htab, g.rint);
  const int64_t i = xcd_tile(blockIdx.x, gridDim.x);
  const int tile = g.only ? g.only[i] : int(i);
  const int part = kSplit > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : 0;
  direct_tile<T, kList, kSplit>(g, tile, i, sm, part, htab);
}

// Batched: job j owns the global tiles [tile_base[j], tile_base[j + 1]); this
// launch covers the n tiles from t0 on (one radius class), kSplit wavefronts
// each.
template <class T, int kList, bool kLdsTable, int kSplit>
__global__ __launch_bounds__(kWave* kSplit, (direct_waves<kList, kSplit>())) void direct_batch_kernel(
    const DirectArgs<T>* jobs, const int64_t* tile_base, int njobs, int64_t t0, int64_t n) {
  __shared__ DirectSmem<T, kList> sm[kSplit];
  const int64_t t = t0 + xcd_chunk_tile(blockIdx.x, n);
  const int j = find_job(tile_base, njobs, t);
  const DirectArgs<T> g = jobs[j];
  const double* htab = stage_htab<kLdsTable>(g.htab, g.rint);
  const int64_t i = t - tile_base[j];
  const int part = kSplit > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : 0;
  direct_tile<T, kList, kSplit>(g, int(i), i, sm, part, htab);
}

}  // namespace vo
