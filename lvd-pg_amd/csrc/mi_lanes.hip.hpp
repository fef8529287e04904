// Pairwise mutual information, a pair per two lanes: a wave holds one variable u and 32 variables v, takes u's examples sorted
// by category, the even ones in one half of its lanes and the odd ones in the other, and keeps, for the category under way, one
// row of counters per v.
//
// The sum over a pair's cells telescopes over its examples (chow_liu.hip), in any order; sorted by u's category only the
// cells (a, .) of one category a are open at a time: C counters, not C^2.  That is 256 bytes per pair (8-bit counters
// of up to 256 categories, 16-bit ones of up to 128), so a pair has a column of the wave's LDS to itself: word r of variable l
// at 128 r + 4 l, the two lanes of a variable in halves of the wave that the LDS takes one after the other (an atomic add takes
// 4.3 cycles, at random addresses of a shared table 7.2, where many examples fall into one cell up to 128), and no barrier keeps
// the waves of a workgroup in step: sixteen waves a compute unit with 256 categories.
//
// Per 64 additions: a request of two examples' rows (a word per variable, 128 bytes each: the staged data lies in blocks of 32
// variables, and the workgroups of a die work on the same one at a time, 2 MB of 16384 examples), an atomic add with
// return, a look-up of the count's term (few counts in a wave: 2.5 cycles), six vector instructions.  A category's counters are
// cleared by a store per example up to 32 examples, else by 8-byte stores over all of them.
//
// 3072 variables, 16384 examples: 256 categories 55 -> 27 ms, 128 categories 38 -> 22, 64 categories 37 -> 20, 256 categories with four
// fifths of the examples in one 241 -> 88.  What bounds it is instruction issue (vector unit, LDS and requests of sixteen waves).
// With 64 variables a wave, one to a lane, eight waves a unit with 256 categories and the vector unit at work for 58 % of the
// time it was 32 ms (1000 examples 4.7 instead of 6.1, the black images 60); tried there: the three steps of a chunk overlapped
// with its neighbours' (35 ms), nine waves a unit (35: the SIMD with three of them is the last), a code of 16 bits a lane (38:
// such a request keeps the data path busy for 16 cycles).
#pragma once

#include <utility>

namespace pcm {

constexpr int kMiChunk = 32;       // examples under way in a wave
constexpr int kMiHalf = kMiChunk / 2;
constexpr int kMiBlock = 32;       // variables v of a wave

// An entry of the list of u's examples: 128 * example, and in the first of each chunk
//   bits 0..4 examples in the chunk - 1 | 5 the category's last chunk | 6 counts may exceed the short counters
constexpr uint32_t kMiLast = 32u, kMiMany = 64u, kMiFlags = 127u;

// What a lane is given per example: byte offset of the counter word's row (128 * row), and in the low bits its shift.
template <int kBits>
__device__ __forceinline__ uint32_t mi_lane_code(uint32_t b) {
  return kBits == 8 ? ((b >> 2) << 7) | ((b & 3u) << 3) : ((b >> 1) << 7) | ((b & 1u) << 4);
}

// xb[V][Np] -> xt[V / 32][N][32], variables past V zero
template <int kBits>
__global__ __launch_bounds__(256) void mi_lane_codes_kernel(const uint8_t* __restrict__ xb, int N, int64_t Np, int V,
                                                            uint32_t* __restrict__ xt) {
  __shared__ uint8_t t[32][68];   // [variable][example]
  const int e0 = blockIdx.x * 64, v0 = blockIdx.y * 32;
  for (int i = threadIdx.x; i < 32 * 16; i += 256) {
    const int v = i >> 4, q = i & 15;
    uint32_t w = 0u;
    if (v0 + v < V) w = *reinterpret_cast<const uint32_t*>(xb + (size_t)(v0 + v) * Np + e0 + 4 * q);   // (Np: a multiple of 64)
    *reinterpret_cast<uint32_t*>(&t[v][4 * q]) = w;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int e = i >> 5, v = i & 31;
    if (e0 + e < N) xt[((size_t)blockIdx.y * N + e0 + e) * 32 + v] = mi_lane_code<kBits>(t[v][e]);
  }
}

// Place of an example in its chunk: the even ones first (one half of a wave's lanes asks for those, the other for the odd ones).
__device__ __forceinline__ int mi_place(int at) {
  return (at & ~(kMiChunk - 1)) | ((at & 1) * kMiHalf) | ((at & (kMiChunk - 1)) >> 1);
}

// One variable's examples sorted by category, every category's padded to whole chunks (with example 0, never counted),
// and where each of `parts` shares of its chunks begins, a category never cut in two.
__global__ __launch_bounds__(1024) void mi_order_kernel(const uint8_t* __restrict__ xb, int N, int64_t Np, int C, int many,
                                                        int parts, int64_t stride, uint32_t* __restrict__ order,
                                                        int* __restrict__ begin) {
  __shared__ int cnt[256], first[257], cur[256];
  const int u = blockIdx.x, t = threadIdx.x;
  const uint8_t* row = xb + (size_t)u * Np;
  uint32_t* out = order + (size_t)u * stride;
  if (t < 256) { cnt[t] = 0; cur[t] = 0; }
  __syncthreads();
  for (int e = t; e < N; e += 1024) atomicAdd(&cnt[row[e]], 1);
  __syncthreads();
  if (t < 256) first[t + 1] = (cnt[t] + kMiChunk - 1) / kMiChunk;
  if (t == 0) first[0] = 0;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    int add = 0;
    if (t < 256 && t + 1 > o) add = first[t + 1 - o];
    __syncthreads();
    if (t < 256) first[t + 1] += add;
    __syncthreads();
  }
  auto entry = [&](int a, int at, int e) {   // at: place among the category's examples
    uint32_t w = (uint32_t)e << 7;
    if (at % kMiChunk == 0) {
      w |= (uint32_t)(min(kMiChunk, cnt[a] - at) - 1);
      if (at + kMiChunk >= cnt[a]) w |= kMiLast;
      if (cnt[a] > many) w |= kMiMany;
    }
    out[first[a] * kMiChunk + mi_place(at)] = w;
  };
  for (int e = t; e < N; e += 1024) {
    const int a = row[e];
    entry(a, atomicAdd(&cur[a], 1), e);
  }
  if (t < 2 * kMiChunk) out[first[256] * kMiChunk + t] = 0u;   // what is asked for ahead of the end
  for (int i = t; i < 256 * kMiChunk; i += 1024) {   // the places past a category's examples
    const int a = i / kMiChunk, at = (cnt[a] & ~(kMiChunk - 1)) + i % kMiChunk;
    if (at >= cnt[a] && cnt[a] % kMiChunk) out[first[a] * kMiChunk + mi_place(at)] = 0u;
  }
  if (t <= parts) {
    const int want = (int)((int64_t)first[256] * t / parts);
    int a = 0;
    while (first[a] < want) ++a;
    begin[(size_t)u * (parts + 1) + t] = first[a];
  }
}

struct MiLanesArgs {
  const uint32_t* xt;
  const uint32_t* order;
  const int* begin;
  const long long* dg;
  const double* stat;
  float* mi;
  unsigned long long* partial;   // [V][32 * blocks] where a pair's categories are shared out (parts > 1)
  int64_t stride;
  int N, V, C, parts, blocks, per_die, items, table, table_bytes, wave_bytes;
  float pc;
};

// r[j]: the word at offset `word` of the row whose offset lane j of the lane's row of sixteen holds in `at`
template <int... kJ>
__device__ __forceinline__ void mi_request_rows(__amdgpu_buffer_rsrc_t rx, int at, int word, uint32_t (&r)[kMiHalf],
                                                std::integer_sequence<int, kJ...>) {
  ((r[kJ] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
        rx, __builtin_amdgcn_update_dpp(0, at, 0x150 + kJ, 0xf, 0xf, true) + word, 0, 0)), ...);
}

template <int kBits>
__global__ __launch_bounds__(1024) void mi_lanes_kernel(MiLanesArgs g) {
  extern __shared__ __align__(16) char mi_lanes_lds[];
  typedef __attribute__((address_space(3))) uint32_t* word_at;
  typedef __attribute__((address_space(3))) double* term_at;
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) u2* pair_at;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int odd = lane >> 5;   // the half of a chunk's examples that the lane takes
  // the workgroups of a die (consecutive ones go round the eight dies) take consecutive items: one block of variables
  int item = (int)(blockIdx.x & 7) * g.per_die + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= g.per_die || item >= g.items) return;
  const int part = item % g.parts;
  item /= g.parts;
  int block = 0, groups;
  for (;; item -= groups, ++block) {
    groups = (min(g.V, kMiBlock * (block + 1)) + waves - 1) / waves;
    if (item < groups) break;
  }
  const int u = item * waves + wave;
  // LDS: terms of the counts 0 .. table - 1 | the waves' counters, each wave's at a multiple of its own size (a power of two)
  for (int i = threadIdx.x; i < g.table; i += blockDim.x) reinterpret_cast<double*>(mi_lanes_lds)[i] = (double)g.dg[i];
  const uint32_t mine = (uint32_t)(g.table_bytes + wave * g.wave_bytes);
  const uint32_t own = mine + 4u * (lane & 31);
  auto sweep = [&](int bytes) {   // multiples of 2 KB
    asm volatile("" ::: "memory");
    for (int o = 0; o < bytes; o += 2048)
#pragma unroll
      for (int i = 0; i < 4; ++i) *(pair_at)(uintptr_t)(mine + 8u * lane + o + 512 * i) = u2{0u, 0u};
    asm volatile("" ::: "memory");
  };
  sweep(g.wave_bytes);
  __syncthreads();
  if (u >= min(g.V, kMiBlock * (block + 1))) return;   // (no barrier from here on)
  const int row_bytes = (((kBits == 8 ? (g.C + 3) / 4 : (g.C + 1) / 2) * 128) + 2047) & ~2047;   // at most wave_bytes
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(g.xt) + (size_t)block * g.N * kMiBlock, 0, (int)((size_t)g.N * 128), 0x00020000);
  const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(g.order) + (size_t)u * g.stride, 0, (int)(g.stride * 4), 0x00020000);
  const int c0 = g.begin[(size_t)u * (g.parts + 1) + part], c1 = g.begin[(size_t)u * (g.parts + 1) + part + 1];
  double acc = 0.0;   // whole numbers below 2^53: exact in any order
  // the list of chunk c: lane i of a row of sixteen lanes holds entry i of its half's sixteen
  const int list_lane = 4 * ((lane & 15) + kMiHalf * odd);
  auto list = [&](int c) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rl, list_lane, min(c, c1 - 1) * (kMiChunk * 4), 0);
  };
  auto flags_of = [&](uint32_t l) { return (uint32_t)__builtin_amdgcn_readfirstlane(l) & kMiFlags; };
  // Two examples a request: one half of the lanes asks for one's row, the other half for the other's, a word a lane
  auto request = [&](uint32_t l, uint32_t (&r)[kMiHalf]) {
    mi_request_rows(rx, (int)(l & ~kMiFlags), 4 * (lane & 31), r, std::make_integer_sequence<int, kMiHalf>{});
  };
  auto term = [&](uint32_t count) { return *(term_at)(uintptr_t)(count << 3); };
  const uint32_t rows = (uint32_t)(g.wave_bytes - 128);
  // A chunk's examples in short counters and the terms in LDS: n of them, of which this lane has the places k with 2 k < n - odd.
  // A place that is not taken adds nothing to its counter and looks up the term of the count 0, which is taken off again at the
  // end (`past` of them).  16-bit counters count in steps of 8, so that a count is its term's place.  watch: true if a counter
  // has overflowed (into its neighbour's bits).
  constexpr uint32_t kOne = kBits == 16 ? 8u : 1u;
  // Only a lane whose sum is stored has a say in that: a variable past the last one counts all of a category in one place, and so
  // does one before u where u has a copy there.  What such a lane's overflow leaves stays in its own column, its sum is given up.
  const int v = block * kMiBlock + (lane & 31);
  const bool stored = v >= u && v < g.V;
  int past = 0;
  auto count = [&](const uint32_t (&d)[kMiHalf], int n, auto watch) {
    uint32_t most = 0u;
    auto places = [&](auto number, auto whole) {
      constexpr int kPlaces = decltype(number)::value;
      constexpr bool kWhole = decltype(whole)::value;
      const int left = n - odd;
      uint32_t old[kPlaces];
#pragma unroll
      for (int k = 0; k < kPlaces; ++k)
        old[k] = __hip_atomic_fetch_add((word_at)(uintptr_t)((d[k] & rows) | own), (kWhole || 2 * k < left ? kOne : 0u) << (d[k] & 31u),
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      double x[kPlaces];
#pragma unroll
      for (int k = 0; k < kPlaces; ++k) {
        const uint32_t c = __builtin_amdgcn_ubfe(old[k], d[k], kWhole || 2 * k < left ? kBits : 0);
        if (decltype(watch)::value) most = max(most, c);
        x[k] = *(term_at)(uintptr_t)(c * (8u / kOne));
      }
      double even = 0.0;
#pragma unroll
      for (int k = 0; k < kPlaces; k += 2) { even += x[k]; acc += x[k + 1]; }
      acc += even;
      if (!kWhole) past += kPlaces - ((left + 1) >> 1);
    };
    if (n == kMiChunk) places(std::integral_constant<int, kMiHalf>{}, std::true_type{});
    else if (n > kMiChunk / 2) places(std::integral_constant<int, kMiHalf>{}, std::false_type{});
    else if (n > kMiChunk / 4) places(std::integral_constant<int, kMiHalf / 2>{}, std::false_type{});
    else places(std::integral_constant<int, kMiHalf / 4>{}, std::false_type{});
    return decltype(watch)::value && __any(stored && most >= (1u << kBits) - 1u);
  };
  auto wipe = [&](const uint32_t (&d)[kMiHalf]) {   // (the places past the chunk's examples hold another's, whose word is zero)
#pragma unroll
    for (int k = 0; k < kMiHalf; ++k) *(word_at)(uintptr_t)((d[k] & rows) | own) = 0u;
  };
  // A category whose counts do exceed them, from chunk c on; returns the chunk behind it.  16-bit counters, with more than 128
  // categories over half of v's categories at a time.
  auto many = [&](int c) {
    int end = c;
    for (int half = 0; half < (kBits == 8 ? 2 : 1); ++half) {
      end = c;
      uint32_t next[2][kMiHalf], l = list(end);
      uint32_t flags = flags_of(l);
      request(l, next[0]);
      l = list(end + 1);
      auto chunk = [&](uint32_t (&d)[kMiHalf], uint32_t (&ahead)[kMiHalf]) {
        const uint32_t next_flags = flags_of(l);
        request(l, ahead);
        l = list(++end + 1);
        const int left = (int)(flags & 31u) + 1 - odd;
        uint32_t old[kMiHalf], most = 0u;
        bool in[kMiHalf];
#pragma unroll
        for (int k = 0; k < kMiHalf; ++k) {
          const uint32_t row = kBits == 8 ? ((d[k] >> 6) & 0x7eu) | ((d[k] >> 4) & 1u) : d[k] >> 7;   // two categories a word
          const uint32_t sh = kBits == 8 ? (d[k] << 1) & 16u : d[k] & 31u;
          in[k] = 2 * k < left && (kBits == 16 || (int)(row >> 6) == half);
          old[k] = __hip_atomic_fetch_add((word_at)(uintptr_t)(((row & 63u) << 7) | own), (in[k] ? 1u : 0u) << sh, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WORKGROUP);
          d[k] = sh;
        }
#pragma unroll
        for (int k = 0; k < kMiHalf; ++k) {
          old[k] = in[k] ? __builtin_amdgcn_ubfe(old[k], d[k], 16) : 0u;
          most = max(most, old[k]);
        }
        double x[kMiHalf];
        if (most >= (uint32_t)g.table) {   // (counts past the terms in LDS)
#pragma unroll
          for (int k = 0; k < kMiHalf; ++k) x[k] = (double)g.dg[old[k]];
        } else {
#pragma unroll
          for (int k = 0; k < kMiHalf; ++k) x[k] = term(old[k]);
        }
#pragma unroll
        for (int k = 0; k < kMiHalf; ++k) acc += in[k] ? x[k] : 0.0;
        const bool more = !(flags & kMiLast);
        flags = next_flags;
        return more;
      };
      while (chunk(next[0], next[1]) && chunk(next[1], next[0])) {
      }
      sweep(kBits == 8 ? g.wave_bytes : row_bytes);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): no load of this path is waited for on the other one
    return end;
  };
  for (int c = c0; c < c1;) {
    // the list two chunks ahead, the examples one
    uint32_t r[2][kMiHalf], l = list(c);
    uint32_t flags = flags_of(l);
    if (kBits == 16 && (flags & kMiMany)) {
      c = many(c);
      continue;
    }
    request(l, r[0]);
    l = list(c + 1);
    int first = c;   // the category's first chunk, and the sums as they were before it
    double acc0 = acc;
    int past0 = past;
    bool over = false;
    // the chunk in r[i]; false: the one behind goes another way
    auto step = [&](int i) {
      const uint32_t next_flags = flags_of(l);
      request(l, r[1 - i]);
      l = list(c + 2);
#pragma unroll
      for (int j = 0; j < kMiHalf; ++j) asm volatile("" : "+v"(r[i][j]));   // (nothing made of them before: it would wait for them)
      const int n = (int)(flags & 31u) + 1;
      if (kBits == 8 && (flags & kMiMany)) {
        // more than 255 examples, which seldom means a count of more: taken for granted, and looked at
        over = count(r[i], n, std::true_type{});
        if (over) return false;
      } else {
        count(r[i], n, std::false_type{});
      }
      if (flags & kMiLast) {
        if (first == c) wipe(r[i]);
        else sweep(row_bytes);
        first = c + 1;
        acc0 = acc;
        past0 = past;
      }
      flags = next_flags;
      return ++c < c1 && !(kBits == 16 && (flags & kMiMany));
    };
    while (step(0) && step(1)) {
    }
    if (over) {
      sweep(row_bytes);
      acc = acc0;
      past = past0;
      __builtin_amdgcn_s_waitcnt(0x0f70);
      c = many(first);
    }
  }
  acc -= (double)past * (double)g.dg[0];
  acc += __shfl_xor(acc, 32);   // both halves' examples
  if (odd || !stored) return;
  const long long total = (long long)acc;
  if (g.parts > 1) {
    atomicAdd(g.partial + (size_t)u * (kMiBlock * g.blocks) + v, (unsigned long long)total);
    return;
  }
  const double Z = (double)g.N + (double)g.pc, s = (double)g.pc / ((double)g.C * g.C);
  const double p0 = s / Z, x0 = p0 > 0.0 ? p0 * log(p0) : 0.0;
  const float val = mi_value(total, g.C, p0, x0, MiStat{g.stat[2 * u], g.stat[2 * u + 1]},
                             MiStat{g.stat[2 * v], g.stat[2 * v + 1]});
  g.mi[(size_t)u * g.V + v] = val;
  g.mi[(size_t)v * g.V + u] = val;
}

__global__ __launch_bounds__(256) void mi_clear_kernel(unsigned long long* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// The shares of a pair put together.
__global__ __launch_bounds__(256) void mi_lanes_finish_kernel(MiLanesArgs g) {
  const int v = blockIdx.x * 256 + threadIdx.x, u = blockIdx.y;
  if (v < u || v >= g.V) return;
  const double Z = (double)g.N + (double)g.pc, s = (double)g.pc / ((double)g.C * g.C);
  const double p0 = s / Z, x0 = p0 > 0.0 ? p0 * log(p0) : 0.0;
  const float val = mi_value((long long)g.partial[(size_t)u * (kMiBlock * g.blocks) + v], g.C, p0, x0,
                             MiStat{g.stat[2 * u], g.stat[2 * u + 1]}, MiStat{g.stat[2 * v], g.stat[2 * v + 1]});
  g.mi[(size_t)u * g.V + v] = val;
  g.mi[(size_t)v * g.V + u] = val;
}

// How the pairs of a call go to lanes; items = 0: they go to workgroups.
struct MiLanesPlan {
  int bits, waves, wave_bytes, table, table_bytes, many, parts, blocks, items, per_die;
  int64_t stride;
};

struct MiLanesScratch {
  uint32_t* xt;                  // [blocks][N][32]
  uint32_t* order;               // [V][stride]
  int* begin;                    // [V][parts + 1]
  unsigned long long* partial;   // [V][32 * blocks] if parts > 1
};

static MiLanesPlan mi_lanes_plan(const MiShape& sh) {
  MiLanesPlan p{};
  int dev = 0, cus = 0, max_lds = 0;
  PCM_HIP(hipGetDevice(&dev));
  PCM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  PCM_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  if (sh.N > 65535 || max_lds < 160 * 1024) return p;   // (16-bit counters)
  MiLanesPlan q{};
  q.bits = sh.C > 128 ? 8 : 16;
  const int rows = q.bits == 8 ? ceil_div(sh.C, 4) : ceil_div(sh.C, 2);
  q.wave_bytes = rows > 32 ? 8192 : rows > 16 ? 4096 : 2048;
  q.table_bytes = 32 * 1024;
  q.waves = 16;
  q.table = std::min(sh.N, q.table_bytes / 8);
  q.many = q.bits == 8 ? 255 : q.table;
  q.blocks = ceil_div(sh.V, kMiBlock);
  int64_t rounds = 0, items = 0;   // waves' rounds of a variable with 32 others, workgroups' worth of them
  for (int b = 0; b < q.blocks; ++b) {
    rounds += std::min(sh.V, kMiBlock * (b + 1));
    items += ceil_div(std::min(sh.V, kMiBlock * (b + 1)), q.waves);
  }
  const int64_t slots = (int64_t)cus * q.waves;
  // Two and a half rounds of the device's waves, or one round of few examples; else a category with most of the examples, which
  // stays with one wave, is what the call waits for.  Workgroups -> lanes, ms, smooth images (four fifths black): 784 variables,
  // 256 categories 3.72 -> 2.84 (16.4 -> 14.5) at 16384 examples, 1.66 -> 1.06 (4.4 -> 3.3) at 4000; 128 categories 2.59 -> 2.28 (14.9 ->
  // 9.3) at 16384; 64 categories 2.58 -> 2.17 (15.3 -> 9.4); 600 variables, 256 categories 1.03 -> 0.64 (2.7 -> 1.3) at 4000.
  if (2 * rounds < 5 * slots && !(rounds >= slots && sh.N <= 4096)) return p;
  q.parts = (int)std::max<int64_t>(1, std::min<int64_t>({16, 6 * cus / items, sh.N / 1024}));
  items *= q.parts;
  if (items > (1 << 28)) return p;
  q.items = (int)items;
  q.per_die = ceil_div(q.items, 8);
  q.stride = ((int64_t)sh.N + (int64_t)(kMiChunk - 1) * std::min(sh.N, sh.C) + 2 * kMiChunk + 63) / 64 * 64;
  return q;
}

// pairs' sums that the shares of a pair add to: whole blocks of variables in every row
static size_t mi_lanes_cells(const MiShape& sh, const MiLanesPlan& p) { return (size_t)sh.V * kMiBlock * p.blocks; }

static void mi_lanes_launch(const uint8_t* d_data, int64_t stride_ex, int64_t stride_var, const MiShape& sh, const MiLanesPlan& p,
                            float pseudocount, const MiScratch& w, const MiLanesScratch& b, float* d_mi, hipStream_t stream) {
  const int N = sh.N, V = sh.V, C = sh.C;
  const int64_t cells = (int64_t)mi_lanes_cells(sh, p);
  pcm_stage(d_data, stride_ex, stride_var, nullptr, N, sh.Np, V, C, w.xb, stream);
  hipLaunchKernelGGL(mi_single_kernel, dim3(V), dim3(256), 0, stream, w.xb, N, sh.Np, C, pseudocount, w.stat);
  hipLaunchKernelGGL(mi_table_kernel, dim3(ceil_div(N, 256)), dim3(256), 0, stream, N, C, pseudocount, w.g);
  const dim3 tiles(ceil_div(N, 64), p.blocks);
  auto codes = p.bits == 8 ? &mi_lane_codes_kernel<8> : &mi_lane_codes_kernel<16>;
  hipLaunchKernelGGL(codes, tiles, dim3(256), 0, stream, w.xb, N, sh.Np, V, b.xt);
  hipLaunchKernelGGL(mi_order_kernel, dim3(V), dim3(1024), 0, stream, w.xb, N, sh.Np, C, p.many, p.parts, p.stride, b.order, b.begin);
  if (p.parts > 1) hipLaunchKernelGGL(mi_clear_kernel, dim3(ceil_div(cells, 256)), dim3(256), 0, stream, b.partial, cells);
  const MiLanesArgs g{b.xt, b.order, b.begin, w.g, w.stat, d_mi, b.partial, p.stride, N, V, C,
                      p.parts, p.blocks, p.per_die, p.items, p.table, p.table_bytes, p.wave_bytes, pseudocount};
  const int lds = p.table_bytes + p.waves * p.wave_bytes;
  auto pairs = p.bits == 8 ? &mi_lanes_kernel<8> : &mi_lanes_kernel<16>;
  PCM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(pairs), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(pairs, dim3(8 * p.per_die), dim3(64 * p.waves), lds, stream, g);
  if (p.parts > 1) hipLaunchKernelGGL(mi_lanes_finish_kernel, dim3(ceil_div(V, 256), V), dim3(256), 0, stream, g);
  check_launch_c("pairwise_mi");
}

}  // namespace pcm
