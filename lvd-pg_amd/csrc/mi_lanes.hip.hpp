// Pairwise mutual information, a pair per lane: a wave holds one variable u and 64 variables v, takes u's examples sorted
// by category and keeps, for the category under way, one row of counters per lane.
//
// The sum over a pair's cells telescopes over its examples (chow_liu.hip), in any order; sorted by u's category only the
// cells (a, .) of one category a are open at a time: C counters, not C^2.  That is 256 bytes per pair (8-bit counters
// where a category of u has up to 255 examples, 16-bit ones otherwise), so a lane has its pair to itself: its counters
// lie in its own bank (word r of lane l at 256 r + 4 l: an atomic add takes the LDS 4.3 cycles, at random addresses of a
// shared table 7.2, where many examples fall into one cell up to 128), sums need no reduction, and no barrier keeps the
// waves of a workgroup in step.
//
// Per 64 examples: half a request (two examples' rows, 128 bytes each: the staged data lies in blocks of 64 variables, and
// the workgroups of a die work on the same one at a time, 2 MB of 16384 examples: 95 % of the rows come from the L2; a code
// of 16 bits a lane, without the change of halves, kept the data path busy for 16 cycles a request), an atomic add with
// return, a look-up of the count's term (few counts in a wave: 2.5 cycles), 7.5 vector instructions.  A category's counters are
// cleared by a store per example up to 16 examples, else by 8-byte stores over all of them.
//
// 3072 variables, 16384 examples: 256 categories 55 -> 32 ms, 64 categories 37 -> 20, 256 categories with four fifths of the
// examples in one 241 -> 60.  What bounds it is instruction issue: the vector unit is at work for 58 % of the time, the LDS
// for half of it, two waves a SIMD (LDS) wait for one or the other.  Tried: the three steps of a chunk overlapped with its
// neighbours' (35 ms), nine waves a compute unit (35: the SIMD with three of them is the last).
#pragma once

namespace pcm {

constexpr int kMiChunk = 16;       // examples under way in a wave

// An entry of the list of u's examples: 128 * example, and in the first of each chunk of sixteen
//   bits 0..3 examples in the chunk - 1 | 4 the category's last chunk | 5 counts may exceed the short counters | 6 its first chunk
constexpr uint32_t kMiLast = 16u, kMiMany = 32u, kMiFirst = 64u, kMiFlags = 127u;

// What a lane is given per example: byte offset of the counter word's row (256 * row), and in the low bits its shift.
template <int kBits>
__device__ __forceinline__ uint16_t mi_lane_code(int b) {
  return kBits == 8 ? (uint16_t)(((b >> 2) << 8) | ((b & 3) << 3)) : (uint16_t)(((b >> 1) << 8) | ((b & 1) << 4));
}

// xb[V][Np] -> xt[V / 64][N][32], word p of a row: the codes of the block's variables p and p + 32 (zero past V)
template <int kBits>
__global__ __launch_bounds__(256) void mi_lane_codes_kernel(const uint8_t* __restrict__ xb, int N, int64_t Np, int V,
                                                            uint32_t* __restrict__ xt) {
  __shared__ uint8_t t[64][68];   // [variable][example]
  const int e0 = blockIdx.x * 64, v0 = blockIdx.y * 64;
  for (int i = threadIdx.x; i < 64 * 16; i += 256) {
    const int v = i >> 4, q = i & 15;
    uint32_t w = 0u;
    if (v0 + v < V) w = *reinterpret_cast<const uint32_t*>(xb + (size_t)(v0 + v) * Np + e0 + 4 * q);   // (Np: a multiple of 64)
    *reinterpret_cast<uint32_t*>(&t[v][4 * q]) = w;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int e = i >> 5, p = i & 31;
    if (e0 + e >= N) continue;
    const uint32_t lo = mi_lane_code<kBits>(t[p][e]), hi = mi_lane_code<kBits>(t[p + 32][e]);
    xt[((size_t)blockIdx.y * N + e0 + e) * 32 + p] = lo | (hi << 16);
  }
}

// Place of an example in its chunk: the even ones first (one half of a wave's lanes asks for those, the other for the odd ones).
__device__ __forceinline__ int mi_place(int at) {
  return (at & ~(kMiChunk - 1)) | ((at & 1) * (kMiChunk / 2)) | ((at & (kMiChunk - 1)) >> 1);
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
      if (at == 0) w |= kMiFirst;
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
  unsigned long long* partial;   // [V][64 * blocks] where a pair's categories are shared out (parts > 1)
  int64_t stride;
  int N, V, C, parts, blocks, per_die, items, table, table_bytes, wave_bytes;
  float pc;
};

// r[j]: the word at offset `word` of the row whose offset lane kFrom + j of the lane's row of sixteen holds in `at`
template <int kFrom, int... kJ>
__device__ __forceinline__ void mi_request_rows(__amdgpu_buffer_rsrc_t rx, int at, int word, uint32_t (&r)[kMiChunk / 2],
                                                std::integer_sequence<int, kJ...>) {
  ((r[kJ] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
        rx, __builtin_amdgcn_update_dpp(0, at, 0x150 + kFrom + kJ, 0xf, 0xf, true) + word, 0, 0)), ...);
}

template <int kBits, int kMost>
__global__ __launch_bounds__(64 * kMost) void mi_lanes_kernel(MiLanesArgs g) {
  extern __shared__ __align__(16) char mi_lanes_lds[];
  typedef __attribute__((address_space(3))) uint32_t* word_at;
  typedef __attribute__((address_space(3))) double* term_at;
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) u2* pair_at;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  // the workgroups of a die (consecutive ones go round the eight dies) take consecutive items: one block of variables
  int item = (int)(blockIdx.x & 7) * g.per_die + (int)(blockIdx.x >> 3);
  if (item >= g.items) return;
  const int part = item % g.parts;
  item /= g.parts;
  int block = 0, groups;
  for (;; item -= groups, ++block) {
    groups = (min(g.V, 64 * (block + 1)) + waves - 1) / waves;
    if (item < groups) break;
  }
  const int u = item * waves + wave;
  // LDS: terms of the counts 0 .. table - 1 | the waves' counters, each wave's at a multiple of its own size (a power of two)
  for (int i = threadIdx.x; i < g.table; i += blockDim.x) reinterpret_cast<double*>(mi_lanes_lds)[i] = (double)g.dg[i];
  const uint32_t mine = (uint32_t)(g.table_bytes + wave * g.wave_bytes);
  const uint32_t own = mine + 4u * lane;
  auto sweep = [&](int bytes) {   // multiples of 4 KB
    asm volatile("" ::: "memory");
    for (int o = 0; o < bytes; o += 4096)
#pragma unroll
      for (int i = 0; i < 8; ++i) *(pair_at)(uintptr_t)(mine + 8u * lane + o + 512 * i) = u2{0u, 0u};
    asm volatile("" ::: "memory");
  };
  sweep(g.wave_bytes);
  __syncthreads();
  if (u >= min(g.V, 64 * (block + 1))) return;   // (no barrier from here on)
  const int row_bytes = (((kBits == 8 ? (g.C + 3) / 4 : (g.C + 1) / 2) * 256) + 4095) & ~4095;   // at most wave_bytes
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(g.xt) + (size_t)block * g.N * 32, 0, (int)((size_t)g.N * 128), 0x00020000);
  const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(g.order) + (size_t)u * g.stride, 0, (int)(g.stride * 4), 0x00020000);
  const int c0 = g.begin[(size_t)u * (g.parts + 1) + part], c1 = g.begin[(size_t)u * (g.parts + 1) + part + 1];
  double acc = 0.0;   // whole numbers below 2^53: exact in any order
  // The list of chunks c and c + 1: lane i of a row of sixteen lanes holds the entry i & 7 of its half's eight of chunk c + (i >> 3)
  const int list_lane = 4 * ((lane & 7) + 8 * (lane >> 5) + 2 * (lane & 8));
  auto list = [&](int c) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rl, list_lane, min(c, c1 - 1) * (kMiChunk * 4), 0);
  };
  auto flags_of = [&](uint32_t l, auto which) {
    return (uint32_t)__builtin_amdgcn_readlane(l, 8 * decltype(which)::value) & kMiFlags;
  };
  using First = std::integral_constant<int, 0>;    // of a list's two chunks
  using Second = std::integral_constant<int, 1>;
  // Two examples a request: one half of the lanes asks for one's row, the other half for the other's, a word (two codes) a lane
  auto request = [&](uint32_t l, auto which, uint32_t (&r)[kMiChunk / 2]) {
    mi_request_rows<8 * decltype(which)::value>(rx, (int)(l & ~kMiFlags), 4 * (lane & 31), r,
                                                std::make_integer_sequence<int, kMiChunk / 2>{});
  };
  // ... and after a change of halves every lane has both examples' code of its own variable (bits 16 .. 31: anything)
  auto codes = [&](const uint32_t (&r)[kMiChunk / 2], uint32_t (&d)[kMiChunk]) {
#pragma unroll
    for (int j = 0; j < kMiChunk / 2; ++j) {
      const auto s = __builtin_amdgcn_permlane32_swap(r[j], r[j] >> 16, false, false);
      d[2 * j] = s[0];
      d[2 * j + 1] = s[1];
    }
  };
  auto term = [&](uint32_t count) { return *(term_at)(uintptr_t)(count << 3); };
  const uint32_t rows = kBits == 8 || g.wave_bytes == 16384 ? 0x3f00u : (uint32_t)(g.wave_bytes - 256);
  // A chunk's examples whose counts fit the short counters and the terms in LDS.  A place past the chunk's n examples adds
  // nothing to its counter and looks up the term of the count 0, which is taken off again at the end (`past` of them).
  // (16-bit counters count in steps of 8, so that a count is its term's place: up to kMiLanesTerms of them)
  constexpr uint32_t kOne = kBits == 16 ? 8u : 1u;
  int past = 0;
  auto count = [&](const uint32_t (&d)[kMiChunk], int n) {
    auto places = [&](auto number, auto&& one) {
      constexpr int kPlaces = decltype(number)::value;
      uint32_t old[kPlaces];
#pragma unroll
      for (int k = 0; k < kPlaces; ++k)
        old[k] = __hip_atomic_fetch_add((word_at)(uintptr_t)((d[k] & rows) | own), (one(k) * kOne) << (d[k] & 31u),
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      double x[kPlaces];
#pragma unroll
      for (int k = 0; k < kPlaces; ++k)
        x[k] = *(term_at)(uintptr_t)(__builtin_amdgcn_ubfe(old[k], d[k], one(k) * kBits) * (8u / kOne));
      double even = 0.0;
#pragma unroll
      for (int k = 0; k < kPlaces; k += 2) { even += x[k]; acc += x[k + 1]; }
      acc += even;
    };
    if (n == kMiChunk) {
      places(std::integral_constant<int, kMiChunk>{}, [](int) { return 1u; });
    } else {
      const uint32_t taken = (1u << n) - 1u;
      auto one = [&](int k) { return (taken >> k) & 1u; };
      if (n > kMiChunk / 2) { places(std::integral_constant<int, kMiChunk>{}, one); past += kMiChunk - n; }
      else { places(std::integral_constant<int, kMiChunk / 2>{}, one); past += kMiChunk / 2 - n; }
    }
  };
  auto wipe = [&](const uint32_t (&d)[kMiChunk]) {   // (the places past the chunk's examples hold another's, whose word is zero)
#pragma unroll
    for (int k = 0; k < kMiChunk; ++k) *(word_at)(uintptr_t)((d[k] & rows) | own) = 0u;
  };
  // A category with more examples than that, from chunk c on; returns the chunk behind it.  16-bit counters; where they are
  // too many for that, half of the variables at a time: the 32 of the rows' low codes, then those of the high ones, the two
  // halves of the wave taking the even and the odd examples (no change of halves) and both adding to a variable's counters.
  double half_acc[2] = {0.0, 0.0};
  auto many = [&](int c) {
    int end = c;
    auto pass = [&](auto which) {
      constexpr int kHalf = decltype(which)::value;   // -1: all 64 variables
      end = c;
      uint32_t next[2][kMiChunk / 2], l = list(end);
      uint32_t flags = flags_of(l, First{});
      request(l, First{}, next[0]);
      const uint32_t pair = mine + 4u * (lane & 31);
      auto chunk = [&](uint32_t (&r)[kMiChunk / 2], uint32_t (&ahead)[kMiChunk / 2]) {
        const uint32_t next_flags = flags_of(l, Second{});
        request(l, Second{}, ahead);
        l = list(++end);
        constexpr int kPlaces = kHalf < 0 ? kMiChunk : kMiChunk / 2;
        const int n = (int)(flags & 15u) + 1;
        const int left = kHalf < 0 ? n : n - (lane >> 5);   // place k is taken if k (2 k) < left
        uint32_t d[kMiChunk], old[kPlaces], sh[kPlaces];
        if (kHalf < 0) codes(r, d);
        uint32_t most = 0u;
#pragma unroll
        for (int k = 0; k < kPlaces; ++k) {
          const uint32_t w = kHalf < 0 ? d[k] : kHalf ? r[k] >> 16 : r[k];
          const uint32_t at = kHalf < 0 ? (w & rows) | own : ((w & 0x3f00u) | pair) + ((w << 3) & 0x80u);
          sh[k] = kHalf < 0 ? w : w << 1;   // (a shift takes the low five bits, of which bit 4 is left)
          if (kHalf >= 0) sh[k] &= 16u;
          const bool in = kHalf < 0 ? k < left : 2 * k < left;
          old[k] = __hip_atomic_fetch_add((word_at)(uintptr_t)at, (in ? 1u : 0u) << (sh[k] & 31u), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WORKGROUP);
        }
#pragma unroll
        for (int k = 0; k < kPlaces; ++k) {
          old[k] = __builtin_amdgcn_ubfe(old[k], sh[k], 16);
          most = max(most, old[k]);
        }
        double x[kPlaces];
        if (most >= (uint32_t)g.table) {   // (counts past the terms in LDS)
#pragma unroll
          for (int k = 0; k < kPlaces; ++k) x[k] = (double)g.dg[old[k]];
        } else {
#pragma unroll
          for (int k = 0; k < kPlaces; ++k) x[k] = term(old[k]);
        }
        double& to = kHalf < 0 ? acc : half_acc[kHalf < 0 ? 0 : kHalf];
        if (n == kMiChunk) {
#pragma unroll
          for (int k = 0; k < kPlaces; ++k) to += x[k];
        } else {
#pragma unroll
          for (int k = 0; k < kPlaces; ++k) to += (kHalf < 0 ? k < left : 2 * k < left) ? x[k] : 0.0;
        }
        const bool more = !(flags & kMiLast);
        flags = next_flags;
        return more;
      };
      while (chunk(next[0], next[1]) && chunk(next[1], next[0])) {
      }
      sweep(kBits == 8 ? g.wave_bytes : row_bytes);
    };
    if constexpr (kBits == 8) {
      pass(std::integral_constant<int, 0>{});
      pass(std::integral_constant<int, 1>{});
    } else {
      pass(std::integral_constant<int, -1>{});
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): no load of this path is waited for on the other one
    return end;
  };
  for (int c = c0; c < c1;) {
    // the list two chunks ahead, the examples one
    uint32_t r[2][kMiChunk / 2], l = list(c);
    uint32_t flags = flags_of(l, First{});
    if (flags & kMiMany) {
      c = many(c);
      continue;
    }
    request(l, First{}, r[0]);
    // the chunk in r[i]; `from`, `which`: the list and the half of it that hold the one behind.  False: no chunk of the same
    // kind follows
    auto step = [&](int i, uint32_t from, auto which) {
      const uint32_t next_flags = flags_of(from, which);
      request(from, which, r[1 - i]);
#pragma unroll
      for (int j = 0; j < kMiChunk / 2; ++j) asm volatile("" : "+v"(r[i][j]));   // (nothing made of them before: it would wait for them)
      uint32_t d[kMiChunk];
      codes(r[i], d);
      count(d, (int)(flags & 15u) + 1);
      if (flags & kMiLast) {
        if (flags & kMiFirst) wipe(d);
        else sweep(row_bytes);
      }
      flags = next_flags;
      return ++c < c1 && !(flags & kMiMany);
    };
    while (true) {
      const uint32_t ahead = list(c + 2);
      if (!step(0, l, Second{}) || !step(1, ahead, First{})) break;
      l = ahead;
    }
  }
  if constexpr (kBits == 8) {   // lane v: its low (v < 32) or high sums of both halves of the wave
    const uint2 lo = __builtin_bit_cast(uint2, half_acc[0]), hi = __builtin_bit_cast(uint2, half_acc[1]);
    const auto x = __builtin_amdgcn_permlane32_swap(lo.x, hi.x, false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(lo.y, hi.y, false, false);
    acc += __builtin_bit_cast(double, make_uint2(x[0], y[0])) + __builtin_bit_cast(double, make_uint2(x[1], y[1]));
  }
  const long long total = (long long)acc - (long long)past * g.dg[0];
  const int v = block * 64 + lane;
  if (v < u || v >= g.V) return;
  if (g.parts > 1) {
    atomicAdd(g.partial + (size_t)u * (64 * g.blocks) + v, (unsigned long long)total);
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
  const float val = mi_value((long long)g.partial[(size_t)u * (64 * g.blocks) + v], g.C, p0, x0,
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
  unsigned long long* partial;   // [V][64 * blocks] if parts > 1
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
  q.wave_bytes = rows > 32 ? 16384 : rows > 16 ? 8192 : 4096;
  q.table_bytes = 32 * 1024;
  q.waves = q.wave_bytes == 16384 ? 8 : 16;
  q.table = std::min(sh.N, q.table_bytes / 8);
  q.many = q.bits == 8 ? 255 : q.table;
  q.blocks = ceil_div(sh.V, 64);
  int64_t rounds = 0, items = 0;   // waves' rounds of a variable with 64 others, workgroups' worth of them
  for (int b = 0; b < q.blocks; ++b) {
    rounds += std::min(sh.V, 64 * (b + 1));
    items += ceil_div(std::min(sh.V, 64 * (b + 1)), q.waves);
  }
  const int64_t slots = (int64_t)cus * q.waves;
  // Two and a half rounds of the device's waves (three with 65 .. 128 categories, whose waves are as few as 256's but whose
  // pairs cost a workgroup less), or one round of few examples; else a category with most of the examples, which stays with one wave, is what the
  // call waits for.  Workgroups -> lanes, ms, smooth images (four fifths black): 784 variables, 256 categories 3.72 -> 3.38
  // (16.4 -> 10.3) at 16384 examples, 1.66 -> 1.00 at 4000; 600 variables 2.29 -> 2.42 at 16384, 1.03 -> 0.73 at 4000; 784
  // variables, 128 categories 2.59 -> 2.67 at 16384; 784 variables, 64 categories 2.58 -> 2.28 (15.3 -> 16.7); 200 variables
  // 0.12 -> 0.22 at 4000.
  const int least = q.bits == 16 && q.waves == 8 ? 6 : 5;
  if (2 * rounds < least * slots && !(rounds >= slots && sh.N <= 4096)) return p;
  q.parts = (int)std::max<int64_t>(1, std::min<int64_t>({16, 6 * cus / items, sh.N / 1024}));
  items *= q.parts;
  if (items > (1 << 28)) return p;
  q.items = (int)items;
  q.per_die = ceil_div(q.items, 8);
  q.stride = ((int64_t)sh.N + (int64_t)(kMiChunk - 1) * std::min(sh.N, sh.C) + 2 * kMiChunk + 63) / 64 * 64;
  return q;
}

static void mi_lanes_launch(const uint8_t* d_data, int64_t stride_ex, int64_t stride_var, const MiShape& sh, const MiLanesPlan& p,
                            float pseudocount, const MiScratch& w, const MiLanesScratch& b, float* d_mi, hipStream_t stream) {
  const int N = sh.N, V = sh.V, C = sh.C;
  const int64_t cells = (int64_t)V * 64 * p.blocks;
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
  auto pairs = p.bits == 8 ? &mi_lanes_kernel<8, 8> : p.waves == 8 ? &mi_lanes_kernel<16, 8> : &mi_lanes_kernel<16, 16>;
  PCM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(pairs), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(pairs, dim3(8 * p.per_die), dim3(64 * p.waves), lds, stream, g);
  if (p.parts > 1) hipLaunchKernelGGL(mi_lanes_finish_kernel, dim3(ceil_div(V, 256), V), dim3(256), 0, stream, g);
  check_launch_c("pairwise_mi");
}

}  // namespace pcm
