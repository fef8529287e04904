// Chow-Liu structure learning: pairwise mutual information of categorical data on the device; maximum spanning tree (of a
// matrix on the device chow_liu_edges.hip finds it where it is the only one) and rooting on the host.
//
// Reference: src/utils/information.jl:3-95 (pairwise and single marginals with a pseudocount
// spread as pc/C per category and pc/C^2 per cell, normalised by Z = N + pc) and :97-141
//   MI[u,v] = sum_{a,b} ( xlogx(P_uv[a,b]) - xlogy(P_uv[a,b], P_u[a] * P_v[b]) ).
// The tree is what src/structures/hclts.jl:17-18 asks ChowLiuTrees.jl / ProbabilisticCircuits.jl
// for: a maximum spanning tree of MI, directed away from the centre of the tree.
//
// The reference fills a dense [V][V][C][C] table with float atomics and reduces it on the host.
// Here a pair's counters never leave the LDS.  With c(a,b) the count of a cell, s = pc/C^2,
// p(c) = (c + s)/Z, la[u][a] = log P_u[a]:
//   MI[u,v] = sum over non-empty cells of g(c(cell))  -  M_u - M_v  +  C^2 * xlogx(p(0))  -  p(0) * C * (L_u + L_v)
//   g(c) = xlogx(p(c)) - xlogx(p(0)),   M_u = (1/Z) sum_e la[u][x_eu],   L_u = sum_a la[u][a]
// (the empty cells' terms are the closed-form remainder).  The sum telescopes over a cell's examples -- the one that
// raises a count from c to c + 1 brings g(c + 1) - g(c) -- so a pair costs ONE pass over its N examples against a C x C
// table of counters in LDS: an atomic add that returns the old count, and a look-up of its difference; then the table is
// cleared.  Up to 65535 examples the counters are 16 bits wide and the whole table fits; beyond, they are 32 bits wide
// and the table is walked in bands of rows.  Many variables go to another kernel, a pair per two lanes (mi_lanes.hip.hpp).
#include "common.hpp"
#include "chow_liu.hpp"
#include "stage_kernel.hip.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <queue>
#include <type_traits>

namespace pcm {

static void check_launch_c(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail(PCM_ERR_HIP, "launch of %s failed: %s", what, hipGetErrorString(e));
}

// Single marginals of one variable per workgroup: with la[a] = log((count_a + pc/C)/Z),
//   stat[v] = {M_v, L_v}
__global__ __launch_bounds__(256) void mi_single_kernel(const uint8_t* __restrict__ xb, int N, int64_t Np, int C, float pc,
                                                        double* __restrict__ stat) {
  __shared__ unsigned cnt[256];
  __shared__ double red[256];
  const int v = blockIdx.x, t = threadIdx.x;
  cnt[t] = 0u;
  __syncthreads();
  const uint8_t* row = xb + (size_t)v * Np;
  for (int64_t b = t; b < N; b += 256) atomicAdd(&cnt[row[b]], 1u);
  __syncthreads();
  const double Z = (double)N + (double)pc;
  double l = 0.0, m = 0.0;
  if (t < C) {
    const double p = ((double)cnt[t] + (double)pc / C) / Z;
    const double lg = p > 0.0 ? log(p) : -INFINITY;
    l = lg;                                        // -inf if a category is empty and pc = 0: only used with pc > 0
    m = cnt[t] ? (double)cnt[t] * lg / Z : 0.0;
  }
  red[t] = m;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) { if (t < o) red[t] += red[t + o]; __syncthreads(); }
  const double M = red[0];
  __syncthreads();
  red[t] = l;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) { if (t < o) red[t] += red[t + o]; __syncthreads(); }
  if (t == 0) { stat[2 * v] = M; stat[2 * v + 1] = red[0]; }
}

// dg[c] = g(c + 1) - g(c) for c = 0 .. N - 1, g(c) = xlogx(p(c)) - xlogx(p(0)) the term of a cell that holds c examples
// as a fixed-point integer of kMiFrac fractional bits: |g| < 0.37, the terms of a pair's cells are fewer than 2^17 and
// add up in 64 bits, and integer sums do not depend on which thread adds which difference (2^-44 per cell is far below
// the float the sum ends as).
constexpr int kMiFrac = 44;
__global__ void mi_table_kernel(int N, int C, float pc, long long* __restrict__ dg) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const double Z = (double)N + (double)pc, s = (double)pc / ((double)C * C);
  const double p0 = s / Z, x0 = p0 > 0.0 ? p0 * log(p0) : 0.0;
  auto g = [&](int64_t n) {
    if (n == 0) return 0ll;
    const double p = ((double)n + s) / Z;
    return (long long)llrint(ldexp(p * log(p) - x0, kMiFrac));
  };
  dg[c] = g(c + 1) - g(c);
}

constexpr int kMiThreads = 1024;   // per workgroup; half of it where several workgroups share a compute unit (mi_launch)

// Calls fn(a, b) for every example of a pair of staged rows; thread t owns examples 4t .. 4t+3
// (+ 4096 per further round).
template <typename F>
__device__ __forceinline__ void mi_each_example(const uint8_t* __restrict__ xu, const uint8_t* __restrict__ xv, int N, int t,
                                                F&& fn) {
  for (int64_t b4 = 4 * (int64_t)t; b4 < N; b4 += 4 * kMiThreads) {
    const uint32_t wu = *reinterpret_cast<const uint32_t*>(xu + b4), wv = *reinterpret_cast<const uint32_t*>(xv + b4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (b4 + i < N) fn((int)((wu >> (8 * i)) & 0xffu), (int)((wv >> (8 * i)) & 0xffu));
  }
}

// Sum of acc over the workgroup, then the closed-form remainder; one lane writes both halves of the matrix.  su, sv: the
// two variables' constants (M, L), read when the pair began -- read here they kept the whole workgroup waiting for a
// trip to memory.  `red` is the pair's own half of a double buffer: nobody writes it again before two further barriers,
// so what the first wave does here is behind no barrier of its own.
struct MiStat { double m, l; };
template <int kCtrl>
__device__ __forceinline__ long long mi_dpp_add(long long x) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)x, kCtrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), kCtrl, 0xf, 0xf, true);
  return x + (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
// every lane: the sum over its row of 16 lanes (rotations by 8, 4, 2, 1: no trips through the LDS, which the table's
// atomics keep busy)
__device__ __forceinline__ long long mi_row_sum(long long x) {
  return mi_dpp_add<0x121>(mi_dpp_add<0x122>(mi_dpp_add<0x124>(mi_dpp_add<0x128>(x))));
}
__device__ __forceinline__ void mi_leave_sum(long long acc, long long* red, int t) {
  const long long x = mi_row_sum(acc);
  long long sum = 0;
#pragma unroll
  for (int l = 0; l < 64; l += 16)
    sum += (long long)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32) |
                       (unsigned)__builtin_amdgcn_readlane((int)(unsigned)x, l));
  if ((t & 63) == 0) red[t >> 6] = sum;
}
__device__ __forceinline__ float mi_value(long long sum, int C, double p0, double x0, MiStat su, MiStat sv) {
  const double tot = ldexp((double)sum, -kMiFrac);
  double val = tot - su.m - sv.m + (double)C * C * x0;
  if (p0 > 0.0) val -= p0 * C * (su.l + sv.l);
  return (float)val;
}
template <int T>
__device__ __forceinline__ void mi_finish_pair(const long long* red, int t, int u, int v, int V, int C, double p0, double x0,
                                               MiStat su, MiStat sv, float* __restrict__ mi) {
  if (t >= 16) return;
  const long long sum = mi_row_sum(t < T / 64 ? red[t] : 0ll);
  if (t == 0) {
    const float val = mi_value(sum, C, p0, x0, su, sv);
    mi[(size_t)u * V + v] = val;
    mi[(size_t)v * V + u] = val;
  }
}

// Rows u, v of the upper triangle's pairs in row-major order, `stride` pairs on at a time.
struct MiPair { int u, v; };
__device__ __forceinline__ void mi_advance(MiPair& p, int stride, int V) {
  p.v += stride;
  while (p.v >= V && p.u < V) { ++p.u; p.v += p.u - V; }   // (past the end of row u: on into row u + 1, which starts at its own diagonal)
}

// Words per row of the 16-bit table, an odd number: with rows of 128 words (C = 256) a cell's bank was that of its
// column alone, and the columns of images bunch around the middle of the grey scale.
__host__ __device__ constexpr int mi_row_words(int C) { return ((C + 1) / 2) | 1; }

// Pairs (u <= v) in row-major order of the upper triangle, dealt round-robin to persistent workgroups.  At most 65535
// examples: a cell's count fits 16 bits, two cells per LDS word.  A thread keeps the words of its first R rounds of four
// examples in registers (R = 1, 2, 4 or 8: the host picks the smallest that covers the examples), all of them requested
// before the first is used, and the next pair's are requested before this pair's pass: where the table fills the LDS
// nothing else hides the latency of the rows.
// What bounds it is the LDS: per 64 examples one atomic with return and one look-up, at 8.5 cycles each without bank
// conflicts.  `sweep`: the table is cleared by 16-byte stores over all of it, else by a store per example into the
// cells it touched.  3072 variables, 256 categories (4.72 M pairs): 36 -> 20 ms at 4096 examples, 88 -> 55 at 16384,
// 170 -> 87 at 32768 against a pass that counts and one that takes the counts away, rows of 128 words and per-pair
// overheads of 64-bit index arithmetic and shuffles through the LDS.
template <int T, int R>
__global__ __launch_bounds__(T) void mi_pair_kernel(const uint8_t* __restrict__ xb, int N, int Np, int V, int C, float pc,
                                                    const long long* __restrict__ dg, int g_lds, int sweep,
                                                    const double* __restrict__ stat, float* __restrict__ mi) {
  extern __shared__ __align__(16) unsigned cells[];   // rows of 16-bit counters | 2 x 16 sums | the first g_lds entries of dg
  const int t = threadIdx.x;
  const int S = mi_row_words(C), words = (C * S + 3) & ~3;
  long long* red2 = reinterpret_cast<long long*>(cells + words);
  long long* gl = red2 + 2 * (kMiThreads / 64);   // what the LDS has left holds the table over counts from its start: a
  auto clear_all = [&] {                          // look-up is then no trip to memory (counts past it are rare)
    uint4* p = reinterpret_cast<uint4*>(cells);
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    int i = t;
    for (; i + 3 * T < words / 4; i += 4 * T) p[i] = p[i + T] = p[i + 2 * T] = p[i + 3 * T] = zero;
    for (; i < words / 4; i += T) p[i] = zero;
  };
  clear_all();
  for (int i = t; i < g_lds; i += T) gl[i] = dg[i];
  __syncthreads();
  const double Z = (double)N + (double)pc, s = (double)pc / ((double)C * C);
  const double p0 = s / Z, x0 = p0 > 0.0 ? p0 * log(p0) : 0.0;
  uint32_t cu[R], cv[R], nu[R], nv[R];   // words of the pair under way and of the next one
  auto request = [&](const MiPair& p, uint32_t (&wu)[R], uint32_t (&wv)[R]) {
    const uint8_t* xu = xb + (size_t)p.u * Np;
    const uint8_t* xv = xb + (size_t)p.v * Np;
#pragma unroll
    for (int r = 0; r < R; ++r) {   // (past the end of a row: its last word, never counted)
      const unsigned at = (unsigned)min(4 * (t + r * T), Np - 4);
      wu[r] = *reinterpret_cast<const uint32_t*>(xu + at);
      wv[r] = *reinterpret_cast<const uint32_t*>(xv + at);
    }
  };
  MiPair p{0, 0};
  mi_advance(p, blockIdx.x, V);
  if (p.u < V) request(p, cu, cv);
  int half = 0;
  while (p.u < V) {
    const MiStat su{stat[2 * p.u], stat[2 * p.u + 1]}, sv{stat[2 * p.v], stat[2 * p.v + 1]};
    MiPair pn = p;
    mi_advance(pn, gridDim.x, V);
    if (pn.u < V) request(pn, nu, nv);   // on their way while this pair is counted
    long long acc = 0;
    // Four examples at a time: their counts are all on the way back before the first is looked up.  Byte i of the words:
    // row byte_i(u) of the table, word byte_i(v) >> 1 of it, the half by the lowest bit.
    auto at = [&](uint32_t wu, uint32_t wv, int i) {
      const uint32_t a = (wu >> (8 * i)) & 0xffu, col = (i ? wv >> (8 * i - 1) : wv << 1) & 0x1fcu;
      return reinterpret_cast<unsigned*>(reinterpret_cast<char*>(cells) + (__umul24(a, 4 * S) + col));
    };
    auto count = [&](uint32_t wu, uint32_t wv, int n) {
      unsigned old[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t sh = (i ? wv >> (8 * i - 4) : wv << 4) & 16u;
        old[i] = 0u;
        if (i < n) old[i] = (atomicAdd(at(wu, wv, i), 1u << sh) >> sh) & 0xffffu;
      }
      long long d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = gl[min(old[i], (unsigned)(g_lds - 1))];
      // (kept apart from the loads below: a choice between the two tables' pointers becomes one flat load, which holds
      // the LDS and the memory path together)
      asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]));
      if (max(max(old[0], old[1]), max(old[2], old[3])) >= (unsigned)g_lds) {
        long long far[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) far[i] = dg[min(old[i], (unsigned)(N - 1))];
        asm volatile("" : "+v"(far[0]), "+v"(far[1]), "+v"(far[2]), "+v"(far[3]));   // waited for in here: the common path
#pragma unroll                                                                             // waits for no memory
        for (int i = 0; i < 4; ++i)
          if (old[i] >= (unsigned)g_lds) d[i] = far[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < n) acc += d[i];
    };
    auto wipe = [&](uint32_t wu, uint32_t wv, int n) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < n) *at(wu, wv, i) = 0u;
    };
    // fn(word of u, word of v, examples in it) for the thread's words of the pair, whole rounds without a test per example
    auto each_word = [&](auto&& fn) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if ((r + 1) * 4 * T <= N) fn(cu[r], cv[r], 4);
        else if (4 * (t + r * T) < N) fn(cu[r], cv[r], min(4, N - 4 * (t + r * T)));
      }
      const uint8_t* xu = xb + (size_t)p.u * Np;
      const uint8_t* xv = xb + (size_t)p.v * Np;
      for (int b4 = 4 * (t + R * T); b4 < N; b4 += 4 * T)
        fn(*reinterpret_cast<const uint32_t*>(xu + b4), *reinterpret_cast<const uint32_t*>(xv + b4), min(4, N - b4));
    };
    each_word(count);
    mi_leave_sum(acc, red2 + half * (kMiThreads / 64), t);
    __syncthreads();   // every example is counted
    if (sweep) clear_all(); else each_word(wipe);
    __syncthreads();
    mi_finish_pair<T>(red2 + half * (kMiThreads / 64), t, p.u, p.v, V, C, p0, x0, su, sv, mi);
    half ^= 1;
    p = pn;
#pragma unroll
    for (int r = 0; r < R; ++r) { cu[r] = nu[r]; cv[r] = nv[r]; }
  }
}

// The same for any number of examples: 32-bit cells.  A C x C table of them can exceed the LDS, so
// the categories of u are cut into bands of `band` rows and the pass runs once per band over
// the examples whose u-category falls into it.
__global__ __launch_bounds__(kMiThreads) void mi_pair_wide_kernel(const uint8_t* __restrict__ xb, int N, int64_t Np, int V,
                                                                  int C, int band, float pc, const long long* __restrict__ dg,
                                                                  const double* __restrict__ stat, float* __restrict__ mi) {
  extern __shared__ __align__(16) unsigned cells[];   // band rows of (C | 1) counters | 2 x 16 sums
  const int t = threadIdx.x;
  const int S = C | 1, words = (band * S + 3) & ~3;
  long long* red2 = reinterpret_cast<long long*>(cells + words);
  auto clear_all = [&] {
    for (int i = 4 * t; i < words; i += 4 * kMiThreads) *reinterpret_cast<uint4*>(cells + i) = make_uint4(0u, 0u, 0u, 0u);
  };
  clear_all();
  __syncthreads();
  const double Z = (double)N + (double)pc, s = (double)pc / ((double)C * C);
  const double p0 = s / Z, x0 = p0 > 0.0 ? p0 * log(p0) : 0.0;
  int half = 0;
  MiPair p{0, 0};
  for (mi_advance(p, blockIdx.x, V); p.u < V; mi_advance(p, gridDim.x, V)) {
    const int u = p.u, v = p.v;
    const uint8_t* xu = xb + (size_t)u * Np;
    const uint8_t* xv = xb + (size_t)v * Np;
    const MiStat su{stat[2 * u], stat[2 * u + 1]}, sv{stat[2 * v], stat[2 * v + 1]};
    long long acc = 0;
    for (int a0 = 0; a0 < C; a0 += band) {
      mi_each_example(xu, xv, N, t, [&](int a, int b) {
        if ((unsigned)(a - a0) < (unsigned)band) acc += dg[atomicAdd(&cells[(a - a0) * S + b], 1u)];
      });
      if (a0 + band >= C) mi_leave_sum(acc, red2 + half * (kMiThreads / 64), t);
      __syncthreads();
      clear_all();
      __syncthreads();
    }
    mi_finish_pair<kMiThreads>(red2 + half * (kMiThreads / 64), t, u, v, V, C, p0, x0, su, sv, mi);
    half ^= 1;
  }
}

static MiShape mi_check_shape(int64_t n_examples, int num_vars, int num_cats) {
  if (n_examples < 1 || n_examples > 2147483584LL)
    fail(PCM_ERR_ARG, "pairwise MI takes 1..2147483584 examples per call, got %lld", (long long)n_examples);
  if (num_vars < 1) fail(PCM_ERR_SHAPE, "num_vars must be positive, got %d", num_vars);
  if (num_cats < 1 || num_cats > 256) fail(PCM_ERR_SHAPE, "num_cats must be in 1..256 (uint8 data), got %d", num_cats);
  MiShape s;
  s.N = (int)n_examples;
  s.V = num_vars;
  s.C = num_cats;
  s.Np = (n_examples + 63) / 64 * 64;
  return s;
}

MiShape mi_check(const uint8_t* d_data, int64_t n_examples, int num_vars, int num_cats, float pseudocount, const float* d_mi) {
  if (!d_data || !d_mi) fail(PCM_ERR_ARG, "data or output pointer is null");
  const MiShape s = mi_check_shape(n_examples, num_vars, num_cats);
  if (pseudocount < 0.f) fail(PCM_ERR_ARG, "pseudocount must not be negative");
  return s;
}

// Queues staging, marginals, the count table and the pair kernel on `stream`; allocates nothing.
void mi_launch(const uint8_t* d_data, int64_t stride_ex, int64_t stride_var, const MiShape& sh, float pseudocount,
               const MiScratch& w, float* d_mi, hipStream_t stream) {
  const int N = sh.N, V = sh.V, C = sh.C;
  int dev = 0, cus = 0, max_lds = 0;
  PCM_HIP(hipGetDevice(&dev));
  PCM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  PCM_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  const size_t red_bytes = 2 * (kMiThreads / 64) * sizeof(long long);
  const bool narrow = N <= 65535;
  int band = C;
  size_t lds;
  int g_lds = 0;
  if (narrow) {
    lds = ((size_t)(C * mi_row_words(C) + 3) & ~(size_t)3) * 4 + red_bytes;
    // The rest of the LDS -- of a workgroup's share of it -- holds the start of the dg table.  As many workgroups as
    // possible, up to four, share a compute unit, each with table space for the counts to expect (a count past it is a
    // trip to memory): their serial parts overlap (C = 64, 3072 variables, 16384 examples: four of 512 threads 37 ms, two
    // of 1024 45 ms).
    const size_t whole = std::min<size_t>((size_t)max_lds, 160 * 1024);
    const size_t counts = std::min<size_t>((size_t)N, 512 + (size_t)32 * N / ((size_t)C * C));
    size_t share = whole;
    for (int n = 4; n > 1 && share == whole; n /= 2)
      if (lds + counts * sizeof(long long) <= whole / n) share = whole / n;
    g_lds = (int)std::min<size_t>((size_t)N, (share - lds) / sizeof(long long));
    lds += (size_t)g_lds * sizeof(long long);
  } else {
    const size_t budget = std::min<size_t>((size_t)max_lds, 160 * 1024) - red_bytes - 16;
    band = (int)std::min<size_t>((size_t)C, budget / ((size_t)(C | 1) * 4));
    if (band < 1) fail(PCM_ERR_UNSUPPORTED, "one row of the pair table does not fit %d bytes of LDS", max_lds);
    band = ceil_div(C, ceil_div(C, band));         // equal bands
    lds = ((size_t)(band * (C | 1) + 3) & ~(size_t)3) * 4 + red_bytes;
  }
  if (lds > (size_t)max_lds) fail(PCM_ERR_UNSUPPORTED, "pair table needs %zu bytes of LDS, device offers %d", lds, max_lds);
  pcm_stage(d_data, stride_ex, stride_var, nullptr, N, sh.Np, V, C, w.xb, stream);
  hipLaunchKernelGGL(mi_single_kernel, dim3(V), dim3(256), 0, stream, w.xb, N, sh.Np, C, pseudocount, w.stat);
  hipLaunchKernelGGL(mi_table_kernel, dim3(ceil_div(N, 256)), dim3(256), 0, stream, N, C, pseudocount, w.g);
  const int64_t n_pairs = (int64_t)V * (V + 1) / 2;
  const int per_cu = std::max<int>(1, (int)(std::min<size_t>((size_t)max_lds, 160 * 1024) / lds));
  const int grid = (int)std::min<int64_t>(n_pairs, (int64_t)cus * std::min(per_cu, 4));
  if (narrow) {
    // clearing the whole table costs what wiping after about this many examples costs: at 64 / 100 / 128 / 256 categories
    // the line is at 790 / 1900 / 3100 / 12400, the two were equal at 500 / 2100 / 4100 / 15500 (700 variables; 256: 1.79 ms
    // wiped, 2.16 swept at 8192, 5.52 and 4.65 at 32768)
    const int sweep = (int64_t)N * 8 > (int64_t)C * mi_row_words(C) * 3 ? 1 : 0;
    const bool small = per_cu > 1;
    auto pairs = [&](auto kernel, int threads) {
      PCM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, stream, w.xb, N, (int)sh.Np, V, C, pseudocount, w.g, g_lds, sweep,
                         w.stat, d_mi);
    };
    // rounds of 4 examples a thread whose words it keeps in registers
    auto by_rounds = [&](auto t) {
      constexpr int T = decltype(t)::value;
      if (N <= 4 * T) pairs(&mi_pair_kernel<T, 1>, T);
      else if (N <= 8 * T) pairs(&mi_pair_kernel<T, 2>, T);
      else if (N <= 16 * T) pairs(&mi_pair_kernel<T, 4>, T);
      else pairs(&mi_pair_kernel<T, 8>, T);
    };
    if (small) by_rounds(std::integral_constant<int, kMiThreads / 2>{});
    else by_rounds(std::integral_constant<int, kMiThreads>{});
  } else {
    PCM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&mi_pair_wide_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(mi_pair_wide_kernel, dim3(grid), dim3(kMiThreads), lds, stream, w.xb, N, sh.Np, V, C, band,
                       pseudocount, w.g, w.stat, d_mi);
  }
  check_launch_c("pairwise_mi");
}

}  // namespace pcm
#include "mi_lanes.hip.hpp"
namespace pcm {

namespace {
// The device memory of a call, in one allocation: each costs more than a small call's kernels.
struct MiMemory {
  size_t xb, stat, terms, xt, order, begin, partial;   // offsets; the last four only where lanes take the pairs
  size_t bytes = 0;
  MiMemory(const MiShape& sh, const MiLanesPlan& p) {
    auto take = [&](size_t n) { const size_t at = bytes; bytes += (n + 255) & ~(size_t)255; return at; };
    xb = take((size_t)sh.V * sh.Np);
    stat = take((size_t)2 * sh.V * sizeof(double));
    terms = take(((size_t)sh.N + 1) * sizeof(long long));
    xt = order = begin = partial = bytes;
    if (!p.items) return;
    xt = take((size_t)p.blocks * sh.N * kMiBlock * sizeof(uint32_t));
    order = take((size_t)sh.V * p.stride * sizeof(uint32_t));
    begin = take((size_t)sh.V * (p.parts + 1) * sizeof(int));
    partial = take(p.parts > 1 ? mi_lanes_cells(sh, p) * sizeof(unsigned long long) : 0);
  }
};
}  // namespace

void pairwise_mi(const uint8_t* d_data, int64_t stride_ex, int64_t stride_var, int64_t n_examples, int num_vars,
                 int num_cats, float pseudocount, float* d_mi, hipStream_t stream) {
  const MiShape sh = mi_check(d_data, n_examples, num_vars, num_cats, pseudocount, d_mi);
  MiLanesPlan p = mi_lanes_plan(sh);
  DevBuf<uint8_t> scratch;
  if (p.items) {
    try {
      scratch.alloc(MiMemory(sh, p).bytes);
    } catch (const Error&) {   // a device that is nearly full: the pairs go to workgroups, whose lists of examples are the data
      (void)hipGetLastError();
      p = MiLanesPlan{};
    }
  }
  const MiMemory m(sh, p);
  if (!p.items) scratch.alloc(m.bytes);
  const MiScratch w{scratch.p + m.xb, reinterpret_cast<double*>(scratch.p + m.stat), reinterpret_cast<long long*>(scratch.p + m.terms)};
  if (p.items)
    mi_lanes_launch(d_data, stride_ex, stride_var, sh, p, pseudocount, w,
                    MiLanesScratch{reinterpret_cast<uint32_t*>(scratch.p + m.xt), reinterpret_cast<uint32_t*>(scratch.p + m.order),
                                   reinterpret_cast<int*>(scratch.p + m.begin),
                                   reinterpret_cast<unsigned long long*>(scratch.p + m.partial)},
                    d_mi, stream);
  else
    mi_launch(d_data, stride_ex, stride_var, sh, pseudocount, w, d_mi, stream);
  PCM_HIP(hipStreamSynchronize(stream));   // the scratch array dies with this call
}

void pairwise_mi_plan(int64_t n_examples, int num_vars, int num_cats, int64_t* plan) {
  if (!plan) fail(PCM_ERR_ARG, "plan pointer is null");
  const MiShape sh = mi_check_shape(n_examples, num_vars, num_cats);
  const MiLanesPlan p = mi_lanes_plan(sh);
  plan[0] = p.items ? 2 : 0;
  plan[1] = p.items ? p.parts : 1;
  plan[2] = (int64_t)MiMemory(sh, p).bytes;
}

// One vertex of Prim's algorithm: its row's better links, and the largest of the vertices still outside (those inside
// hold +inf in `best`, which no row beats, and are capped at -inf in `key`, the comparison).  Eight vertices at a time.
using f8 = float __attribute__((ext_vector_type(8)));
using i8 = int32_t __attribute__((ext_vector_type(8)));
static float prim_take_row(const float* row, int32_t pick, int V, float* best, int32_t* link, const float* cap, float* key) {
  f8 top = -INFINITY;
  int v = 0;
  for (; v + 8 <= V; v += 8) {
    f8 r, b, c;
    i8 l;
    std::memcpy(&r, row + v, sizeof r);
    std::memcpy(&b, best + v, sizeof b);
    std::memcpy(&c, cap + v, sizeof c);
    std::memcpy(&l, link + v, sizeof l);
    const i8 better = r > b;
    b = better ? r : b;
    l = better ? (i8)pick : l;
    const f8 k = b < c ? b : c;
    top = k > top ? k : top;
    std::memcpy(best + v, &b, sizeof b);
    std::memcpy(link + v, &l, sizeof l);
    std::memcpy(key + v, &k, sizeof k);
  }
  float most = -INFINITY;
  for (int q = 0; q < 8; ++q) most = std::max(most, top[q]);
  for (; v < V; ++v) {
    if (row[v] > best[v]) { best[v] = row[v]; link[v] = pick; }
    key[v] = std::min(best[v], cap[v]);
    most = std::max(most, key[v]);
  }
  return most;
}

// The tree with these links directed away from its lowest-numbered centre (the vertex of least eccentricity).
static void root_at_centre(std::vector<std::vector<int32_t>>& adj, int32_t* parent_out) {
  const int V = (int)adj.size();
  for (auto& a : adj) std::sort(a.begin(), a.end());
  // centre: peel leaves layer by layer; the last one or two vertices are the centres
  std::vector<int> deg(V);
  std::vector<int32_t> layer, next;
  int left = V;
  for (int v = 0; v < V; ++v) { deg[v] = (int)adj[v].size(); if (deg[v] <= 1) layer.push_back(v); }
  while (left > 2) {
    left -= (int)layer.size();
    next.clear();
    for (int32_t v : layer)
      for (int32_t w : adj[v])
        if (--deg[w] == 1) next.push_back(w);
    layer.swap(next);
  }
  const int root = *std::min_element(layer.begin(), layer.end());
  std::fill(parent_out, parent_out + V, -2);
  std::queue<int32_t> q;
  parent_out[root] = -1;
  q.push(root);
  while (!q.empty()) {
    const int32_t v = q.front();
    q.pop();
    for (int32_t w : adj[v])
      if (parent_out[w] == -2) { parent_out[w] = v; q.push(w); }
  }
}

// Maximum spanning tree of a dense symmetric weight matrix (Prim; among equal weights the
// lowest vertex index wins), rooted at the lowest-numbered centre of the tree (the vertex of
// least eccentricity), as a parent array with -1 at the root.
void chow_liu_tree(const float* mi, int V, int32_t* parent_out) {
  if (!mi || !parent_out) fail(PCM_ERR_ARG, "matrix or output pointer is null");
  if (V < 1) fail(PCM_ERR_SHAPE, "num_vars must be positive, got %d", V);
  for (int v = 1; v < V; ++v)   // (the first vertex's links start the tree; a later row's NaN is a link that is not there)
    if (std::isnan(mi[v])) fail(PCM_ERR_ARG, "mutual information matrix holds NaN or -inf in row %d", v);
  std::vector<float> best(V, -INFINITY);
  std::vector<int32_t> link(V, 0);
  std::vector<std::vector<int32_t>> adj(V);
  best[0] = INFINITY;
  std::vector<float> cap(V, INFINITY), key(V);
  cap[0] = -INFINITY;
  int pick = 0;
  for (int it = 1; it < V; ++it) {
    const float most = prim_take_row(mi + (size_t)pick * V, pick, V, best.data(), link.data(), cap.data(), key.data());
    if (!(most > -INFINITY)) fail(PCM_ERR_ARG, "mutual information matrix holds NaN or -inf in row %d",
                                  (int)(std::find(cap.begin(), cap.end(), INFINITY) - cap.begin()));
    pick = (int)(std::find(key.begin(), key.end(), most) - key.begin());
    best[pick] = INFINITY;
    cap[pick] = -INFINITY;
    adj[pick].push_back(link[pick]);
    adj[link[pick]].push_back(pick);
  }
  root_at_centre(adj, parent_out);
}

// The same from the V - 1 edges of a spanning tree.
void chow_liu_root(const int32_t* edges, int V, int32_t* parent_out) {
  if (!edges || !parent_out) fail(PCM_ERR_ARG, "edges or output pointer is null");
  if (V < 1) fail(PCM_ERR_SHAPE, "num_vars must be positive, got %d", V);
  std::vector<std::vector<int32_t>> adj(V);
  std::vector<int32_t> part(V);   // (a cycle or an edge out of range is refused: the peeling below would not end)
  std::iota(part.begin(), part.end(), 0);
  auto find = [&](int32_t v) {
    while (part[v] != v) v = part[v] = part[part[v]];
    return v;
  };
  for (int i = 0; i < V - 1; ++i) {
    const int32_t a = edges[2 * i], b = edges[2 * i + 1];
    if (a < 0 || b < 0 || a >= V || b >= V || find(a) == find(b)) fail(PCM_ERR_ARG, "edge %d (%d, %d) does not belong to a tree", i, a, b);
    part[find(a)] = find(b);
    adj[a].push_back(b);
    adj[b].push_back(a);
  }
  root_at_centre(adj, parent_out);
}

}  // namespace pcm
