// Lean tree-walk kernels: the same slice-persistent forward / backward walks as in
// hclt_kernels.hip.hpp, for the common case (no tile ever leaves LDS, at most three children
// per tree node, every array below 2 GiB), written for the fewest instructions per step.
//
// Why a second pair of kernels.  With one 16-example tile per wave and step, a step is only
// ~100 useful vector instructions (8 exp, 8 log, 16 MFMA, a few adds), and four waves share a
// SIMD: measured on gfx950 the general walk kernels are bound by instruction issue, not by
// memory -- their schedule decoding and 64-bit address arithmetic cost more instructions
// than the arithmetic.  Here
//   * every array is addressed through ONE buffer descriptor built before the loop; a node's
//     byte offset comes precomputed from the schedule and goes into the instruction's scalar
//     offset, the lane part is a per-thread constant, the tile row an immediate;
//   * operands are typed by position (own leaf row, own value tile, up to three children), so
//     an absent operand is a scalar branch around its loads and its adds -- nothing is
//     zero-filled, selected or copied;
//   * the parameter block is requested right after the contraction that used its
//     predecessor, into the same registers, so nothing rotates between steps.
//   * a wave follows a chain of the tree (lean_schedule.hpp): the tile of its last node is in registers when the next one
//     needs it, and four tiles in five go through no LDS slot, no wait and no post;
//   * idle steps only keep the requests going.
// What bounds a step (forward walk with pieces left out, 784 variables, K = 32, 512 examples, 53 steps, then 97 us): all its
// memory requests without the arithmetic 95 us, all the arithmetic without the requests 84, neither 33.  The fp32 matrix
// instructions of a SIMD's four waves (4 x 512 cycles) and their vector instructions (4 x 600) add up, as both use the same
// units; the requests of a compute unit (140 KB a step) do so beside them.
#pragma once

#include "hclt_kernels.hip.hpp"
#include "lean_rows.hpp"

namespace pcm {

constexpr int kLeanFlagWords = 256;        // one state word per LDS slot, behind the slots
constexpr int kLeanSpinLimit = 1 << 22;    // polls before a wave gives up on a tile (never reached by a sound schedule)

constexpr int kLeanChunk = 60;   // steps per refill (even): 64 lanes minus what the last two steps look ahead

struct LeanChunk {
  int v[kLeanFields];
  int base;
};

__device__ __forceinline__ void lean_refill(const int32_t* __restrict__ fields, int stride, int wave, int lane, int base,
                                            LeanChunk& c) {
#pragma unroll
  for (int f = 0; f < kLeanFields; ++f) c.v[f] = fields[((size_t)f * kWalkWaves + wave) * stride + base + lane];
  // the rows are used as landed from here on: no step waits for them (a step's own waits
  // then count only the requests of the steps)
#pragma unroll
  for (int f = 0; f < kLeanFields; ++f) asm volatile("" : "+v"(c.v[f]));
  c.base = base;
}

__device__ __forceinline__ int lean_get(const LeanChunk& c, int field, int step) {
  return __builtin_amdgcn_readlane(c.v[field], step - c.base);
}

template <int K>
__device__ __forceinline__ void lean_row_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, Tile<K>& t) {
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
    t.v[kt] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(voff + kt * 64), soff, 0));
}

template <int K>
__device__ __forceinline__ void lean_tile_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, Tile<K>& t) {
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
    t.v[kt] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(voff + kt * 1024), soff, kStreamLoad));
}

template <int K>
__device__ __forceinline__ void lean_tile_store(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, const Tile<K>& t) {
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, t.v[kt]), r, (int)(voff + kt * 1024), soff, kStreamStore);
}

template <int K>
__device__ __forceinline__ void lean_w_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, WTile<K>& w) {
#pragma unroll
  for (int i = 0; i < (K / 16) * (K / 16); ++i)
    w.a[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(voff + (i & 3) * 1024), soff + (i >> 2) * 4096, 0));
}

// The same where the block may be absent (-1: idle steps; going down, nodes without inner children): the requests go out
// all the same, past the end of the array, where the buffer unit answers with zeros and fetches nothing.  Behind a branch
// they would cost more than they save: the compiler counts the requests in flight for the shorter way, so the wait for
// the next step's rows would also wait for this block, two steps early.
constexpr uint32_t kLeanNowhere = 0x80000000u;   // (every array is shorter: lean_array_fits)
template <int K>
__device__ __forceinline__ void lean_w_load_if(__amdgpu_buffer_rsrc_t r, uint32_t vtile, int soff, WTile<K>& w) {
  lean_w_load<K>(r, soff < 0 ? kLeanNowhere + vtile : vtile, max(soff, 0), w);
}

// Places the requests of the block of code it stands in between the block's matrix instructions: three reads (words, rows) and
// the first half of the next parameter block behind every second one, the other half as its registers are through.  A wave
// that issues a matrix instruction waits for the one before; these slots are free.  (K = 32; a K = 16 contraction is four
// instructions.)  632 nodes in four parts, 512 examples, forward: 96 -> 91 us.  The same in the backward walk, whose requests
// would then stand in three branches, loses: the compiler no longer knows how many are in flight where they join (75 -> 118).
template <int K>
__device__ __forceinline__ void lean_between() {
  if constexpr (K == 32) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // matrix instructions
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // reads
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
  }
}

// byte offset of this lane's part of leaf row x (byte `sel` of the packed word)
template <int K>
__device__ __forceinline__ uint32_t lean_row_off(uint32_t xpack, int sel, uint32_t vleaf) {
  return ((xpack >> (8 * sel)) & 0xffu) * (K * 4) + vleaf;
}

// Waits until the slot's state word reads `want`.  The walks have no barrier between steps: a wave goes on as
// soon as the tiles it needs are there, and hands its own tile on by advancing the slot's state.  Every wait is
// for a tile of an earlier step of the host's schedule, and every wave works through its steps in order, so the
// earliest unfinished step can always proceed.  The wait is bounded all the same: a wave that runs out of polls
// raises *err and carries on, so the kernel ends whatever the schedule holds.
__device__ __forceinline__ void lean_wait(const unsigned* state, unsigned want, const HcltDev& d) {
  int polls = 0;
  while (__builtin_amdgcn_readfirstlane(
             (int)__hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != (int)want) {
    if (++polls > kLeanSpinLimit) {
      if ((threadIdx.x & 63) == 0) {
        __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(d.err_dev, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Advances a slot's state once everything this wave did to the slot's tile before is in LDS order (a wave's
// LDS accesses execute in the order they were issued; the fence keeps the compiler to that order too).
__device__ __forceinline__ void lean_post(unsigned* state, unsigned value) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __hip_atomic_store(state, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---- a tree over several workgroups ----------------------------------------------------------
// A batch of few slices leaves most compute units idle while one of them per slice walks the whole tree.  So a single tree
// is also scheduled in 2, 4, 8 .. parts (lean_parts), blockIdx.y of the walk: the top of the tree and, dealt to the parts,
// the subtrees below it.  A tile that crosses goes through memory, once on the way up or down, with a flag per (tile, slice)
// that its one reader puts back to zero, so that a launch leaves the flags as it found them (also one that a graph replays).
// The data is written and read with device-scope accesses of its own, which pass the L2s of the eight dies; a release or
// acquire fence would write back or drop a whole L2 each time.  Only the top waits going up, only the others going down,
// and whoever is waited for comes first in the grid.  Workgroups go to the dies in turn and are dispatched in order within a
// die, so the grid's first dimension is a multiple of their number: the parts of a slice are then on one die, and a
// workgroup never holds a compute unit while the one it waits for still queues behind another stream's.  The waits are
// bounded like those for LDS tiles.  3072 variables, K = 32, 512 examples: forward 322 -> 156 us, backward 368 -> 171 in
// eight parts; 1024 examples 322 -> 173 and 394 -> 221 in four; 784 variables, 512 examples: 105 -> 70 and 107 -> 76.
struct LeanAway {
  float* tiles;        // [tile][slice][16 * K]
  unsigned* flags;     // [tile][slice]
  double* sums;        // [part][Bp] a part's share of the log-likelihood
  unsigned* sum_flags; // [part][slice]
};

__device__ __forceinline__ void away_wait(unsigned* flag, const HcltDev& d) {
  int polls = 0;
  while (__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 1) {
    if (++polls > kLeanSpinLimit) {
      if ((threadIdx.x & 63) == 0) {
        __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(d.err_dev, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      break;
    }
    __builtin_amdgcn_s_sleep(2);
  }
  asm volatile("" ::: "memory");   // (what the flag announces is read behind this)
}

// everything this wave has written or read so far is through before the flag changes
__device__ __forceinline__ void away_flag(unsigned* flag, unsigned value) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if ((threadIdx.x & 63) == 0) __hip_atomic_store(flag, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr int kDeviceScope = 16;   // (sc1)
template <int K>
__device__ __forceinline__ void away_put(const LeanAway& x, const HcltDev& d, int tile, int slice, uint32_t vtile, const Tile<K>& t) {
  const int at = tile * d.nslices + slice;
  const __amdgpu_buffer_rsrc_t r = make_rsrc(x.tiles + (size_t)at * (kSlice * K), kSlice * K * 4);
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, t.v[kt]), r, (int)(vtile + kt * 1024), 0, kDeviceScope);
  away_flag(x.flags + at, 1u);
}

template <int K>
__device__ __forceinline__ void away_get(const LeanAway& x, const HcltDev& d, int tile, int slice, uint32_t vtile, Tile<K>& t) {
  const int at = tile * d.nslices + slice;
  const __amdgpu_buffer_rsrc_t r = make_rsrc(x.tiles + (size_t)at * (kSlice * K), kSlice * K * 4);
  away_wait(x.flags + at, d);
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
    t.v[kt] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(vtile + kt * 1024), 0, kDeviceScope));
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt) asm volatile("" : "+v"(t.v[kt]));   // (waited for here, not where the ways join)
  away_flag(x.flags + at, 0u);
}

// ---- forward ------------------------------------------------------------------------------
// A node's value is kept in two parts: the tile holds O'_v[k] = log S_v[k] = log sum_j W[k,j] exp(Z'_v[j] - m_v), numbers
// of order one, and the row of maxima holds m_v = max_j Z'_v[j], where Z'_v is the sum of the node's leaf rows and of its
// inner children's TILES (not of their full values).  The full value is O'_v[k] plus the maxima of all nodes of the
// subtree, a number that grows with the size of the subtree and is the same for all K states: nothing below needs it
// but the log-likelihood at the root.  Stored as one float32 it would cost every state of a 3000-variable circuit
// (values near -14000) an absolute error of 1e-3, which is a relative error of 1e-3 on every flow; in two parts the
// flows keep float32's relative accuracy at any depth.
//
// The lowest bit of a stored maximum is not part of the number: m is rounded to an even last place before anything is scaled
// by it (any number near the maximum does), and the bit says that some example of the slice has a state of probability zero
// (a value of -inf) at this node.  A node with one inner child then needs that child's tile on the way down only where the
// bit is set: its ratio tile is made of the OTHER operands, and of its own values only "is it zero" counts.
__device__ __forceinline__ float lean_scale(float m) { return __builtin_bit_cast(float, __builtin_bit_cast(int, m) & ~1); }
template <int K>
__device__ __forceinline__ float lean_mark(float m, const Tile<K>& o) {
  float least = o.v[0][0];
#pragma unroll
  for (int kt = 0; kt < K / 16; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) least = fminf(least, o.v[kt][i]);
  return __builtin_bit_cast(float, __builtin_bit_cast(int, m) | (__ballot(least == -INFINITY) != 0ull ? 1 : 0));
}

// kKeep: what the walk leaves in memory.  kKeepAll: every node's tile and row of maxima, for the passes behind it;
// kKeepRoots: the maxima and the roots' tiles, what the head kernel of a multi-head circuit reads; kKeepNone: nothing
// but the log-likelihoods: a scoring pass has nobody behind it, and value stores are 512 of a step's 1340 requests.
// 10300 examples of 3072 variables (K = 32), which no longer need tile arrays and so go through 4096 at a time
// whatever the caller's batch size: 3.93 ms in batches of 1000 -> 1.08 ms.
//
// Measured (us; the schedule that picked the sixteen most urgent nodes of every step anew and put a tile per node through LDS /
// chains in registers / and requests that never wait for a store, two steps ahead, waves that leave when they are through):
// 784 variables, 512 examples 111 / 97 / 70, 192 variables 55 / 42 / 37, 64 variables (K = 16) 19 / 16.5 / 13; 3072 variables
// at 512 examples (in parts) 336 / 194 / 141, at 4096, where the stores of the tiles count, 390 / 384 / 372.
//
// kRows: the packed categories come from the caller's rows, each workgroup packing its slice's into LDS before it starts
// (small trees, scores of small batches: the kernel in front that packs them took a quarter as long as the walk; 64 variables,
// K = 16, 100 examples 14.6 -> 11.1 us).
struct LeanRows {
  const int4* vars;   // per inner node: its own variable and its first three leaf children (-1: none)
  const uint8_t* data;
  int64_t stride_ex, stride_var;
  const int32_t* idx;
};
// Most inner nodes of a tree whose categories a workgroup packs and keeps, 64 bytes each (0: never).  What packing takes grows with the
// nodes, a lookup per variable and example; the kernel in front takes 5 us whatever they are.  At K = 16 steps are short and
// the categories out of LDS shorten them: 64 / 171 / 225 nodes, 200 examples 24.7 -> 19.2 / 77.9 -> 61.1 / 94.1 -> 75.1 us.  At K = 32
// they do not: 72 / 93 / 115 / 130 / 219 nodes 46.1 -> 45.1 / 59.1 -> 58.1 / 64.8 -> 64.5 / 72.7 -> 73.0 / 116.4 -> 118.2.  (All lookups of a
// thread requested at once, those of missing children too: 119.3; a lane's lookups are a cache line each.)
constexpr int lean_row_nodes(int K) { return K == 16 ? 256 : K == 32 ? 112 : 0; }

template <int K, int kKeep, bool kRows>
__global__ __launch_bounds__(kWalkWaves * 64) void hclt_forward_lean_kernel(
    HcltDev d, const int32_t* __restrict__ fields, int stride, float* __restrict__ ll_out, int n_slots, LeanAway away, LeanRows rows) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slice = blockIdx.x;
  if (slice >= d.nslices) return;   // (the grid of a tree in parts is rounded up)
  unsigned* state = reinterpret_cast<unsigned*>(lds + (size_t)n_slots * (kSlice * K));
  for (int i = threadIdx.x; i < kLeanFlagWords; i += blockDim.x) state[i] = 0u;
  uint32_t* const xs = state + kLeanFlagWords;   // kRows: [n_inner + 1][16 examples], behind the state words
  if constexpr (kRows) {
    const int b = slice * kSlice + (int)(threadIdx.x & 15);
    const uint8_t* row = rows.data + (b < d.B ? (int64_t)(rows.idx ? rows.idx[b] : b) * rows.stride_ex : 0);
    auto category = [&](int var) -> uint32_t {
      return var >= 0 && b < d.B ? min((uint32_t)row[var * rows.stride_var], (uint32_t)(d.C - 1)) : 0u;   // (in range whatever the caller sent)
    };
    for (int n = threadIdx.x >> 4; n <= d.n_inner; n += kWalkWaves * 4) {
      const int4 v = n < d.n_inner ? rows.vars[n] : make_int4(-1, -1, -1, -1);
      xs[n * kSlice + (threadIdx.x & 15)] = category(v.x) | category(v.y) << 8 | category(v.z) << 16 | category(v.w) << 24;
    }
  }
  __syncthreads();
  const uint32_t vtile = (uint32_t)lane * 16, vleaf = (uint32_t)(lane >> 4) * 16, vx = (uint32_t)(lane & 15) * 4;
  const int bcol = slice * kSlice + (lane & 15);
  const uint32_t slice_bytes = (uint32_t)slice * (kSlice * K * 4);
  const __amdgpu_buffer_rsrc_t rO =   // (kKeepNone: the arrays may not exist, and nothing is stored)
      make_rsrc(reinterpret_cast<const char*>(d.O) + slice_bytes, (uint32_t)(d.n_inner + 1) * d.tile_stride - slice_bytes);
  const __amdgpu_buffer_rsrc_t rW = make_rsrc(d.Wf, (uint32_t)d.n_inner * (K * K * 4));
  const __amdgpu_buffer_rsrc_t rL = make_rsrc(d.leaf, (uint32_t)d.V * d.leaf_stride);
  const __amdgpu_buffer_rsrc_t rX =
      make_rsrc(d.xn + (size_t)slice * kSlice, (uint32_t)d.n_inner * (uint32_t)d.Bp * 4u - (uint32_t)slice * (kSlice * 4));
  const int xrow = d.Bp * 4;
  // the row maxima M[node][example] go out beside the value tiles: the backward walk and the statistics
  // kernel scale by exactly these numbers (lanes 16..63 hold copies: their stores fall outside the buffer)
  const __amdgpu_buffer_rsrc_t rM =
      make_rsrc(d.M + (size_t)slice * kSlice, (uint32_t)(d.n_inner + 1) * (uint32_t)d.Bp * 4u - (uint32_t)slice * (kSlice * 4));
  const uint32_t vm = lane < 16 ? vx : 0x70000000u;   // (past the end with kLeanNowhere added, too)

  fields += (size_t)blockIdx.y * (kLeanFields * kWalkWaves * (size_t)stride + kWalkWaves);   // groups of trees, parts: a schedule each
  const int n_steps = __builtin_amdgcn_readfirstlane(fields[(size_t)kLeanFields * kWalkWaves * stride + wave]);
  LeanChunk sc;
  lean_refill(fields, stride, wave, lane, 0, sc);
  // What is in flight: a node's own leaf rows and its parameter block are requested two steps ahead, into the registers of
  // the step that has just used them (so there are two sets, of the even and the odd steps), the rows of its leaf children
  // one step ahead, the categories three.
  Tile<K> PA, PB, P1, P2;   // (a third leaf child is rare: its rows are fetched at the point of use)
  WTile<K> wA, wB;
  uint32_t x0, x1, x2;  // packed categories of this step, of the next and of the one after
  int a1, a2, a3;       // leaf children of the step whose operands are in flight
  auto load_x = [&](int s) {
    if constexpr (kRows) return xs[lean_get(sc, kLNode, s) * kSlice + (lane & 15)];
    else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rX, (int)vx, lean_get(sc, kLNode, s) * xrow, 0);
  };
  {
    x0 = load_x(0);
    x1 = load_x(1);
    x2 = load_x(2);
    lean_row_load<K>(rL, lean_row_off<K>(x0, 0, vleaf), lean_get(sc, kLA0, 0), PA);
    a1 = lean_get(sc, kLA1, 0); a2 = lean_get(sc, kLA2, 0); a3 = lean_get(sc, kLA3, 0);
    if (a1 >= 0) lean_row_load<K>(rL, lean_row_off<K>(x0, 1, vleaf), a1, P1);
    if (a2 >= 0) lean_row_load<K>(rL, lean_row_off<K>(x0, 2, vleaf), a2, P2);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, 0), wA);
    __builtin_amdgcn_sched_barrier(0);   // (in this order: the waits inside the loop are counted for both ways into it)
    lean_row_load<K>(rL, lean_row_off<K>(x1, 0, vleaf), lean_get(sc, kLA0, 1), PB);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, 1), wB);
    __builtin_amdgcn_sched_barrier(0);
  }
  float ll = 0.f;
  bool root_here = false;
  double msum = 0.0;   // sum of the row maxima of this wave's nodes: the part of the log-likelihood the tiles leave out
  Tile<K> o;           // the value tile of this wave's last node: its parent takes it from here if it comes next in the wave
  tile_zero<K>(o);
  // what of it is to be stored, in the step after (kLeanNowhere: nothing)
  uint32_t keep_o = kLeanNowhere, keep_m = kLeanNowhere;
  int o_at = 0, m_at = 0;
  float m_prev = 0.f;

  // A step sends its requests whatever it does, those with nothing to fetch or to store past the end of their array: the wait
  // for one is then for a known number of requests behind it, and none is waited for less than a step after it went out.
  auto ahead = [&](const int s, WTile<K>& w, Tile<K>& P) {
    const uint32_t x3 = load_x(s + 3);
    lean_row_load<K>(rL, lean_row_off<K>(x2, 0, vleaf), lean_get(sc, kLA0, s + 2), P);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, s + 2), w);
    x0 = x1;
    x1 = x2;
    x2 = x3;
  };
  auto step = [&](const int s, WTile<K>& w, Tile<K>& P) {
    // (1) the leaf rows of this step have landed
    Tile<K> z = P;
    if (a1 >= 0) {
      tile_add<K>(z, P1);
      if (a2 >= 0) tile_add<K>(z, P2);
      if (a3 >= 0) {
        Tile<K> t;
        lean_row_load<K>(rL, lean_row_off<K>(x0, 3, vleaf), a3, t);
        tile_add<K>(z, t);
#pragma unroll
        for (int kt = 0; kt < K / 16; ++kt) asm volatile("" : "+v"(z.v[kt]));   // (waited for here, not where the ways join)
      }
    }
    // (2) request the rows of the next step's leaf children, the node's own of the step after, the categories of the third;
    // the previous step's tile goes out
    a1 = lean_get(sc, kLA1, s + 1);
    if (a1 >= 0) {
      a2 = lean_get(sc, kLA2, s + 1); a3 = lean_get(sc, kLA3, s + 1);
      lean_row_load<K>(rL, lean_row_off<K>(x1, 1, vleaf), a1, P1);
      if (a2 >= 0) lean_row_load<K>(rL, lean_row_off<K>(x1, 2, vleaf), a2, P2);
    }
    if (kKeep != kKeepNone) {
      lean_tile_store<K>(rO, keep_o + vtile, o_at, o);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, m_prev), rM, (int)(keep_m + vm), m_at, kStreamStore);
      keep_o = keep_m = kLeanNowhere;
    }
    const int node = lean_get(sc, kLNode, s);
    if (node != d.n_inner) {   // (idle steps only keep the requests going)
      // (3) inner children, from LDS or, the one this wave computed last, from registers; logsumexp through the matrix cores
      const uint32_t slots = (uint32_t)lean_get(sc, kLSlots, s), turns = (uint32_t)lean_get(sc, kLTurns, s);
      if ((slots >> 8) == (0xffff00u | kLeanKept)) {   // (most nodes: one inner child, and this wave has it)
        tile_add<K>(z, o);
      } else {
        int next_away = lean_get(sc, kLAway, s);
#pragma unroll
        for (int c = 1; c <= 3; ++c) {
          const uint32_t sl = (slots >> (8 * c)) & 0xffu, tn = (turns >> (8 * c)) & 0x7fu;
          if (sl == 0xffu) break;
          if (sl == kLeanKept) {
            tile_add<K>(z, o);
          } else if (sl == kLeanAway) {
            Tile<K> t;
            away_get<K>(away, d, next_away++, slice, vtile, t);
            tile_add<K>(z, t);
          } else {
            lean_wait(state + sl, (2 * tn + 1) & 0xffu, d);
            Tile<K> t;
            lds_tile_load<K>(lds, (int)sl, lane, t);
            tile_add<K>(z, t);
            lean_post(state + sl, (2 * tn + 2) & 0xffu);   // read: the slot may take its next tile
          }
        }
      }
      const float m = lean_scale(tile_rowmax<K>(z));
      tile_exp_sub<K>(z, m);
      // the requests go out between the matrix instructions, which leave the wave's issue slots free
      contract<K>(w, z, o);
      ahead(s, w, P);
      lean_between<K>();
#pragma unroll
      for (int kt = 0; kt < K / 16; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o.v[kt][i] = __builtin_amdgcn_logf(o.v[kt][i]) * kLn2;
      // hand the tile on (the root's, and one whose reader is this wave's next node, go nowhere)
      const uint32_t so = slots & 0xffu;
      if (so <= kLeanAway) {
        const uint32_t tn = turns & 0x7fu;
        if (so == kLeanAway) {
          away_put<K>(away, d, lean_get(sc, kLAway, s), slice, vtile, o);
        } else {
          lean_wait(state + so, (2 * tn) & 0xffu, d);
          lds_tile_store<K>(lds, (int)so, lane, o);
          lean_post(state + so, (2 * tn + 1) & 0xffu);
        }
      }
      msum += (double)m;
      const bool root = (turns & 0x80u) != 0;
      if (root) {
        ll = o.v[0][0];
        root_here = true;
      }
      if (kKeep == kKeepAll || (kKeep == kKeepRoots && root)) keep_o = 0;
      if (kKeep != kKeepNone) {
        keep_m = 0;
        m_prev = lean_mark<K>(m, o);
      }
      o_at = (int)((uint32_t)node * d.tile_stride);
      m_at = node * xrow;
    } else {
      ahead(s, w, P);
    }
  };
  // The schedule is consumed in chunks of kLeanChunk steps (a chunk's registers also serve the
  // two steps of look-ahead past its end), two steps per trip: the parameter blocks alternate
  // between two register sets, each reloaded two steps ahead right after its use.  An odd
  // step count runs one idle step of the padding.
  for (int base = 0; base < n_steps; base += kLeanChunk) {
    if (base) lean_refill(fields, stride, wave, lane, base, sc);
    const int s_end = min(base + kLeanChunk, n_steps);
    for (int s = base; s < s_end; s += 2) {
      step(s, wA, PA);
      step(s + 1, wB, PB);
    }
  }
  if (kKeep != kKeepNone) {
    lean_tile_store<K>(rO, keep_o + vtile, o_at, o);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, m_prev), rM, (int)(keep_m + vm), m_at, kStreamStore);
  }
  // log-likelihood of a single-root circuit: the root's (scaled) value plus the row maxima of all nodes, the
  // waves' sums added in wave order (a multi-head circuit's head kernel adds up the stored maxima per tree)
  if (!ll_out) return;
  __syncthreads();   // every wave is through its steps: the slots are free
  double* part = reinterpret_cast<double*>(lds);
  float* top = lds + 2 * kWalkWaves * 16;
  if (lane < 16) {
    part[wave * 16 + lane] = msum;
    if (root_here) top[lane] = ll;
  }
  __syncthreads();
  if (wave == 0) {
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < kWalkWaves; ++w) tot += part[w * 16 + (lane & 15)];
    // (a tree over several workgroups: the top, which comes last, adds up the shares of the others in order)
    const int last = (int)gridDim.y - 1;
    if ((int)blockIdx.y < last) {
      if (lane < 16) __hip_atomic_store(away.sums + (size_t)blockIdx.y * d.Bp + bcol, tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      away_flag(away.sum_flags + (size_t)blockIdx.y * d.nslices + slice, 1u);
    } else {
      for (int g = 0; g < last; ++g) {
        unsigned* flag = away.sum_flags + (size_t)g * d.nslices + slice;
        away_wait(flag, d);
        tot += __hip_atomic_load(away.sums + (size_t)g * d.Bp + bcol, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        away_flag(flag, 0u);
      }
      if (lane < 16 && bcol < d.B) ll_out[bcol] = (float)(tot + (double)top[lane]);
    }
  }
}

// ---- backward -----------------------------------------------------------------------------
// What travels down the tree through LDS is not the flow of a child's sum nodes but already their
// ratio tile R_c = F_c / S_c, built by the parent: with t = W_v^T R_v, F_c = G_v = exp(Z'_v - m_v) .* t
// and S_c = exp(O'_c) (the tiles hold log S, see the forward walk),
//   R_c[j] = t[j] * exp((Z'_v[j] - O'_c[j]) - m_v),
// where Z'_v - O'_c is the sum of v's OTHER operands (own leaf row, leaf children, further inner
// children's tiles): the child's own values cancel, so a node never reads its own value tile, and the
// exponent is formed from small numbers.  m_v are the row maxima the forward walk stored.  A state the
// child gives probability zero (O'_c = -inf) has flow 0 and keeps ratio 0.  A node without inner children
// only stores its tile.
// kHeads: multi-head circuit, whose head kernel has left the root's ratio tile in memory.
// Measured as above: 192 variables at 4096 examples 77 / 53 / 43 us, 784 at 4096 184 / 170 / 151, at 512 125 / 107 / 75; 3072
// at 4096 625 / 625 / 572 (the tiles of only children, 0.8 of 1.3 GB of the value tiles, are no longer read).
template <int K, bool kHeads>
__global__ __launch_bounds__(kWalkWaves * 64) void hclt_backward_lean_kernel(
    HcltDev d, const int32_t* __restrict__ fields, int stride, int n_slots, LeanAway away) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slice = blockIdx.x;
  if (slice >= d.nslices) return;   // (the grid of a tree in parts is rounded up)
  unsigned* state = reinterpret_cast<unsigned*>(lds + (size_t)n_slots * (kSlice * K));
  for (int i = threadIdx.x; i < kLeanFlagWords; i += blockDim.x) state[i] = 0u;
  __syncthreads();
  const uint32_t vtile = (uint32_t)lane * 16, vleaf = (uint32_t)(lane >> 4) * 16, vx = (uint32_t)(lane & 15) * 4;
  const int bcol = slice * kSlice + (lane & 15);
  const uint32_t slice_bytes = (uint32_t)slice * (kSlice * K * 4);
  const uint32_t arr_bytes = (uint32_t)(d.n_inner + 1) * d.tile_stride - slice_bytes;
  const __amdgpu_buffer_rsrc_t rO = make_rsrc(reinterpret_cast<const char*>(d.O) + slice_bytes, arr_bytes);
  const __amdgpu_buffer_rsrc_t rR = make_rsrc(reinterpret_cast<const char*>(d.R) + slice_bytes, arr_bytes);
  const __amdgpu_buffer_rsrc_t rW = make_rsrc(d.Wb, (uint32_t)d.n_inner * (K * K * 4));
  const __amdgpu_buffer_rsrc_t rL = make_rsrc(d.leaf, (uint32_t)d.V * d.leaf_stride);
  const __amdgpu_buffer_rsrc_t rX =
      make_rsrc(d.xn + (size_t)slice * kSlice, (uint32_t)d.n_inner * (uint32_t)d.Bp * 4u - (uint32_t)slice * (kSlice * 4));
  const __amdgpu_buffer_rsrc_t rM =
      make_rsrc(d.M + (size_t)slice * kSlice, (uint32_t)(d.n_inner + 1) * (uint32_t)d.Bp * 4u - (uint32_t)slice * (kSlice * 4));
  const int xrow = d.Bp * 4;

  // a child operand: value tile of an inner child, or leaf row of a leaf child
  auto child_load = [&](int c, uint32_t xpack, Tile<K>& t) {
    if (c & 1) lean_row_load<K>(rL, lean_row_off<K>(xpack, (c >> 1) & 3, vleaf), c & ~7, t);
    else lean_tile_load<K>(rO, vtile, (c >> 3) * (int)d.tile_stride, t);
  };
  auto is_inner = [](int c) { return c >= 0 && !(c & 1); };

  fields += (size_t)blockIdx.y * (kLeanFields * kWalkWaves * (size_t)stride + kWalkWaves);   // groups of trees, parts: a schedule each
  const int n_steps = __builtin_amdgcn_readfirstlane(fields[(size_t)kLeanFields * kWalkWaves * stride + wave]);
  LeanChunk sc;
  lean_refill(fields, stride, wave, lane, 0, sc);
  // in flight: a node's own leaf rows, row maxima and parameter block two steps ahead, its children's operands one, the
  // categories three (see the forward walk)
  Tile<K> PA, PB, C1, C2, C3;
  WTile<K> wA, wB;
  uint32_t x1, x2;
  int c1, c2, c3;
  float m0, m1;   // row maxima of this step and of the next, as stored
  auto load_x = [&](int s) { return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rX, (int)vx, lean_get(sc, kLNode, s) * xrow, 0); };
  auto load_m = [&](int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rM, (int)vx, lean_get(sc, kLNode, s) * xrow, 0));
  };
  auto load_children = [&](int s, uint32_t xpack) {
    c1 = lean_get(sc, kLA1, s); c2 = lean_get(sc, kLA2, s); c3 = lean_get(sc, kLA3, s);
    if (c1 >= 0) {
      if ((c1 & 3) != 2) child_load(c1, xpack, C1);
      if (c2 >= 0) child_load(c2, xpack, C2);
      if (c3 >= 0) child_load(c3, xpack, C3);
    }
  };
  {
    const uint32_t x0 = load_x(0);
    x1 = load_x(1);
    x2 = load_x(2);
    m0 = load_m(0);
    m1 = load_m(1);
    lean_row_load<K>(rL, lean_row_off<K>(x0, 0, vleaf), lean_get(sc, kLA0, 0), PA);
    load_children(0, x0);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, 0), wA);
    __builtin_amdgcn_sched_barrier(0);   // (in this order: the waits inside the loop are counted for both ways into it)
    lean_row_load<K>(rL, lean_row_off<K>(x1, 0, vleaf), lean_get(sc, kLA0, 1), PB);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, 1), wB);
    __builtin_amdgcn_sched_barrier(0);
  }
  Tile<K> r;   // the ratio tile of the node under way; behind a step, that of its first child, which comes next in this wave (or is away)
  tile_zero<K>(r);

  auto step = [&](const int s, WTile<K>& w, Tile<K>& P) {
    // (1) from the landed operands: what an inner child's ratio tile is made of besides t, exp of the other operands minus
    // m_v, zero where the child's own value is -inf.  The inner children come first; the first's factors stay in registers,
    // a second's and third's wait in the LDS slots their ratio tiles will take.
    const int node = lean_get(sc, kLNode, s);
    const bool in1 = is_inner(c1), in2 = is_inner(c2), in3 = is_inner(c3), alone = (c1 & 3) == 2 && in1;
    const int own1 = c1;
    const uint32_t slots = (uint32_t)lean_get(sc, kLSlots, s), turns = (uint32_t)lean_get(sc, kLTurns, s);
    const float dm = -lean_scale(m0) * kLog2e;
    auto factor = [&](bool check, const Tile<K>& own, bool has_a, const Tile<K>& a, bool has_b, const Tile<K>& b, Tile<K>& x) {
      Tile<K> rest = P;
      if (has_a) tile_add<K>(rest, a);
      if (has_b) tile_add<K>(rest, b);
#pragma unroll
      for (int kt = 0; kt < K / 16; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = fminf(__builtin_amdgcn_exp2f(fmaf(rest.v[kt][i], kLog2e, dm)), kFlowRatioCap);
          x.v[kt][i] = check && own.v[kt][i] == -INFINITY ? 0.f : e;
        }
    };
    Tile<K> X1;
    if (in1) {
      if (alone) factor(false, C1, c2 >= 0, C2, c3 >= 0, C3, X1);
      else factor(true, C1, c2 >= 0, C2, c3 >= 0, C3, X1);
    }
    if (in2) {   // the children's slots are this wave's from here (scratch first, their ratio tiles at the end)
      Tile<K> x;
      factor(true, C2, true, C1, c3 >= 0, C3, x);
      lean_wait(state + ((slots >> 16) & 0xffu), (2 * ((turns >> 16) & 0x7fu)) & 0xffu, d);
      lds_tile_store<K>(lds, (int)((slots >> 16) & 0xffu), lane, x);
      if (in3) {
        factor(true, C3, true, C1, true, C2, x);
        lean_wait(state + ((slots >> 24) & 0xffu), (2 * ((turns >> 24) & 0x7fu)) & 0xffu, d);
        lds_tile_store<K>(lds, (int)((slots >> 24) & 0xffu), lane, x);
      }
    }
    // (2) requests: the operands of the next step's children, own rows and maxima of the step after, categories of the third
    load_children(s + 1, x1);
    {
      const uint32_t x3 = load_x(s + 3);
      m0 = m1;
      m1 = load_m(s + 2);
      lean_row_load<K>(rL, lean_row_off<K>(x2, 0, vleaf), lean_get(sc, kLA0, s + 2), P);
      x1 = x2;
      x2 = x3;
    }
    if (node != d.n_inner) {   // (idle steps only keep the requests going)
      // (3) this node's ratio tile: in registers from the step before, or left in LDS by the parent
      const uint32_t so = slots & 0xffu;
      if (so != kLeanKept) {
        if (so == kLeanAway) {
          away_get<K>(away, d, lean_get(sc, kLAway, s), slice, vtile, r);
        } else if (so < kLeanAway) {
          lean_wait(state + so, (2 * (turns & 0x7fu) + 1) & 0xffu, d);
          lds_tile_load<K>(lds, (int)so, lane, r);
          lean_post(state + so, (2 * (turns & 0x7fu) + 2) & 0xffu);
        } else if (kHeads) {   // a root of a multi-head circuit: the head kernel has left its ratio tile in memory
          lean_tile_load<K>(rR, vtile, node * (int)d.tile_stride, r);
#pragma unroll
          for (int kt = 0; kt < K / 16; ++kt) asm volatile("" : "+v"(r.v[kt]));   // (waited for here, not where the ways join)
        } else {   // flow 1 into the single root sum node of every live example: R = 1 / S = exp(-O')
          const float o00 = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(rO, (int)vtile, node * (int)d.tile_stride, 0));
          const bool live = lane < 16 && bcol < d.B;
          const float wgt = (d.w && live) ? d.w[bcol] : 1.f;   // per-example weights: the flow the example starts with
          float r00 = live ? wgt * fminf(__builtin_amdgcn_exp2f(o00 * -kLog2e), kFlowRatioCap) : 0.f;
          asm volatile("" : "+v"(r00));
          tile_zero<K>(r);
          r.v[0][0] = r00;
        }
      }
      lean_tile_store<K>(rR, vtile, node * (int)d.tile_stride, r);
      // (4) the inner children's ratio tiles; the first child is this wave's next node
      if (in1) {
        Tile<K> t;
        contract<K>(w, r, t);
        // (alone: the child comes next, so m0 is its row of maxima by now, with the mark of a state of probability zero)
        if (alone && (__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, m0)) & 1)) {
          Tile<K> own;
          lean_tile_load<K>(rO, vtile, (own1 >> 3) * (int)d.tile_stride, own);
#pragma unroll
          for (int kt = 0; kt < K / 16; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) X1.v[kt][i] = own.v[kt][i] == -INFINITY ? 0.f : X1.v[kt][i];
#pragma unroll
          for (int kt = 0; kt < K / 16; ++kt) asm volatile("" : "+v"(X1.v[kt]));
        }
        auto ratio = [&](const Tile<K>& x, Tile<K>& rc) {
#pragma unroll
          for (int kt = 0; kt < K / 16; ++kt) rc.v[kt] = t.v[kt] * x.v[kt];
        };
        const bool first_away = (turns & 0x8000u) != 0;
        if (in2) {
          int next_away = lean_get(sc, kLAway, s) + (first_away ? 1 : 0);
          auto hand_on = [&](int c) {
            const uint32_t sl = (slots >> (8 * c)) & 0xffu;
            Tile<K> x;
            lds_tile_load<K>(lds, (int)sl, lane, x);
            ratio(x, x);
            if ((turns >> (8 * c)) & 0x80u) {   // away: the slot was only to work in
              away_put<K>(away, d, next_away++, slice, vtile, x);
              lean_post(state + sl, (2 * ((turns >> (8 * c)) & 0x7fu) + 2) & 0xffu);
            } else {
              lds_tile_store<K>(lds, (int)sl, lane, x);
              lean_post(state + sl, (2 * ((turns >> (8 * c)) & 0x7fu) + 1) & 0xffu);
            }
          };
          hand_on(2);
          if (in3) hand_on(3);
        }
        ratio(X1, r);
        if (first_away) away_put<K>(away, d, lean_get(sc, kLAway, s), slice, vtile, r);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    lean_w_load_if<K>(rW, vtile, lean_get(sc, kLW, s + 2), w);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int base = 0; base < n_steps; base += kLeanChunk) {
    if (base) lean_refill(fields, stride, wave, lane, base, sc);
    const int s_end = min(base + kLeanChunk, n_steps);
    for (int s = base; s < s_end; s += 2) {
      step(s, wA, PA);
      step(s + 1, wB, PB);
    }
  }
}

// ---- statistics -----------------------------------------------------------------------------
// Same job as hclt_stats_kernel (a workgroup takes a tree node over all slices; edge flows summed
// over the batch with the matrix cores, leaf histograms with integer LDS atomics), for nodes
// with at most three children, written like the lean walks: one descriptor per array, a node's
// byte offsets as scalars, typed operands behind scalar branches, every register reloaded right
// after its last use, the waves' partial edge-flow blocks combined by a plain LDS sum.  The LDS
// holds up to `nh_pass` histograms (two where they fit: a node's own variable and its first leaf
// child then need one pass over the batch).  Pass 0 does all the arithmetic; a node with more
// variables than that leaves the child-flow tiles G where it read R from, and further passes
// re-read G only.
//
// The workgroups are persistent: one per compute unit, each working through nodes it claims from a
// counter in memory (the first two by its index), and a wave's stream of slices runs on from one
// node into the next: in its last two slices of a node the requests it sends ahead are the first
// operands of the next node, so that they land while the histograms are written out and the
// partial blocks are combined.  A node that needs several passes, and a batch of fewer than
// 32 slices, ends the stream: the node after it starts with requests of its own.
//
// LDS layouts, both without padding so that two histograms of 256 x 32 cells and sixteen pads fill
// 160 KB exactly: histogram cell (category x, state j) sits in word x*K + (j ^ (x % K)) of its limb
// (equal states of different categories spread over the banks); a wave's 16 x K transposition pad
// rotates row r by 8*r floats (column reads of four rows then cover every bank twice).  The
// histogram area is all zero whenever a node begins: whoever reads a cell out clears it.
constexpr int kStatLeanWaves = 16;

// A node's scalars as the statistics kernel uses them.
struct StatRef {
  int node;          // the node's index
  int tile_off;      // byte offset of the node's tiles in the value and ratio arrays
  int x_off;         // ... of its row of packed categories (and of row maxima)
  int leaf_off;      // ... of its own variable's leaf table
  int w_off;         // ... of its parameter block
  int c1, c2, c3;    // children as in StatNode
  int n_hist;
};

__device__ __forceinline__ StatRef stat_ref(const HcltDev& d, const StatNode* __restrict__ nodes, int pos, int kk4) {
  const StatNode* __restrict__ np = nodes + pos;
  const int n = np->node;
  StatRef r;
  r.node = n;
  r.tile_off = n * (int)d.tile_stride;
  r.x_off = n * d.Bp * 4;
  r.leaf_off = np->var * (int)d.leaf_stride;
  r.w_off = n * kk4;
  r.c1 = np->c[0];
  r.c2 = np->c[1];
  r.c3 = np->c[2];
  r.n_hist = np->n_hist;
  return r;
}

// Next node of a workgroup (-1: none left).  Tickets count from the third node of every workgroup; each
// workgroup draws until its first miss, so a launch hands out n_nodes - gridDim.x tickets in all, and whoever
// draws the last one puts the counter back to zero for the next launch.
__device__ __forceinline__ int stat_claim(unsigned* counter, int n_nodes) {
  const unsigned t = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (t + 1u == (unsigned)n_nodes - gridDim.x) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned n = 2u * gridDim.x + t;
  return n < (unsigned)n_nodes ? (int)n : -1;
}

template <int K>
__global__ __launch_bounds__(kStatLeanWaves * 64) void hclt_stats_lean_kernel(
    HcltDev d, const StatNode* __restrict__ nodes, float* __restrict__ edge_aggr, float* __restrict__ leaf_flow,
    float rate, int hist_words, int nh_pass, int limb, const int* __restrict__ flow_shift, unsigned* __restrict__ counter,
    int n_nodes) {
  constexpr int KT = K / 16;
  extern __shared__ float smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = lane & 15, g = lane >> 4;
  const uint32_t vtile = (uint32_t)lane * 16, vleaf = (uint32_t)g * 16, vx = (uint32_t)b * 4;
  const int hist_sz = d.C * K;           // words per limb; a histogram is two limbs
  unsigned* hist = reinterpret_cast<unsigned*>(smem);
  float* pad = smem + hist_words + (size_t)wave * (kSlice * K);
  int* claim_word = reinterpret_cast<int*>(smem + hist_words);   // wave 0's pad, which is idle between two nodes
  // flows lie in [0, 2^shift]: 1 per example in a single-head circuit, the largest total head
  // mask of an example (found on the device by the head kernel) in a multi-head one
  const int shift = flow_shift ? __builtin_amdgcn_readfirstlane(*flow_shift) : 0;
  const float scale = __builtin_ldexpf(1.f, limb), scale_in = __builtin_ldexpf(1.f, limb - shift);
  const float hi_inv = __builtin_ldexpf(1.f, shift - limb), lo_inv = __builtin_ldexpf(1.f, shift - 2 * limb);

  const uint32_t tiles_bytes = (uint32_t)(d.n_inner + 1) * d.tile_stride;
  const __amdgpu_buffer_rsrc_t rR = make_rsrc(d.R, tiles_bytes);
  const __amdgpu_buffer_rsrc_t rO = make_rsrc(d.O, tiles_bytes);
  const __amdgpu_buffer_rsrc_t rL = make_rsrc(d.leaf, (uint32_t)d.V * d.leaf_stride);
  const __amdgpu_buffer_rsrc_t rX = make_rsrc(d.xn, (uint32_t)d.n_inner * (uint32_t)d.Bp * 4u);
  const __amdgpu_buffer_rsrc_t rM = make_rsrc(d.M, (uint32_t)(d.n_inner + 1) * (uint32_t)d.Bp * 4u);   // row maxima of the forward walk
  const __amdgpu_buffer_rsrc_t rW = make_rsrc(d.Wb, (uint32_t)d.n_inner * (K * K * 4));
  auto child_load = [&](int c, uint32_t xpack, int slice_off, Tile<K>& t) {
    if (c & 1) lean_row_load<K>(rL, lean_row_off<K>(xpack, (c >> 1) & 3, vleaf), (c >> 3) * (int)d.leaf_stride, t);
    else lean_tile_load<K>(rO, vtile, (c >> 3) * (int)d.tile_stride + slice_off, t);
  };
  auto load_x = [&](const StatRef& r, int s) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rX, (int)vx, r.x_off + s * (kSlice * 4), 0);
  };
  auto load_m = [&](const StatRef& r, int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rM, (int)vx, r.x_off + s * (kSlice * 4), 0));
  };

  // fixed-point limbs of this lane's K/4 flows (clamped to [0, 2^shift]) into row x of histogram h
  auto histogram = [&](const Tile<K>& t, uint32_t xpack, int sel, int h) {
    const uint32_t x = (xpack >> (8 * sel)) & 0xffu;
    unsigned* hrow = hist + (size_t)h * 2 * hist_sz + x * K;
    const uint32_t sw = x & (K - 1);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = __builtin_amdgcn_fmed3f(t.v[kt][i] * scale_in, 0.f, scale);
        const unsigned hi = (unsigned)v;
        const unsigned lo = (unsigned)(__builtin_amdgcn_fractf(v) * scale);
        const uint32_t col = (uint32_t)(kt * 16 + 4 * g + i) ^ sw;
        __hip_atomic_fetch_add(&hrow[col], hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_add(&hrow[hist_sz + col], lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
  };
  // a pass's histograms out to memory; every cell read is cleared for whoever uses the area next
  auto flush = [&](const StatNode* __restrict__ np, int h0, int nh) {
    for (int h = 0; h < nh; ++h) {
      float* dst = leaf_flow + (size_t)np->hvar[h0 + h] * d.C * K;
      unsigned* hh = hist + (size_t)h * 2 * hist_sz;
      for (int i = threadIdx.x; i < d.C * K; i += blockDim.x) {
        const int c = i / K, j = i % K;
        const int cell = c * K + (j ^ (c & (K - 1)));
        const float val = (float)hh[cell] * hi_inv + (float)hh[hist_sz + cell] * lo_inv;
        hh[cell] = 0u;
        hh[hist_sz + cell] = 0u;
        const float old = rate != 0.f ? rate * dst[i] : 0.f;
        __builtin_nontemporal_store(old + val, &dst[i]);   // read once more, by the update
      }
    }
  };
  // pad positions: this lane's float4 of example row b (states kt*16 + 4g ..), and the element
  // (example 4q + g, state kt*16 + b) of the transposed read
  auto pad_w = [&](int kt) { return b * K + ((kt * 16 + 4 * g + 8 * b) & (K - 1)); };
  auto pad_r = [&](int q, int kt) { return (4 * q + g) * K + ((kt * 16 + b + 8 * g) & (K - 1)); };

  const int last = d.nslices - 1;
  const bool stream_on = d.nslices >= 2 * kStatLeanWaves;   // every wave then has two slices of a node at least
  const int n_it = (d.nslices - wave + kStatLeanWaves - 1) / kStatLeanWaves;   // this wave's slices of a node
  constexpr int kTileBytes = kSlice * K * 4;

  int cur = blockIdx.x;
  int nxt = cur + (int)gridDim.x < n_nodes ? cur + (int)gridDim.x : -1;
  StatRef A = stat_ref(d, nodes, cur, K * K * 4);
  // loop-carried requests: operands of the wave's next slice, categories and row maxima of the one after
  Tile<K> P0, R, C1, C2;   // (a third child is rare: it is fetched at the point of use)
  uint32_t xc, xn;
  float mc, mn;
  WTile<K> w;
  // categories and row maxima of the wave's first two slices: requested before the histograms are cleared, so
  // that the leaf rows that depend on them can go out right behind the barrier
  xc = load_x(A, min(wave, last));
  xn = load_x(A, min(wave + kStatLeanWaves, last));
  mc = load_m(A, min(wave, last));
  mn = load_m(A, min(wave + kStatLeanWaves, last));
  lean_w_load<K>(rW, vtile, A.w_off, w);
  for (int i = threadIdx.x; i < hist_words; i += blockDim.x) hist[i] = 0u;
  __syncthreads();
  bool warm = false;   // the first slice's operands of `cur` are on their way already

  while (true) {
    const StatNode* __restrict__ np = nodes + cur;
    const StatRef B = stat_ref(d, nodes, max(nxt, 0), K * K * 4);
    const int n_pass = (A.n_hist + nh_pass - 1) / nh_pass;
    const bool cross = stream_on && nxt >= 0 && n_pass == 1;   // this wave's stream runs on into `nxt`
    if (!warm) {
      // operands of the wave's first slice (slices past the end are clamped: harmless repeated loads)
      const int so = min(wave, last) * kTileBytes;
      lean_row_load<K>(rL, lean_row_off<K>(xc, 0, vleaf), A.leaf_off, P0);
      if (A.c1 >= 0) child_load(A.c1, xc, so, C1);
      if (A.c2 >= 0) child_load(A.c2, xc, so, C2);
      lean_tile_load<K>(rR, vtile, A.tile_off + so, R);
    }
    v4f accA[KT][KT];
#pragma unroll
    for (int a = 0; a < KT; ++a)
#pragma unroll
      for (int c = 0; c < KT; ++c) accA[a][c] = v4f{0.f, 0.f, 0.f, 0.f};

    {
      const int nh = min(nh_pass, A.n_hist);   // pass 0 fills the histograms of the first nh variables
      for (int it = 0; it < n_it; ++it) {
        const int s0 = wave + it * kStatLeanWaves;
        // where the requests of this turn go: the next slice of this node, or the first of the next node
        const bool over1 = it + 1 >= n_it, over2 = it + 2 >= n_it;
        const bool x1 = cross && over1, x2 = cross && over2;
        const int s1 = x1 ? wave : min(s0 + kStatLeanWaves, last);
        const int s2 = x2 ? wave + (it + 2 - n_it) * kStatLeanWaves : min(s0 + 2 * kStatLeanWaves, last);
        const int t_tile = x1 ? B.tile_off : A.tile_off, t_leaf = x1 ? B.leaf_off : A.leaf_off;
        const int t_c1 = x1 ? B.c1 : A.c1, t_c2 = x1 ? B.c2 : A.c2;
        const int t_x = x2 ? B.x_off : A.x_off;
        const int so1 = s1 * kTileBytes;
        // (1) E (unnormalised) from the landed operands; request the next slice's
        Tile<K> e = P0;
        if (A.c1 >= 0) tile_add<K>(e, C1);
        if (A.c2 >= 0) tile_add<K>(e, C2);
        const uint32_t xh = xc;   // categories of the slice computed now
        if (A.c3 >= 0) {
          Tile<K> t3;
          child_load(A.c3, xh, s0 * kTileBytes, t3);
          tile_add<K>(e, t3);
        }
        xc = xn;
        xn = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rX, (int)vx, t_x + s2 * (kSlice * 4), 0);
        const float m = mc;   // the scale the backward walk built R with
        mc = mn;
        mn = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rM, (int)vx, t_x + s2 * (kSlice * 4), 0));
        lean_row_load<K>(rL, lean_row_off<K>(xc, 0, vleaf), t_leaf, P0);
        if (t_c1 >= 0) child_load(t_c1, xc, so1, C1);
        if (t_c2 >= 0) child_load(t_c2, xc, so1, C2);
        // (2) E, the edge flows, then G = E .* (R W)
        tile_exp_sub<K>(e, lean_scale(m));
        {
          // A += R^T E over the 16 examples of the tile (contraction over examples): both operands
          // go through the wave's pad to reach the [state][example] operand layout.  A wave's LDS
          // accesses execute in order, so the pad needs no barrier between its phases.
          float ra[4][KT];
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) *reinterpret_cast<v4f*>(&pad[pad_w(kt)]) = R.v[kt];
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) ra[q][kt] = pad[pad_r(q, kt)];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) *reinterpret_cast<v4f*>(&pad[pad_w(kt)]) = e.v[kt];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float eb[KT];
#pragma unroll
            for (int jt = 0; jt < KT; ++jt) eb[jt] = pad[pad_r(q, jt)];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
              for (int jt = 0; jt < KT; ++jt)
                accA[kt][jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[q][kt], eb[jt], accA[kt][jt], 0, 0, 0);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        Tile<K> t;
        contract<K>(w, R, t);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) t.v[kt] *= e.v[kt];
        lean_tile_load<K>(rR, vtile, t_tile + so1, R);   // next slice's ratios, after the last use of these
        if (n_pass > 1) {
          // the later passes only need G: it replaces the tile of R just consumed
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, t.v[kt]), rR, (int)(vtile + kt * 1024),
                                                   A.tile_off + s0 * kTileBytes, 0);
        }
        // (3) histograms: the node's own variable, and its first leaf child if the LDS holds two
        if (s0 * kSlice + b < d.B) {
          histogram(t, xh, 0, 0);
          if (nh > 1) histogram(t, xh, 1, 1);
        }
      }
      __syncthreads();
      // the node after next is drawn while the histograms go out
      if (threadIdx.x == 0) *claim_word = nxt >= 0 ? stat_claim(counter, n_nodes) : -1;
      flush(np, 0, nh);
      __syncthreads();
    }
    const int nxt2 = __builtin_amdgcn_readfirstlane(*claim_word);
    for (int pass = 1; pass < n_pass; ++pass) {
      // further leaf children: G comes back from where pass 0 left it; only the categories differ
      const int h0 = pass * nh_pass, nh = min(nh_pass, A.n_hist - h0);
      Tile<K> T;
      uint32_t yc = load_x(A, min(wave, last)), yn = load_x(A, min(wave + kStatLeanWaves, last));
      lean_tile_load<K>(rR, vtile, A.tile_off + min(wave, last) * kTileBytes, T);
      for (int s0 = wave; s0 < d.nslices; s0 += kStatLeanWaves) {
        const int s1 = min(s0 + kStatLeanWaves, last), s2 = min(s0 + 2 * kStatLeanWaves, last);
        const uint32_t xh = yc;
        yc = yn;
        yn = load_x(A, s2);
        if (s0 * kSlice + b < d.B) {
          histogram(T, xh, h0, 0);
          if (nh > 1) histogram(T, xh, h0 + 1, 1);
        }
        lean_tile_load<K>(rR, vtile, A.tile_off + s1 * kTileBytes, T);
      }
      __syncthreads();
      flush(np, h0, nh);
      __syncthreads();
    }

    // combine the waves' partial blocks: every wave parks its accumulators in LDS (the histogram area is free
    // now), then each thread adds up the waves' copies of its elements in wave order.  The edge weight of an
    // element is already in the lane that holds it -- the block as the backward contraction's operand has
    // element (k, j) where the accumulator tile has it -- so the partial sums are parked weighted and the
    // parameters are not read again.
    v4f* park = reinterpret_cast<v4f*>(smem);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int jt = 0; jt < KT; ++jt)
        park[((size_t)wave * KT * KT + kt * KT + jt) * 64 + lane] = accA[kt][jt] * w.a[jt * KT + kt];
    if (nxt >= 0) lean_w_load<K>(rW, vtile, B.w_off, w);   // the next node's block, into the registers just freed
    __syncthreads();
    {
      float* dst = edge_aggr + (size_t)A.node * K * K;
      float* parkf = smem;
      for (int t = threadIdx.x; t < K * K; t += blockDim.x) {   // one element a thread: (tile q, component v)
        const int q = t >> 2, v = t & 3;
        float sum = parkf[t];
        parkf[t] = 0.f;
#pragma unroll
        for (int wv = 1; wv < kStatLeanWaves; ++wv) {
          sum += parkf[wv * (K * K) + t];
          parkf[wv * (K * K) + t] = 0.f;
        }
        const int kt = q / (KT * 64), jt = (q / 64) % KT, l = q % 64;
        const int idx = (kt * 16 + 4 * (l >> 4) + v) * K + jt * 16 + (l & 15);
        const float old = rate != 0.f ? rate * dst[idx] : 0.f;
        dst[idx] = old + sum;
      }
    }
    if (nxt < 0) break;
    if (!cross) {
      // the stream ended with this node: first categories and row maxima of the next one
      xc = load_x(B, min(wave, last));
      xn = load_x(B, min(wave + kStatLeanWaves, last));
      mc = load_m(B, min(wave, last));
      mn = load_m(B, min(wave + kStatLeanWaves, last));
    }
    __syncthreads();   // the area is clear again before anyone counts into it
    warm = cross;
    cur = nxt;
    nxt = nxt2;
    A = B;
  }
}

}  // namespace pcm
