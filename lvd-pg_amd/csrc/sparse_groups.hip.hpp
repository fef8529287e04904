// Dense groups of the layered engine: sum nodes of one layer over ONE set of (prime, sub) children.
//
// Every structure builder of the reference emits them -- the K sum nodes of an HCLT's tree node over its K
// products (src/structures/hclts.jl:133), the heads of a multi-head circuit over the root's products, the
// doubled sums of grow_heads_by_flows over the doubled products -- and per edge they cost the layer kernels an
// exponential and two row reads per example.  A group of G sums over C children is the block algebra of the HCLT
// kernels instead:
//   X[c] = sum of the values of child c's factors,  m = max_c X[c],  E[c] = exp(X[c] - m)
//   S[g] = sum_c W[g,c] E[c],  value of sum g = m + log S[g]                       (forward; W = exp(log-parameters))
//   R[g] = flow of sum g / S[g],  flow into child c = E[c] * sum_g W[g,c] R[g]      (backward)
//   edge flow (g, c) summed over the batch = W[g,c] * sum_b R[b,g] E[b,c]
// (tempered flows, fscale != 1: going down W, E and the shares of R to the power 1 / fscale, R over the tempered sum)
// with the three contractions on v_mfma_f32_16x16x4_f32: C exponentials per example instead of G * C.  The two that
// sit in the chain of layers are one wave per (group, 16 examples) with everything in registers; the edge flows, which
// nothing waits for, are one launch per shape of group after the pass.
//
// A child whose prime is a product node of up to three factors that only groups use (as a prime) is taken apart: the
// group reads the product's factors, writes the product's value next to its own, and the product leaves the forward
// layers (in an HCLT: the product of a tree node's children, which otherwise is a layer between any two levels).  Going down, a
// group's row for child c is the whole flow of every node that nothing else reaches -- the product, its factors, their
// only children -- and the kernel writes those rows itself (`copies`), so they leave the backward layers; where some
// other node still adds the row to flows from elsewhere it is kept behind the node rows of the flow array (row
// n_nodes + slot), which the layer kernels read like the flow of a product parent.  In an HCLT this leaves one group
// launch per tree level and direction and nothing else between the leaves and the root.
// The edge flows go to the same rows of partial sums as the layer kernels' (one row per 64 examples, added in order
// afterwards), so results do not depend on the order in which workgroups run.
#pragma once

namespace pcm {

typedef float g4f __attribute__((ext_vector_type(4)));

// The tables the kernels index are padded to the tile sizes, group after group in launch order: Gp = 16 GT entries of
// sums (node id -1 past G), Cp = 16 CT entries of children (own = -2 past C: a child that is not there, X = -inf) and
// Gp x Cp of W (0 outside G x C), so a kernel finds its group's entries from its block index and tests no bounds.
struct GroupRec {
  int32_t G, C;
  int32_t pnode0;   // the group's first entry in the per-sum tables
  int32_t pslot0;   // ... in the per-child tables
  int64_t pw0;      // ... in the W tables
  int32_t gt, ct;   // Gp / 16, Cp / 16
};

constexpr int kGroupCopies = 8;   // rows a group's kernel writes per child: two int4 of row numbers, -1: none

struct GroupDev {
  const GroupRec* rec;
  const int32_t* node;    // per sum entry: node id
  const int32_t* edge;    // per entry of the padded Gp x Cp, [g][c]: the up edge of sum g to child c (the sums list their
                          // children in orders of their own); -1 outside G x C
  const int4* rows;       // per child entry: the value rows whose sum is X: three for the prime, one for the sub (the row of zeros where there are fewer)
  const int32_t* own;     // per child entry: the product node that is the prime taken apart, whose value the forward kernel writes; -1: none
  const int4* copies;     // per child entry: kGroupCopies rows of the flow array that take the child's flow
  const int32_t* order;   // groups by shape, for the launches that are not per layer
  const float* wf;        // W in the order the forward kernel's lanes take it: [gt][q][lane] = W[16 gt + lo][4 q + hi]
  const float* wb;        // ... and the backward kernel's: [ct][k][lane] = W[4 k + hi][16 ct + lo]
  float* m;               // [groups][Bp]: the maximum the forward kernel took out, per example
  float* xm;              // [child entries][Bp]: X - m as the forward kernel formed it (-inf: an impossible child), for the way down
  const float* logp;
  float* mars;
  float* flows;           // [n_nodes + slots][Bp]
  float* edge_part;       // [Bp / 64][n_edges]
  int64_t n_nodes, n_edges;
  int32_t B, Bp;
  uint32_t flow_bytes;    // size of the flow array, 0 from 2 GiB on (its rows are then addressed by pointers)
  // tempered flows (fscale of mini_batch_em_beta): shares to the power inv_f = 1 / fscale, normalised again by the
  // sums' rows of `norm` (row norm_row for every sum if it is >= 0: the row of zeros of a pass that is not tempered)
  float inv_f;
  const float* norm;
  int64_t norm_row;
};

// where the kernels of one launch find their groups' entries: group = group0 + block, entries at base + block * stride
struct GroupBase {
  int32_t group0, pnode0, pslot0;
  int64_t pw0;
};

constexpr int kGroupPad = 65;   // row length of the [.][64 examples] tiles in LDS

// LDS of a statistics workgroup, in floats: E [Cp][65] | R [Gp][65]
__host__ __device__ inline size_t group_lds_floats(int Gp, int Cp) { return (size_t)(Cp + Gp) * kGroupPad; }

__host__ __device__ inline int64_t group_wf_index(int g, int c, int ct) {   // ct = Cp / 16
  return ((int64_t)(g >> 4) * (ct * 4) + (c >> 2)) * 64 + (c & 3) * 16 + (g & 15);
}
__host__ __device__ inline int64_t group_wb_index(int g, int c, int gt) {   // gt = Gp / 16
  return ((int64_t)(c >> 4) * (gt * 4) + (g >> 2)) * 64 + (g & 3) * 16 + (c & 15);
}

// W below float's normal range is kept as -0: nothing to a product, and the mark by which sums that may hang on such an
// edge (see kLowSum) find it and take its logarithm.  NaN stays NaN for the way up; going down, a sum it made NaN has no flow.
__device__ __forceinline__ bool group_tiny_w(float w) { return __builtin_bit_cast(uint32_t, w) == 0x80000000u; }
__device__ __forceinline__ float group_w(float lw) {
  const float w = __expf(lw);
  return w >= __FLT_MIN__ ? w : lw > -INFINITY ? -0.f : lw == lw ? 0.f : lw;
}

// exp of the groups' log-parameters in both orders, once per pass (the parameters may have moved): thread = (group,
// entry of its padded Gp x Cp)
__global__ __launch_bounds__(256) void sparse_group_w_kernel(GroupDev d, const int32_t* __restrict__ group_of_elem, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const GroupRec r = d.rec[group_of_elem[i]];
  const int64_t local = i - r.pw0;
  const int g = (int)(local / (16 * r.ct)), c = (int)(local % (16 * r.ct));
  const int e = d.edge[i];
  const float w = e >= 0 ? group_w(d.logp[e] * d.inv_f) : 0.f;
  const_cast<float*>(d.wf)[r.pw0 + group_wf_index(g, c, r.ct)] = w;
  const_cast<float*>(d.wb)[r.pw0 + group_wb_index(g, c, r.gt)] = w == w ? w : 0.f;
}

// exp(x) * y with a product in float's range, whatever exp(x) alone would be
__device__ __forceinline__ float group_exp_times(float x, float y) {
  const float a = fmaxf(x, -2000.f) * 1.44269504f, n = rintf(a);   // (log2 e; -inf: far enough down)
  return ldexpf(__builtin_amdgcn_exp2f(a - n) * y, (int)n);
}

__device__ __forceinline__ int guni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// maximum over the four lanes that hold one example (lane, lane ^ 16, lane ^ 32, lane ^ 48)
__device__ __forceinline__ float group_max4(float v) {
  const int a = __builtin_bit_cast(int, v);
  const auto r16 = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  v = fmaxf(__builtin_bit_cast(float, (int)r16[0]), __builtin_bit_cast(float, (int)r16[1]));
  const int b = __builtin_bit_cast(int, v);
  const auto r32 = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__builtin_bit_cast(float, (int)r32[0]), __builtin_bit_cast(float, (int)r32[1]));
}

// How the group kernels reach memory: `at` is the same for a wave, `own` a lane's, `row` a row of values or flows of which
// the lane's example is taken (row -1: a store goes nowhere).  By pointers, whatever the arrays' sizes:
struct GroupPointers {
  const GroupDev& d;
  int64_t col;
  __device__ __forceinline__ GroupPointers(const GroupDev& dev, int slice, int lane) : d(dev), col((int64_t)slice * 16 + (lane & 15)) {}
  __device__ __forceinline__ int4 rows(int at, int own) const { return d.rows[(int64_t)at + own]; }
  __device__ __forceinline__ int own(int at, int own_) const { return d.own[(int64_t)at + own_]; }
  __device__ __forceinline__ int node(int at, int own) const { return d.node[(int64_t)at + own]; }
  __device__ __forceinline__ int4 node4(int at, int own) const { return *reinterpret_cast<const int4*>(d.node + at + own); }
  __device__ __forceinline__ int4 copies(int64_t at, int own) const { return d.copies[at + own]; }
  __device__ __forceinline__ float wf(int64_t at, int own) const { return d.wf[at + own]; }
  __device__ __forceinline__ float wb(int64_t at, int own) const { return d.wb[at + own]; }
  __device__ __forceinline__ float m(int group) const { return d.m[(int64_t)group * d.Bp + col]; }
  __device__ __forceinline__ void put_m(int group, float v) const { d.m[(int64_t)group * d.Bp + col] = v; }
  __device__ __forceinline__ float xm(int at, int own) const { return d.xm[((int64_t)at + own) * d.Bp + col]; }
  __device__ __forceinline__ void put_xm(int at, int own, float v) const { d.xm[((int64_t)at + own) * d.Bp + col] = v; }
  __device__ __forceinline__ float value(int row) const { return d.mars[(int64_t)row * d.Bp + col]; }
  __device__ __forceinline__ void put_value(int row, float v) const { if (row >= 0) d.mars[(int64_t)row * d.Bp + col] = v; }
  __device__ __forceinline__ float flow(int row) const { return d.flows[(int64_t)row * d.Bp + col]; }
  __device__ __forceinline__ float norm(int row) const { return d.norm[(int64_t)row * d.Bp + col]; }
};
// ... and by buffer descriptors where every array stays below 2 GiB and a row below 64 KB: a row's address is one
// 24-bit multiply-add, the tables' offsets are in the requests.
struct GroupBuffers {
  __amdgpu_buffer_rsrc_t r_rows, r_own, r_node, r_copies, r_wf, r_wb, r_m, r_xm, r_mars, r_flows, r_norm;
  int bp4, col4;
  template <typename T>
  __device__ __forceinline__ static __amdgpu_buffer_rsrc_t all(const T* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, 0x7fffffff, 0x00020000);
  }
  __device__ __forceinline__ GroupBuffers(const GroupDev& d, int slice, int lane)
      : r_rows(all(d.rows)), r_own(all(d.own)), r_node(all(d.node)), r_copies(all(d.copies)), r_wf(all(d.wf)), r_wb(all(d.wb)),
        r_m(all(d.m)), r_xm(all(d.xm)), r_mars(all(d.mars)), r_flows(all(d.flows)), r_norm(all(d.norm)), bp4(d.Bp * 4),
        col4(slice * 64 + (lane & 15) * 4) {}
  __device__ __forceinline__ static float one(__amdgpu_buffer_rsrc_t r, int own, int at) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, own, at, 0));
  }
  __device__ __forceinline__ static int4 four(__amdgpu_buffer_rsrc_t r, int own, int at) {
    return __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(r, own, at, 0));
  }
  __device__ __forceinline__ int at_row(int row) const { return (int)__umul24(row, bp4) + col4; }
  __device__ __forceinline__ int4 rows(int at, int own) const { return four(r_rows, 16 * own, 16 * at); }
  __device__ __forceinline__ int own(int at, int own_) const { return (int)__builtin_amdgcn_raw_buffer_load_b32(r_own, 4 * own_, 4 * at, 0); }
  __device__ __forceinline__ int node(int at, int own) const { return (int)__builtin_amdgcn_raw_buffer_load_b32(r_node, 4 * own, 4 * at, 0); }
  __device__ __forceinline__ int4 node4(int at, int own) const { return four(r_node, 4 * own, 4 * at); }
  __device__ __forceinline__ int4 copies(int64_t at, int own) const { return four(r_copies, 16 * own, (int)(16 * at)); }
  __device__ __forceinline__ float wf(int64_t at, int own) const { return one(r_wf, 4 * own, (int)(4 * at)); }
  __device__ __forceinline__ float wb(int64_t at, int own) const { return one(r_wb, 4 * own, (int)(4 * at)); }
  __device__ __forceinline__ float m(int group) const { return one(r_m, col4, group * bp4); }
  __device__ __forceinline__ void put_m(int group, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r_m, col4, group * bp4, 0);
  }
  __device__ __forceinline__ float xm(int at, int own) const { return one(r_xm, own * bp4 + col4, at * bp4); }
  __device__ __forceinline__ void put_xm(int at, int own, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r_xm, own * bp4 + col4, at * bp4, 0);
  }
  __device__ __forceinline__ float value(int row) const { return one(r_mars, at_row(row), 0); }
  __device__ __forceinline__ void put_value(int row, float v) const {   // (past the descriptor's end: nowhere)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r_mars, row >= 0 ? at_row(row) : -1, 0, 0);
  }
  __device__ __forceinline__ float flow(int row) const { return one(r_flows, at_row(row), 0); }
  __device__ __forceinline__ float norm(int row) const { return one(r_norm, at_row(row), 0); }
};

// Sums far below their group's maximum.  E = exp(X - m) leaves float's range 87 below m, and a sum without a share in
// the children near m -- masked groups (build_groups) have many -- may own nothing above that.  A sum that comes out
// below kLowSum is added up again with E = exp(X - m + off) for an offset raised step by step (per example, so the
// matrix instruction's columns stay independent).  A step raises the highest child that has not had its turn to
// kHighShare, and with it the children up to kTurn below, which are then at kHighShare - kTurn = 20 or more: as W >= FLT_MIN,
// W E >= 5.8e-30 shows any of them that the sum has.  So when E is cut off at exp(kMaxRaise), for children far above, no sum
// that is still looked for has one of those, and every step takes in a child more, so the loop ends.
// Only such sums can hang on a parameter below float's range; where a block has one (group_tiny_w) they are added up in
// logarithms, edge by edge.  So are sums that come out NaN: of the children's NaNs only those of a sum's own make it NaN.
// Going down, the shares of all sums with m - value > kHighShare are added in logarithms.
constexpr float kLowSum = 1e-30f, kHighShare = 60.f, kTurn = 40.f, kMaxRaise = 88.f;

template <int NK>
__device__ __forceinline__ void group_low_sums(const GroupDev& d, const float* xm, int hi, const float* w, const int32_t* edge, float mx,
                                               bool (&low)[4], float (&val)[4]) {
  float xs[NK], a[NK];
  bool tiny = false;
#pragma unroll
  for (int q = 0; q < NK; ++q) {
    xs[q] = xm[(int64_t)(4 * q + hi) * d.Bp];   // (what this lane has just written)
    a[q] = w[q * 64];
    tiny |= group_tiny_w(a[q]) || !(a[q] == a[q]) || !(xs[q] == xs[q]);
  }
  if (__any(tiny)) {   // edge: the tile's rows of d.edge, [16][4 NK]
    __threadfence_block();   // (X - m of the children that the other lanes of the example hold)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!low[i]) continue;
      const int32_t* row = edge + (4 * hi + i) * (4 * NK);
      float top = -INFINITY, sum = 0.f;
#pragma clang loop unroll(disable)
      for (int c = 0; c < 4 * NK; ++c)
        if (row[c] >= 0) top = fmaxf(top, xm[(int64_t)c * d.Bp] + d.logp[row[c]] * d.inv_f);
      if (top > -INFINITY) {
#pragma clang loop unroll(disable)
        for (int c = 0; c < 4 * NK; ++c)
          if (row[c] >= 0) sum += __expf(xm[(int64_t)c * d.Bp] + d.logp[row[c]] * d.inv_f - top);
      }
      val[i] = mx + (top > -INFINITY ? top + __logf(sum) : -INFINITY);
    }
    return;
  }
  float turned = INFINITY;   // the children from here up have had their turn
  for (int it = 0; it <= 4 * NK; ++it) {
    float next = -INFINITY;
#pragma unroll
    for (int q = 0; q < NK; ++q) if (xs[q] < turned) next = fmaxf(next, xs[q]);
    next = group_max4(next);
    if (!(next > -INFINITY)) low[0] = low[1] = low[2] = low[3] = false;   // nothing further down: what S was, it is
    if (!__any(low[0] | low[1] | low[2] | low[3])) break;
    const float off = next > -INFINITY ? kHighShare - next : 0.f;
    turned = next - kTurn;
    g4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NK; ++q)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], xs[q] > -INFINITY ? __expf(fminf(xs[q] + off, kMaxRaise)) : 0.f, acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (low[i] && acc[i] >= kLowSum) {
        val[i] = mx - off + __logf(acc[i]);
        low[i] = false;
      }
  }
}

// Forward: values of the group's sums.  One wave per (group, 16 examples), nothing shared: lane 16 * hi + lo takes
// example lo and the children c = 4 q + hi, which is the B-operand layout of the matrix instruction's k-step q, so
// X, the maximum (two lane swaps), E and the contraction stay in the wave's registers.  GT = Gp / 16, CT = Cp / 16.
// What the kernel reads is requested in two rounds (row numbers, W and node ids; then the rows), everything of a round
// before anything of it is used and no branch around a load: a layer's launch lasts as long as its longest chain of
// requests.  The maximum goes to d.m for the backward kernels.
template <int GT, int CT>
struct GroupUpTables {   // what the forward kernel reads of a group in its first round
  static constexpr int NK = CT * 4;
  static constexpr bool kPre = GT * NK <= 64;   // W in registers before the rows arrive
  int4 rw[NK], nd4[GT];
  int own[NK];
  float a[kPre ? GT : 1][kPre ? NK : 1];
  template <typename M>
  __device__ __forceinline__ void load(const M& mem, const GroupBase& base, int bx, int lane) {
    constexpr int Gp = GT * 16, Cp = CT * 16;
    const int hi = lane >> 4;
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      rw[q] = mem.rows(base.pslot0 + bx * Cp + 4 * q, hi);
      own[q] = mem.own(base.pslot0 + bx * Cp + 4 * q, hi);
    }
    if constexpr (kPre) {
#pragma unroll
      for (int gt = 0; gt < GT; ++gt)
#pragma unroll
        for (int q = 0; q < NK; ++q) a[gt][q] = mem.wf(base.pw0 + (int64_t)bx * Gp * Cp + (gt * NK + q) * 64, lane);
    }
#pragma unroll   // (the four sums of a lane's output rows are neighbours in the table: one request per tile)
    for (int gt = 0; gt < GT; ++gt) nd4[gt] = mem.node4(base.pnode0 + bx * Gp + gt * 16, 4 * hi);
  }
};
// A group going up, in two steps: the sums' values, which the groups above wait for, and what later passes read.
template <int GT, int CT>
struct GroupUp {
  static constexpr int NK = CT * 4;
  float xs[NK], pv[NK], mx;   // X - m and the value of the prime, per child; m
  bool kept;                  // X - m is in memory
  template <typename M>
  __device__ __forceinline__ void keep_xm(const M& mem, const GroupBase& base, int bx, int lane) {
#pragma unroll
    for (int q = 0; q < NK; ++q) mem.put_xm(base.pslot0 + bx * CT * 16 + 4 * q, lane >> 4, xs[q]);
  }
  // X of a child: the value of its prime (the first three rows: the prime itself and two rows of zeros, or the factors of a
  // product the group computes) plus its sub's (the last row; zeros: none).  kAll: what later passes read is stored on the
  // way, where it takes the fewest registers, and there is no rest.
  template <bool kAll, typename M>
  __device__ __forceinline__ void values(const GroupDev& d, const GroupBase& base, int bx, int lane, int slice, const M& mem,
                                         const GroupUpTables<GT, CT>& tb) {
    constexpr int Gp = GT * 16, Cp = CT * 16;
    constexpr bool kPre = GroupUpTables<GT, CT>::kPre;
    const int lo = lane & 15, hi = lane >> 4;
    float e[NK];
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      pv[q] = (mem.value(tb.rw[q].x) + mem.value(tb.rw[q].y)) + mem.value(tb.rw[q].z);
      xs[q] = pv[q] + mem.value(tb.rw[q].w);
    }
#pragma unroll
    for (int q = 0; q < NK; ++q) if (tb.own[q] == -2) xs[q] = -INFINITY;
    mx = xs[0];
#pragma unroll
    for (int q = 1; q < NK; ++q) mx = fmaxf(mx, xs[q]);
    mx = group_max4(mx);
    if (!(mx > -INFINITY)) mx = 0.f;   // every child impossible: E = 0, the sums come out as -inf
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      xs[q] -= mx;   // (-inf stays -inf)
      e[q] = __expf(xs[q]);
    }
    kept = false;
    if constexpr (kAll) {
      rest(base, bx, lane, mem, tb);
      kept = true;
    }
    float val[GT][4];
    bool low[GT][4], any = false;
    g4f acc[GT];
#pragma unroll
    for (int gt = 0; gt < GT; ++gt) acc[gt] = g4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NK; ++q)
#pragma unroll
      for (int gt = 0; gt < GT; ++gt) {
        float av;
        if constexpr (kPre) av = tb.a[gt][q];
        else av = mem.wf(base.pw0 + (int64_t)bx * Gp * Cp + (gt * NK + q) * 64, lane);
        acc[gt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, e[q], acc[gt], 0, 0, 0);
      }
#pragma unroll
    for (int gt = 0; gt < GT; ++gt) {
      const int nd[4] = {tb.nd4[gt].x, tb.nd4[gt].y, tb.nd4[gt].z, tb.nd4[gt].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        val[gt][i] = mx + __logf(acc[gt][i]);
        low[gt][i] = nd[i] >= 0 && !(acc[gt][i] >= kLowSum);
        any |= low[gt][i];
      }
    }
    if (__any(any)) {
      if (!kept) keep_xm(mem, base, bx, lane);
      kept = true;
      const float* xm = d.xm + (base.pslot0 + (int64_t)bx * Cp) * d.Bp + (int64_t)slice * 16 + lo;
      const float* wg = d.wf + base.pw0 + (int64_t)bx * Gp * Cp + lane;
#pragma unroll
      for (int gt = 0; gt < GT; ++gt)
        if (__any(low[gt][0] | low[gt][1] | low[gt][2] | low[gt][3]))
          group_low_sums<NK>(d, xm, hi, wg + gt * NK * 64, d.edge + base.pw0 + ((int64_t)bx * Gp + gt * 16) * Cp, mx, low[gt], val[gt]);
    }
#pragma unroll
    for (int gt = 0; gt < GT; ++gt) {
      const int nd[4] = {tb.nd4[gt].x, tb.nd4[gt].y, tb.nd4[gt].z, tb.nd4[gt].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) mem.put_value(nd[i], val[gt][i]);
    }
  }
  template <typename M>
  __device__ __forceinline__ void rest(const GroupBase& base, int bx, int lane, const M& mem, const GroupUpTables<GT, CT>& tb) {
    if (!kept) keep_xm(mem, base, bx, lane);
#pragma unroll
    for (int q = 0; q < NK; ++q) mem.put_value(tb.own[q], pv[q]);
    if ((lane >> 4) == 0) mem.put_m(base.group0 + bx, mx);
  }
};
template <int GT, int CT>
__device__ __forceinline__ void group_forward_body(const GroupDev& d, const GroupBase& base, int bx, int lane, int slice) {
  const GroupPointers mem(d, slice, lane);
  GroupUpTables<GT, CT> tb;
  tb.load(mem, base, bx, lane);
  GroupUp<GT, CT> up;
  up.template values<true>(d, base, bx, lane, slice, mem, tb);
}

template <int GT, int CT>
__global__ __launch_bounds__(64) void sparse_group_forward_kernel(GroupDev d, GroupBase base) {
  group_forward_body<GT, CT>(d, base, blockIdx.x, threadIdx.x, blockIdx.y);
}

// The part of the children's rows that the product on the matrix cores leaves out, edge by edge with the exponent of the
// share: what comes from sums with m - value > kHighShare (see kLowSum; flow * W and exp(X - m) * share / W both leave
// float's range on the way to a share that does not) and, where the tile has such edges (tiny), what goes through a W below
// float's range from sums with m - value > kTinyShare (from others: shares below e^-67).
constexpr float kTinyShare = 20.f;

// out[i]: the rows of the four children whose X - m are e[i]; edge: the group's [4 NG][Cp] entries of d.edge from these
// four children on (16-byte words).
template <int NG, int Cp>
__device__ __forceinline__ void group_shares_by_edge(const GroupDev& d, const int32_t* node, int64_t col, float mb, bool tiny,
                                                     const int32_t* edge, const float (&e)[4], float (&out)[4]) {
#pragma clang loop unroll(disable)
  for (int k = 0; k < NG; ++k) {
    const int4 n4 = *reinterpret_cast<const int4*>(node + 4 * k);
    const int nd[4] = {n4.x, n4.y, n4.z, n4.w};
    float f[4], t[4];
    bool take = false;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t n = nd[g] < 0 ? 0 : nd[g];
      f[g] = d.flows[n * d.Bp + col];
      const float v = d.mars[n * d.Bp + col];
      t[g] = (mb - v) * d.inv_f - (d.norm_row < 0 ? d.norm[n * d.Bp + col] : 0.f);
      if (!(nd[g] >= 0 && f[g] > 0.f && v > -INFINITY && t[g] > (tiny ? kTinyShare : kHighShare))) f[g] = 0.f;
      take |= f[g] > 0.f;
    }
    if (!__any(take)) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int4 e4 = *reinterpret_cast<const int4*>(edge + (int64_t)(4 * k + g) * Cp);
      const int ed[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (ed[i] < 0) continue;
        const float lw = d.logp[ed[i]] * d.inv_f;
        if (f[g] > 0.f && (t[g] > kHighShare || group_tiny_w(group_w(lw)))) out[i] += f[g] * __expf(e[i] * d.inv_f + lw + t[g]);
      }
    }
  }
}

// Backward, per layer: the rows the group hands its children, E[c] * sum_g W[g,c] R[g].  One wave per (group, 16
// examples) as going up: R of the sums g = 4 k + hi is the B operand of k-step k as it is loaded.  The same two
// rounds of requests where the registers hold a group's W and row numbers (kPre); 16 children at a time otherwise.
template <int GT, int CT>
struct GroupDownTables {   // what the backward kernel reads of a group without waiting for anything
  static constexpr int NG = GT * 4;
  static constexpr bool kPre = CT <= 2 && GT * CT <= 16;
  static constexpr int CL = kPre ? CT : 1;
  int nd[NG];
  int4 cpa[CL][4], cpb[CL][4];
  float a[CL][NG], e[CL][4], mb, v[NG];
  template <typename M>   // row numbers and W for the children 16 ct + 4 hi + i
  __device__ __forceinline__ void numbers(const M& mem, const GroupBase& base, int bx, int lane, int ct, int s) {
    constexpr int Gp = GT * 16, Cp = CT * 16;
    const int hi = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t at = 2 * (base.pslot0 + (int64_t)bx * Cp + ct * 16);
      cpa[s][i] = mem.copies(at + 2 * i, 8 * hi);
      cpb[s][i] = mem.copies(at + 2 * i + 1, 8 * hi);
    }
#pragma unroll
    for (int k = 0; k < NG; ++k) a[s][k] = mem.wb(base.pw0 + (int64_t)bx * Gp * Cp + (ct * NG + k) * 64, lane);
  }
  template <typename M>
  __device__ __forceinline__ void load(const M& mem, const GroupBase& base, int bx, int lane) {
    mb = mem.m(base.group0 + bx);
#pragma unroll
    for (int k = 0; k < NG; ++k) nd[k] = mem.node(base.pnode0 + bx * GT * 16 + 4 * k, lane >> 4);
    if constexpr (kPre) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) numbers(mem, base, bx, lane, ct, ct);
    }
  }
  template <typename M>   // X - m as the forward kernel left it (a child that is not there: -inf)
  __device__ __forceinline__ void children(const M& mem, const GroupBase& base, int bx, int lane, int ct, int s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) e[s][i] = mem.xm(base.pslot0 + bx * CT * 16 + ct * 16 + i, 4 * (lane >> 4));
  }
  template <typename M>   // the sums' values, and the children's where the registers hold them
  __device__ __forceinline__ void values(const M& mem, const GroupBase& base, int bx, int lane) {
#pragma unroll
    for (int k = 0; k < NG; ++k) v[k] = mem.value(max(nd[k], 0));
    if constexpr (kPre) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) children(mem, base, bx, lane, ct, ct);
    }
  }
};
template <int GT, int CT, typename M>
__device__ __forceinline__ void group_backward_body(const GroupDev& d, const GroupBase& base, int bx, int lane, int slice,
                                                    const M& mem, GroupDownTables<GT, CT>& tb) {
  constexpr int NG = GT * 4, Gp = GT * 16, Cp = CT * 16;
  constexpr bool kPre = GroupDownTables<GT, CT>::kPre;
  constexpr int CL = GroupDownTables<GT, CT>::CL;
  const int lo = lane & 15, hi = lane >> 4;
  const int64_t col = (int64_t)slice * 16 + lo;
  const int32_t* node = d.node + base.pnode0 + (int64_t)bx * Gp;
  const float mb = tb.mb;
  const int (&nd)[NG] = tb.nd;
  const auto& cpa = tb.cpa;
  const auto& cpb = tb.cpb;
  const auto& a = tb.a;
  const auto& e = tb.e;
  const auto& v = tb.v;
  float rv[NG];
  bool high = false, middle = false;
  {   // R = F / S = F * exp(m - value): no flow stays no flow where the value is -inf.  (All rows requested, then used:
      // written as one loop the compiler waits for every sum's rows in turn.)
    float f[NG], nv[NG];
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const int n = max(nd[k], 0);
      f[k] = mem.flow(n);
      nv[k] = 0.f;
    }
    if (d.norm_row < 0) {   // tempered flows only (the same for every lane: a branch around requests, none around a wait)
#pragma unroll
      for (int k = 0; k < NG; ++k) nv[k] = mem.norm(max(nd[k], 0));
    }
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const float t = (mb - v[k]) * d.inv_f - nv[k];
      const bool some = nd[k] >= 0 && f[k] > 0.f && v[k] > -INFINITY;
      high |= some && t > kHighShare;
      middle |= some && t > kTinyShare;
      rv[k] = some && !(t > kHighShare) ? f[k] * __expf(t) : 0.f;
    }
  }
  high = __any(high);
  middle = __any(middle);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int s = kPre ? ct : 0;
    if constexpr (!kPre) { tb.numbers(mem, base, bx, lane, ct, 0); tb.children(mem, base, bx, lane, ct, 0); }
    g4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NG; ++k) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][k], rv[k], acc, 0, 0, 0);
    float out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = group_exp_times(e[s][i] * d.inv_f, acc[i]);   // (sum_g W R reaches e^kHighShare)
    uint32_t signs = 0;   // W >= 0 but for the mark of a tiny one, -0
#pragma unroll
    for (int k = 0; k < NG; ++k) signs |= __builtin_bit_cast(uint32_t, a[s][k]);
    const bool tiny = middle && __any((int32_t)signs < 0);
    if (high || tiny)
      group_shares_by_edge<NG, Cp>(d, node, col, mb, tiny, d.edge + base.pw0 + (int64_t)bx * Gp * Cp + ct * 16 + 4 * hi, e[s], out);
    if (d.flow_bytes) {
      // Row -1 of a buffer lies past its end and a store there goes nowhere, so the copies go out without a branch per row;
      // one test in eight is left, whether any child of the tile has a copy of that rank (they fill up from the front).
      // (A branch per row, 32 a tile: 192 variables, 128 heads, 512 examples: a walk down 37 layers 137 us, without 102.  The
      // same for the rows read and written on the way up loses, 48 -> 102 us a walk.)
      const __amdgpu_buffer_rsrc_t rf = __builtin_amdgcn_make_buffer_rsrc(d.flows, 0, (int)d.flow_bytes, 0x00020000);
      const int col4 = (int)col * 4;
      auto put = [&](const int r0, const int r1, const int r2, const int r3) {
        if (!__any((r0 & r1 & r2 & r3) >= 0)) return false;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, out[0]), rf, r0 * (d.Bp * 4) + col4, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, out[1]), rf, r1 * (d.Bp * 4) + col4, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, out[2]), rf, r2 * (d.Bp * 4) + col4, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, out[3]), rf, r3 * (d.Bp * 4) + col4, 0, 0);
        return true;
      };
      const int4* const p = cpa[s];
      const int4* const q = cpb[s];
      (void)(put(p[0].x, p[1].x, p[2].x, p[3].x) && put(p[0].y, p[1].y, p[2].y, p[3].y) && put(p[0].z, p[1].z, p[2].z, p[3].z) &&
             put(p[0].w, p[1].w, p[2].w, p[3].w) && put(q[0].x, q[1].x, q[2].x, q[3].x) && put(q[0].y, q[1].y, q[2].y, q[3].y) &&
             put(q[0].z, q[1].z, q[2].z, q[3].z) && put(q[0].w, q[1].w, q[2].w, q[3].w));
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float f = out[i];
      const int4 p = cpa[s][i], q = cpb[s][i];
      if (p.x >= 0) d.flows[(int64_t)p.x * d.Bp + col] = f;
      if (p.y >= 0) d.flows[(int64_t)p.y * d.Bp + col] = f;
      if (p.z >= 0) d.flows[(int64_t)p.z * d.Bp + col] = f;
      if (p.w >= 0) d.flows[(int64_t)p.w * d.Bp + col] = f;
      if (q.x >= 0) d.flows[(int64_t)q.x * d.Bp + col] = f;
      if (q.y >= 0) d.flows[(int64_t)q.y * d.Bp + col] = f;
      if (q.z >= 0) d.flows[(int64_t)q.z * d.Bp + col] = f;
      if (q.w >= 0) d.flows[(int64_t)q.w * d.Bp + col] = f;
    }
  }
}

template <int GT, int CT>
__device__ __forceinline__ void group_backward_body(const GroupDev& d, const GroupBase& base, int bx, int lane, int slice) {
  const GroupPointers mem(d, slice, lane);
  GroupDownTables<GT, CT> tb;
  tb.load(mem, base, bx, lane);
  tb.values(mem, base, bx, lane);
  group_backward_body<GT, CT>(d, base, bx, lane, slice, mem, tb);
}

template <int GT, int CT>
__global__ __launch_bounds__(64) void sparse_group_backward_kernel(GroupDev d, GroupBase base) {
  group_backward_body<GT, CT>(d, base, blockIdx.x, threadIdx.x, blockIdx.y);
}

// Walks: several consecutive layers of groups in ONE launch.  A launch that depends on the one before costs 4 to 5 us
// however little it does, and a circuit over a tree has as many layers of groups as the tree has levels; but everything
// a group reads and writes for 16 examples is read and written for those 16 examples only.  So a workgroup takes one
// slice of 16 examples through all the layers of a run (layers that hold groups of one shape and nothing else): a layer's
// groups dealt to its waves, a barrier between layers.  What a layer stores the next one reads through the same compute
// unit's cache, which the waves of a workgroup share: the barrier's wait for the stores is all the ordering it needs.
// Used where a layer's groups would not fill the device anyway (the host decides).
struct GroupWalk {
  const int2* levels;   // per layer of the run, in the order of the walk: {its first group, counted from the run's first; groups}
  int n_levels;
  GroupBase base;       // of the run's first group (the tables are padded: group i's entries are i strides further on)
};

template <int GT, int CT, int WV, bool kForward>
__global__ __launch_bounds__(WV * 64) void sparse_group_walk_kernel(GroupDev d, GroupWalk w) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int l = 0; l < w.n_levels; ++l) {
    const int2 lv = w.levels[l];
    for (int i = wave; i < lv.y; i += WV) {
      if constexpr (kForward) group_forward_body<GT, CT>(d, w.base, lv.x + i, lane, blockIdx.x);
      else group_backward_body<GT, CT>(d, w.base, lv.x + i, lane, blockIdx.x);
    }
    __syncthreads();
  }
}

// The same where a batch has few slices.  What a compute unit spends on a layer grows with the layer's groups (each is 70
// to 100 requests of four cache lines), while most compute units have nothing to do.  Groups that nothing of some
// consecutive layers connects can be walked by workgroups of their own, so a run is cut into stages, a launch each, whose
// groups are dealt to several workgroups per slice (blockIdx.y), whole connected sets to one of them.  With few groups left in
// a layer, its time is that of one group's chain of requests and instructions (up: rows 500 + 230 cycles, values 1500), so what
// no group of the next layer waits for -- rows for later passes, the tables of the wave's next group -- is left for behind the
// barrier, where the next layer's groups are other waves' (a part's groups go round its waves).
// 192 variables, K = 32, 512 examples, 25 layers: up 96 us (two walks) -> 53 (four launches), down 100 -> 54 (three); a layer of
// one group takes 1.7 us, of which its own instructions are the most.  Tried: the next tables asked for behind the rows under
// way (2.0 us), the rows of earlier launches asked for at the start (to no effect: 1 us a launch longer).
constexpr int kPartWaves = 4;
struct GroupParts {
  const int2* items;   // [part][wave][n_items]: {group, counted from the run's first, or -1: no more; its layer of the stage}
  int n_items, n_levels;
  GroupBase base;
};

template <int GT, int CT, bool kForward>
__global__ __launch_bounds__(kPartWaves * 64) void sparse_group_parts_kernel(GroupDev d, GroupParts w) {
  const int lane = threadIdx.x & 63, wave = guni(threadIdx.x >> 6);
  // (read as constants: by the scalar unit, beside the requests that are under way)
  typedef const __attribute__((address_space(4))) int* list_at;
  const list_at items = (list_at)(uintptr_t)(w.items + ((size_t)blockIdx.y * kPartWaves + wave) * w.n_items);
  using Tables = std::conditional_t<kForward, GroupUpTables<GT, CT>, GroupDownTables<GT, CT>>;
  const GroupBuffers mem(d, blockIdx.x, lane);
  Tables tb;
  int level = 0;
  int2 item{guni(items[0]), guni(items[1])};
  if (item.x >= 0) tb.load(mem, w.base, item.x, lane);
  for (int k = 1; item.x >= 0; ++k) {
    const int2 after = k < w.n_items ? int2{guni(items[2 * k]), guni(items[2 * k + 1])} : int2{-1, 0};
    if constexpr (!kForward) tb.values(mem, w.base, item.x, lane);
    for (; level < item.y; ++level) __syncthreads();
    // what the next layer waits for; then, unless this wave has more of the layer, the layer is over for it
    auto over = [&] {
      if ((after.x < 0 || after.y > level) && level + 1 < w.n_levels) { __syncthreads(); ++level; }
    };
    if constexpr (kForward) {
      GroupUp<GT, CT> up;
      up.template values<false>(d, w.base, item.x, lane, blockIdx.x, mem, tb);
      over();
      up.rest(w.base, item.x, lane, mem, tb);
    } else {
      group_backward_body<GT, CT>(d, w.base, item.x, lane, blockIdx.x, mem, tb);
      over();
    }
    item = after;
    if (item.x >= 0) tb.load(mem, w.base, item.x, lane);
  }
  for (; level + 1 < w.n_levels; ++level) __syncthreads();   // (as many barriers for every wave)
}

// Edge flows of the groups of one shape, after the backward pass: W[g,c] * sum_b R[b,g] E[b,c] over a block of 64
// examples, from the values and flows the pass has left.  A workgroup takes (group, 64 examples): E and R in LDS (a
// wave stages every fourth child, whose row numbers are the same for its 64 lanes: scalar loads, the rows of eight
// children requested before the first is used), the GT x CT tiles of the result dealt out over its four waves.
// R E is share / W and is added up over the examples before W comes in, so the product only takes pairs (sum, example)
// with m - value up to kEdgeShare; E is kept 2^kEdgeUp (e^kEdgeShare) up, so that it reaches down to X - m = -125 and no
// share falls out for it, and R 2^kEdgeDown down, so that 64 pairs stay in range for flows of up to 1e9; what falls out for
// that are flows of less than e^-73.  The other pairs, and for an edge with a W below float's range (kept as -0) all of
// them, are added in logarithms, example by example: X and log R in the same LDS, every exponent then that of a share.
// 192 variables, 128 heads, K = 32, batches of 512: 11 us for the bodies' groups and 20 for the heads' with parameters as
// training starts from, 15 and 20 after 20 epochs (30 as the limit: 19 and 20; whole sums added up again instead of their
// pairs above the limit: 18 and 21).
constexpr float kEdgeShare = 38.f;
constexpr int kEdgeUp = 55, kEdgeDown = 20;

template <int GT, int CT>
__global__ __launch_bounds__(256) void sparse_group_stats_kernel(GroupDev d, int first) {
  extern __shared__ float glds[];
  __shared__ uint64_t row_some[GT * 16], row_high[GT * 16];   // of a sum: the examples with flow, those above kEdgeShare
  __shared__ int any_again;
  const int group = d.order[first + blockIdx.x];
  const GroupRec r = d.rec[group];
  constexpr int Gp = GT * 16, Cp = CT * 16;
  const int gt0 = GT * blockIdx.z / gridDim.z, gt1 = GT * (blockIdx.z + 1) / gridDim.z;   // the workgroup's tiles of sums
  float* E = glds;
  float* R = E + Cp * kGroupPad;
  const int b0 = blockIdx.y * 64;
  const int t = threadIdx.x;
  const int b = t & 63, part = guni(t >> 6);
  const float mb = d.m[(int64_t)group * d.Bp + b0 + b];
  const int lane = t & 63, wave = t >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  float* part_row = d.edge_part + (size_t)blockIdx.y * d.n_edges;
  // child(c, X - m) for the wave's children, sum(g, flow (0: none), m - value) for its sums
  auto stage = [&](auto&& child, auto&& sum) {
    for (int cb = part; cb < Cp; cb += 32) {
      float x[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int c = cb + 4 * q;
        x[q] = c < Cp ? d.xm[(int64_t)(r.pslot0 + c) * d.Bp + b0 + b] : -INFINITY;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (cb + 4 * q < Cp) child(cb + 4 * q, x[q] > -INFINITY ? x[q] * d.inv_f : -INFINITY);
    }
    for (int gb = 16 * gt0 + part; gb < 16 * gt1; gb += 32) {   // (eight sums' rows requested before the first is used, as above)
      float f[8], v[8], nv[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int g = gb + 4 * q;
        f[q] = 0.f;
        v[q] = 0.f;
        nv[q] = 0.f;
        if (g < min(r.G, 16 * gt1)) {
          const int64_t n = guni(d.node[r.pnode0 + g]);
          f[q] = d.flows[n * d.Bp + b0 + b];
          v[q] = d.mars[n * d.Bp + b0 + b];
          nv[q] = d.norm[(d.norm_row >= 0 ? d.norm_row : n) * d.Bp + b0 + b];
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (gb + 4 * q < 16 * gt1) sum(gb + 4 * q, f[q] > 0.f && v[q] > -INFINITY ? f[q] : 0.f, (mb - v[q]) * d.inv_f - nv[q]);
    }
  };
  if (t == 0) any_again = 0;
  stage([&](int c, float x) {
          const bool far = x < -64.f;   // (where exp(x) alone would run out of float's range on its way up)
          E[c * kGroupPad + b] = __expf(far ? x + kEdgeUp * 0.69314718f : x) * (far ? 1.f : __builtin_ldexpf(1.f, kEdgeUp));
        },
        [&](int g, float f, float tq) {
          const bool high = f > 0.f && tq > kEdgeShare;
          R[g * kGroupPad + b] = f > 0.f && !high ? f * __expf(tq) * __builtin_ldexpf(1.f, -kEdgeDown) : 0.f;
          const uint64_t some = __ballot(f > 0.f), above = __ballot(high);
          if (b == 0) {
            row_some[g] = some;
            row_high[g] = above;
          }
        });
  __syncthreads();
  uint64_t again = 0;   // a bit per (tile of the wave, i): edges with something to be added in logarithms
  int nth = 0;
  for (int tile = gt0 * CT + wave; tile < gt1 * CT; tile += 4, ++nth) {
    const int gt = tile / CT, ct = tile % CT;
    g4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(R[(gt * 16 + lo) * kGroupPad + kk * 4 + hi], E[(ct * 16 + lo) * kGroupPad + kk * 4 + hi],
                                                 acc, 0, 0, 0);
    const int c = ct * 16 + lo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = gt * 16 + 4 * hi + i;
      const int edge = g < r.G && c < r.C ? d.edge[r.pw0 + g * Cp + c] : -1;
      if (edge < 0) continue;   // (in a masked group also a child the sum does not have)
      const float w = d.wf[r.pw0 + group_wf_index(g, c, CT)];
      part_row[edge] = w > 0.f ? w * acc[i] * __builtin_ldexpf(1.f, kEdgeDown - kEdgeUp) : 0.f;
      if (group_tiny_w(w) ? row_some[g] : row_high[g]) again |= (uint64_t)1 << (4 * nth + i);
    }
  }
  if (again) any_again = 1;
  __syncthreads();
  if (!any_again) return;
  stage([&](int c, float x) {
          E[c * kGroupPad + b] = x;
          if (b == 0) E[c * kGroupPad + 64] = 0.f;   // (column 64 stands for no example)
        },
        [&](int g, float f, float tq) {
          R[g * kGroupPad + b] = f > 0.f ? __logf(f) + tq : -INFINITY;
          if (b == 0) R[g * kGroupPad + 64] = -INFINITY;
        });
  __syncthreads();
  nth = 0;
  for (int tile = gt0 * CT + wave; tile < gt1 * CT; tile += 4, ++nth) {
    const int mine = (int)(again >> (4 * nth)) & 15;
    if (!__any(mine)) continue;
    const int gt = tile / CT, ct = tile % CT, c = ct * 16 + lo;
    const float* Ec = E + c * kGroupPad;
    const float* Rg = R + (gt * 16 + 4 * hi) * kGroupPad;
    int edge[4];
    float lw[4], flow[4];
    uint64_t own[4], examples = 0;   // the examples of each edge, and of any of the tile's
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = gt * 16 + 4 * hi + i;
      edge[i] = mine >> i & 1 ? d.edge[r.pw0 + g * Cp + c] : -1;
      lw[i] = edge[i] >= 0 ? d.logp[edge[i]] * d.inv_f : 0.f;
      own[i] = edge[i] < 0 ? 0 : group_tiny_w(group_w(lw[i])) ? row_some[g] : row_high[g];
      flow[i] = 0.f;
      examples |= own[i];
    }
    uint32_t half[2] = {(uint32_t)examples, (uint32_t)(examples >> 32)};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      half[0] |= (uint32_t)__shfl_xor((int)half[0], o);
      half[1] |= (uint32_t)__shfl_xor((int)half[1], o);
    }
    examples = (uint64_t)(uint32_t)guni((int)half[1]) << 32 | (uint32_t)guni((int)half[0]);
    // four at a time
    while (examples) {
      int x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = examples ? __builtin_ctzll(examples) : 64;
        examples &= examples - 1;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float e = Ec[x[u]];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float share = __expf(e + Rg[i * kGroupPad + x[u]] + lw[i]);
          flow[i] += own[i] >> (x[u] & 63) & 1 ? share : 0.f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (edge[i] >= 0) part_row[edge[i]] += flow[i];
  }
}

}  // namespace pcm
