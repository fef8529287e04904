// Maximum spanning tree of a weight matrix that is on the device, where it is the only one.
//
// Boruvka: every component takes the largest edge that leaves it, ceil(log2 V) rounds at most, a pass over the matrix each.  An
// edge that is strictly the largest across a cut is in every maximum spanning tree, so if no component in any round has
// two largest edges the tree is unique, and the one that the host's Prim (chow_liu.hip) gives, ties or no ties elsewhere.
// If one has, or if the matrix is not symmetric and finite, the result says so and the caller takes the matrix to the host.
//
// Reference: ChowLiuTrees.jl as src/structures/hclts.jl:17-18 calls it.  3072 vertices: host 5.0 ms (Prim, a vector pass per
// vertex, and 36 MB out), here 0.40 ms: 12 rounds of a row pass (the matrix from the last-level cache) and one workgroup that
// puts the components together.
#include "common.hpp"


namespace pcm {

namespace {
constexpr int kEdgeVertices = 8192;   // most vertices: the components of one workgroup in LDS
constexpr int kRowThreads = 256, kJoinThreads = 1024;

struct EdgeState { int failed, edges; };   // edges: found so far

// a total order of finite floats as unsigned numbers
__device__ __forceinline__ uint32_t edge_order(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  return b & 0x80000000u ? ~b : b | 0x80000000u;
}

__global__ __launch_bounds__(256) void edge_start_kernel(int V, int* __restrict__ label, EdgeState* __restrict__ st) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v < V) label[v] = v;
  if (v == 0) { st->failed = 0; st->edges = 0; }
}

// symmetric and finite off the diagonal: a workgroup takes the tile (i, j) and its mirror
__global__ __launch_bounds__(256) void edge_check_kernel(const float* __restrict__ w, int V, EdgeState* __restrict__ st) {
  __shared__ float t[64][65];
  const int i0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
  if (j0 < i0) return;
  const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
  for (int y = y0; y < 64; y += 4) t[y][x] = i0 + y < V && j0 + x < V ? w[(size_t)(i0 + y) * V + j0 + x] : 0.f;
  __syncthreads();
  bool bad = false;
  for (int y = y0; y < 64; y += 4) {
    const int r = j0 + y, c = i0 + x;   // the mirror's element
    if (r >= V || c >= V || r == c) continue;
    const float m = w[(size_t)r * V + c], o = t[x][y];
    bad |= !(m == o) || !(fabsf(m) < INFINITY);
  }
  if (bad) st->failed = 1;
}

// per vertex: the largest edge to another component, and whether another is as large
__global__ __launch_bounds__(kRowThreads) void edge_row_kernel(const float* __restrict__ w, int V, const int* __restrict__ label,
                                                               const EdgeState* __restrict__ st, float* __restrict__ best_of,
                                                               int* __restrict__ arg_of, int* __restrict__ tie_of) {
  if (st->failed || st->edges == V - 1) return;
  const int v = blockIdx.x, own = label[v];
  const float* row = w + (size_t)v * V;
  float best = -INFINITY;
  int arg = -1, tie = 0;
  auto take = [&](float x, int u, int also) {
    if (u < 0) return;
    if (arg < 0 || x > best) { best = x; arg = u; tie = also; }
    else if (x == best) tie = 1;
  };
  for (int u0 = threadIdx.x; u0 < V; u0 += 4 * kRowThreads) {   // four requests of either kind under way
    float x[4];
    int l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int u = min(u0 + q * kRowThreads, V - 1);
      x[q] = row[u];
      l[q] = label[u];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int u = u0 + q * kRowThreads;
      take(x[q], u < V && l[q] != own ? u : -1, 0);
    }
  }
  __shared__ float bs[kRowThreads / 64];
  __shared__ int as[kRowThreads / 64], ts[kRowThreads / 64];
  for (int o = 32; o > 0; o >>= 1) {
    const float x = __shfl_xor(best, o);
    const int u = __shfl_xor(arg, o), also = __shfl_xor(tie, o);
    if (u >= 0) take(x, u, also);   // (both sides end with the same best and tie; the vertex is only used where there is no tie)
  }
  if ((threadIdx.x & 63) == 0) { bs[threadIdx.x >> 6] = best; as[threadIdx.x >> 6] = arg; ts[threadIdx.x >> 6] = tie; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < kRowThreads / 64; ++q) take(bs[q], as[q], ts[q]);
    best_of[v] = best;
    arg_of[v] = arg;
    tie_of[v] = tie;
  }
}

// one workgroup: every component's largest edge, the components joined over them
__global__ __launch_bounds__(kJoinThreads) void edge_join_kernel(int V, int* __restrict__ label, EdgeState* __restrict__ st,
                                                                 const float* __restrict__ best_of, const int* __restrict__ arg_of,
                                                                 const int* __restrict__ tie_of, int* __restrict__ edges) {
  extern __shared__ uint32_t join_lds[];   // per vertex (a component goes by one of its own): largest | its row | joined to
  __shared__ int found, bad, changed;
  uint32_t* const top = join_lds;
  int* const pick = reinterpret_cast<int*>(join_lds + V);
  int* const to = pick + V;
  const int t = threadIdx.x;
  if (st->failed || st->edges == V - 1) return;
  if (t == 0) { found = st->edges; bad = 0; }
  for (int v = t; v < V; v += kJoinThreads) { top[v] = 0u; pick[v] = -1; to[v] = v; }
  __syncthreads();
  for (int v = t; v < V; v += kJoinThreads)
    if (arg_of[v] >= 0) atomicMax(&top[label[v]], edge_order(best_of[v] + 0.f));   // (+ 0: the two zeros are one weight)
  __syncthreads();
  for (int v = t; v < V; v += kJoinThreads) {
    const int c = label[v];
    if (arg_of[v] < 0 || edge_order(best_of[v] + 0.f) != top[c]) continue;
    if (tie_of[v] || atomicCAS(&pick[c], -1, v) != -1) bad = 1;   // two edges as large: the tree may not be the only one
  }
  __syncthreads();
  if (bad) {
    if (t == 0) st->failed = 1;
    return;
  }
  for (int v = t; v < V; v += kJoinThreads) {
    if (label[v] != v) continue;
    const int a = pick[v];
    if (a < 0) continue;
    const int b = arg_of[a], other = label[b];
    const bool both = pick[other] == b && arg_of[b] == a;   // the other component takes the same edge: one of the two keeps it
    if (both && v > other) { to[v] = other; continue; }
    const int at = atomicAdd(&found, 1);
    if (at < V - 1) { edges[2 * at] = a; edges[2 * at + 1] = b; }
    if (!both) to[v] = other;
  }
  __syncthreads();
  // every component to the end of its chain: it ends at the pair that took one edge, as the largest edges grow along it
  for (int turn = 0; turn < 16; ++turn) {   // (log2 of the vertices at most)
    if (t == 0) changed = 0;
    __syncthreads();
    for (int v = t; v < V; v += kJoinThreads) {
      const int next = to[to[v]];
      if (next != to[v]) { to[v] = next; changed = 1; }
    }
    __syncthreads();
    const int more = changed;
    __syncthreads();
    if (!more) break;
  }
  for (int v = t; v < V; v += kJoinThreads) label[v] = to[label[v]];
  if (t == 0) st->edges = found;
}

__global__ void edge_result_kernel(int V, const EdgeState* __restrict__ st, int* __restrict__ out) {
  out[0] = !st->failed && st->edges == V - 1 ? 1 : 0;
}

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }
}  // namespace

int64_t chow_liu_edges_workspace(int V) { return V < 2 || V > kEdgeVertices ? 0 : (int64_t)(256 + 4 * up256((size_t)V * 4)); }

// out: {1 if the tree is the only one, else 0; then its V - 1 edges}.  Queued on `stream`; waits for nothing, allocates nothing.
void chow_liu_edges(const float* d_w, int V, int32_t* d_out, void* d_work, hipStream_t stream) {
  if (!d_w || !d_out || !d_work) fail(PCM_ERR_ARG, "matrix, output or workspace pointer is null");
  if (V < 2 || V > kEdgeVertices) fail(PCM_ERR_UNSUPPORTED, "2 to %d vertices, got %d", kEdgeVertices, V);
  char* p = static_cast<char*>(d_work);
  EdgeState* st = reinterpret_cast<EdgeState*>(p);
  const size_t row = up256((size_t)V * 4);
  int* label = reinterpret_cast<int*>(p + 256);
  float* best = reinterpret_cast<float*>(p + 256 + row);
  int* arg = reinterpret_cast<int*>(p + 256 + 2 * row);
  int* tie = reinterpret_cast<int*>(p + 256 + 3 * row);
  const int lds = 3 * V * 4, tiles = ceil_div(V, 64);
  PCM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&edge_join_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(edge_start_kernel, dim3(ceil_div(V, 256)), dim3(256), 0, stream, V, label, st);
  hipLaunchKernelGGL(edge_check_kernel, dim3(tiles, tiles), dim3(256), 0, stream, d_w, V, st);
  for (int left = V; left > 1; left = (left + 1) / 2) {   // (a round at least halves the components)
    hipLaunchKernelGGL(edge_row_kernel, dim3(V), dim3(kRowThreads), 0, stream, d_w, V, label, st, best, arg, tie);
    hipLaunchKernelGGL(edge_join_kernel, dim3(1), dim3(kJoinThreads), lds, stream, V, label, st, best, arg, tie, d_out + 1);
  }
  hipLaunchKernelGGL(edge_result_kernel, dim3(1), dim3(1), 0, stream, V, st, d_out);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail(PCM_ERR_HIP, "launch of chow_liu_edges failed: %s", hipGetErrorString(e));
}

}  // namespace pcm
