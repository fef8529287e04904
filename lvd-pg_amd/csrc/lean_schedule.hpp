// Step schedules of the lean tree walks (hclt_walk_lean.hip.hpp): which tree node each of the sixteen waves of a
// workgroup takes in which step, and which LDS slot a tile passes through on its way from one wave to another.
//
// A wave follows a chain: going up it takes the parent of the node it has just done as soon as that parent's other
// children are there too; going down it takes the first child (the one with the longest chain below) of the node it has
// just done.  The tile handed from the one to the other then never leaves the wave's registers, and only the tiles that
// change waves -- one per end of a chain -- take a slot.  Trees learned from images are mostly chains: of the 2507 inner
// nodes of a 3072-variable one 2030 are handed on in registers, in as many steps (167, the fewest 16 waves can do) as a
// schedule that picks the most urgent sixteen nodes of each step anew (619 in registers by luck), and 32 tiles wait in LDS
// at a time instead of 57.  An idle wave starts the most urgent node that is ready: the deepest going up, the one with the
// longest chain below going down.  That order opens many subtrees at once, so with more than half of the slots taken the
// order is the one that finishes subtrees instead.
//
// Plain C++ (no HIP): also compiled into a host test.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace pcm {

constexpr int kLeanSchedWaves = 16;
constexpr int32_t kLeanSlotKept = 0xfe;   // the tile stays in the registers of the wave
constexpr int32_t kLeanSlotNone = 0xff;   // nobody hands this tile on (a root)

struct LeanTree {   // inner nodes, children before their parents
  std::vector<int32_t> parent;               // -1: a root
  std::vector<std::vector<int32_t>> inner;   // inner children, longest chain first
  std::vector<int32_t> tree, depth;
  std::vector<int32_t> chain, below;         // longest chain of inner nodes below; inner nodes below
  std::vector<int32_t> order;                // place in a depth-first order that takes the larger subtree first

  // parent, inner, tree and depth are there; fills the rest and puts the children in order
  void complete() {
    const int n = (int)parent.size();
    chain.assign(n, 0);
    below.assign(n, 0);
    order.assign(n, 0);
    for (int v = 0; v < n; ++v) {
      for (int c : inner[v]) {
        chain[v] = std::max(chain[v], chain[c] + 1);
        below[v] += below[c] + 1;
      }
      std::stable_sort(inner[v].begin(), inner[v].end(), [&](int a, int b) { return chain[a] > chain[b]; });
    }
    // post-order places: a node's subtree ends at its own place; the larger child's subtree comes first
    for (int v = n - 1; v >= 0; --v) {
      if (parent[v] < 0) order[v] = v;   // (trees are runs of node numbers that end with their root)
      std::vector<int32_t> c = inner[v];
      std::stable_sort(c.begin(), c.end(), [&](int a, int b) { return below[a] < below[b]; });
      int at = order[v] - 1;
      for (int k : c) {
        order[k] = at;
        at -= below[k] + 1;
      }
    }
  }
};

struct LeanSchedule {
  std::vector<int32_t> item;   // [steps][16 waves] node, -1: idle
  std::vector<int32_t> slot;   // by node: the slot of its tile (going down: of its ratio tile), kLeanSlotKept or kLeanSlotNone
  int steps = 0;
  bool ok = false;             // false: the slots do not do
};

// Nodes that wait for a wave, by a key of two numbers (smallest first, then the lower node).  A node may be in several
// heaps; whoever takes it marks it, and the others drop it when it comes to their top.
struct LeanHeap {
  struct Entry {
    int32_t a, b, node;
    bool operator<(const Entry& o) const { return a != o.a ? a > o.a : b != o.b ? b > o.b : node > o.node; }
  };
  std::vector<Entry> e;
  void push(int32_t a, int32_t b, int32_t node) {
    e.push_back({a, b, node});
    std::push_heap(e.begin(), e.end());
  }
  int top(const std::vector<char>& waiting) {   // -1: empty
    while (!e.empty() && !waiting[e.front().node]) {
      std::pop_heap(e.begin(), e.end());
      e.pop_back();
    }
    return e.empty() ? -1 : e.front().node;
  }
};

// The slot that has been free longest is taken first: a wave then hardly ever waits for the reader of the tile before.
inline bool lean_place(const LeanTree& t, LeanSchedule& s, int n_slots, bool up) {
  std::vector<int32_t> ring(n_slots), freed;   // the free slots, first in first out
  for (int i = 0; i < n_slots; ++i) ring[i] = i;
  size_t head = 0;
  int n_free = n_slots;
  auto take = [&](int tile) {
    if (s.slot[tile] >= 0) return true;   // (kept, or nobody's)
    if (!n_free) return false;
    s.slot[tile] = ring[head];
    head = (head + 1) % n_slots;
    --n_free;
    return true;
  };
  auto free_after = [&](int tile) {
    if (s.slot[tile] < kLeanSlotKept) freed.push_back(s.slot[tile]);
  };
  for (int st = 0; st < s.steps; ++st) {
    freed.clear();
    for (int w = 0; w < kLeanSchedWaves; ++w) {
      const int n = s.item[(size_t)st * kLeanSchedWaves + w];
      if (n < 0) continue;
      if (up) {
        for (int c : t.inner[n]) free_after(c);
        if (!take(n)) return false;
      } else {
        free_after(n);
        for (int c : t.inner[n])
          if (!take(c)) return false;
      }
    }
    for (int x : freed) ring[(head + n_free++) % n_slots] = x;
  }
  return true;
}

// Nodes g0 .. g1 - 1 (whole trees) from the leaves up.
inline LeanSchedule lean_schedule_up(const LeanTree& t, int g0, int g1, int n_slots) {
  constexpr int W = kLeanSchedWaves;
  LeanSchedule s;
  s.slot.assign(t.parent.size(), -1);
  std::vector<int32_t> pending(t.parent.size(), 0), last(W, -1);
  std::vector<char> waiting(t.parent.size(), 0);
  // [0]: nodes without inner children, [1]: the others; the most urgent first (a forest: earlier trees first) / in the order
  // that finishes subtrees
  LeanHeap by_depth[2], by_order[2];
  auto add = [&](int v) {
    const int kind = t.inner[v].empty() ? 0 : 1;
    waiting[v] = 1;
    by_depth[kind].push(t.tree[v], -t.depth[v], v);
    by_order[kind].push(t.order[v], 0, v);
  };
  for (int v = g0; v < g1; ++v) {
    pending[v] = (int32_t)t.inner[v].size();
    if (!pending[v]) add(v);
  }
  int live = 0;   // tiles nobody has taken yet, those in registers among them
  for (int done = 0; done < g1 - g0;) {
    std::vector<int32_t> now(W, -1);
    int taken = 0;
    for (int w = 0; w < W; ++w) {   // chains first; of several children that could hand on in registers the first does
      const int c = last[w], p = c < 0 ? -1 : t.parent[c];
      if (p < 0 || !waiting[p]) continue;   // (its other children are not there yet, or it is done)
      bool mine = true;
      for (int o : t.inner[p]) {
        if (o == c) break;
        if (std::find(last.begin(), last.end(), o) != last.end()) mine = false;
      }
      if (mine) now[w] = p;
    }
    for (int w = 0; w < W; ++w)
      if (now[w] >= 0) {
        waiting[now[w]] = 0;
        ++taken;
      }
    for (int w = 0; w < W; ++w) {
      if (now[w] >= 0) continue;
      LeanHeap* const heap = 2 * live <= n_slots ? by_depth : by_order;
      // a node without inner children adds a tile: it leaves a slot per wave to the nodes that take tiles
      const int start = live + taken + 1 <= n_slots - W ? heap[0].top(waiting) : -1, merge = heap[1].top(waiting);
      int pick = merge < 0 ? start : merge;
      if (start >= 0 && merge >= 0 && heap[1].e.front() < heap[0].e.front()) pick = start;
      if (pick < 0) break;
      now[w] = pick;
      waiting[pick] = 0;
      ++taken;
    }
    if (!taken) return s;   // only nodes that need a slot, and none is left
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      if (v < 0) continue;
      for (int c : t.inner[v]) {
        if (last[w] == c) s.slot[c] = kLeanSlotKept;
        --live;
      }
      if (t.parent[v] >= 0) ++live; else s.slot[v] = kLeanSlotNone;
    }
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      s.item.push_back(v);
      if (v < 0) continue;
      last[w] = v;
      ++done;
      const int p = t.parent[v];
      if (p >= 0 && --pending[p] == 0) add(p);
    }
    ++s.steps;
  }
  s.ok = lean_place(t, s, n_slots, true);
  return s;
}

// Nodes g0 .. g1 - 1 (whole trees) from the roots down.  A node's first child always follows it on its wave, and its other
// children take a slot each.  A chain that finds none waits, its tile in registers; `careful`: so that not all waves end up
// waiting, a chain is only started if the slots do for what it and the chains under way (but the greediest) still take.
inline LeanSchedule lean_schedule_down(const LeanTree& t, int g0, int g1, int n_slots, bool careful) {
  constexpr int W = kLeanSchedWaves;
  LeanSchedule s;
  s.slot.assign(t.parent.size(), -1);
  std::vector<int32_t> last(W, -1), rest(t.parent.size(), 0);
  std::vector<char> waiting(t.parent.size(), 0);
  auto extra = [&](int v) { return std::max(0, (int)t.inner[v].size() - 1); };   // slots a node's children take
  for (int v = g0; v < g1; ++v) rest[v] = extra(v) + (t.inner[v].empty() ? 0 : rest[t.inner[v][0]]);   // ... a chain's
  LeanHeap by_chain, by_size;   // longest chain first (a forest: earlier trees first) / those soonest gone again first
  auto add = [&](int v) {
    waiting[v] = 1;
    by_chain.push(t.tree[v], -t.chain[v], v);
    by_size.push(t.below[v], -s.steps, v);
  };
  for (int v = g0; v < g1; ++v)
    if (t.parent[v] < 0) {
      add(v);
      s.slot[v] = kLeanSlotNone;
    }
  int live = 0;
  for (int done = 0; done < g1 - g0; ++s.steps) {
    std::vector<int32_t> now(W, -1);
    std::vector<char> held(W, 0);
    int taken = 0, freed = 0, open = 0, widest = 0;
    for (int w = 0; w < W; ++w) {
      if (last[w] < 0 || t.inner[last[w]].empty()) continue;
      held[w] = 1;
      const int c = t.inner[last[w]][0];
      int left = rest[c];
      if (live + extra(c) <= n_slots) {
        live += extra(c);
        left -= extra(c);
        now[w] = c;
        s.slot[c] = kLeanSlotKept;
        ++taken;
      }
      open += left;
      widest = std::max(widest, left);
    }
    for (int w = 0; w < W; ++w) {
      if (held[w]) continue;
      last[w] = -1;
      const int v = (2 * live <= n_slots && !careful ? by_chain : by_size).top(waiting);
      if (v < 0) continue;
      const int left = rest[v] - extra(v);
      const bool fits = rest[v] == 0 || (careful ? live + open + rest[v] - std::max(widest, left) <= n_slots
                                                 : live + extra(v) <= n_slots - W / 2);
      if (!fits) continue;
      waiting[v] = 0;
      live += extra(v);
      open += left;
      widest = std::max(widest, left);
      if (t.parent[v] >= 0) ++freed;   // its slot is free again after the step
      now[w] = v;
      ++taken;
    }
    if (!taken) return s;
    live -= freed;
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      s.item.push_back(v);
      if (v < 0) continue;
      last[w] = v;
      ++done;
      for (size_t i = 1; i < t.inner[v].size(); ++i) add(t.inner[v][i]);
    }
  }
  s.ok = lean_place(t, s, n_slots, false);
  return s;
}

inline LeanSchedule lean_schedule_down(const LeanTree& t, int g0, int g1, int n_slots) {
  LeanSchedule s = lean_schedule_down(t, g0, g1, n_slots, false);
  return s.ok ? s : lean_schedule_down(t, g0, g1, n_slots, true);
}

}  // namespace pcm
