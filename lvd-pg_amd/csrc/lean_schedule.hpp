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
// A chain never leaves its wave, so a few chains more than waves, all about equally long, run one behind the other: 17 rows of
// 60 nodes off a column take 121 steps where the most urgent sixteen of every step, picked anew, would take 77.  That costs
// little, as a step's time goes with the waves at work in it (0.3 of a full step's with one), and a tree with
// such schedules (K <= 32) runs on the lean walks whatever the general walk kernels' would be: scores of 4096 examples
// of those 17 rows 149 us against 220, 18 rows of 170 386 against 576.  Letting a chain give up its wave to a more
// urgent node, its tile in a slot, saves the steps but hardly time: 140 us there, and where chains and turns are closer it
// loses (32 rows of 32: 81 steps 136 us, 75 steps 144).  Of 20000 trees of rows, crowns and random ones none costs more
// than 1.27 times the fewest steps there could be; the general walk kernels take about 1.7 times as long per step.
//
// Plain C++ (no HIP): also compiled into a host test.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace pcm {

constexpr int kLeanSchedWaves = 16;
constexpr int32_t kLeanSlotKept = 0xfe;   // the tile stays in the registers of the wave
constexpr int32_t kLeanSlotNone = 0xff;   // nobody hands this tile on (a root)
constexpr int32_t kLeanSlotAway = 0xfd;   // the tile goes to or comes from another workgroup

// The lean kernels reach every array with a 32-bit offset from one descriptor, and send a request that is to fetch or store
// nothing 2 GiB further on, past the end: so each array -- parameter blocks and leaf tables here, tiles and categories by the
// batch -- has to be shorter than that.
inline bool lean_array_fits(size_t rows, size_t floats_per_row) { return rows * floats_per_row * 4 < ((size_t)1 << 31); }

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
      if (inner[v].size() > 1)
        std::stable_sort(inner[v].begin(), inner[v].end(), [&](int a, int b) { return chain[a] > chain[b]; });
    }
    std::vector<int32_t> c;
    // post-order places: a node's subtree ends at its own place; the larger child's subtree comes first
    for (int v = n - 1; v >= 0; --v) {
      if (parent[v] < 0) order[v] = v;   // (trees are runs of node numbers that end with their root)
      c.assign(inner[v].begin(), inner[v].end());
      if (c.size() > 1) std::stable_sort(c.begin(), c.end(), [&](int a, int b) { return below[a] < below[b]; });
      int at = order[v] - 1;
      for (int k : c) {
        order[k] = at;
        at -= below[k] + 1;
      }
    }
  }
};

// The nodes one workgroup walks: whole trees, or a part of one whose other parts other workgroups walk.
struct LeanScope {
  std::vector<int32_t> nodes;     // in ascending order
  std::vector<char> in;           // by node
  std::vector<int32_t> release;   // by node: the step before which a tile from another part is not to be expected; may be empty

  LeanScope(const LeanTree& t, int g0, int g1) : in(t.parent.size(), 0) {
    for (int v = g0; v < g1; ++v) add(v);
  }
  LeanScope(const std::vector<int32_t>& part, int g) : in(part.size(), 0) {
    for (int v = 0; v < (int)part.size(); ++v)
      if (part[v] == g) add(v);
  }
  void add(int v) { nodes.push_back(v); in[v] = 1; }
  int ready_at(int v) const { return release.empty() ? 0 : release[v]; }
};

struct LeanSchedule {
  std::vector<int32_t> item;   // [steps][16 waves] node, -1: idle
  // by node: the slot of its tile (going down: of its ratio tile), kLeanSlotKept, kLeanSlotNone or kLeanSlotAway.  Going down,
  // a node's second and third child that are away have a slot too: their parent works there before it sends the tile.
  std::vector<int32_t> slot;
  std::vector<int32_t> step_of;   // by node
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
inline bool lean_place(const LeanTree& t, const LeanScope& in, LeanSchedule& s, int n_slots, bool up) {
  std::vector<int32_t> ring(n_slots), freed;   // the free slots, first in first out
  for (int i = 0; i < n_slots; ++i) ring[i] = i;
  size_t head = 0;
  int n_free = n_slots;
  auto take = [&](int tile) {
    if (s.slot[tile] >= 0) return true;   // (kept, away or nobody's)
    if (!n_free) return false;
    s.slot[tile] = ring[head];
    head = (head + 1) % n_slots;
    --n_free;
    return true;
  };
  auto free_after = [&](int tile) {
    if (s.slot[tile] >= 0 && s.slot[tile] < kLeanSlotAway) freed.push_back(s.slot[tile]);
  };
  for (int st = 0; st < s.steps; ++st) {
    freed.clear();
    for (int w = 0; w < kLeanSchedWaves; ++w) {
      const int n = s.item[(size_t)st * kLeanSchedWaves + w];
      if (n < 0) continue;
      if (up) {
        for (int c : t.inner[n])
          if (in.in[c]) free_after(c);
        if (!take(n)) return false;
      } else {
        free_after(n);
        for (int c : t.inner[n]) {
          if (!take(c)) return false;
          if (!in.in[c]) free_after(c);   // (a slot to work in)
        }
      }
    }
    for (int x : freed) ring[(head + n_free++) % n_slots] = x;
  }
  return true;
}

// From the leaves up.
inline LeanSchedule lean_schedule_up(const LeanTree& t, const LeanScope& in, int n_slots) {
  constexpr int W = kLeanSchedWaves;
  LeanSchedule s;
  s.slot.assign(t.parent.size(), -1);
  s.step_of.assign(t.parent.size(), -1);
  std::vector<int32_t> pending(t.parent.size(), 0), last(W, -1);
  std::vector<char> waiting(t.parent.size(), 0), all(t.parent.size(), 1), starts(t.parent.size(), 0);
  // [0]: nodes without inner children here, [1]: the others; the most urgent first (a forest: earlier trees first) / in the
  // order that finishes subtrees; `later`: nodes that would be ready but for a tile from another part
  LeanHeap by_depth[2], by_order[2], later;
  auto add = [&](int v) {
    if (in.ready_at(v) > s.steps) return later.push(in.ready_at(v), 0, v);
    const int kind = starts[v] ? 0 : 1;
    waiting[v] = 1;
    by_depth[kind].push(t.tree[v], -t.depth[v], v);
    by_order[kind].push(t.order[v], 0, v);
  };
  for (int v : in.nodes) {
    for (int c : t.inner[v]) {
      pending[v] += in.in[c];
      if (!in.in[c]) s.slot[c] = kLeanSlotAway;
    }
    starts[v] = pending[v] == 0;
    if (starts[v]) add(v);
    if (t.parent[v] < 0) s.slot[v] = kLeanSlotNone;
    else if (!in.in[t.parent[v]]) s.slot[v] = kLeanSlotAway;
  }
  int32_t now[W];
  int live = 0;   // tiles nobody has taken yet, those in registers among them
  for (size_t done = 0; done < in.nodes.size(); ++s.steps) {
    for (int v; (v = later.top(all)) >= 0 && in.ready_at(v) <= s.steps;) {
      std::pop_heap(later.e.begin(), later.e.end());
      later.e.pop_back();
      add(v);
    }
    std::fill_n(now, W, -1);
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
    if (!taken && later.top(all) < 0) {
      // tiles wait for a subtree that has not begun (its nodes came late): the deepest node may use the slots left free
      const int start = by_depth[0].top(waiting);
      if (start < 0 || live + 2 > n_slots) return s;
      now[0] = start;
      waiting[start] = 0;
    }
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      if (v < 0) continue;
      for (int c : t.inner[v]) {
        if (!in.in[c]) continue;
        if (last[w] == c) s.slot[c] = kLeanSlotKept;
        --live;
      }
      if (s.slot[v] != kLeanSlotNone && s.slot[v] != kLeanSlotAway) ++live;
    }
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      s.item.push_back(v);
      if (v < 0) continue;
      last[w] = v;
      s.step_of[v] = s.steps;
      ++done;
      const int p = t.parent[v];
      if (p >= 0 && in.in[p] && --pending[p] == 0) add(p);
    }
  }
  s.ok = lean_place(t, in, s, n_slots, true);
  return s;
}

// From the roots down.  A node's first child always follows it on its wave (unless it is away), and its other children take
// a slot each.  A chain that finds none waits, its tile in registers; `careful`: so that not all waves end up waiting, a
// chain is only started if the slots do for what it and the chains under way (but the greediest) still take.
inline LeanSchedule lean_schedule_down(const LeanTree& t, const LeanScope& in, int n_slots, bool careful) {
  constexpr int W = kLeanSchedWaves;
  LeanSchedule s;
  s.slot.assign(t.parent.size(), -1);
  s.step_of.assign(t.parent.size(), -1);
  std::vector<int32_t> last(W, -1), rest(t.parent.size(), 0);
  std::vector<char> waiting(t.parent.size(), 0), all(t.parent.size(), 1);
  auto next = [&](int v) { return t.inner[v].empty() || !in.in[t.inner[v][0]] ? -1 : t.inner[v][0]; };   // on the same wave
  std::vector<int32_t> extra(t.parent.size(), 0);   // slots a node's children take
  for (int v : in.nodes) {
    for (size_t i = 1; i < t.inner[v].size(); ++i) extra[v] += in.in[t.inner[v][i]];
    rest[v] = extra[v] + (next(v) < 0 ? 0 : rest[next(v)]);   // ... a chain's
    if (!t.inner[v].empty() && next(v) < 0) s.slot[t.inner[v][0]] = kLeanSlotAway;
  }
  LeanHeap by_chain, by_size, later;   // longest chain first (a forest: earlier trees first) / those soonest gone again first
  auto add = [&](int v) {
    if (in.ready_at(v) > s.steps) return later.push(in.ready_at(v), 0, v);
    waiting[v] = 1;
    by_chain.push(t.tree[v], -t.chain[v], v);
    by_size.push(t.below[v], -s.steps, v);
  };
  for (int v : in.nodes)
    if (t.parent[v] < 0 || !in.in[t.parent[v]]) {
      add(v);
      s.slot[v] = t.parent[v] < 0 ? kLeanSlotNone : kLeanSlotAway;
    }
  int32_t now[W];
  bool held[W];
  int live = 0;
  for (size_t done = 0; done < in.nodes.size(); ++s.steps) {
    for (int v; (v = later.top(all)) >= 0 && in.ready_at(v) <= s.steps;) {
      std::pop_heap(later.e.begin(), later.e.end());
      later.e.pop_back();
      add(v);
    }
    std::fill_n(now, W, -1);
    std::fill_n(held, W, false);
    int taken = 0, freed = 0, open = 0, widest = 0;
    for (int w = 0; w < W; ++w) {
      const int c = last[w] < 0 ? -1 : next(last[w]);
      if (c < 0) continue;
      held[w] = 1;
      int left = rest[c];
      if (live + extra[c] <= n_slots) {
        live += extra[c];
        left -= extra[c];
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
      const int left = rest[v] - extra[v];
      const bool fits = rest[v] == 0 || (careful ? live + open + rest[v] - std::max(widest, left) <= n_slots
                                                 : live + extra[v] <= n_slots - W / 2);
      if (!fits) continue;
      waiting[v] = 0;
      live += extra[v];
      open += left;
      widest = std::max(widest, left);
      if (s.slot[v] == -1) ++freed;   // its slot is free again after the step
      now[w] = v;
      ++taken;
    }
    if (!taken && later.top(all) < 0) return s;
    live -= freed;
    for (int w = 0; w < W; ++w) {
      const int v = now[w];
      s.item.push_back(v);
      if (v < 0) continue;
      last[w] = v;
      s.step_of[v] = s.steps;
      ++done;
      for (size_t i = 1; i < t.inner[v].size(); ++i)
        if (in.in[t.inner[v][i]]) add(t.inner[v][i]);
    }
  }
  s.ok = lean_place(t, in, s, n_slots, false);
  return s;
}

inline LeanSchedule lean_schedule_down(const LeanTree& t, const LeanScope& in, int n_slots) {
  LeanSchedule s = lean_schedule_down(t, in, n_slots, false);
  return s.ok ? s : lean_schedule_down(t, in, n_slots, true);
}

// One tree cut for `G` workgroups: part 0 has the top of the tree, everything more than 1 / (2 G) of the nodes hang from,
// and the subtrees below it are dealt to the parts, largest first, each to the part with the fewest nodes.  So a tile
// crosses at most once on its way up or down, and only part 0 waits (going up) or is waited for (going down).  A subtree of
// fewer than kLeanCutNodes nodes is not worth the crossing and stays with the top.  `*largest`: nodes of the largest part.
constexpr int kLeanCutNodes = 6;
inline std::vector<int32_t> lean_parts(const LeanTree& t, int G, int* largest) {
  const int n = (int)t.parent.size(), most = std::max(kLeanCutNodes, n / (2 * G));
  std::vector<int32_t> part(n, 0), load(G, 0), cut;
  for (int v = 0; v < n; ++v) {
    const bool small = t.below[v] + 1 <= most;
    if (!small || t.parent[v] < 0) ++load[0];
    else if (t.below[t.parent[v]] + 1 > most || t.parent[t.parent[v]] < 0) {
      if (t.below[v] + 1 < kLeanCutNodes) load[0] += t.below[v] + 1;
      else cut.push_back(v);
    }
  }
  std::stable_sort(cut.begin(), cut.end(), [&](int a, int b) { return t.below[a] > t.below[b]; });
  for (int v : cut) {
    const int g = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    part[v] = g;
    load[g] += t.below[v] + 1;
  }
  for (int v = n - 1; v >= 0; --v)   // (parents have higher numbers)
    if (t.parent[v] >= 0 && part[v] == 0) part[v] = part[t.parent[v]];
  *largest = *std::max_element(load.begin(), load.end());
  return part;
}

// What a walk up one tree in such parts takes, in us (K = 16 or 32): as long as its longest chain or as the sixteen waves of the
// largest part need, or a little more where the two are close.  A node that merges two chains or more waits for the others'
// tiles; one with children in other parts fetches their tiles from memory, one behind the other, and that is all on the chain
// where a spine has a branch at every node: 200 nodes with 8 below each, K = 16, 170 us in one part, 208 in two, 292 in eight
// (K = 32: 251, 261, 289).  So more parts are taken only while this says that they gain.  Fitted to 121 measured walks of 256
// examples through 19 trees (spines, crowns, random and Chow-Liu trees of 200 to 2500 nodes) in 1 to 16 parts, off by 9 % on
// average; of those trees, taking as many parts as their nodes allow costs 13 % more than the best number of parts on average and
// 72 % at worst at the scores (5 and 32 % for a whole EM step), taking them by this 1.4 and 11 % (1.1 and 14).
inline double lean_walk_us(const LeanTree& t, const std::vector<int32_t>& part, int largest, int K) {
  const double node = 0.4, merge = K > 16 ? 0.95 : 0.75, away = K > 16 ? 0.33 : 0.7, late = 4.0, full_step = K > 16 ? 1.9 : 1.0;
  const int n = (int)t.parent.size();
  std::vector<double> at(n, 0.0);   // when a node's tile is there
  double chain = 0.0;
  for (int v = 0; v < n; ++v) {
    int crossing = 0;
    for (int c : t.inner[v]) {
      const bool crosses = part[c] != part[v];
      crossing += crosses;
      at[v] = std::max(at[v], at[c] + (crosses ? late : 0.0));
    }
    at[v] += (t.inner[v].size() < 2 ? node : merge) + away * crossing;
    chain = std::max(chain, at[v]);
  }
  const double waves = full_step * largest / kLeanSchedWaves;
  return std::cbrt(chain * chain * chain + waves * waves * waves);
}

}  // namespace pcm
