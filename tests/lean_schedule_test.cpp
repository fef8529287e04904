// Host test of csrc/lean_schedule.hpp and csrc/lean_rows.hpp: schedules of chains, stars, binary and random trees, one tree or several, for many
// and few slots.  Every schedule is replayed step by step.  Prints "<name> <number>" lines.
#include <cstdio>
#include <random>

#include "lean_rows.hpp"
#include "lean_schedule_check.hpp"

using namespace pcm;

// What the steps of a walk over so many nodes cost, a step with all sixteen waves at work being 1.  (17 rows of 60 nodes against
// 16: 45 steps with one wave more, 22 us more; the 76 others take 128.)
static double steps_cost(int steps, size_t nodes) { return 0.3 * steps + 0.7 * (double)nodes / kLeanSchedWaves; }

// inner nodes only, children before their parents: parent[v] > v, or -1
static LeanTree make(const std::vector<int>& parent) {
  LeanTree t;
  const int n = (int)parent.size();
  t.parent.assign(parent.begin(), parent.end());
  t.inner.resize(n);
  t.tree.assign(n, 0);
  t.depth.assign(n, 0);
  for (int v = 0; v < n; ++v)
    if (parent[v] >= 0) t.inner[parent[v]].push_back(v);
  for (int v = n - 1; v >= 0; --v) t.depth[v] = parent[v] < 0 ? 0 : t.depth[parent[v]] + 1;
  for (int v = 0, k = 0; v < n; ++v) {
    t.tree[v] = k;
    if (parent[v] < 0) ++k;
  }
  t.complete();
  return t;
}

// the same tree, given from the root (up_to[v] < v), with children before their parents
static std::vector<int> from_root(const std::vector<int>& up_to) {
  const int n = (int)up_to.size();
  std::vector<std::vector<int>> ch(n);
  for (int v = 1; v < n; ++v) ch[up_to[v]].push_back(v);
  std::vector<int> id(n), parent(n, -1);
  std::vector<std::pair<int, size_t>> st{{0, 0}};
  for (int k = 0; !st.empty();) {
    auto& top = st.back();
    if (top.second < ch[top.first].size()) { const int c = ch[top.first][top.second++]; st.push_back({c, 0}); }
    else { id[top.first] = k++; st.pop_back(); }
  }
  for (int v = 1; v < n; ++v) parent[id[v]] = id[up_to[v]];
  return parent;
}

// 0 if the schedule is right: every node of the scope once, what a node reads was written in an earlier step and is where it
// looks for it (tiles from other workgroups excepted)
static int fault(const LeanTree& t, const LeanSchedule& s, const LeanScope& in, int n_slots, bool up) {
  std::vector<int> step(t.parent.size(), -1), in_slot(n_slots, -1), last(kLeanSchedWaves, -1);
  size_t done = 0;
  for (int st = 0; st < s.steps; ++st) {
    std::vector<std::pair<int, int>> put;
    std::vector<int> scratch;
    for (int w = 0; w < kLeanSchedWaves; ++w) {
      const int v = s.item[(size_t)st * kLeanSchedWaves + w];
      if (v < 0) continue;
      if (!in.in[v] || step[v] >= 0 || s.step_of[v] != st) return 1;
      const std::vector<int32_t> reads = up ? t.inner[v] : std::vector<int32_t>{v};
      for (int r : reads) {
        const int from = up ? r : t.parent[v];
        if (from < 0) { if (s.slot[v] != kLeanSlotNone) return 2; continue; }
        if (!in.in[from]) { if (s.slot[r] != kLeanSlotAway) return 8; continue; }
        if (step[from] < 0 || step[from] >= st) return 3;
        if (s.slot[r] == kLeanSlotKept) {
          if (last[w] != from || (!up && t.inner[from][0] != v)) return 4;
        } else {
          if (s.slot[r] < 0 || s.slot[r] >= n_slots || in_slot[s.slot[r]] != r) return 5;
          in_slot[s.slot[r]] = -1;
        }
      }
      if (up && t.parent[v] >= 0 && !in.in[t.parent[v]] && s.slot[v] != kLeanSlotAway) return 9;
      const std::vector<int32_t> writes = up ? std::vector<int32_t>{v} : t.inner[v];
      for (int x : writes)
        if (s.slot[x] < kLeanSlotAway) {
          put.push_back({s.slot[x], x});
          if (!up && !in.in[x]) scratch.push_back(s.slot[x]);
        } else if (!up && !in.in[x] && x != t.inner[v][0]) {
          return 10;
        }
      step[v] = st;
      ++done;
      last[w] = v;
    }
    for (auto& p : put) {
      if (p.first < 0 || p.first >= n_slots || in_slot[p.first] >= 0) return 6;
      in_slot[p.first] = p.second;
    }
    for (int x : scratch) in_slot[x] = -1;
  }
  return done == in.nodes.size() ? 0 : 7;
}

int main() {
  std::mt19937 rng(3);
  auto chain = [](int n) { std::vector<int> p(n); for (int v = 0; v < n; ++v) p[v] = v + 1 < n ? v + 1 : -1; return p; };
  {
    const LeanTree t = make(chain(40));
    const LeanSchedule a = lean_schedule_up(t, LeanScope(t, 0, 40), 20), b = lean_schedule_down(t, LeanScope(t, 0, 40), 20);
    int kept = 0;
    for (int v = 0; v < 40; ++v) kept += (a.slot[v] == kLeanSlotKept) + (b.slot[v] == kLeanSlotKept);
    std::printf("chain_steps %d\nchain_kept %d\n", a.steps + b.steps, kept);
  }
  // arrays the lean kernels can address: blocks of K = 32 are 4 KB, 2^19 of them 2 GiB
  std::printf("array_fits %d\narray_too_long %d\n", lean_array_fits((1 << 19) - 1, 32 * 32) + lean_array_fits((1 << 21) - 1, 16 * 16) + lean_array_fits(1, 1),
              !lean_array_fits(1 << 19, 32 * 32) + !lean_array_fits(1 << 21, 16 * 16) + !lean_array_fits((size_t)1 << 30, (size_t)1 << 31));
  int faults = 0, refused_many = 0, refused_few = 0, long_ones = 0, handed = 0;
  for (int i = 0; i < 600; ++i) {
    const int n = 1 + (int)(rng() % (i % 10 == 0 ? 1500 : 200));
    const int span = i % 3 == 0 ? n : 1 + (int)(rng() % 12), trees = i % 4 == 0 ? 1 + (int)(rng() % 6) : 1;
    std::vector<int> p(n), kids(n, 0);
    for (int v = 0; v < n; ++v) {   // parents with fewer than three children, within `span` of the node
      p[v] = -1;
      for (int tries = 0; tries < 40 && p[v] < 0 && v + 1 < n; ++tries) {
        const int q = std::min(n - 1, v + 1 + (int)(rng() % span));
        if (kids[q] < 3 && q != v) { p[v] = q; ++kids[q]; }
      }
      for (int q = v + 1; q < n && p[v] < 0; ++q)
        if (kids[q] < 3) { p[v] = q; ++kids[q]; }
    }
    // post-order numbering, tree after tree: relabel a forest of `trees` copies
    std::vector<int> all;
    {
      std::vector<std::vector<int>> ch(n);
      for (int v = 0; v < n; ++v) if (p[v] >= 0) ch[p[v]].push_back(v);
      std::vector<int> id(n, -1), post;
      std::vector<std::pair<int, size_t>> st{{n - 1, 0}};
      while (!st.empty()) {
        auto& top = st.back();
        if (top.second < ch[top.first].size()) { const int c = ch[top.first][top.second++]; st.push_back({c, 0}); }
        else { id[top.first] = (int)post.size(); post.push_back(top.first); st.pop_back(); }
      }
      for (int k = 0; k < trees; ++k)
        for (size_t v = 0; v < post.size(); ++v) all.push_back(p[post[v]] < 0 ? -1 : id[p[post[v]]] + k * (int)post.size());
    }
    const LeanTree t = make(all);
    const int m = (int)all.size();
    int deep = 0;
    for (int v = 0; v < m; ++v) deep = std::max(deep, t.depth[v] + 1);
    for (int n_slots : {79, 24}) {
      const LeanSchedule a = lean_schedule_up(t, LeanScope(t, 0, m), n_slots), b = lean_schedule_down(t, LeanScope(t, 0, m), n_slots);
      for (const LeanSchedule* s : {&a, &b}) {
        if (!s->ok) { ++(n_slots == 79 ? refused_many : refused_few); continue; }
        const int f = fault(t, *s, LeanScope(t, 0, m), n_slots, s == &a);
        if (f) { ++faults; std::fprintf(stderr, "tree %d (%d nodes), %d slots, %s: fault %d\n", i, m, n_slots, s == &a ? "up" : "down", f); }
        if (n_slots == 79 && s->steps > std::max(deep, (m + 15) / 16) * 1.4 + 4) ++long_ones;
        for (int v = 0; v < m; ++v) handed += s->slot[v] == kLeanSlotKept;
      }
    }
  }
  // rows of equally long chains off a column, crowns with chains below: what the steps cost, over the fewest there could be
  double worst = 0;
  int shapes = 0, shape_faults = 0;
  auto look = [&](const std::vector<int>& up_to) {   // numbered from the root
    const int n = (int)up_to.size();
    const LeanTree t = make(from_root(up_to));
    int deep = 0;
    for (int v = 0; v < n; ++v) deep = std::max(deep, t.depth[v] + 1);
    const LeanScope in(t, 0, n);
    const LeanSchedule a = lean_schedule_up(t, in, 79), b = lean_schedule_down(t, in, 79);
    if (!a.ok || !b.ok || fault(t, a, in, 79, true) || fault(t, b, in, 79, false)) ++shape_faults;
    worst = std::max(worst, steps_cost(a.steps + b.steps, 2 * n) / steps_cost(2 * std::max(deep, (n + 15) / 16), 2 * n));
    ++shapes;
  };
  auto chain_at = [](std::vector<int>& up, int p, int length) {
    for (int i = 0; i < length; ++i) { up.push_back(p); p = (int)up.size() - 1; }
    return p;
  };
  for (int rows : {2, 15, 16, 17, 18, 20, 24, 31, 32, 33, 40, 47, 48, 49, 64, 100})
    for (int length : {1, 9, 20, 28, 32, 60, 170}) {
      std::vector<int> up{-1}, column{0};
      for (int r = 1; r < rows; ++r) column.push_back(chain_at(up, column.back(), 1));
      for (int r = 0; r < rows; ++r) chain_at(up, column[r], length);
      if (up.size() < 4000) look(up);
    }
  for (int levels : {1, 3, 5, 7})
    for (int above : {0, 50, 150})
      for (int length : {0, 3, 10, 40}) {
        std::vector<int> up{-1}, now;
        now.push_back(chain_at(up, 0, above));
        for (int l = 0; l < levels; ++l) {
          std::vector<int> next;
          for (int p : now) { next.push_back(chain_at(up, p, 1)); next.push_back(chain_at(up, p, 1)); }
          now.swap(next);
        }
        for (int p : now) chain_at(up, p, length);
        look(up);
      }
  std::printf("shapes %d\nshape_faults %d\nshape_cost %d\n", shapes, shape_faults, (int)(worst * 100));
  // trees over several workgroups: a tile crosses once, between the top and another part, every part's schedule is right, and
  // the field rows of all parts together let every wave through and leave the exchange empty.  taken[G]: cuts the engine's
  // rule takes at K = 32 (the largest part no more than three quarters of that of the cut before, and the walk shorter).
  int cut_trees = 0, cut_pairs = 0, cut_faults = 0, cut_refused = 0, cut_stuck = 0, taken[17] = {0};
  for (int i = 0; i < 120; ++i) {
    const int n = 60 + (int)(rng() % 2500), span = i % 3 == 0 ? n : i % 3 == 1 ? 2 + (int)(rng() % 10) : 20 + (int)(rng() % 200);
    std::vector<int> up_to(n, -1), kids(n, 0);   // numbered from the root, every node below one of its `span` predecessors
    for (int v = 1; v < n; ++v) {
      int q = std::max(0, v - 1 - (int)(rng() % span));
      while (kids[q] >= 3) q = q + 1 < v ? q + 1 : 0;
      up_to[v] = q;
      ++kids[q];
    }
    const LeanTree t = make(from_root(up_to));
    LeanNodes nd;
    nd.K = 32;
    nd.leaf_stride = 512;
    for (int v = 0, var = 0; v < n; ++v) {
      nd.var.push_back(var++);
      nd.leaves.push_back({});
      for (size_t room = 3 - t.inner[v].size(), k = t.inner[v].empty() ? 1 + rng() % room : rng() % (room + 1); k > 0; --k) nd.leaves[v].push_back(var++);
    }
    ++cut_trees;
    int before = n;
    bool going = true;
    double us = lean_walk_us(t, std::vector<int32_t>(n, 0), n, 32);
    for (int G : {2, 4, 8, 16}) {
      int largest = 0, most = 0;
      const std::vector<int32_t> part = lean_parts(t, G, &largest);
      for (int g = 0; g < G; ++g) most = std::max(most, (int)std::count(part.begin(), part.end(), g));
      if (most != largest) ++cut_faults;
      const double part_us = lean_walk_us(t, part, largest, 32);
      going = going && largest <= 3 * before / 4 && part_us <= us;
      before = largest;
      us = part_us;
      taken[G] += going;
      ++cut_pairs;
      for (int v = 0; v < n; ++v)
        if (part[v] < 0 || part[v] >= G || (t.parent[v] >= 0 && part[v] != part[t.parent[v]] && part[t.parent[v]] != 0)) ++cut_faults;
      std::vector<LeanScope> scopes;
      for (int g = 0; g < G; ++g) {
        scopes.push_back(LeanScope(part, g));
        LeanScope in = scopes.back(), late = in;   // tiles from other parts: the top waits for them going up, the others going down
        late.release.assign(n, 0);
        for (int v = 0; v < n; ++v)
          if (t.parent[v] >= 0 && part[v] != part[t.parent[v]]) {
            const int x = g == 0 ? t.parent[v] : v;
            late.release[x] = std::max(late.release[x], (int32_t)(rng() % 40));
          }
        const LeanSchedule a = lean_schedule_up(t, g == 0 ? late : in, 79), b = lean_schedule_down(t, g == 0 ? in : late, 79);
        for (const LeanSchedule* s : {&a, &b}) {
          if (!s->ok) { ++cut_refused; continue; }
          const int f = fault(t, *s, in, 79, s == &a);
          if (f) { ++cut_faults; std::fprintf(stderr, "cut tree %d (%d nodes), part %d of %d, %s: fault %d\n", i, n, g, G, s == &a ? "up" : "down", f); }
        }
      }
      LeanPlanRows p;
      if (!lean_plan_rows(t, nd, scopes, part, 79, p)) { ++cut_refused; continue; }
      int crossing = 0;
      for (int v = 0; v < n; ++v) crossing += t.parent[v] >= 0 && part[v] != part[t.parent[v]];
      if (crossing != p.n_away) ++cut_faults;
      for (const bool forward : {true, false}) {
        std::vector<uint8_t> flags;
        const int stuck = lean_rows_stuck_at(p.rows[!forward].data(), G, p.stride[!forward], p.steps[!forward], forward, kLeanSlotNone, &flags);
        if (stuck >= 0 || (int)flags.size() != p.n_away || std::count(flags.begin(), flags.end(), 0) != p.n_away) {
          ++cut_stuck;
          std::fprintf(stderr, "cut tree %d (%d nodes), %d parts, %s: stuck at %d, %d flags of %d\n", i, n, G, forward ? "up" : "down", stuck,
                       (int)flags.size(), p.n_away);
        }
        // every node in one group, a wave's last step where the row behind says
        std::vector<int> seen(n, 0);
        const size_t per_group = (size_t)kLeanFields * kLeanSchedWaves * p.stride[!forward] + kLeanSchedWaves;
        for (int g = 0; g < G; ++g)
          for (int w = 0; w < kLeanSchedWaves; ++w) {
            const int32_t* const f = p.rows[!forward].data() + g * per_group;
            for (int st = 0; st < p.stride[!forward]; ++st) {
              const int v = f[((size_t)kLNode * kLeanSchedWaves + w) * p.stride[!forward] + st];
              if ((v != n) != (st < f[per_group - kLeanSchedWaves + w])) ++cut_faults;
              if (v != n) ++seen[v];
            }
          }
        cut_faults += (int)(n - std::count(seen.begin(), seen.end(), 1));
      }
    }
  }
  std::printf("cut_trees %d\ncut_pairs %d\ncut_faults %d\ncut_refused %d\ncut_stuck %d\n", cut_trees, cut_pairs, cut_faults, cut_refused, cut_stuck);
  for (int G : {2, 4, 8, 16}) std::printf("taken_%d %d\n", G, taken[G]);
  // a spine with a branch at every node waits for what crosses, a crown of chains does not: parts that gain, of 2, 4, 8 and 16
  auto gains = [&](int spine, int branch, int levels, int K) {
    std::vector<int> up{-1}, ends{0};
    if (spine)
      for (int i = 0, p = 0; i < spine; ++i, p = (int)up.size() - 1) {
        chain_at(up, p, branch);
        up.push_back(p);
      }
    for (int l = 0; l < levels; ++l) {
      std::vector<int> below;
      for (int u : ends)
        for (int k = 0; k < 2; ++k) below.push_back(chain_at(up, u, l + 1 < levels ? 1 : branch));
      ends = below;
    }
    const LeanTree t = make(from_root(up));
    const int n = (int)up.size();
    double us = lean_walk_us(t, std::vector<int32_t>(n, 0), n, K);
    int best = 1;
    for (int G : {2, 4, 8, 16}) {
      int largest = 0;
      const std::vector<int32_t> part = lean_parts(t, G, &largest);
      const double x = lean_walk_us(t, part, largest, K);
      if (x > us) break;
      us = x;
      best = G;
    }
    return best;
  };
  std::printf("gain_spine_16 %d\ngain_spine_32 %d\ngain_crown_16 %d\ngain_crown_32 %d\n", gains(200, 7, 0, 16), gains(200, 7, 0, 32),
              gains(0, 40, 5, 16), gains(0, 40, 5, 32));
  std::printf("faults %d\nrefused_many %d\nrefused_few %d\nlong %d\nhanded %d\n", faults, refused_many, refused_few, long_ones, handed > 0);
  return 0;
}
