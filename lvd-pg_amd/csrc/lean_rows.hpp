// Field rows of the lean tree walks: what the schedules of lean_schedule.hpp become for the kernels of
// hclt_walk_lean.hip.hpp, for whole trees side by side or one tree in parts.
//
// Plain C++ (no HIP): also compiled into a host test, which replays the rows with lean_schedule_check.hpp.
#pragma once

#include "lean_schedule.hpp"

namespace pcm {

// Field rows of a lean schedule, [field][wave][stride], and behind them [wave] the number of steps up
// to the wave's last node: a wave that is through leaves the compute unit to the others.
//   kLW     byte offset of the node's parameter block (-1: none wanted)
//   kLA0    byte offset of the node's own leaf rows (variable * leaf_stride)
//   kLA1..3 forward: leaf children's rows (-1: none; their categories are bytes 1..3 of the
//           packed word).  backward: children, inner ones first, -1: none, leaf child: row
//           offset | 1 | category byte << 1, inner child: node index << 3 (its value tile), | 2
//           if it is the only one and comes next in this wave: its value tile is not wanted
//   kLNode  node index (value / flow tile, packed-category row, row of maxima); idle waves:
//           n_inner (that category row is out of range and reads as zero)
//   kLSlots forward: out slot | child slots << 8, 16, 24 (0xff: none); backward: slot holding
//           this node's ratio tile | slots of the inner children's ratio tiles << 8, 16, 24
//           (0xff: that child is a leaf or absent); kLeanKept: in registers
//   kLTurns which use of its slot a tile is, modulo 128, in the byte layout of kLSlots: a slot passes through
//           the states 2t (free for its t-th tile), 2t + 1 (that tile is there), 2t + 2 (read, free again).  Bit 7 of byte 0:
//           the root; bit 7 of bytes 1..3, backward: that child is away
//   kLAway  place in the exchange of this node's tile, or of the first of its children's, that crosses workgroups
enum { kLW = 0, kLA0, kLA1, kLA2, kLA3, kLNode, kLSlots, kLTurns, kLAway, kLeanFields };
// in place of a slot: the tile comes from or goes to another workgroup / stays in the wave's registers (one that stays nowhere: 0xff)
constexpr uint32_t kLeanAway = kLeanSlotAway, kLeanKept = kLeanSlotKept;

// A tile from another workgroup is expected this many steps after the step it is sent in.
constexpr int kLeanAwaySteps = 4;

struct LeanNodes {   // what the rows say of the inner nodes besides the tree
  std::vector<std::vector<int32_t>> leaves;   // leaf children (variables)
  std::vector<int32_t> var;                   // the node's own variable
  int K = 0;
  size_t leaf_stride = 0;                     // bytes of a variable's leaf table
};

// The rows of one group behind those in `dst`, with padding up to `stride` steps (at least 64 more than the schedule has: a
// chunk refill reads 64 steps starting anywhere below it).  xid: by node, its tile's place in the exchange.  False if some node
// has more operands than the lean kernels hold.
inline bool lean_field_rows(const LeanTree& t, const LeanNodes& nd, const LeanScope& in, const LeanSchedule& sched,
                            const std::vector<int32_t>& xid, bool forward, int stride, std::vector<int32_t>& dst) {
  constexpr int W = kLeanSchedWaves;
  const size_t f0 = dst.size(), block = (size_t)nd.K * nd.K * sizeof(float);
  dst.resize(f0 + (size_t)kLeanFields * W * stride + W, 0);
  int32_t* const f = dst.data() + f0;
  auto at = [&](int field, int w, int st) -> int32_t& { return f[((size_t)field * W + w) * stride + st]; };
  auto item = [&](int st, int w) { return sched.item[(size_t)st * W + w]; };
  // A wave takes its nodes one behind the other: where the schedule has it idle it is the tile it waits for that holds it
  // up.  place[st][w]: the step of the wave itself.  The rest of the rows is padding: no node, leaf rows of variable 0.
  std::vector<int32_t> place((size_t)sched.steps * W, 0);
  int32_t* const n_own = f + (size_t)kLeanFields * W * stride;
  for (int st = 0; st < sched.steps; ++st)
    for (int w = 0; w < W; ++w)
      if (item(st, w) >= 0) place[(size_t)st * W + w] = n_own[w]++;
  const size_t field = (size_t)W * stride;
  for (const int none : {kLW, kLA1, kLA2, kLA3, kLSlots}) std::fill_n(f + none * field, field, -1);
  std::fill_n(f + kLNode * field, field, (int32_t)t.parent.size());
  // how often each slot has been filled so far: a step's reads see the fills of earlier steps only, so the
  // readers of a step are numbered before its writers
  std::vector<int32_t> fills(256, 0);
  for (int st = 0; st < sched.steps; ++st)
    for (int pass = 0; pass < 2; ++pass)
      for (int w = 0; w < W; ++w) {
        const int n = item(st, w);
        if (n < 0) continue;
        int32_t& turns = at(kLTurns, w, place[(size_t)st * W + w]);
        auto turn = [&](int tile, int byte) {
          const int sl = sched.slot[tile];
          if (sl < kLeanSlotAway) turns |= ((pass == 0 ? fills[sl] - 1 : fills[sl]++) & 0x7f) << (8 * byte);
        };
        if (t.inner[n].size() > 3) return false;
        if ((pass == 0) == forward)   // the children's tiles are bytes 1 .. 3, the node's own is byte 0
          for (size_t i = 0; i < t.inner[n].size(); ++i) turn(t.inner[n][i], 1 + (int)i);
        else
          turn(n, 0);
      }
  for (int st = 0; st < sched.steps; ++st)
    for (int w = 0; w < W; ++w) {
      const int n = item(st, w), i = place[(size_t)st * W + w];
      if (n < 0) continue;
      const std::vector<int32_t>&inner = t.inner[n], &leaves = nd.leaves[n];
      at(kLNode, w, i) = n;
      if (inner.size() + (forward ? 0 : leaves.size()) > 3 || leaves.size() > 3) return false;
      if (forward || !inner.empty()) at(kLW, w, i) = (int32_t)(n * block);
      at(kLA0, w, i) = (int32_t)(nd.var[n] * nd.leaf_stride);
      if (t.parent[n] < 0) at(kLTurns, w, i) |= 0x80;
      uint32_t slots = 0xffffff00u | (uint32_t)sched.slot[n];
      int q = 0;
      for (int c : inner) {
        slots = (slots & ~(0xffu << (8 * (q + 1)))) | ((uint32_t)sched.slot[c] << (8 * (q + 1)));
        if (!forward) at(kLA1 + q, w, i) = c << 3 | (inner.size() == 1 && in.in[c] ? 2 : 0);
        ++q;
      }
      at(kLSlots, w, i) = (int32_t)slots;
      if (t.parent[n] >= 0 && !in.in[t.parent[n]]) at(kLAway, w, i) = xid[n];
      for (size_t k = inner.size(); k-- > 0;) {
        if (in.in[inner[k]]) continue;
        at(kLAway, w, i) = xid[inner[k]];   // (those of one node are numbered in order)
        if (!forward) at(kLTurns, w, i) |= (int32_t)(0x80u << (8 * (k + 1)));
      }
      if (forward) q = 0;
      for (size_t k = 0; k < leaves.size(); ++k)
        at(kLA1 + q++, w, i) = (int32_t)(leaves[k] * nd.leaf_stride) | (forward ? 0 : 1 | (int32_t)((k + 1) << 1));
    }
  return true;
}

struct LeanPlanRows {   // [0]: up, [1]: down
  int n_groups = 0, n_away = 0;
  int steps[2] = {0, 0}, stride[2] = {0, 0};
  std::vector<int32_t> rows[2];
};

// The rows of a walk in groups: whole trees (`part` empty), or the parts of one tree, where going up the top, part 0, is
// the last group and going down the first.
inline bool lean_plan_rows(const LeanTree& t, const LeanNodes& nd, const std::vector<LeanScope>& scopes, const std::vector<int32_t>& part,
                           int n_slots, LeanPlanRows& p) {
  const int n = (int)t.parent.size(), G = p.n_groups = (int)scopes.size();
  std::vector<int32_t> xid(n, -1);
  if (!part.empty())
    for (int v = 0; v < n; ++v)
      for (int c : t.inner[v])
        if (part[c] != part[v]) xid[c] = p.n_away++;
  for (const bool forward : {true, false}) {
    std::vector<LeanScope> in = scopes;
    std::vector<LeanSchedule> sched(G);
    int steps = 0;
    for (int i = 0; i < G; ++i) {
      const int g = forward ? (i + 1) % G : i;   // (the top is scheduled as it runs)
      if (!part.empty() && (g == 0) == forward) {
        in[g].release.assign(n, 0);
        for (int v = 0; v < n; ++v)
          for (int c : t.inner[v])
            if (part[c] != part[v]) {
              const int from = forward ? c : v;
              int32_t& at = in[g].release[forward ? v : c];
              for (const LeanSchedule& sc : sched)
                if (!sc.step_of.empty() && sc.step_of[from] >= 0) at = std::max(at, sc.step_of[from] + 1 + kLeanAwaySteps);
            }
      }
      sched[g] = forward ? lean_schedule_up(t, in[g], n_slots) : lean_schedule_down(t, in[g], n_slots);
      if (!sched[g].ok) return false;
      steps = std::max(steps, sched[g].steps);
    }
    p.steps[!forward] = steps;
    p.stride[!forward] = steps + 64;   // the shorter groups idle at the end
    p.rows[!forward].reserve((size_t)G * (kLeanFields * kLeanSchedWaves * (size_t)(steps + 64) + kLeanSchedWaves));
    for (int i = 0; i < G; ++i) {
      const int g = forward && !part.empty() ? (i + 1) % G : i;
      if (!lean_field_rows(t, nd, in[g], sched[g], xid, forward, steps + 64, p.rows[!forward])) return false;
    }
  }
  return true;
}

}  // namespace pcm
