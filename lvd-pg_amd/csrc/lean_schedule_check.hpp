// Host-side proof that a lean walk schedule cannot leave a wave waiting for ever.
//
// The lean walk kernels have no barrier between steps: tiles pass from wave to wave through LDS slots whose
// state words go 2t (free for the slot's t-th tile) -> 2t + 1 (tile there) -> 2t + 2 (read, free again), all
// modulo 256; a producer waits for 2t, the one consumer for 2t + 1, and every wave works through its steps in
// order.  Whether that terminates depends on the schedule alone, so it is checked when the schedule is built:
// the waits and posts of every wave are replayed on the host, each wave advancing whenever the state it waits
// for is there.  A slot's state is only ever changed by the one operation that is next in the slot's chain, so
// the replay's order does not matter: either every wave reaches its end, or the waves that are left wait for
// states nobody will post -- on the device they would run into their poll limit and void the pass.  The workgroups of a
// tree in parts are replayed together, the flags of the tiles they exchange among the states.
//
// Plain C++ (no HIP): also compiled into a host test.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace pcm {

// field rows of a lean schedule, [field][wave][stride]; the names are those of lean_rows.hpp
constexpr int kLeanCheckA1 = 2, kLeanCheckSlots = 6, kLeanCheckTurns = 7, kLeanCheckAway = 8, kLeanCheckFields = 9, kLeanCheckWaves = 16;
constexpr uint8_t kLeanCheckKept = 0xfd;   // from here on a slot byte names no slot (another workgroup's / kept in registers / nobody's)

struct LeanSlotOp {
  int slot;            // an LDS slot of the workgroup, or kLeanCheckFlag + place in the exchange
  uint8_t value;
  bool wait;   // wait until the slot's state equals value / set the slot's state to value
};
constexpr int kLeanCheckFlag = 256;   // (a tile in the exchange: 0 not there, 1 there; back at 0 behind its one reader)

// the slot operations of wave w in step s, in the order the kernels issue them
inline void lean_step_ops(const int32_t* f, int stride, int w, int s, bool forward, int trash_slot, std::vector<LeanSlotOp>& ops) {
  auto get = [&](int field) { return (uint32_t)f[((size_t)field * kLeanCheckWaves + w) * stride + s]; };
  const uint32_t slots = get(kLeanCheckSlots), turns = get(kLeanCheckTurns);
  if (slots == 0xffffffffu) return;   // (an idle step, or nothing to hand over)
  auto sl = [&](int c) { return (uint8_t)((slots >> (8 * c)) & 0xffu); };
  auto st = [&](int c, int add) { return (uint8_t)((2u * ((turns >> (8 * c)) & 0x7fu) + (uint32_t)add) & 0xffu); };
  auto is_away = [&](int c) { return sl(c) == kLeanCheckKept && sl(c) != (uint8_t)trash_slot; };
  int next_away = kLeanCheckFlag + (int)get(kLeanCheckAway);
  auto take = [&](int flag) { ops.push_back({flag, 1, true}); ops.push_back({flag, 0, false}); };
  auto send = [&](int flag) { ops.push_back({flag, 0, true}); ops.push_back({flag, 1, false}); };
  if (forward) {
    const int own_away = next_away;
    for (int c = 1; c <= 3; ++c)
      if (sl(c) < kLeanCheckKept) {   // a child's tile: wait for it, read it, free the slot
        ops.push_back({sl(c), st(c, 1), true});
        ops.push_back({sl(c), st(c, 2), false});
      } else if (is_away(c)) {
        take(next_away++);
      }
    if (is_away(0)) {
      send(own_away);
    } else if (sl(0) != (uint8_t)trash_slot && sl(0) < kLeanCheckKept) {   // the node's own tile goes into its slot once that is free
      ops.push_back({sl(0), st(0, 0), true});
      ops.push_back({sl(0), st(0, 1), false});
    }
    return;
  }
  bool inner[4] = {false, false, false, false};
  for (int c = 1; c <= 3; ++c) {
    const int32_t a = (int32_t)get(kLeanCheckA1 + c - 1);
    inner[c] = a >= 0 && !(a & 1);
  }
  for (int c = 1; c <= 3; ++c)
    if (inner[c] && sl(c) < kLeanCheckKept) ops.push_back({sl(c), st(c, 0), true});   // the children's slots must be free
  if (is_away(0)) {   // the node's ratio tile, left by its parent
    take(next_away);
  } else if (sl(0) != (uint8_t)trash_slot && sl(0) < kLeanCheckKept) {
    ops.push_back({sl(0), st(0, 1), true});
    ops.push_back({sl(0), st(0, 2), false});
  }
  if (!inner[1]) return;
  const int first_away = next_away;
  if (is_away(1)) ++next_away;
  for (int c = 1; c <= 3; ++c) {
    if (!inner[c] || sl(c) >= kLeanCheckKept) continue;
    const bool away = (turns >> (8 * c)) & 0x80u;
    if (away) send(next_away++);
    ops.push_back({sl(c), st(c, away ? 2 : 1), false});   // (a child in another workgroup: its slot is free again at once)
  }
  if (is_away(1)) send(first_away);   // (the first child's tile is in registers until here)
}

// The rows of `n_groups` workgroups of one slice, one behind the other as lean_rows.hpp leaves them.  -1 if every wave gets
// through its `n_steps` steps; otherwise (step * n_groups + group) * 16 + wave of the first wave found stuck.  `flags` (may be
// null): what is left in the exchange, all zero if every tile was read.
inline int lean_rows_stuck_at(const int32_t* f, int n_groups, int stride, int n_steps, bool forward, int trash_slot,
                              std::vector<uint8_t>* flags = nullptr) {
  const size_t per_group = (size_t)kLeanCheckFields * kLeanCheckWaves * stride + kLeanCheckWaves;
  const int n_waves = n_groups * kLeanCheckWaves;
  std::vector<std::vector<LeanSlotOp>> ops(n_waves);
  std::vector<std::vector<uint32_t>> step_end(n_waves, std::vector<uint32_t>(n_steps));   // operations up to a step's end
  int n_flags = 0;
  for (int w = 0; w < n_waves; ++w)
    for (int s = 0; s < n_steps; ++s) {
      const size_t before = ops[w].size();
      lean_step_ops(f + (size_t)(w / kLeanCheckWaves) * per_group, stride, w % kLeanCheckWaves, s, forward, trash_slot, ops[w]);
      step_end[w][s] = (uint32_t)ops[w].size();
      for (size_t i = before; i < ops[w].size(); ++i) {
        if (ops[w][i].slot < kLeanCheckFlag) ops[w][i].slot += w / kLeanCheckWaves * kLeanCheckFlag;
        else n_flags = std::max(n_flags, (ops[w][i].slot += (n_groups - 1) * kLeanCheckFlag) - n_groups * kLeanCheckFlag + 1);
      }
    }
  std::vector<uint8_t> state((size_t)n_groups * kLeanCheckFlag + n_flags, 0);
  std::vector<size_t> pos(n_waves, 0);
  for (bool moved = true; moved;) {
    moved = false;
    for (int w = 0; w < n_waves; ++w)
      while (pos[w] < ops[w].size()) {
        const LeanSlotOp& o = ops[w][pos[w]];
        if (o.wait && state[o.slot] != o.value) break;
        if (!o.wait) state[o.slot] = o.value;
        ++pos[w];
        moved = true;
      }
  }
  if (flags) flags->assign(state.begin() + (size_t)n_groups * kLeanCheckFlag, state.end());
  for (int w = 0; w < n_waves; ++w)
    if (pos[w] < ops[w].size()) {
      const int step = (int)(std::upper_bound(step_end[w].begin(), step_end[w].end(), (uint32_t)pos[w]) - step_end[w].begin());
      return (step * n_groups + w / kLeanCheckWaves) * kLeanCheckWaves + w % kLeanCheckWaves;
    }
  return -1;
}

// one workgroup's rows, without those of others
inline int lean_schedule_stuck_at(const int32_t* f, int stride, int n_steps, bool forward, int trash_slot) {
  return lean_rows_stuck_at(f, 1, stride, n_steps, forward, trash_slot);
}

}  // namespace pcm
