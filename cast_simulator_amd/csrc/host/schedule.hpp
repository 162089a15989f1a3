// Passes of a gate list over one statevector.
//
// The device applies a group of gates in one pass over the statevector when
// their targets together lie in few qubits (cast_hip_gate_apply_group).
// PassPlanner cuts a gate list into such groups.  Gates on disjoint qubits
// commute, so a pass may take a later gate along as long as none of its
// qubits is touched by an earlier gate that stays behind.
#pragma once

#include "cast_hip.h"

#include <cstdint>
#include <functional>
#include <vector>

namespace cast::hip {

struct PlannedGate {
  uint64_t qubits = 0;   // mask of the targets
  bool may_join = false; // the device can run it in a group
};

struct PassLimits {
  uint32_t n_qubits = 0;   // of the statevector
  uint32_t max_qubits = 0; // of a pass, the low_qubits lowest always among them
  uint32_t low_qubits = 0;
  uint32_t max_gates = 0;
};

class PassPlanner {
public:
  PassPlanner(std::vector<PlannedGate> gates, PassLimits limits);
  // Indices of the gates of the next pass, ascending; false when none is left.
  bool next(std::vector<uint32_t> &pass);

private:
  // Gates that a pass over the qubits of `set` takes; their indices when
  // `taken` is given, and in `ready` the qubits of each gate outside the set
  // that could run now.
  uint32_t collect(uint64_t set, std::vector<uint32_t> *taken, std::vector<uint64_t> *ready) const;

  // A pass takes gates among the next kWindow only.  A list that leaves a qubit
  // idle never blocks every qubit, and each pass would look through all of it:
  // 16000 gates on 19 of 20 qubits took 222 ms to plan, now 20 (all 20
  // qubits: 10), with as many passes.
  static constexpr size_t kWindow = 512;

  std::vector<PlannedGate> gates_;
  PassLimits lim_;
  std::vector<uint32_t> left_; // from head_ on: not yet in a pass, in order
  size_t head_ = 0;
};

// The passes of `plans` on one statevector, as indices; `all_join`:
// whether every gate can run in a group.
std::vector<std::vector<uint32_t>> plan_passes(const std::vector<const void *> &plans,
                                               uint32_t n_qubits, bool &all_join);

// Enqueues `plans` in order on `stream`, the groups that the planner finds as
// one pass each, where that pays, and every other gate i by `single(i)`.
void apply_in_passes(const std::vector<const void *> &plans, void *stream, uint64_t sv_dptr,
                     uint32_t n_qubits, const std::function<void(uint32_t)> &single);

} // namespace cast::hip
