// Cutting gate lists into passes; see schedule.hpp.
#include "schedule.hpp"

#include "hip_backend.hpp"

#include <algorithm>

namespace cast::hip {

namespace {
constexpr size_t kErr = 1024; // src/cuda/types.rs:72
}

PassPlanner::PassPlanner(std::vector<PlannedGate> gates, PassLimits limits)
    : gates_(std::move(gates)), lim_(limits), left_(gates_.size()) {
  for (uint32_t i = 0; i < left_.size(); ++i)
    left_[i] = i;
}

uint32_t PassPlanner::collect(uint64_t set, std::vector<uint32_t> *taken,
                              std::vector<uint64_t> *ready) const {
  const uint64_t all = (uint64_t(1) << lim_.n_qubits) - 1;
  const size_t end = std::min(left_.size(), head_ + kWindow);
  uint64_t blocked = 0;
  uint32_t count = 0;
  for (size_t at = head_; at < end; ++at) {
    const uint32_t i = left_[at];
    const PlannedGate &g = gates_[i];
    if (!(g.qubits & blocked) && g.may_join) {
      if (!(g.qubits & ~set)) {
        if (taken)
          taken->push_back(i);
        if (++count == lim_.max_gates)
          break;
        continue;
      }
      if (ready)
        ready->push_back(g.qubits);
    }
    blocked |= g.qubits;
    if (blocked == all)
      break;
  }
  return count;
}

// Greedy: the first gate left, then, as long as a gate that could run next
// fits, the one that brings the most gates per added qubit.
bool PassPlanner::next(std::vector<uint32_t> &pass) {
  pass.clear();
  if (head_ == left_.size())
    return false;
  const PlannedGate &first = gates_[left_[head_]];
  if (!first.may_join) {
    pass.push_back(left_[head_++]);
    return true;
  }
  uint64_t set = first.qubits | ((uint64_t(1) << lim_.low_qubits) - 1);
  std::vector<uint64_t> ready;
  for (;;) {
    ready.clear();
    const uint32_t have = collect(set, nullptr, &ready);
    const int used = __builtin_popcountll(set);
    uint64_t best = 0;
    double best_score = -1.0;
    for (uint64_t q : ready) {
      const uint64_t grown = set | q;
      const int size = __builtin_popcountll(grown);
      if (size > int(lim_.max_qubits))
        continue;
      const double score = double(collect(grown, nullptr, nullptr) - have) / double(size - used);
      if (score > best_score) {
        best_score = score;
        best = grown;
      }
    }
    if (!best)
      break;
    set = best;
  }
  collect(set, &pass, nullptr);
  // The gates that stay behind move up to the last one taken.
  size_t at = head_;
  for (size_t t = 0; t < pass.size(); ++at)
    t += left_[at] == pass[t];
  size_t to = at;
  for (size_t t = pass.size(); at-- > head_;) {
    if (t > 0 && left_[at] == pass[t - 1])
      --t;
    else
      left_[--to] = left_[at];
  }
  head_ = to;
  return true;
}

namespace {
PassPlanner planner_of(const std::vector<const void *> &plans, uint32_t n_qubits, bool &all_join) {
  char err[kErr];
  std::vector<PlannedGate> gates(plans.size());
  PassLimits lim;
  all_join = true;
  for (size_t i = 0; i < plans.size(); ++i) {
    cast_hip_group_info_t info{};
    throw_if(cast_hip_gate_group_info(plans[i], n_qubits, &info, err, kErr), err);
    gates[i].qubits = info.targets;
    gates[i].may_join = info.targets != 0;
    all_join = all_join && gates[i].may_join;
    if (gates[i].may_join) {
      lim = {n_qubits, info.max_qubits, info.low_qubits, info.max_gates};
      continue;
    }
    cast_hip_gate_plan_info_t p{};
    throw_if(cast_hip_gate_plan_info(plans[i], &p, err, kErr), err);
    for (uint32_t b = 0; b < p.n_qubits; ++b)
      gates[i].qubits |= uint64_t(1) << p.qubits[b];
  }
  lim.n_qubits = n_qubits;
  return PassPlanner(std::move(gates), lim);
}
} // namespace

std::vector<std::vector<uint32_t>> plan_passes(const std::vector<const void *> &plans,
                                               uint32_t n_qubits, bool &all_join) {
  PassPlanner planner = planner_of(plans, n_qubits, all_join);
  std::vector<std::vector<uint32_t>> passes;
  std::vector<uint32_t> pass;
  while (planner.next(pass))
    passes.push_back(pass);
  return passes;
}

void apply_in_passes(const std::vector<const void *> &plans, void *stream, uint64_t sv_dptr,
                     uint32_t n_qubits, const std::function<void(uint32_t)> &single) {
  char err[kErr];
  bool all_join;
  PassPlanner planner = planner_of(plans, n_qubits, all_join);
  std::vector<uint32_t> pass;
  std::vector<const void *> group;
  while (planner.next(pass)) { // the device works on a pass while the next is planned
    group.clear();
    for (uint32_t i : pass)
      group.push_back(plans[i]);
    if (pass.size() == 1 || !cast_hip_gate_group_pays(group.data(), group.size(), n_qubits)) {
      for (uint32_t i : pass)
        single(i);
      continue;
    }
    throw_if(cast_hip_gate_apply_group(group.data(), group.size(), stream, sv_dptr, n_qubits, err,
                                       kErr),
             err);
  }
}

} // namespace cast::hip
