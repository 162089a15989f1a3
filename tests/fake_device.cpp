// Stands in front of libcast_hip.so, without a device, for host tests of the kernel
// manager: statevectors are tokens, gates are only counted, and a gate or copy
// on a statevector that has been freed is recorded instead of run.
#include "cast_hip.h"

#include <cstdio>
#include <cstring>
#include <set>

namespace {
struct Plan {
  uint32_t k, q[8], precision;
  bool dense;
};
std::set<uint64_t> live;
uint64_t next_sv = 4096;
} // namespace

extern "C" {
struct cast_fake_counts {
  long plans, syncs, singles, grouped, on_freed, allocs, fail_alloc, pays; // fail_alloc: -1 or which
} cast_fake = {0, 0, 0, 0, 0, 0, -1, 1};

uint64_t cast_hip_sv_alloc(size_t, uint8_t, char *err, size_t len) {
  if (cast_fake.allocs++ == cast_fake.fail_alloc) {
    std::snprintf(err, len, "out of memory");
    return 0;
  }
  live.insert(next_sv += 4096);
  return next_sv;
}
void cast_hip_sv_free(uint64_t p) { live.erase(p); }
int cast_hip_sv_zero(uint64_t, size_t, uint8_t, char *, size_t) { return 0; }
int cast_hip_sv_download(uint64_t, double *h, size_t n, uint8_t, char *, size_t) {
  std::memset(h, 0, n * sizeof(double));
  return 0;
}
int cast_hip_memcpy_dtod_async(uint64_t d, uint64_t s, size_t, void *, char *, size_t) {
  cast_fake.on_freed += !live.count(d) || !live.count(s);
  return 0;
}
uint64_t cast_hip_malloc(size_t, char *, size_t) { return 64; }
void cast_hip_free(uint64_t) {}
int cast_hip_marginal_probabilities(uint64_t, uint32_t, uint8_t, const uint32_t *, size_t m,
                                    double *out, void *, char *, size_t) {
  for (size_t i = 0; i < size_t(1) << m; ++i)
    out[i] = i == 0;
  return 0;
}

void *cast_hip_stream_create(char *, size_t) { return &live; }
void cast_hip_stream_destroy(void *) {}
int cast_hip_stream_sync(void *, char *, size_t) { return ++cast_fake.syncs, 0; }
void *cast_hip_event_create(char *, size_t) { return &live; }
int cast_hip_event_record(void *, void *, char *, size_t) { return 0; }
int cast_hip_event_synchronize(void *, char *, size_t) { return ++cast_fake.syncs, 0; }
void cast_hip_event_destroy(void *) {}
int cast_hip_event_elapsed_ms(void *, void *, float *ms, char *, size_t) { return *ms = 1.f, 0; }

int cast_hip_gate_plan_create(const cast_hip_kernel_gen_spec_t *spec, const cast_complex64_t *m,
                              size_t, const uint32_t *q, size_t k, void **out, char *, size_t) {
  Plan *p = new Plan{uint32_t(k), {}, uint32_t(spec->precision), false};
  const size_t K = size_t(1) << k;
  for (size_t r = 0; r < K; ++r)
    for (size_t c = 0; c < K; ++c)
      p->dense = p->dense || (r != c && (m[r * K + c].re != 0 || m[r * K + c].im != 0));
  for (size_t b = 0; b < k; ++b)
    p->q[b] = q[b];
  ++cast_fake.plans;
  *out = p;
  return 0;
}
void cast_hip_gate_plan_destroy(void *p) { delete static_cast<Plan *>(p); }
int cast_hip_gate_plan_info(const void *plan, cast_hip_gate_plan_info_t *out, char *, size_t) {
  const Plan &p = *static_cast<const Plan *>(plan);
  std::memset(out, 0, sizeof(*out));
  out->n_qubits = p.k;
  out->precision = p.precision;
  out->variant = p.dense ? CAST_HIP_VARIANT_DENSE : CAST_HIP_VARIANT_MONOMIAL;
  std::memcpy(out->qubits, p.q, sizeof(p.q));
  return 0;
}
int cast_hip_gate_plan_family(const void *, uint32_t, uint32_t *v, char *, size_t) {
  static uint32_t next = 0;
  *v = 1 + next++ % 2; // two candidates differ
  return 0;
}
// f64: up to 5 qubits join.
int cast_hip_gate_group_info(const void *plan, uint32_t n, cast_hip_group_info_t *out, char *,
                             size_t) {
  const Plan &p = *static_cast<const Plan *>(plan);
  std::memset(out, 0, sizeof(*out));
  if (n < 9 || p.k > 5)
    return 0;
  for (uint32_t b = 0; b < p.k; ++b)
    out->targets |= uint64_t(1) << p.q[b];
  out->max_qubits = 12;
  out->low_qubits = 2;
  out->max_gates = 64;
  return 0;
}
int cast_hip_gate_group_pays(const void *const *, size_t, uint32_t) { return int(cast_fake.pays); }
int cast_hip_gate_apply(const void *, void *, uint64_t sv, uint32_t, char *, size_t) {
  cast_fake.on_freed += !live.count(sv);
  return ++cast_fake.singles, 0;
}
int cast_hip_gate_apply_group(const void *const *, size_t n, void *, uint64_t sv, uint32_t, char *,
                              size_t) {
  cast_fake.on_freed += !live.count(sv);
  return cast_fake.grouped += long(n), 0;
}
size_t cast_hip_group_batch_scratch_bytes(size_t g, size_t p) { return 64 * (g + p); }
int cast_hip_gate_apply_group_batch(const cast_hip_group_item_t *items, size_t n, uint32_t,
                                    uint64_t, void *, char *, size_t) {
  for (size_t i = 0; i < n; ++i) {
    cast_fake.on_freed += !live.count(items[i].sv);
    cast_fake.grouped += long(items[i].n_plans);
  }
  return 0;
}
}
