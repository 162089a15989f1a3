// Gate groups: several consecutive gates in one pass over the statevector.
//
// A single-gate kernel reads and writes every amplitude from HBM for each
// gate, so below the matrix-core ridge a circuit costs one HBM round trip per
// gate.  A group is a list of gates whose targets together lie in a set S of
// m qubits (m <= 12 at f64, 13 at f32).  A workgroup owns one tile of 2^m
// amplitudes (the S bits vary, the others are fixed by the tile index),
// loads it into LDS (64 KiB), applies every gate of the list there with a
// barrier between gates, and writes it back: one HBM round trip per group.
//
// LDS layout: 16-byte units (one f64 amplitude, two f32 ones) at unit index
// u ^ (u >> 4 & 15) ^ (u >> 8 & 15).  The map is linear over GF(2), so the
// address of an amplitude is the XOR of one constant per index bit; the host
// puts these constants (byte offsets) into the gate's descriptor in the order
// in which the kernel consumes them.  Consecutive lanes get index bits that
// fall on different banks.
//
// A thread holds 2^R amplitudes at a time (f64 R = 3 or 4, f32 one more):
//   k <= 3        one combo per lane and register group on the VALU, matrix
//                 rows by scalar loads, each row used for 2^(R-k) combos;
//   k = 4, f64 5  three real products on the matrix cores, 16 combos per
//                 MFMA tile, operands laid out by lane when the plan is built;
//   f32 k = 5, 6  bf16 split products as in the single-gate kernel;
//   monomial      phases and diagonal gates (any k) multiply in place,
//                 permutations (k <= 4) move amplitudes between LDS slots.
//
// What bounds it (30 qubits, f64): loading and storing the tiles alone takes
// 6.0-7.5 ms a pass, depending on where the tile's qubits fall on the memory
// channels (an in-place stream takes 5.3).  Two workgroups share a CU, so one
// works while the other loads; a further k = 3, 4, 5 gate adds 0.9, 1.6, 3.0
// ms (matrix cores alone 1.3 and 2.6 for k = 4, 5), where its own pass would
// take 5.9-6.5.  Measured and not kept: tiles of 2^11 (379 ms against 350 for
// 90 gates), workgroups that stay and fetch their next tile during the gates
// (409 against 372 then; one of 512 threads per CU with all operands in LDS,
// so that no gate waits for the tile fetch, 379 against 339), operands in LDS
// instead of in registers (the same time), one workgroup per CU (474-540), wave
// priorities and staggered starts (no change).

#include "cast_hip.h"
#include "common.hpp"
#include "device_core.hpp"

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

namespace cast_hip {
namespace {

using dev::bf16x8_t;
using dev::f32x4_t;
using dev::fma_t;
using dev::insert_zero;
using dev::NV;
using dev::Split3;
using dev::split3;

constexpr uint32_t kMaxOffsets = 13; // one per tile bit
constexpr int kMaxGroupGates = 64;
constexpr uint32_t kMaxGroupQubits = 34; // 2^22 workgroups at most

enum Kind : uint32_t { kDense = 0, kDiagonal = 1, kPermutation = 2, kPhase = 3 };

struct GroupGate {
  const void *mat;       // dense k <= 3: the matrix; else matrix-core operands or, of a
                         // monomial gate, the entry of each row (plan.d_op)
  uint64_t cols;         // monomial k <= 4: source column of row r in nibble r;
                         // above (diagonal), bit r: row r is not the identity's
  uint32_t off2[7];      // LDS byte offsets of the index bits, two per word, in use order
  uint32_t k;
  uint32_t kind;
};

// A group on one statevector.
struct GroupHead {
  uint32_t n_gates;
  uint32_t thread_bits;  // log2(threads per workgroup)
  uint32_t m;            // tile qubits
  uint32_t xcd_bits;     // 0, or log2(tiles): tiles in XCD order
  uint32_t s[16];        // tile qubits, ascending (words: a byte is no scalar load)
  void *sv;
  uint64_t first;        // of its gates, in a table of several groups
};

struct GroupArgs {
  GroupHead h;
  GroupGate g[kMaxGroupGates];
};

// Whether a 16-byte unit holds two amplitudes.
template <typename T> struct Shape;
template <> struct Shape<double> {
  static constexpr int P = 0;
};
template <> struct Shape<float> {
  static constexpr int P = 1;
};

typedef float Unit __attribute__((ext_vector_type(4))); // 16 bytes

template <typename T> using Const = const __attribute__((address_space(4))) T *;
template <typename T> using Global = const __attribute__((address_space(1))) T *;
// A pointer read from a table, known to be one to global memory.
template <typename T> __device__ __forceinline__ Global<T> global_ptr(const void *p) {
  return (Global<T>)(reinterpret_cast<uintptr_t>(p));
}

// G: a GroupGate in the kernel's arguments or in constant memory.
template <typename G> __device__ __forceinline__ uint32_t offset_of(G &g, int b) {
  return (g.off2[b >> 1] >> (16 * (b & 1))) & 0xffffu;
}

template <typename T>
__device__ __forceinline__ typename NV<T>::type lds_get(const unsigned char *lds, uint32_t a) {
  return *reinterpret_cast<const typename NV<T>::type *>(lds + a);
}
template <typename T>
__device__ __forceinline__ void lds_put(unsigned char *lds, uint32_t a, typename NV<T>::type v) {
  *reinterpret_cast<typename NV<T>::type *>(lds + a) = v;
}

// XOR of the offsets first .. first + N - 1 selected by the bits of v.
template <int N, typename G>
__device__ __forceinline__ uint32_t select_offsets(G &g, int first, uint32_t v) {
  uint32_t a = 0;
#pragma unroll
  for (int b = 0; b < N; ++b)
    a ^= (0u - ((v >> b) & 1u)) & offset_of(g, first + b);
  return a;
}

// Dense gate on k <= 3 targets.  Offsets: k targets, R - k combos of the
// thread, then the thread index bits.  Row r + 1 of the matrix is requested
// (scalar loads) before row r is used.
template <typename T, int R, int KL, typename G>
__device__ __forceinline__ void small_gate(unsigned char *lds, G &g, uint32_t tid) {
  constexpr int K = 1 << KL, U = 1 << (R - KL);
  using V = typename NV<T>::type;
  typedef T Row __attribute__((ext_vector_type(2 * K)));
  const uint32_t base = select_offsets<12 - R + Shape<T>::P>(g, R, tid);
  Const<Row> rows = (Const<Row>)(reinterpret_cast<uintptr_t>(g.mat));
  Row next = rows[0];
  __syncthreads();
  V x[U][K];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int c = 0; c < K; ++c)
      x[u][c] = lds_get<T>(lds, base ^ select_offsets<R>(g, 0, uint32_t(u << KL | c)));
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const Row row = next;
    if (r + 1 < K)
      next = rows[r + 1];
    T ar0[U], ar1[U], ai0[U], ai1[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      ar0[u] = ar1[u] = ai0[u] = ai1[u] = T(0);
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const T mr = row[2 * c], mi = row[2 * c + 1];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ar0[u] = fma_t(mr, x[u][c].x, ar0[u]);
        ar1[u] = fma_t(mi, x[u][c].y, ar1[u]);
        ai0[u] = fma_t(mr, x[u][c].y, ai0[u]);
        ai1[u] = fma_t(mi, x[u][c].x, ai1[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      V o;
      o.x = ar0[u] - ar1[u];
      o.y = ai0[u] + ai1[u];
      lds_put<T>(lds, base ^ select_offsets<R>(g, 0, uint32_t(u << KL | r)), o);
    }
  }
}

// Dense gate on the matrix cores, three real products per complex one.
// Offsets: k targets, 4 column bits (combo of the MFMA tile), R + 2 - k tiles
// of the wave, wave index bits.  The contraction index is c = j KS + s (j =
// lane / 16); rows follow the accumulator layout (f64: j + 4 i, f32: 4 j + i,
// + 16 rb).  A wave reads all its inputs before it writes any output.
//
// f64: with P = Re M (vr + vi), Re = P - (Re M + Im M) vi and Im = P + (Im M -
// Re M) vr: both continue P's accumulator, so no output needs a vector
// instruction (an f64 MFMA keeps the vector unit busy too).  f32: t1 = Re M
// vr, t2 = Im M vi, t3 = (Re M + Im M)(vr + vi), Re = t1 - t2, Im = t3 - t1 -
// t2, the form of the single-gate kernels.
template <int R, int KL, typename G>
__device__ __forceinline__ void mfma_gate(unsigned char *lds, G &g, uint32_t tid,
                                          double) {
  constexpr int K = 1 << KL, RB = K / 16, KS = K / 4, LB = R + 2 - KL, NT = 1 << LB;
  using AV = dev::Acc4<double>::type;
  typedef double Pair __attribute__((ext_vector_type(2)));
  const uint32_t lane = tid & 63u, col = lane & 15u, j = lane >> 4, wave = tid >> 6;
  const uint32_t base = select_offsets<4>(g, KL, col) ^ select_offsets<6 - R>(g, R + 6, wave);
  const uint32_t in = base ^ select_offsets<2>(g, KL - 2, j);
  const uint32_t out = base ^ select_offsets<2>(g, 0, j);
  const Global<Pair> op = global_ptr<Pair>(g.mat) + lane;
  Pair a[3][KS / 2];
  auto load_rows = [&](int rb) {
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int s = 0; s < KS / 2; ++s)
        a[m][s] = op[64 * ((m * RB + rb) * (KS / 2) + s)];
  };
  load_rows(0);
  __syncthreads();
  dev::d2v x[NT][KS];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      x[t][s] = lds_get<double>(lds, in ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                                         select_offsets<KL - 2>(g, 0, uint32_t(s)));
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    if (rb > 0)
      load_rows(rb);
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += 2) { // two tiles: independent accumulator chains
      constexpr int W = NT < 2 ? NT : 2;
      AV p[W];
#pragma unroll
      for (int w = 0; w < W; ++w)
        p[w] = AV{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int w = 0; w < W; ++w)
          p[w] = dev::mfma16(a[0][s / 2][s & 1], x[t0 + w][s].x + x[t0 + w][s].y, p[w]);
      AV re[W], im[W];
#pragma unroll
      for (int w = 0; w < W; ++w)
        re[w] = im[w] = p[w];
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int w = 0; w < W; ++w) {
          re[w] = dev::mfma16(a[1][s / 2][s & 1], x[t0 + w][s].y, re[w]);
          im[w] = dev::mfma16(a[2][s / 2][s & 1], x[t0 + w][s].x, im[w]);
        }
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const uint32_t ro = out ^ select_offsets<LB>(g, KL + 4, uint32_t(t0 + w)) ^
                            select_offsets<KL - 4>(g, 4, uint32_t(rb));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dev::d2v o;
          o.x = re[w][i];
          o.y = im[w][i];
          lds_put<double>(lds, ro ^ select_offsets<2>(g, 2, uint32_t(i)), o);
        }
      }
    }
  }
}

template <int R, int KL, typename G>
__device__ __forceinline__ void mfma_gate(unsigned char *lds, G &g, uint32_t tid,
                                          float) {
  static_assert(KL == 4, "f32 k = 5 has the split products");
  constexpr int LB = R + 2 - KL, NT = 1 << LB;
  using AV = dev::Acc4<float>::type;
  const uint32_t lane = tid & 63u, col = lane & 15u, j = lane >> 4, wave = tid >> 6;
  const uint32_t base = select_offsets<4>(g, KL, col) ^ select_offsets<7 - R>(g, R + 6, wave);
  const uint32_t in = base ^ select_offsets<2>(g, 2, j); // rows and columns alike
  const Global<Unit> op = global_ptr<Unit>(g.mat) + lane;
  const Unit ar = op[0], ai = op[64], as = op[128];
  __syncthreads();
  dev::f2v x[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int s = 0; s < 4; ++s)
      x[t][s] = lds_get<float>(lds, in ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                                        select_offsets<2>(g, 0, uint32_t(s)));
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    AV t1 = {0, 0, 0, 0}, t2 = {0, 0, 0, 0}, t3 = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      t1 = dev::mfma16(ar[s], x[t][s].x, t1);
      t2 = dev::mfma16(ai[s], x[t][s].y, t2);
      t3 = dev::mfma16(as[s], x[t][s].x + x[t][s].y, t3);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dev::f2v o;
      o.x = t1[i] - t2[i];
      o.y = t3[i] - t1[i] - t2[i];
      lds_put<float>(lds, in ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                              select_offsets<2>(g, 0, uint32_t(i)),
                     o);
    }
  }
}

// f32 k = 5 as bf16 split products (the partial products and their order are
// those of dev::split_tile); the operands are the splits of Re M and Im M.
// Offsets as in mfma_gate.
template <int R, typename G>
__device__ __forceinline__ void split_gate5(unsigned char *lds, G &g, uint32_t tid) {
  constexpr int KL = 5, LB = R + 2 - KL, NT = 1 << LB;
  const uint32_t lane = tid & 63u, col = lane & 15u, j = lane >> 4, wave = tid >> 6;
  const Global<bf16x8_t> op = global_ptr<bf16x8_t>(g.mat) + lane;
  bf16x8_t a[2][3][2]; // [Re, Im][split][row block]
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        a[m][s][h] = op[dev::SplitOperands<5>::at(m, s, h, 0)];
  const uint32_t base = select_offsets<4>(g, KL, col) ^ select_offsets<7 - R>(g, R + 6, wave);
  const uint32_t in = base ^ select_offsets<2>(g, 3, j);
  const uint32_t out = base ^ select_offsets<2>(g, 2, j);
  __syncthreads();
  dev::f2v x[NT][8];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[t][e] = lds_get<float>(lds, in ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                                        select_offsets<3>(g, 0, uint32_t(e)));
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    bf16x8_t br[3], bi[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const Split3 sr = split3(x[t][e].x), si = split3(x[t][e].y);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        br[s][e] = sr.p[s];
        bi[s][e] = si.p[s];
      }
    }
    f32x4_t t1[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, t2[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}},
            t3[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int sa = 2; sa >= 0; --sa)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int sb = 2 - sa; sb >= 0; --sb) {
          t1[h] = dev::mfma_bf16(a[0][sa][h], br[sb], t1[h]);
          t3[h] = dev::mfma_bf16(a[0][sa][h], bi[sb], t3[h]);
          t2[h] = dev::mfma_bf16(a[1][sa][h], bi[sb], t2[h]);
          t3[h] = dev::mfma_bf16(a[1][sa][h], br[sb], t3[h]);
        }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dev::f2v o;
        o.x = t1[h][i] - t2[h][i];
        o.y = t3[h][i];
        lds_put<float>(lds,
                       out ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                           select_offsets<2>(g, 0, uint32_t(i)) ^
                           select_offsets<1>(g, 4, uint32_t(h)),
                       o);
      }
  }
}

// f32 k = 6 likewise.  Its 48 KiB of operands neither fit the registers nor,
// beside two tiles, the LDS: they stream from the caches in 12 steps (row
// block, split), each step's 4 KiB requested D steps before its products.
// Bound by the products (41 us at 25 qubits at the chip's bf16 rate): it adds
// about 55 us to a pass there, where its own pass takes 130-155.  25 qubits,
// 37 gates of which 13 have k = 6: 2829 us with those alone, 2515 in groups.
template <int R, typename G>
__device__ __forceinline__ void split_gate6(unsigned char *lds, G &g, uint32_t tid) {
  constexpr int KL = 6, LB = R + 2 - KL, NT = 1 << LB, D = R == 5 ? 2 : 1, STEPS = 12;
  const uint32_t lane = tid & 63u, col = lane & 15u, j = lane >> 4, wave = tid >> 6;
  const Global<bf16x8_t> op = global_ptr<bf16x8_t>(g.mat) + lane;
  bf16x8_t a[D + 1][2][2]; // ring of steps, [Re, Im][k step]
  auto fetch = [&](int step) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        a[step % (D + 1)][m][ks] =
            op[dev::SplitOperands<6>::at(m, 2 - step % 3, step / 3, ks)];
  };
#pragma unroll
  for (int s = 0; s < D; ++s)
    fetch(s);
  const uint32_t base = select_offsets<4>(g, KL, col) ^ select_offsets<7 - R>(g, R + 6, wave);
  const uint32_t in = base ^ select_offsets<2>(g, 3, j);
  const uint32_t out = base ^ select_offsets<2>(g, 2, j);
  __syncthreads();
  bf16x8_t br[NT][3][2], bi[NT][3][2];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const dev::f2v x =
            lds_get<float>(lds, in ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                                    select_offsets<3>(g, 0, uint32_t(e)) ^
                                    select_offsets<1>(g, 5, uint32_t(ks)));
        const Split3 sr = split3(x.x), si = split3(x.y);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          br[t][s][ks][e] = sr.p[s];
          bi[t][s][ks][e] = si.p[s];
        }
      }
  f32x4_t t1[NT], t2[NT], t3[NT];
#pragma unroll
  for (int step = 0; step < STEPS; ++step) {
    const int sa = 2 - step % 3, rb = step / 3;
    if (step + D < STEPS)
      fetch(step + D);
    __builtin_amdgcn_sched_barrier(0);
    if (sa == 2)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        t1[t] = t2[t] = t3[t] = {0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8_t ar = a[step % (D + 1)][0][ks], ai = a[step % (D + 1)][1][ks];
#pragma unroll
      for (int sb = 2 - sa; sb >= 0; --sb)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          t1[t] = dev::mfma_bf16(ar, br[t][sb][ks], t1[t]);
          t3[t] = dev::mfma_bf16(ar, bi[t][sb][ks], t3[t]);
          t2[t] = dev::mfma_bf16(ai, bi[t][sb][ks], t2[t]);
          t3[t] = dev::mfma_bf16(ai, br[t][sb][ks], t3[t]);
        }
    }
    if (sa == 0)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dev::f2v o;
          o.x = t1[t][i] - t2[t][i];
          o.y = t3[t][i];
          lds_put<float>(lds,
                         out ^ select_offsets<LB>(g, KL + 4, uint32_t(t)) ^
                             select_offsets<2>(g, 0, uint32_t(i)) ^
                             select_offsets<2>(g, 4, uint32_t(rb)),
                         o);
        }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// v times an entry (re, im).
template <typename T>
__device__ __forceinline__ typename NV<T>::type times(typename NV<T>::type v, T re, T im) {
  typename NV<T>::type o;
  o.x = re * v.x - im * v.y;
  o.y = re * v.y + im * v.x;
  return o;
}

// Monomial gate on k <= R targets (diagonal or permutation): row r takes
// entry (r, col(r)) times amplitude col(r).  Rows equal to the identity's
// touch nothing.  Offsets as in small_gate; the mask of the other rows is in
// the upper half of off2[6].
template <typename T, int R, int KL, typename G>
__device__ __forceinline__ void monomial_gate(unsigned char *lds, G &g,
                                              uint32_t tid) {
  constexpr int K = 1 << KL, U = 1 << (R - KL);
  using V = typename NV<T>::type;
  const uint32_t base = select_offsets<12 - R + Shape<T>::P>(g, R, tid), active = g.off2[6] >> 16;
  typedef T Entries __attribute__((ext_vector_type(2 * K)));
  const Entries e = *(Const<Entries>)(reinterpret_cast<uintptr_t>(g.mat));
  __syncthreads();
  V x[U][K];
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (active >> r & 1u) {
      const uint32_t c = uint32_t(g.cols >> (4 * r)) & 15u;
      const uint32_t co = select_offsets<KL>(g, 0, c);
#pragma unroll
      for (int u = 0; u < U; ++u)
        x[u][r] = lds_get<T>(lds, base ^ co ^ select_offsets<R>(g, 0, uint32_t(u << KL)));
    }
#pragma unroll
  for (int r = 0; r < K; ++r)
    if (active >> r & 1u) {
      const T re = e[2 * r], im = e[2 * r + 1];
#pragma unroll
      for (int u = 0; u < U; ++u)
        lds_put<T>(lds, base ^ select_offsets<R>(g, 0, uint32_t(u << KL | r)),
                   times<T>(x[u][r], re, im));
    }
}

// Monomial gate on more than R targets: the targets from the R-th on are the
// lowest thread index bits, so a wave holds whole combos and reads them
// before it writes.
template <typename T, int R, typename G>
__device__ __forceinline__ void wide_monomial_gate(unsigned char *lds, G &g,
                                                   uint32_t tid, uint32_t k, bool diagonal) {
  constexpr int N = 1 << R;
  using V = typename NV<T>::type;
  const uint32_t base = select_offsets<12 - R + Shape<T>::P>(g, R, tid);
  const uint32_t hi = tid & ((1u << (k - R)) - 1);
  const Global<V> mat = global_ptr<V>(g.mat);
  __syncthreads();
  V x[N], e[N];
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const uint32_t r = hi << R | uint32_t(c);
    const uint32_t col = diagonal ? r : uint32_t(g.cols >> (4 * r)) & 15u;
    e[c] = mat[r];
    x[c] = lds_get<T>(lds, base ^ select_offsets<R>(g, 0, col) ^
                               select_offsets<6 - R>(g, R, (col >> R) ^ hi));
  }
  // Rows equal to the identity's leave the amplitude as it is.  (With R >= 4 only
  // diagonal gates are this wide.)  The mask instead of a look at each entry and
  // column also leaves the other gates of the kernel more registers: 13 qubits
  // f64 in gates of k = 2 175.4 -> 170.3 us, 12 qubits of k <= 4 65.2 -> 63.8.
  const uint32_t active = uint32_t((k > 4 ? g.cols : uint64_t(g.off2[6] >> 16)) >> (hi << R));
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const bool keep = R < 4 ? !(active >> c & 1u) : diagonal && e[c].x == T(1) && e[c].y == T(0);
    const V o = times<T>(x[c], e[c].x, e[c].y);
    lds_put<T>(lds, base ^ select_offsets<R>(g, 0, uint32_t(c)), keep ? x[c] : o);
  }
}

// Diagonal gate with one entry other than 1 (a phase, controlled or not; any
// k): multiplies the amplitudes of that row, 2^(R-k) per thread or one in each
// of the first threads.  The targets' positions are the nibbles of `cols`,
// off2[0] is the offset of the row; free index bit j of the tile is bit j of
// (combo, thread), and off2[1 + b] the offset of the b-th one above the
// thread's (b < 4).  The entry itself is in `mat` and off2[5, 6]: a load of it
// would be a cache miss per gate.  Bound by its
// instructions: as a diagonal gate on two targets, with a test per row and
// offsets by table, it took 0.85 us on a CU, now 0.5; the 20-qubit Fourier
// transform (180 such gates) 292 -> 235 us.
template <typename T, int R, int KL>
__device__ __forceinline__ void phase_gate(unsigned char *lds, const GroupGate &g, uint32_t tid,
                                           uint32_t k) {
  constexpr int P = Shape<T>::P, LU = KL < R ? R - KL : 0, U = 1 << LU;
  uint32_t i = tid;
  for (uint32_t b = 0; b < (KL < 4 ? uint32_t(KL) : k); ++b)
    i = uint32_t(insert_zero(i, uint32_t(g.cols >> (4 * b)) & 15u));
  const uint32_t u = i >> P;
  uint32_t at = 16 * (u ^ ((u >> 4) & 15u) ^ ((u >> 8) & 15u)) ^ g.off2[0];
  if (P)
    at ^= (i & 1u) << 3;
  const uint64_t re = reinterpret_cast<uintptr_t>(g.mat), im = uint64_t(g.off2[6]) << 32 | g.off2[5];
  typename NV<T>::type e;
  if constexpr (sizeof(T) == 8) {
    e.x = __builtin_bit_cast(double, re);
    e.y = __builtin_bit_cast(double, im);
  } else {
    e.x = __builtin_bit_cast(float, uint32_t(re));
    e.y = __builtin_bit_cast(float, uint32_t(im));
  }
  __syncthreads();
  if (KL >= 4 && k > uint32_t(R) && tid >= blockDim.x >> (k - R))
    return;
  typename NV<T>::type x[U];
  uint32_t a[U];
#pragma unroll
  for (int c = 0; c < U; ++c) {
    a[c] = at;
#pragma unroll
    for (int b = 0; b < LU; ++b)
      a[c] ^= c >> b & 1 ? g.off2[1 + b] : 0u;
    x[c] = lds_get<T>(lds, a[c]);
  }
#pragma unroll
  for (int c = 0; c < U; ++c)
    lds_put<T>(lds, a[c], times<T>(x[c], e.x, e.y));
}

// The 16-byte units of a thread: unit i * threads + tid of a tile, i < 2^RU.
template <typename T, int RU> struct TileUnits {
  static constexpr int P = Shape<T>::P, N = 1 << RU;
  Unit *p;          // global address of unit tid
  uint64_t reg[RU]; // global unit offsets of the bits of i
  uint32_t lds_t, thread_bits;

  template <typename H>
  __device__ __forceinline__ TileUnits(T *sv, H &a, uint64_t tile, uint32_t tid) {
    for (uint32_t b = 0; b < a.m; ++b)
      tile = insert_zero(tile, a.s[b]);
#pragma unroll
    for (int b = 0; b < 12 - RU; ++b)
      tile |= uint64_t((tid >> b) & 1u) << a.s[b + P];
    thread_bits = a.thread_bits;
#pragma unroll
    for (int b = 0; b < RU; ++b)
      reg[b] = (uint64_t(1) << a.s[thread_bits + b + P]) >> P;
    p = reinterpret_cast<Unit *>(sv) + (tile >> P);
    lds_t = tid ^ ((tid >> 4) & 15u) ^ ((tid >> 8) & 15u);
  }
  __device__ __forceinline__ Unit *global(int i) const {
    uint64_t o = 0;
#pragma unroll
    for (int b = 0; b < RU; ++b)
      o |= (i >> b & 1) ? reg[b] : 0;
    return p + o;
  }
  __device__ __forceinline__ uint32_t local(int i) const { // LDS byte offset
    const uint32_t u = uint32_t(i) << thread_bits;
    return 16 * (lds_t ^ u ^ ((u >> 4) & 15u) ^ ((u >> 8) & 15u));
  }
};

template <typename G> __device__ __forceinline__ GroupGate fetch(G &from) {
  GroupGate g;
  g.mat = from.mat;
  g.cols = from.cols;
#pragma unroll
  for (int i = 0; i < 7; ++i)
    g.off2[i] = from.off2[i];
  g.k = from.k;
  g.kind = from.kind;
  return g;
}

// R amplitude bits per thread.  The gate functions begin with the barrier that
// orders them after the previous gate; what they need from global memory is
// requested before it.
template <typename T, int R, typename H, typename G>
__device__ __forceinline__ void run_group(T *sv, H &a, G *gates, unsigned char *lds) {
  using Units = TileUnits<T, R - Shape<T>::P>;
  const uint32_t tid = threadIdx.x;
  uint64_t tile = blockIdx.x;
  if (a.xcd_bits)
    tile = ((tile & 7u) << (a.xcd_bits - 3)) | (tile >> 3);
  {
    const Units t(sv, a, tile, tid);
    Unit x[Units::N];
#pragma unroll
    for (int i = 0; i < Units::N; ++i)
      x[i] = __builtin_nontemporal_load(t.global(i));
#pragma unroll
    for (int i = 0; i < Units::N; ++i)
      *reinterpret_cast<Unit *>(lds + t.local(i)) = x[i];
  }
  // The next descriptor is requested a gate ahead.
  GroupGate ahead = fetch(gates[0]);
  asm volatile("" ::"s"(ahead.kind)); // arrived: the loop's first wait is not for the next one
  for (uint32_t gi = 0; gi < a.n_gates; ++gi) {
    const GroupGate g = ahead;
    ahead = fetch(gates[gi + 1 < a.n_gates ? gi + 1 : gi]);
    if (g.kind == kPhase) {
      switch (g.k) {
      case 1:
        phase_gate<T, R, 1>(lds, g, tid, 1);
        break;
      case 2:
        phase_gate<T, R, 2>(lds, g, tid, 2);
        break;
      case 3:
        phase_gate<T, R, 3>(lds, g, tid, 3);
        break;
      case 4:
        phase_gate<T, R, 4>(lds, g, tid, 4);
        break;
      default:
        phase_gate<T, R, 6>(lds, g, tid, g.k);
        break;
      }
    } else if (g.kind != kDense) {
      switch (g.k) {
      case 1:
        monomial_gate<T, R, 1>(lds, g, tid);
        break;
      case 2:
        monomial_gate<T, R, 2>(lds, g, tid);
        break;
      case 3:
        monomial_gate<T, R, 3>(lds, g, tid);
        break;
      default:
        if (g.k == 4 && R >= 4)
          monomial_gate<T, R, R < 4 ? R : 4>(lds, g, tid);
        else
          wide_monomial_gate<T, R>(lds, g, tid, g.k, g.kind == kDiagonal);
        break;
      }
    } else {
      switch (g.k) {
      case 1:
        small_gate<T, R, 1>(lds, g, tid);
        break;
      case 2:
        small_gate<T, R, 2>(lds, g, tid);
        break;
      case 3:
        small_gate<T, R, 3>(lds, g, tid);
        break;
      case 4:
        mfma_gate<R, 4>(lds, g, tid, T(0));
        break;
      case 5:
        if constexpr (sizeof(T) == 8)
          mfma_gate<R, 5>(lds, g, tid, T(0));
        else
          split_gate5<R>(lds, g, tid);
        break;
      default: // f32 only
        if constexpr (sizeof(T) == 4)
          split_gate6<R>(lds, g, tid);
        break;
      }
    }
  }
  __syncthreads();
  // Addresses again from the thread index: kept over the gates they would
  // take the registers that the gates need.
  uint32_t again = tid;
  asm volatile("" : "+v"(again));
  const Units t(sv, a, tile, again);
#pragma unroll
  for (int i = 0; i < Units::N; ++i)
    __builtin_nontemporal_store(*reinterpret_cast<const Unit *>(lds + t.local(i)), t.global(i));
}

template <typename T, int R>
__global__ void __launch_bounds__(1 << (12 + Shape<T>::P - R), R == 3 + Shape<T>::P ? 4 : 2)
    k_group(T *__restrict__ sv, GroupArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const GroupHead &h = a.h;
  run_group<T, R>(sv, h, static_cast<const GroupGate *>(a.g), lds);
}

// Groups on several statevectors, one per grid row, from a table.  A small
// statevector has few tiles (16 qubits f64: 16), and its pass is a chain of
// gates of about 1 us each on that many CUs; here they run side by side.
// 16 members of a noisy 16-qubit ensemble, 3 layers: 6447 us with a launch
// per member and pass (950 launches), 1666 with these.
template <typename T, int R>
__global__ void __launch_bounds__(1 << (12 + Shape<T>::P - R), R == 3 + Shape<T>::P ? 4 : 2)
    k_group_batch(Const<GroupHead> heads, Const<GroupGate> gates) {
  extern __shared__ __align__(16) unsigned char lds[];
  auto &h = heads[blockIdx.y];
  using GT = __attribute__((address_space(1))) T;
  T *sv = (T *)((GT *)(reinterpret_cast<uintptr_t>(h.sv)));
  run_group<T, R>(sv, h, gates + h.first, lds);
}

// ── Host side ───────────────────────────────────────────────────────────────

bool is_diagonal(const GatePlan &p) {
  for (uint32_t i = 0; i < p.n_active; ++i)
    if (p.act_row[i] != p.act_col[i])
      return false;
  return true;
}

uint32_t max_tile(uint8_t precision) { return precision == 0 ? 13 : 12; }
// Lowest qubits that every tile holds: 64-byte rows.  Fewer leave more qubits
// to the gates, so fewer passes, and tiles that share 128-byte lines run on
// one XCD at about the same time (XCD order).  90 gates at 30 qubits, ms at
// 16, 32, 64, 128 and 256 bytes: f64 380, 346, 350, 361, 379; f32 (32 to 128
// bytes) 162, 160, 162.
uint32_t low_qubits(uint8_t precision) { return precision == 0 ? 3 : 2; }
uint32_t regs_log2(uint8_t precision) { return precision == 0 ? 4 : 3; }

bool can_join(const GatePlan &p, uint32_t n) {
  if (n < regs_log2(p.precision) + 6 || n > kMaxGroupQubits || n < p.k || p.q[p.k - 1] >= n)
    return false;
  if (p.variant == 2)
    return is_diagonal(p) || p.k <= 4;
  return p.k <= (p.precision == 0 ? 6u : 5u);
}

// LDS byte offset of local index bit `p` (see the file comment).
uint32_t bit_offset(uint32_t p, bool f32) {
  if (f32 && p == 0)
    return 8;
  const uint32_t u = f32 ? p - 1 : p;
  return 16 * ((1u << u) | (u >= 4 ? 1u << (u & 3) : 0u));
}

template <typename T, int R>
void launch_k_group(dim3 grid, dim3 block, size_t lds, hipStream_t stream, void *sv,
                    const GroupArgs &a) {
  hipLaunchKernelGGL((k_group<T, R>), grid, block, lds, stream, static_cast<T *>(sv), a);
}

template <typename T, int R>
void launch_k_group_batch(dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                          const GroupHead *heads, const GroupGate *gates) {
  hipLaunchKernelGGL((k_group_batch<T, R>), grid, block, lds, stream,
                     (Const<GroupHead>)(reinterpret_cast<uintptr_t>(heads)),
                     (Const<GroupGate>)(reinterpret_cast<uintptr_t>(gates)));
}

} // namespace

// Operand vector x of lane l is 16-byte unit x * 64 + l, so that a wave reads
// 1 KiB in order.
//   f64: x = (matrix * RB + rb) * KS / 2 + s / 2, two entries of row 16 rb + l %
//        16 from column (l / 16) KS + s on, matrices Re M, -(Re M + Im M), Im M -
//        Re M;
//   f32 k = 4: x = matrix, four entries of row l % 16 from column 4 (l / 16)
//        on, matrices Re M, Im M, Re M + Im M;
//   f32 k = 5, 6: the bf16 fragments of dev::split_stage.
size_t group_operand_bytes(uint32_t k, uint8_t precision) {
  const size_t K = size_t(1) << k;
  if (precision == 0)
    return k == 4   ? 3 * K * K * sizeof(float)
           : k == 5 ? dev::SplitOperands<5>::kFragments * 16
                    : dev::SplitOperands<6>::kFragments * 16;
  return 3 * K * K * sizeof(double);
}

namespace {
// The bf16 parts of 8 values, each rounded to nearest even as the device's
// conversion does (without branches, for the vectoriser).
void split8(const float *x, uint16_t out[3][8]) {
  float rest[8];
  std::memcpy(rest, x, sizeof(rest));
  for (int s = 0; s < 3; ++s) {
    uint32_t b[8], h[8];
    float part[8];
    std::memcpy(b, rest, sizeof(b));
    for (int e = 0; e < 8; ++e) {
      const uint32_t nan = b[e] | 0x400000u, round = b[e] + 0x7fffu + (b[e] >> 16 & 1u);
      // magnitudes are positive as signed numbers
      h[e] = (int32_t(b[e] & 0x7fffffffu) > 0x7f800000 ? nan : round) & 0xffff0000u;
    }
    std::memcpy(part, h, sizeof(part));
    for (int e = 0; e < 8; ++e)
      rest[e] -= part[e];
    for (int e = 0; e < 8; ++e)
      out[s][e] = uint16_t(h[e] >> 16);
  }
}
} // namespace

void group_operands(const double *m, uint32_t k, uint8_t precision, void *out) {
  const uint32_t K = 1u << k, RB = K / 16, KS = K / 4;
  auto re = [&](uint32_t r, uint32_t c) { return m[2 * (r * K + c)]; };
  auto im = [&](uint32_t r, uint32_t c) { return m[2 * (r * K + c) + 1]; };
  if (precision == 1) {
    double *d = static_cast<double *>(out);
    for (uint32_t x = 0; x < 3; ++x)
      for (uint32_t rb = 0; rb < RB; ++rb)
        for (uint32_t s = 0; s < KS; ++s)
          for (uint32_t l = 0; l < 64; ++l) {
            const uint32_t r = 16 * rb + (l & 15u), c = (l >> 4) * KS + s;
            const double v = x == 0   ? re(r, c)
                             : x == 1 ? -(re(r, c) + im(r, c))
                                      : im(r, c) - re(r, c);
            d[(((x * RB + rb) * (KS / 2) + s / 2) * 64 + l) * 2 + (s & 1u)] = v;
          }
  } else if (k == 4) {
    float *f = static_cast<float *>(out);
    for (uint32_t x = 0; x < 3; ++x)
      for (uint32_t l = 0; l < 64; ++l)
        for (uint32_t s = 0; s < 4; ++s) {
          const uint32_t r = l & 15u, c = (l >> 4) * 4 + s;
          f[(x * 64 + l) * 4 + s] =
              float(x == 0 ? re(r, c) : x == 1 ? im(r, c) : re(r, c) + im(r, c));
        }
  } else {
    unsigned char *h = static_cast<unsigned char *>(out);
    const uint32_t n_ks = K / 32;
    std::vector<float> part(K * K);
    for (uint32_t x = 0; x < 2; ++x) {
      for (uint32_t i = 0; i < K * K; ++i)
        part[i] = float(m[2 * i + x]);
      for (uint32_t rb = 0; rb < RB; ++rb)
        for (uint32_t ks = 0; ks < n_ks; ++ks)
          for (uint32_t l = 0; l < 64; ++l) {
            uint16_t b[3][8];
            split8(&part[(16 * rb + (l & 15u)) * K + 32 * ks + 8 * (l >> 4)], b);
            for (uint32_t s = 0; s < 3; ++s) {
              const int at = k == 5
                                 ? dev::SplitOperands<5>::at(int(x), int(s), int(rb), int(ks))
                                 : dev::SplitOperands<6>::at(int(x), int(s), int(rb), int(ks));
              std::memcpy(h + (size_t(at) + l) * 16, b[s], 16);
            }
          }
    }
  }
}

GroupLimits group_limits(const GatePlan &p, uint32_t n) {
  GroupLimits l{};
  if (!can_join(p, n))
    return l;
  for (uint32_t b = 0; b < p.k; ++b)
    l.targets |= uint64_t(1) << p.q[b];
  l.max_qubits = std::min(n, max_tile(p.precision));
  l.low_qubits = low_qubits(p.precision);
  l.max_gates = kMaxGroupGates;
  return l;
}

namespace {

// Amplitudes per thread: twice as many, with half the threads, from 2^10
// tiles on.  There the tiles are enough to fill the chip and a wave that
// runs more MFMA tiles per operand load is the faster one (30 qubits f64,
// 90 gates in 44 passes: 373 ms against 393); below it the latency of a
// gate counts (12 qubits f64, 23 gates: 64 us against 74).
bool many_tiles(uint32_t n, uint8_t prec) { return n >= max_tile(prec) + 10; }

// Head and gates (identities left out) of a group; `gates` holds n_plans.
void describe_group(const GatePlan *const *plans, size_t n_plans, uint32_t n, GroupHead &a,
                    GroupGate *gates) {
  if (n_plans > size_t(kMaxGroupGates))
    throw Error("a gate group holds at most " + std::to_string(kMaxGroupGates) + " gates");
  if (n > 40)
    throw Error("statevector qubit count " + std::to_string(n) + " is out of range");
  const uint8_t prec = plans[0]->precision;
  const bool f32 = prec == 0;
  uint64_t set = 0;
  for (size_t i = 0; i < n_plans; ++i) {
    const GatePlan &p = *plans[i];
    if (p.precision != prec)
      throw Error("grouped plans must share the precision");
    if (!can_join(p, n))
      throw Error("gate " + std::to_string(i) + " cannot join a group on a " + std::to_string(n) +
                  "-qubit statevector");
    for (uint32_t b = 0; b < p.k; ++b)
      set |= uint64_t(1) << p.q[b];
  }
  const uint32_t m = std::min(n, max_tile(prec));
  const uint32_t R = regs_log2(prec) + many_tiles(n, prec);
  const uint32_t low = low_qubits(prec);
  set |= (uint64_t(1) << low) - 1;
  if (uint32_t(__builtin_popcountll(set)) > m)
    throw Error("grouped gates act on more than " + std::to_string(m) + " qubits (the lowest " +
                std::to_string(low) + " included)");
  // The rest of the tile: the lowest free qubits, which lengthens its rows.
  for (uint32_t q = 0; uint32_t(__builtin_popcountll(set)) < m; ++q)
    set |= uint64_t(1) << q;

  a = {};
  a.m = m;
  a.thread_bits = m - R;
  uint8_t local[64] = {};
  {
    uint32_t i = 0;
    for (uint32_t q = 0; q < n; ++q)
      if (set >> q & 1u) {
        local[q] = uint8_t(i);
        a.s[i++] = q;
      }
  }
  for (size_t i = 0; i < n_plans; ++i) {
    const GatePlan &p = *plans[i];
    const bool mono = p.variant == 2;
    if (mono && p.n_active == 0)
      continue; // identity
    GroupGate &g = gates[a.n_gates++];
    g = {};
    const bool diag = mono && is_diagonal(p);
    const bool mfma = !mono && p.k >= 4;
    g.mat = mfma || mono ? p.d_op : p.d_mat;
    g.k = p.k;
    g.kind = mono ? (diag ? kDiagonal : kPermutation) : kDense;
    uint32_t used = 0;
    for (uint32_t b = 0; b < p.k; ++b)
      used |= 1u << local[p.q[b]];
    if (diag && p.n_active == 1) {
      // (identity entries take no part, so the row is not the identity's)
      g.kind = kPhase;
      uint64_t part[2] = {};
      const float fl[2] = {float(p.act_re[0]), float(p.act_im[0])};
      for (int x = 0; x < 2; ++x)
        f32 ? std::memcpy(&part[x], &fl[x], 4)
            : std::memcpy(&part[x], x ? &p.act_im[0] : &p.act_re[0], 8);
      g.mat = reinterpret_cast<const void *>(uintptr_t(part[0]));
      g.off2[5] = uint32_t(part[1]);
      g.off2[6] = uint32_t(part[1] >> 32);
      for (uint32_t b = 0; b < p.k; ++b) {
        g.cols |= uint64_t(local[p.q[b]]) << (4 * b);
        g.off2[0] ^= p.act_row[0] >> b & 1u ? bit_offset(local[p.q[b]], f32) : 0u;
      }
      uint32_t free_bit = 0;
      for (uint32_t b = 0; b < m; ++b)
        if (!(used >> b & 1u)) {
          if (free_bit >= a.thread_bits && free_bit - a.thread_bits < 4)
            g.off2[1 + free_bit - a.thread_bits] = bit_offset(b, f32);
          ++free_bit;
        }
      continue;
    }
    if (mono && p.k <= 4) {
      for (uint32_t r = 0; r < (1u << p.k); ++r)
        g.cols |= uint64_t(r) << (4 * r);
      for (uint32_t x = 0; x < p.n_active; ++x) {
        g.cols &= ~(uint64_t(15) << (4 * p.act_row[x]));
        g.cols |= uint64_t(p.act_col[x]) << (4 * p.act_row[x]);
        g.off2[6] |= 0x10000u << p.act_row[x];
      }
    } else if (mono) {
      for (uint32_t x = 0; x < p.n_active; ++x)
        g.cols |= uint64_t(1) << p.act_row[x];
    }
    // The other positions, those whose banks differ first (they go to
    // consecutive lanes).
    uint32_t order[kMaxOffsets] = {}, lanes = 0, rest[kMaxOffsets] = {}, n_rest = 0, banks = 0;
    for (uint32_t b = 0; b < m; ++b) {
      if (used >> b & 1u)
        continue;
      const uint32_t bank = f32 ? (b == 0 ? 4u : (b - 1) & 3u) : b & 3u;
      if (!(banks >> bank & 1u)) {
        banks |= 1u << bank;
        order[lanes++] = b;
      } else {
        rest[n_rest++] = b;
      }
    }
    for (uint32_t b = 0; b < n_rest; ++b)
      order[lanes + b] = rest[b];
    const uint32_t free_bits = m - p.k;
    uint32_t off[kMaxOffsets + 1] = {}, w = 0;
    for (uint32_t b = 0; b < p.k; ++b)
      off[w++] = bit_offset(local[p.q[b]], f32);
    if (mfma) { // columns, tiles of the wave, waves: as ordered
      for (uint32_t b = 0; b < free_bits; ++b)
        off[w++] = bit_offset(order[b], f32);
    } else { // combos of the thread last in the order, threads first
      const uint32_t u = p.k < R ? R - p.k : 0;
      for (uint32_t b = 0; b < u; ++b)
        off[w++] = bit_offset(order[free_bits - u + b], f32);
      for (uint32_t b = 0; b < free_bits - u; ++b)
        off[w++] = bit_offset(order[b], f32);
    }
    for (uint32_t b = 0; b < kMaxOffsets; ++b)
      g.off2[b >> 1] |= off[b] << (16 * (b & 1));
  }
  const uint32_t tile_bits = n - m;
  a.xcd_bits = tile_bits >= 6 ? tile_bits : 0;
}

size_t tile_bytes(uint32_t m, uint8_t prec) { return size_t(prec == 0 ? 8 : 16) << m; }

} // namespace

// A pass reads and writes every amplitude, a monomial gate by itself only the
// lines with rows other than the identity's.  On states that fill the chip a
// few such gates (controlled phases, Toffolis) are therefore faster one by
// one.  With T the time of a read and a write of the state at 6.55 TB/s, a pass
// takes about 5 us + T (1.12 T above 512 MiB) and a quarter of a microsecond
// per gate, a launch 5 us + a T times the share of lines touched, and with four
// targets and more at least the share `least` of T (its rows are gathered).
// Up to 512 MiB the caches serve lines of 64 bytes: a = 1 behind another pass
// (two gates of four targets, 6 rows of 16, 24 qubits f64: 108 us, 74 in a
// pass), 0.75 where the state was read before; above, lines of 128 bytes, a =
// 1.15 up to 2 GiB, then 1.4.  us, one by one / in a pass: two phases with 1,
// 2, 4 controls on high qubits, f64 24 qubits 36 / 90, 23 / 99, 53 / 99, 28
// qubits 850 / 1500, 393 / 1591, 270 / 1593, 30 qubits 3772 / 5882, 1788 /
// 6342, 872 / 6301; five with one control 88 / 100, 2105 / 1579, 9579 / 6460.
bool group_pays(const GatePlan *const *plans, size_t n_plans, uint32_t n) {
  constexpr double least[2][3] = {{0.1, 0.25, 0.7}, {0.06, 0.12, 0.35}}; // k = 4, 5, 6
  if (n_plans < 2 || n > kMaxGroupQubits)
    return false;
  const uint8_t prec = plans[0]->precision;
  if (!many_tiles(n, prec))
    return true;
  const double bytes = double(prec == 0 ? 8 : 16) * double(uint64_t(1) << n);
  const double mib = bytes / (1 << 20), t = 2.0 * bytes / 6.55e6;
  const bool cached = mib <= 512;
  const double a = cached ? 1.0 : mib <= 2048 ? 1.15 : 1.4;
  const uint32_t line_bits = (prec == 0 ? 4 : 3) - cached;
  double alone = 0.0;
  for (size_t i = 0; i < n_plans; ++i) {
    const GatePlan &p = *plans[i];
    if (p.variant != 2)
      return true;
    double share = a * touched_lines(p, line_bits);
    if (p.k >= 4 && p.k <= 6)
      share = std::max(share, least[n >= 27][p.k - 4]);
    if (p.n_active > 0)
      alone += 5.0 + share * t;
  }
  return alone >= 5.0 + (cached ? 1.0 : 1.12) * t + 0.25 * double(n_plans);
}

void launch_group(const GatePlan *const *plans, size_t n_plans, hipStream_t stream, void *sv,
                  uint32_t n) {
  if (n_plans == 0)
    return;
  const uint8_t prec = plans[0]->precision;
  GroupArgs a;
  describe_group(plans, n_plans, n, a.h, a.g);
  if (a.h.n_gates == 0)
    return;
  const size_t lds = tile_bytes(a.h.m, prec);
  const dim3 grid(1u << (n - a.h.m)), block(1u << a.h.thread_bits);
  if (prec == 0)
    many_tiles(n, prec) ? launch_k_group<float, 5>(grid, block, lds, stream, sv, a)
                        : launch_k_group<float, 4>(grid, block, lds, stream, sv, a);
  else
    many_tiles(n, prec) ? launch_k_group<double, 4>(grid, block, lds, stream, sv, a)
                        : launch_k_group<double, 3>(grid, block, lds, stream, sv, a);
  check(hipGetLastError(), "hipLaunchKernelGGL(k_group)");
}

size_t group_batch_bytes(size_t n_groups, size_t n_plans) {
  return n_groups * sizeof(GroupHead) + n_plans * sizeof(GroupGate);
}

void launch_group_batch(const GroupItem *items, size_t n_items, uint32_t n, void *table,
                        hipStream_t stream) {
  if (n_items == 0)
    return;
  const uint8_t prec = items[0].plans[0]->precision;
  if (many_tiles(n, prec))
    throw Error("grouped gates on a " + std::to_string(n) +
                "-qubit statevector fill the chip by themselves");
  size_t n_plans = 0;
  for (size_t i = 0; i < n_items; ++i)
    n_plans += items[i].n_plans;
  std::vector<unsigned char> host(group_batch_bytes(n_items, n_plans));
  GroupHead *heads = reinterpret_cast<GroupHead *>(host.data());
  GroupGate *gates = reinterpret_cast<GroupGate *>(heads + n_items);
  uint64_t at = 0;
  for (size_t i = 0; i < n_items; ++i) {
    const GroupItem &it = items[i];
    if (it.plans[0]->precision != prec)
      throw Error("grouped plans must share the precision");
    if (i && it.round < items[i - 1].round)
      throw Error("rounds of grouped gates must not decrease");
    describe_group(it.plans, it.n_plans, n, heads[i], gates + at);
    heads[i].sv = it.sv;
    heads[i].first = at;
    at += it.n_plans;
  }
  check(hipMemcpyAsync(table, host.data(), host.size(), hipMemcpyHostToDevice, stream),
        "hipMemcpyAsync(group table)");
  const auto *d_heads = static_cast<const GroupHead *>(table);
  const auto *d_gates = reinterpret_cast<const GroupGate *>(d_heads + n_items);
  const size_t lds = tile_bytes(heads[0].m, prec);
  const dim3 block(1u << heads[0].thread_bits);
  for (size_t i = 0; i < n_items;) {
    size_t end = i + 1;
    while (end < n_items && items[end].round == items[i].round && end - i < 32768)
      ++end;
    const dim3 grid(1u << (n - heads[0].m), unsigned(end - i));
    if (prec == 0)
      launch_k_group_batch<float, 4>(grid, block, lds, stream, d_heads + i, d_gates);
    else
      launch_k_group_batch<double, 3>(grid, block, lds, stream, d_heads + i, d_gates);
    check(hipGetLastError(), "hipLaunchKernelGGL(k_group_batch)");
    i = end;
  }
  // Pageable memory: the copy has read it when hipMemcpyAsync returns.
}

} // namespace cast_hip
