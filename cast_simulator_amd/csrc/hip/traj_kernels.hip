// Batched-trajectory kernels for gfx950: a persistent launch (k_traj) for many
// tasks or small statevectors, a launch per gate step (k_traj_step,
// k_traj_finish) for few tasks on larger ones.
//
// k_traj: one workgroup owns one statevector slot and takes whole tasks from a
// global counter until the list is exhausted; no workgroup ever waits on
// another, so any grid size drains.  A task is (checkpoint, gate list): the
// first applied gate reads the checkpoint statevector and writes the slot,
// every later gate updates the slot in place, with a workgroup barrier
// between gates.  Gates use wave tiles (coalesced 64-amplitude rows, cross-
// lane exchange of targets below bit 6) when n >= k + 6, else one combo per
// thread.  A wave keeps 16 amplitude loads in flight per lane whatever k is
// (16 / K tiles per step for k <= 4), since one workgroup alone must cover
// the memory latency of its statevector.  Gates of k = 4 to 6 (k = 5, 6 in
// f32 only) use the three-product form, the pool holding [Re M | Im M | Re M
// + Im M]: k = 4 on the VALU, k = 5 and 6 on the matrix cores.  At the end the workgroup reduces, in f64, the
// squared norm and sum |amp|^2 (-1)^(bit a xor bit b) for each requested
// pair (a, b), and can copy the final state out.
//
// The gate update is the one of src/cpp/cuda/cuda_gen.cpp:241-283 (local
// basis i sets bit q[b] for bit b of i; new[r] = sum_c M[r][c] old[c]).

#include "cast_hip.h"
#include "common.hpp"
#include "device_core.hpp"

#include <algorithm>
#include <string>

namespace cast_hip {
namespace {

using dev::combo_base;
using dev::insert_zero;
using dev::local_delta;
using dev::V2;

constexpr int kMaxPairs = 32;
constexpr int kMaxBlock = 512;
constexpr int kMaxWaves = kMaxBlock / 64;
constexpr uint32_t kMaxTrajGateQubits = 6; // 4 at f64
// A step is cut into this many workgroups of at most 256 threads: two share a
// CU, so that one stages its operands while the other multiplies.  Several
// rounds of the CUs even out gates of different size; f32 stages operands per
// workgroup, so fewer.  188 tasks of 20 qubits, ms in 2048, 4096, 8192 groups:
// f32 15.4, 14.9, 15.0 (512 threads 15.8, 15.9, 16.5), f64 38.8, 37.5, 36.0
// (512: 38.1, 36.6, 36.1); 128 threads 16.4-18.6 and 38.1-42.0.
template <typename T> constexpr uint32_t kStepGroups = sizeof(T) == 4 ? 4096 : 8192;
constexpr uint32_t kStepBlock = 256;
// ... and the closing sums into this many.
constexpr uint32_t kSumGroups = 2048;
// Host lengths of tasks that k_traj_lengths takes, in its arguments (4 KiB at most).
constexpr uint32_t kMaxLengths = 960;

// Layouts the host bindings rely on (no padding surprises across compilers).
static_assert(sizeof(cast_hip_traj_gate_t) == 12, "cast_hip_traj_gate_t layout");
static_assert(sizeof(cast_hip_traj_task_t) == 16, "cast_hip_traj_task_t layout");
static_assert(sizeof(cast_hip_traj_launch_t) == 376, "cast_hip_traj_launch_t layout");

struct TrajScalars {
  uint64_t n_matrix_elems;
  uint32_t n_tasks, n_gates, n_checkpoints, n_qubits, n_pairs, log2_block, flags;
  uint32_t pairs[2 * kMaxPairs];
};

// Gate operands staged in LDS by the k = 6 (f32 products) and the split-
// product gates, one buffer shared by both: 48 KiB at f32, none at f64.
template <typename T> constexpr size_t kGateLdsBytes = sizeof(T) == 4 ? 48 * 1024 : 16;

__global__ void k_fill_u32(uint32_t *__restrict__ p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = v;
}

using dev::opaque_u32;

// The calling wave's place among the waves that share a gate: those of the
// workgroup that owns the statevector, or of all its parts.
struct Share {
  uint32_t wave, n_waves;
};

// One gate over the waves' share of the statevector, wave tiles.  q[] are
// the ascending targets, of which exactly L are below 6.
template <typename T, int KL, int L>
__device__ __forceinline__ void wg_tile_gate(const T *src, T *dst, const T *__restrict__ mat,
                                             const uint32_t *q, uint32_t n, Share sh) {
  constexpr int U = KL >= 4 ? 1 : (16 >> KL); // tiles per step
  // Tile layout: register bit j < L -> the j-th non-target position >= 6,
  // register bit j >= L -> target q[j] (targets >= 6); the tile index is
  // deposited around the ascending set of those positions.
  uint64_t tmask = 0;
#pragma unroll
  for (int b = 0; b < KL; ++b)
    tmask |= uint64_t(1) << q[b];
  uint32_t reg_pos[KL], low_t[L > 0 ? L : 1], ins[KL];
  uint64_t f = ~tmask & ~uint64_t(63), fmask = 0;
#pragma unroll
  for (int j = 0; j < L; ++j) {
    low_t[j] = q[j];
    reg_pos[j] = uint32_t(__builtin_ctzll(f));
    fmask |= uint64_t(1) << reg_pos[j];
    f &= f - 1;
  }
#pragma unroll
  for (int j = L; j < KL; ++j)
    reg_pos[j] = q[j];
  uint64_t im = fmask | (tmask & ~uint64_t(63));
#pragma unroll
  for (int b = 0; b < KL; ++b) {
    ins[b] = uint32_t(__builtin_ctzll(im)) - 6;
    im &= im - 1;
  }

  const uint32_t lane = threadIdx.x & 63u, wave = sh.wave, n_waves = sh.n_waves;
  const uint64_t n_tiles = uint64_t(1) << (n - 6 - KL);
  auto tile_ptr = [&](uint64_t tile) {
#pragma unroll
    for (int b = 0; b < KL; ++b)
      tile = insert_zero(tile, ins[b]);
    return 2 * ((tile << 6) | lane);
  };
  if (n_tiles >= uint64_t(U)) {
    // n_tiles and U are powers of two, so every step is whole.
    for (uint64_t t0 = uint64_t(wave) * U; t0 < n_tiles; t0 += uint64_t(n_waves) * U) {
      // Re-derived each step so the K*K matrix entries are read by scalar
      // loads inside the loop rather than hoisted into VGPRs.
      const T *m = mat + opaque_u32(0);
      const T *s[U];
      T *d[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t off = tile_ptr(t0 + u);
        s[u] = src + off;
        d[u] = dst + off;
      }
      dev::tile_step<T, KL, L, U, (KL >= 4)>(s, d, m, reg_pos, low_t, lane);
    }
  } else {
    for (uint64_t t = wave; t < n_tiles; t += n_waves) {
      const T *m = mat + opaque_u32(0);
      const uint64_t off = tile_ptr(t);
      dev::tile_update<T, KL, L, (KL >= 4)>(src + off, dst + off, m, reg_pos, low_t, lane);
    }
  }
}

// Small statevectors (n < k + 6): one combo per thread.
template <typename T, int KL>
__device__ __forceinline__ void wg_dense_gate(const T *src, T *dst, const T *__restrict__ mat,
                                              const uint32_t *q, uint32_t n, Share sh) {
  constexpr int K = 1 << KL;
  using VT = typename V2<T>::type;
  uint64_t delta[K];
#pragma unroll
  for (int i = 0; i < K; ++i)
    delta[i] = local_delta<KL>(uint32_t(i), q);
  const uint64_t combos = uint64_t(1) << (n - KL);
  for (uint64_t c = sh.wave * 64u + (threadIdx.x & 63u); c < combos; c += sh.n_waves * 64u) {
    const T *m = mat + opaque_u32(0);
    const VT *in = reinterpret_cast<const VT *>(src);
    VT *out = reinterpret_cast<VT *>(dst);
    const uint64_t base = combo_base<KL>(c, q);
    if constexpr (KL >= 4) { // three real matrices [Re | Im | Re + Im]
      T vr[K], vi[K];
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const VT x = in[base + delta[i]];
        vr[i] = x.x;
        vi[i] = x.y;
      }
#pragma unroll
      for (int r = 0; r < K; ++r) {
        T t1 = T(0), t2 = T(0), t3 = T(0);
#pragma unroll
        for (int cc = 0; cc < K; ++cc) {
          t1 = dev::fma_t(m[r * K + cc], vr[cc], t1);
          t2 = dev::fma_t(m[K * K + r * K + cc], vi[cc], t2);
          t3 = dev::fma_t(m[2 * K * K + r * K + cc], vr[cc] + vi[cc], t3);
        }
        VT o;
        o.x = t1 - t2;
        o.y = t3 - t1 - t2;
        out[base + delta[r]] = o;
      }
    } else {
      dev::dense_combo<T, KL>(in, out, m, base, delta);
    }
  }
}

// k = 5 at f32 on the matrix cores: the three-product contraction of the
// plain-path matrix-core kernel (Out = M V over tiles of 16 combos with
// v_mfma_f32_16x16x4), run by the workgroup's waves over the statevector.
// Lane l owns combo l % 16 of a tile and loads inputs 4 s + l / 16; the
// three real K x K matrices ([Re | Im | Re + Im] from the pool) stay in
// registers for the whole gate.  Two tiles per step keep 16 loads per lane
// in flight.  Any target set: addresses come from the combo's bit deposit.
// (The VALU three-product update of k = 5 costs 12 flops per byte at f32,
// above the 9.8 flop/B VALU ridge of the chip; here it is MFMA work.)
template <int KL>
__device__ __forceinline__ void wg_mfma_gate(const float *src, float *dst,
                                             const float *__restrict__ m3, const uint32_t *q,
                                             uint32_t n, Share sh) {
  constexpr int K = 1 << KL, RB = K / 16, KS = K / 4, U = 2;
  using VT = typename V2<float>::type;
  using AV = dev::Acc4<float>::type;
  const VT *in = reinterpret_cast<const VT *>(src);
  VT *out = reinterpret_cast<VT *>(dst);
  const uint32_t lane = threadIdx.x & 63u, j = lane >> 4, col = lane & 15u;
  const uint32_t wave = sh.wave, n_waves = sh.n_waves;
  float a[3][RB][KS];
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        a[m][rb][s] = m3[m * K * K + (16 * rb + col) * K + 4 * s + j];
  uint64_t din[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    din[s] = local_delta<KL>(4 * s + j, q);
  // accumulator register i of lane l holds output row 16 rb + 4 (l / 16) + i
  uint64_t dout[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dout[rb][i] = local_delta<KL>(16 * rb + 4 * j + i, q);
  // n >= KL + 5, so n_tiles = 2^(n - KL - 4) is a multiple of U
  const uint64_t n_tiles = uint64_t(1) << (n - KL - 4);
  for (uint64_t t0 = uint64_t(wave) * U; t0 < n_tiles; t0 += uint64_t(n_waves) * U) {
    uint64_t base[U];
    float br[U][KS], bi[U][KS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      base[u] = combo_base<KL>((t0 + u) * 16 + col, q);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const VT x = in[base[u] + din[s]];
        br[u][s] = x.x;
        bi[u][s] = x.y;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        AV t1 = {0, 0, 0, 0}, t2 = {0, 0, 0, 0}, t3 = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          t1 = dev::mfma16(a[0][rb][s], br[u][s], t1);
          t2 = dev::mfma16(a[1][rb][s], bi[u][s], t2);
          t3 = dev::mfma16(a[2][rb][s], br[u][s] + bi[u][s], t3);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          VT o;
          o.x = t1[i] - t2[i];
          o.y = t3[i] - t1[i] - t2[i];
          out[base[u] + dout[rb][i]] = o;
        }
      }
  }
}

// k = 6 at f32 on the matrix cores, as the plain path's k = 6 kernel: Re M
// and Im M (32 KiB) are staged in LDS once per gate, laid out so that the
// operand (m, rb, s) of lane l is element ((m * 4 + rb) * 16 + s) * 64 + l
// (every read is 64 consecutive values); Re M + Im M is formed on the fly.
// A lane owns combo l % 16 of a 16-combo tile and keeps its 16 inputs in
// registers while two 16-row output blocks are produced per pass (six
// independent accumulator chains).  Needs n >= 12 (checked by the caller).
// The caller's barrier after every gate keeps the next gate's staging from
// overwriting operands still in use.
__device__ __forceinline__ void wg_mfma6_gate(const float *src, float *dst,
                                              const float *__restrict__ m3, const uint32_t *q,
                                              uint32_t n, Share sh, float *a_lds) {
  constexpr int KL = 6, K = 64, RB = 4, KS = 16;
  using VT = typename V2<float>::type;
  using AV = dev::Acc4<float>::type;
  for (uint32_t i = threadIdx.x; i < 2 * RB * KS * 64; i += blockDim.x) {
    const uint32_t l = i & 63u, s = (i >> 6) & (KS - 1), rb = (i >> 10) & (RB - 1), m = i >> 12;
    a_lds[i] = m3[m * K * K + (16 * rb + (l & 15u)) * K + 4 * s + (l >> 4)];
  }
  __syncthreads();
  const VT *in = reinterpret_cast<const VT *>(src);
  VT *out = reinterpret_cast<VT *>(dst);
  const uint32_t lane = threadIdx.x & 63u, j = lane >> 4, col = lane & 15u;
  const uint32_t wave = sh.wave, n_waves = sh.n_waves;
  uint64_t din[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    din[s] = local_delta<KL>(4 * s + j, q);
  const uint64_t n_tiles = uint64_t(1) << (n - KL - 4);
  for (uint64_t t = wave; t < n_tiles; t += n_waves) {
    const uint64_t base = combo_base<KL>(t * 16 + col, q);
    float br[KS], bi[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const VT x = in[base + din[s]];
      br[s] = x.x;
      bi[s] = x.y;
    }
#pragma unroll
    for (int rp = 0; rp < RB; rp += 2) {
      // Re-read per tile (not hoisted out of the tile loop into registers).
      const float *a = a_lds + rp * KS * 64 + lane + opaque_u32(0);
      AV t1[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, t2[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}},
         t3[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float ar = a[h * KS * 64 + s * 64];
          const float ai = a[RB * KS * 64 + h * KS * 64 + s * 64];
          t1[h] = dev::mfma16(ar, br[s], t1[h]);
          t2[h] = dev::mfma16(ai, bi[s], t2[h]);
          t3[h] = dev::mfma16(ar + ai, br[s] + bi[s], t3[h]);
        }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          VT o;
          o.x = t1[h][i] - t2[h][i];
          o.y = t3[h][i] - t1[h][i] - t2[h][i];
          out[base + local_delta<KL>(16 * (rp + h) + 4 * j + i, q)] = o;
        }
    }
  }
}

// k = 5, 6 at f32 through bf16 split products (dev::split_tile): the splits
// of Re M and Im M are staged in LDS once per gate (k = 6: 48 KiB, k = 5:
// 12 KiB of the shared gate buffer); the workgroup's waves take 16-combo
// tiles in turn.  Needs n >= KL + 4.  The caller's barrier after every gate
// keeps the next gate's staging from overwriting operands still in use.
template <int KL>
__device__ __forceinline__ void wg_split_gate(const float *src, float *dst,
                                              const float *__restrict__ m3, const uint32_t *q,
                                              uint32_t n, Share sh,
                                              dev::bf16x8_t *a_lds) {
  // k = 5: two tiles per step, so that each lane keeps 16 loads in flight as
  // at k = 6 (one workgroup streams the whole statevector).
  constexpr int U = KL == 5 ? 2 : 1;
  dev::split_stage<KL>(m3, a_lds);
  __syncthreads();
  const dev::SplitLane<KL> sl(q);
  const uint32_t wave = sh.wave, n_waves = sh.n_waves;
  // n >= KL + 5 for k = 5 (checked by the caller), so n_tiles is a multiple of U
  const uint64_t n_tiles = uint64_t(1) << (n - KL - 4);
  for (uint64_t t = uint64_t(wave) * U; t < n_tiles; t += uint64_t(n_waves) * U)
    dev::split_tile<KL, U>(reinterpret_cast<const float2 *>(src),
                           reinterpret_cast<float2 *>(dst), a_lds, q, sl, t);
}

template <typename T, int KL>
__device__ __forceinline__ void wg_gate_k(const T *src, T *dst, const T *__restrict__ mat,
                                          const uint32_t *q, uint32_t n, Share sh) {
  if (n < uint32_t(KL) + 6)
    return wg_dense_gate<T, KL>(src, dst, mat, q, n, sh);
  uint32_t n_low = 0;
#pragma unroll
  for (int b = 0; b < KL; ++b)
    n_low += q[b] < 6;
  if constexpr (KL == 5) { // f32 only: matrix cores, any targets
    if constexpr (sizeof(T) == 4)
      wg_mfma_gate<KL>(src, dst, mat, q, n, sh);
  } else {
    switch (n_low) {
    case 0:
      return wg_tile_gate<T, KL, 0>(src, dst, mat, q, n, sh);
    case 1:
      if constexpr (KL >= 1)
        return wg_tile_gate<T, KL, 1>(src, dst, mat, q, n, sh);
      break;
    case 2:
      if constexpr (KL >= 2)
        return wg_tile_gate<T, KL, 2>(src, dst, mat, q, n, sh);
      break;
    case 3:
      if constexpr (KL == 3 || KL == 4)
        return wg_tile_gate<T, KL, 3>(src, dst, mat, q, n, sh);
      break;
    case 4:
      if constexpr (KL == 4)
        return wg_tile_gate<T, KL, 4>(src, dst, mat, q, n, sh);
      break;
    default:
      break;
    }
  }
}

// Squared norm and the pair sums of the workgroup's final state, written to
// out_row[0 .. 1 + n_pairs).  Amplitude i = tid + B r (B = blockDim.x = 2^bB).
// The sign of pair (a, b) at i factors into a per-thread part (positions
// below bB), applied once at the end, and the parity of r & m for the pair's
// row mask m.  16 rows are taken at a time: the 16-point Walsh-Hadamard
// transform of their probabilities (64 additions) holds the sums under every
// mask of the low 4 row bits, and the parity of the others is the same for the
// whole workgroup, so a pair costs one f64 FMA for 16 amplitudes instead of
// one each: the sums of 188 states of 20 qubits (f32, 19 pairs, one workgroup
// each) 1.67 -> 1.1 ms.  Rows [first_row, first_row + n_rows) are summed.
template <typename T>
__device__ __forceinline__ void wg_observe(const T *sv, uint32_t n, uint32_t n_pairs, uint32_t bB,
                           const uint32_t *s_pairs, uint32_t first_row, uint32_t n_rows,
                           double *out_row, double *red) {
  using VT = typename V2<T>::type;
  constexpr int R = 16;
  const VT *amp = reinterpret_cast<const VT *>(sv);
  const uint32_t tid = threadIdx.x;
  uint32_t rmask[kMaxPairs];
  uint32_t tneg = 0; // bit j: the per-thread sign of pair j is -1
#pragma unroll
  for (int j = 0; j < kMaxPairs; ++j) {
    rmask[j] = 0;
    if (uint32_t(j) < n_pairs) {
      const uint32_t qa = __builtin_amdgcn_readfirstlane(s_pairs[2 * j]);
      const uint32_t qb = __builtin_amdgcn_readfirstlane(s_pairs[2 * j + 1]);
      rmask[j] = (qa >= bB ? 1u << (qa - bB) : 0u) ^ (qb >= bB ? 1u << (qb - bB) : 0u);
      const uint32_t tb = (qa < bB ? (tid >> qa) & 1u : 0u) ^ (qb < bB ? (tid >> qb) & 1u : 0u);
      tneg |= tb << j;
    }
  }
  double acc[1 + kMaxPairs];
#pragma unroll
  for (int j = 0; j < 1 + kMaxPairs; ++j)
    acc[j] = 0.0;
  const uint64_t len = uint64_t(1) << n;
  const uint32_t rows = first_row + n_rows;
  typedef double Rows __attribute__((ext_vector_type(R)));
  for (uint32_t r0 = first_row; r0 < rows; r0 += R) {
    double p[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const uint64_t i = tid + (uint64_t(r0 + u) << bB);
      p[u] = 0.0;
      if (r0 + u < rows && i < len) {
        const VT x = amp[i];
        const double re = double(x.x), im = double(x.y);
        p[u] = re * re + im * im;
      }
    }
    Rows w;
#pragma unroll
    for (int u = 0; u < R; ++u)
      w[u] = p[u];
#pragma unroll
    for (int b = 1; b < R; b <<= 1)
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (!(u & b)) {
          const double lo = w[u], hi = w[u | b];
          w[u] = lo + hi;
          w[u | b] = lo - hi;
        }
    acc[0] += w[0];
#pragma unroll
    for (int j = 0; j < kMaxPairs; ++j)
      if (uint32_t(j) < n_pairs) { // uniform
        const bool neg = __builtin_popcount(r0 & rmask[j]) & 1;
        acc[1 + j] = __builtin_fma(neg ? -1.0 : 1.0, w[rmask[j] & (R - 1)], acc[1 + j]);
      }
  }
#pragma unroll
  for (int j = 0; j < kMaxPairs; ++j)
    if ((tneg >> j) & 1u)
      acc[1 + j] = -acc[1 + j];

  // Workgroup reduction in a fixed order: xor-shuffle within each wave, then
  // thread j sums entry j over the waves.
  const uint32_t lane = tid & 63u, wave = tid >> 6, n_waves = blockDim.x >> 6;
  const uint32_t cnt = 1 + n_pairs;
#pragma unroll
  for (int j = 0; j < 1 + kMaxPairs; ++j) {
    if (uint32_t(j) < cnt) {
      double x = acc[j];
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1)
        x += __shfl_xor(x, m, 64);
      if (lane == 0)
        red[wave * (1 + kMaxPairs) + j] = x;
    }
  }
  __syncthreads();
  if (tid < cnt) {
    double s = 0.0;
    for (uint32_t w = 0; w < n_waves; ++w)
      s += red[w * (1 + kMaxPairs) + tid];
    out_row[tid] = s;
  }
  __syncthreads();
}

// One gate of a task by the waves `sh` describes; false for a descriptor that
// is out of range (nothing is done then).  `gate_lds` holds kGateLdsBytes<T>.
template <typename T>
__device__ __forceinline__ bool wg_gate(const cast_hip_traj_gate_t &d, const T *src, T *dst,
                                        const T *__restrict__ matrices, const TrajScalars &a,
                                        uint32_t n, Share sh, unsigned char *gate_lds) {
  const bool f32_products = a.flags & CAST_HIP_TRAJ_FLAG_MFMA_F32;
  // The descriptor is the same for the whole workgroup; readfirstlane
  // states that, so geometry and matrix address live in SGPRs.
  const uint32_t k = __builtin_amdgcn_readfirstlane(d.k);
  const uint32_t moff = __builtin_amdgcn_readfirstlane(d.matrix_offset);
  uint32_t q[kMaxTrajGateQubits];
  bool ok = k >= 1 && k <= (sizeof(T) == 4 ? kMaxTrajGateQubits : 4u);
  ok = ok && (k < 6 || n >= 12); // the k = 6 path needs 64 tiles of 16 combos
#pragma unroll
  for (uint32_t b = 0; b < kMaxTrajGateQubits; ++b) {
    q[b] = __builtin_amdgcn_readfirstlane(d.q[b]);
    if (b < k)
      ok = ok && q[b] < n && (b == 0 || q[b] > q[b - 1]);
  }
  // k = 4, 5 entries hold three real K x K matrices: 3 K^2 / 2 complex slots.
  const uint64_t entries = k >= 4 ? uint64_t(3) << (2 * k - 1) : (uint64_t(1) << (2 * k));
  ok = ok && uint64_t(moff) + entries <= a.n_matrix_elems;
  if (!ok)
    return false;
  const T *mat = matrices + 2 * uint64_t(moff);
  switch (k) {
  case 1:
    wg_gate_k<T, 1>(src, dst, mat, q, n, sh);
    break;
  case 2:
    wg_gate_k<T, 2>(src, dst, mat, q, n, sh);
    break;
  case 3:
    wg_gate_k<T, 3>(src, dst, mat, q, n, sh);
    break;
  case 4:
    wg_gate_k<T, 4>(src, dst, mat, q, n, sh);
    break;
  case 5: // f32 only (checked above)
    if constexpr (sizeof(T) == 4) {
      if (f32_products || n < 11)
        wg_gate_k<T, 5>(src, dst, mat, q, n, sh);
      else
        wg_split_gate<5>(src, dst, mat, q, n, sh, reinterpret_cast<dev::bf16x8_t *>(gate_lds));
    }
    break;
  default: // k = 6, f32 only, n >= 12 (checked above)
    if constexpr (sizeof(T) == 4) {
      if (f32_products)
        wg_mfma6_gate(src, dst, mat, q, n, sh, reinterpret_cast<float *>(gate_lds));
      else
        wg_split_gate<6>(src, dst, mat, q, n, sh, reinterpret_cast<dev::bf16x8_t *>(gate_lds));
    }
    break;
  }
  return true;
}

// The task order[t] of the launch, checked; false (and the error flag set, by
// every lane: no lane-dependent branch) when it is out of range.
__device__ __forceinline__ bool fetch_task(const cast_hip_traj_task_t *tasks,
                                           const uint32_t *order, uint32_t t, uint32_t *work,
                                           const TrajScalars &a, uint32_t &ti,
                                           cast_hip_traj_task_t &task) {
  ti = __builtin_amdgcn_readfirstlane(order[t]);
  bool ok = ti < a.n_tasks;
  if (ok) {
    const cast_hip_traj_task_t tk = tasks[ti];
    task.first_gate = __builtin_amdgcn_readfirstlane(tk.first_gate);
    task.n_gates = __builtin_amdgcn_readfirstlane(tk.n_gates);
    task.checkpoint = __builtin_amdgcn_readfirstlane(tk.checkpoint);
    ok = task.checkpoint < a.n_checkpoints && task.first_gate <= a.n_gates &&
         task.n_gates <= a.n_gates - task.first_gate;
  }
  if (!ok)
    atomicOr(&work[1], 1u);
  return ok;
}

// Rows of wg_observe in a whole statevector.
__host__ __device__ __forceinline__ uint32_t observe_rows(uint32_t n, uint32_t log2_block) {
  return n > log2_block ? 1u << (n - log2_block) : 1u;
}

// The workgroup's copy of (a part of) a final state.
template <typename T> __device__ __forceinline__ void wg_dump(const T *cur, T *to, uint64_t len) {
  using VT = typename V2<T>::type;
  const VT *src = reinterpret_cast<const VT *>(cur);
  VT *dst = reinterpret_cast<VT *>(to);
  for (uint64_t i0 = threadIdx.x; i0 < len; i0 += uint64_t(blockDim.x) * 8) {
    VT x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint64_t i = i0 + uint64_t(u) * blockDim.x;
      if (i < len)
        x[u] = src[i];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint64_t i = i0 + uint64_t(u) * blockDim.x;
      if (i < len)
        dst[i] = x[u];
    }
  }
}

// Built for OCC waves per SIMD (second launch-bound argument): 2 allows 256
// VGPRs (no spills, one 512-thread workgroup per CU), 4 allows 128 (spills,
// but two workgroups per CU keep twice the loads in flight).
template <typename T, int OCC>
__global__ void __launch_bounds__(kMaxBlock, OCC)
    k_traj(const cast_hip_traj_task_t *__restrict__ tasks, const uint32_t *__restrict__ order,
           const cast_hip_traj_gate_t *__restrict__ gates, const T *__restrict__ matrices,
           const T *__restrict__ checkpoints, T *__restrict__ slots, double *__restrict__ out,
           T *__restrict__ dump, uint32_t *__restrict__ work, TrajScalars a) {
  __shared__ uint32_t s_task;
  __shared__ uint32_t s_pairs[2 * kMaxPairs];
  __shared__ double red[kMaxWaves * (1 + kMaxPairs)];
  __shared__ __align__(16) unsigned char gate_lds[kGateLdsBytes<T>];
  const Share sh{threadIdx.x >> 6, blockDim.x >> 6};
  if (threadIdx.x < 2 * a.n_pairs)
    s_pairs[threadIdx.x] = a.pairs[threadIdx.x];
  for (;;) {
    // The leading barrier keeps every path into the lane-0 fetch below
    // convergent: without it the compiler may thread lanes that skipped a
    // lane-0-only branch straight to the next barrier, into a loop that waits
    // for a task index lane 0 never gets to fetch.
    __syncthreads();
    if (threadIdx.x == 0)
      s_task = atomicAdd(&work[0], 1u);
    __syncthreads();
    const uint32_t t = __builtin_amdgcn_readfirstlane(s_task);
    __syncthreads();
    if (t >= a.n_tasks)
      break;
    const uint32_t n = opaque_u32(a.n_qubits);
    const uint64_t len = uint64_t(1) << n;
    T *slot = slots + 2 * len * blockIdx.x;
    uint32_t ti;
    cast_hip_traj_task_t task{};
    if (!fetch_task(tasks, order, t, work, a, ti, task))
      continue;
    const T *cur = checkpoints + 2 * len * task.checkpoint; // state the next gate reads
    for (uint32_t g = 0; g < task.n_gates; ++g) {
      if (!wg_gate<T>(gates[task.first_gate + g], cur, slot, matrices, a, n, sh, gate_lds)) {
        atomicOr(&work[1], 1u);
        continue;
      }
      cur = slot;
      __syncthreads();
    }
    wg_observe<T>(cur, n, a.n_pairs, a.log2_block, s_pairs, 0, observe_rows(n, a.log2_block),
                  out + uint64_t(ti) * (1 + a.n_pairs), red);
    if (dump) {
      wg_dump<T>(cur, dump + 2 * len * ti, len);
      __syncthreads();
    }
  }
}

// Gate g of the tasks order[first ...), every statevector shared by `parts`
// workgroups; slot t belongs to the task order[first + t].  A workgroup that
// owns a statevector (k_traj) is held to what one CU can do, and the launch to
// its longest task: 188 tasks of 20 qubits and up to 40 gates at f32 took
// 29.4 ms with 0.73 ms per gate on each of 188 CUs.  With a launch per step all
// CUs share the tasks that are left: 14.9 ms (3.9 us per gate of 16.8 MB moved,
// 4.3 TB/s, k = 5 and 6 bound by the split products), 32 tasks 23.6 -> 2.7 ms.
// Each amplitude goes through the same operations as in k_traj.
template <typename T, int OCC>
__global__ void __launch_bounds__(kMaxBlock, OCC)
    k_traj_step(const cast_hip_traj_task_t *__restrict__ tasks, const uint32_t *__restrict__ order,
                const cast_hip_traj_gate_t *__restrict__ gates, const T *__restrict__ matrices,
                const T *__restrict__ checkpoints, T *__restrict__ slots,
                uint32_t *__restrict__ work, TrajScalars a, uint32_t first, uint32_t g,
                uint32_t parts) {
  __shared__ __align__(16) unsigned char gate_lds[kGateLdsBytes<T>];
  const uint32_t slot_i = blockIdx.x / parts, part = blockIdx.x % parts;
  uint32_t ti;
  cast_hip_traj_task_t task{};
  if (!fetch_task(tasks, order, first + slot_i, work, a, ti, task) || g >= task.n_gates)
    return;
  const uint32_t n = opaque_u32(a.n_qubits);
  const uint64_t len = uint64_t(1) << n;
  T *slot = slots + 2 * len * slot_i;
  const T *src = g == 0 ? checkpoints + 2 * len * task.checkpoint : slot;
  const uint32_t waves = blockDim.x >> 6;
  const Share sh{part * waves + (threadIdx.x >> 6), parts * waves};
  if (wg_gate<T>(gates[task.first_gate + g], src, slot, matrices, a, n, sh, gate_lds))
    return;
  atomicOr(&work[1], 1u);
  if (g == 0) { // left out: the next gate reads the slot
    using VT = typename V2<T>::type;
    for (uint64_t i = uint64_t(part) * blockDim.x + threadIdx.x; i < len;
         i += uint64_t(parts) * blockDim.x)
      reinterpret_cast<VT *>(slot)[i] = reinterpret_cast<const VT *>(src)[i];
  }
}

// Sums and dump of the tasks order[first ...) after their last step, `parts`
// workgroups each.  With several, a part leaves its sums at the start of the
// range of the slot that it alone has read (or that holds nothing, for a task
// without gates); k_traj_sum adds them up.  188 states of 20 qubits, f32: 1.1
// ms in one part, 0.56 in eight.
template <typename T>
__global__ void __launch_bounds__(kMaxBlock, 2)
    k_traj_finish(const cast_hip_traj_task_t *__restrict__ tasks,
                  const uint32_t *__restrict__ order, const T *__restrict__ checkpoints, T *slots,
                  double *__restrict__ out, T *__restrict__ dump, uint32_t *__restrict__ work,
                  TrajScalars a, uint32_t first, uint32_t parts) {
  __shared__ uint32_t s_pairs[2 * kMaxPairs];
  __shared__ double red[kMaxWaves * (1 + kMaxPairs)];
  if (threadIdx.x < 2 * a.n_pairs)
    s_pairs[threadIdx.x] = a.pairs[threadIdx.x];
  __syncthreads();
  const uint32_t slot_i = blockIdx.x / parts, part = blockIdx.x % parts;
  uint32_t ti;
  cast_hip_traj_task_t task{};
  if (!fetch_task(tasks, order, first + slot_i, work, a, ti, task))
    return;
  const uint64_t len = uint64_t(1) << a.n_qubits, mine = len / parts;
  T *slot = slots + 2 * len * slot_i;
  const T *cur = task.n_gates == 0 ? checkpoints + 2 * len * task.checkpoint : slot;
  if (dump) {
    wg_dump<T>(cur + 2 * mine * part, dump + 2 * (len * ti + mine * part), mine);
    __syncthreads();
  }
  const uint32_t n_rows = observe_rows(a.n_qubits, a.log2_block) / parts;
  // Every read of the range is over at the barrier before the sums go out.
  double *sums = parts == 1 ? out + uint64_t(ti) * (1 + a.n_pairs)
                            : reinterpret_cast<double *>(slot + 2 * mine * part);
  wg_observe<T>(cur, a.n_qubits, a.n_pairs, a.log2_block, s_pairs, n_rows * part, n_rows, sums,
                red);
}

// Sets the error flag for tasks of order[first ...) with more gates than the
// host says: these gates would be left out, since the steps follow the host's
// lengths.  One launch a run (about 3 us) for every 960 tasks.
struct TrajLengths {
  uint32_t n;
  uint32_t n_gates[kMaxLengths];
};
__global__ void __launch_bounds__(256)
    k_traj_lengths(const cast_hip_traj_task_t *__restrict__ tasks,
                   const uint32_t *__restrict__ order, uint32_t n_tasks, uint32_t first,
                   uint32_t *__restrict__ work, TrajLengths a) {
  for (uint32_t i = threadIdx.x; i < a.n; i += blockDim.x) {
    const uint32_t ti = order[first + i];
    if (ti < n_tasks && tasks[ti].n_gates > a.n_gates[i])
      atomicOr(&work[1], 1u);
  }
}

template <typename T>
__global__ void k_traj_sum(const cast_hip_traj_task_t *__restrict__ tasks,
                           const uint32_t *__restrict__ order, const T *__restrict__ slots,
                           double *__restrict__ out, uint32_t *__restrict__ work, TrajScalars a,
                           uint32_t first, uint32_t parts) {
  uint32_t ti;
  cast_hip_traj_task_t task{};
  const uint32_t slots_n = 1 + a.n_pairs;
  if (!fetch_task(tasks, order, first + blockIdx.x, work, a, ti, task) || threadIdx.x >= slots_n)
    return; // k_traj_finish left no sums for a task out of range
  const uint64_t len = uint64_t(1) << a.n_qubits, mine = len / parts;
  double s = 0.0;
  for (uint32_t p = 0; p < parts; ++p)
    s += reinterpret_cast<const double *>(slots + 2 * (len * blockIdx.x + mine * p))[threadIdx.x];
  out[uint64_t(ti) * slots_n + threadIdx.x] = s;
}

template <typename T, int OCC>
void launch_traj_t(const cast_hip_traj_launch_t &L, const TrajScalars &a, hipStream_t s) {
  hipLaunchKernelGGL((k_traj<T, OCC>), dim3(L.n_slots), dim3(L.block), 0, s,
                     reinterpret_cast<const cast_hip_traj_task_t *>(L.tasks),
                     reinterpret_cast<const uint32_t *>(L.order),
                     reinterpret_cast<const cast_hip_traj_gate_t *>(L.gates),
                     reinterpret_cast<const T *>(L.matrices),
                     reinterpret_cast<const T *>(L.checkpoints), reinterpret_cast<T *>(L.slots),
                     reinterpret_cast<double *>(L.out), reinterpret_cast<T *>(L.dump),
                     reinterpret_cast<uint32_t *>(L.work), a);
  check(hipGetLastError(), "hipLaunchKernelGGL(k_traj)");
}

template <typename T, int OCC>
void launch_steps_t(const cast_hip_traj_launch_t &L, const TrajScalars &a, const uint32_t *n_gates,
                    hipStream_t s) {
  const auto *tasks = reinterpret_cast<const cast_hip_traj_task_t *>(L.tasks);
  const auto *order = reinterpret_cast<const uint32_t *>(L.order);
  const auto *gates = reinterpret_cast<const cast_hip_traj_gate_t *>(L.gates);
  const T *mats = reinterpret_cast<const T *>(L.matrices);
  const T *ckpt = reinterpret_cast<const T *>(L.checkpoints);
  T *slots = reinterpret_cast<T *>(L.slots);
  uint32_t *work = reinterpret_cast<uint32_t *>(L.work);
  const uint32_t block = std::min(L.block, kStepBlock), waves = block / 64;
  // At most as many parts as leave every wave a k = 6 tile of 2^10 amplitudes.
  const uint32_t most =
      L.n_qubits > 10 ? std::max(1u, (1u << std::min(L.n_qubits - 10, 20u)) / waves) : 1u;
  // Parts of the closing sums: four or more groups of 16 rows (4096 amplitudes) each.
  auto parts_of = [&](uint32_t tasks_here) {
    const uint32_t rows = observe_rows(L.n_qubits, a.log2_block);
    uint32_t parts = 1;
    while (parts * tasks_here < kSumGroups && rows / (2 * parts) >= 64)
      parts *= 2;
    return parts;
  };
  for (uint32_t first = 0; first < L.n_tasks; first += kMaxLengths) {
    TrajLengths lengths;
    lengths.n = std::min(kMaxLengths, L.n_tasks - first);
    std::copy_n(n_gates + first, lengths.n, lengths.n_gates);
    hipLaunchKernelGGL(k_traj_lengths, dim3(1), dim3(256), 0, s, tasks, order, L.n_tasks, first,
                       work, lengths);
    check(hipGetLastError(), "hipLaunchKernelGGL(k_traj_lengths)");
  }
  for (uint32_t first = 0; first < L.n_tasks; first += L.n_slots) {
    const uint32_t here = std::min(L.n_slots, L.n_tasks - first);
    uint32_t active = here;
    const uint32_t n_steps = n_gates[first];
    for (uint32_t g = 0; g < n_steps; ++g) {
      while (n_gates[first + active - 1] <= g)
        --active;
      const uint32_t parts = std::min(most, std::max(1u, kStepGroups<T> / active));
      hipLaunchKernelGGL((k_traj_step<T, OCC>), dim3(active * parts), dim3(block), 0, s, tasks,
                         order, gates, mats, ckpt, slots, work, a, first, g, parts);
      check(hipGetLastError(), "hipLaunchKernelGGL(k_traj_step)");
    }
    const uint32_t parts = parts_of(here);
    hipLaunchKernelGGL((k_traj_finish<T>), dim3(here * parts), dim3(L.block), 0, s, tasks, order,
                       ckpt, slots, reinterpret_cast<double *>(L.out),
                       reinterpret_cast<T *>(L.dump), work, a, first, parts);
    check(hipGetLastError(), "hipLaunchKernelGGL(k_traj_finish)");
    if (parts == 1)
      continue;
    hipLaunchKernelGGL((k_traj_sum<T>), dim3(here), dim3(64), 0, s, tasks, order, slots,
                       reinterpret_cast<double *>(L.out), work, a, first, parts);
    check(hipGetLastError(), "hipLaunchKernelGGL(k_traj_sum)");
  }
}

} // namespace

void launch_traj(const cast_hip_traj_launch_t &L, const uint32_t *n_gates, hipStream_t stream) {
  if (L.precision > 1)
    throw Error("trajectory launch: precision must be 0 (F32) or 1 (F64)");
  if (L.n_qubits < 1 || L.n_qubits > 34)
    throw Error("trajectory launch: n_qubits must be in 1..34");
  if (L.n_slots < 1 || L.n_slots > (1u << 20))
    throw Error("trajectory launch: n_slots must be in 1..2^20");
  if (L.block != 64 && L.block != 128 && L.block != 256 && L.block != 512)
    throw Error("trajectory launch: block must be 64, 128, 256 or 512");
  if (L.n_pairs > kMaxPairs)
    throw Error("trajectory launch: at most 32 qubit pairs");
  if (L.waves_per_simd != 0 && L.waves_per_simd != 2 && L.waves_per_simd != 4)
    throw Error("trajectory launch: waves_per_simd must be 0, 2 or 4");
  for (uint32_t j = 0; j < L.n_pairs; ++j) {
    const uint32_t qa = L.pairs[2 * j], qb = L.pairs[2 * j + 1];
    if (qa >= L.n_qubits || qb >= L.n_qubits || qa == qb)
      throw Error("trajectory launch: pair " + std::to_string(j) + " = (" + std::to_string(qa) +
                  ", " + std::to_string(qb) + ") is not two distinct qubits below n");
  }
  if (!L.work)
    throw Error("trajectory launch: work buffer is null");
  if (L.n_tasks > 0 && (!L.tasks || !L.order || !L.out || !L.slots || !L.checkpoints ||
                        L.n_checkpoints == 0))
    throw Error("trajectory launch: null task, order, output, slot or checkpoint buffer");
  if (L.n_gates > 0 && (!L.gates || !L.matrices))
    throw Error("trajectory launch: null gate table or matrix pool");
  uint32_t *work = reinterpret_cast<uint32_t *>(L.work);
  hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, stream, work, 2u, 0u);
  check(hipGetLastError(), "hipLaunchKernelGGL(k_fill_u32)");
  if (L.n_tasks == 0)
    return;
  TrajScalars a{};
  a.n_matrix_elems = L.n_matrix_elems;
  a.n_tasks = L.n_tasks;
  a.n_gates = L.n_gates;
  a.n_checkpoints = L.n_checkpoints;
  a.n_qubits = L.n_qubits;
  a.n_pairs = L.n_pairs;
  a.log2_block = uint32_t(__builtin_ctz(L.block));
  if (L.flags & ~CAST_HIP_TRAJ_FLAG_MFMA_F32)
    throw Error("trajectory launch: unknown flags " + std::to_string(L.flags));
  a.flags = L.flags;
  for (uint32_t j = 0; j < 2 * L.n_pairs; ++j)
    a.pairs[j] = L.pairs[j];
  const bool occ4 = L.waves_per_simd == 4;
  if (n_gates) {
    for (uint32_t t = 1; t < L.n_tasks; ++t)
      if (n_gates[t] > n_gates[t - 1])
        throw Error("trajectory launch: task lengths must not increase along the order");
    if (L.precision == 0)
      occ4 ? launch_steps_t<float, 4>(L, a, n_gates, stream)
           : launch_steps_t<float, 2>(L, a, n_gates, stream);
    else
      occ4 ? launch_steps_t<double, 4>(L, a, n_gates, stream)
           : launch_steps_t<double, 2>(L, a, n_gates, stream);
    return;
  }
  if (L.precision == 0)
    occ4 ? launch_traj_t<float, 4>(L, a, stream) : launch_traj_t<float, 2>(L, a, stream);
  else
    occ4 ? launch_traj_t<double, 4>(L, a, stream) : launch_traj_t<double, 2>(L, a, stream);
}

} // namespace cast_hip
