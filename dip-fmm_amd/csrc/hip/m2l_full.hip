// M2L in the type's own precision on the matrix cores
// (v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64, FMA chains), for plans whose
// class matrices factor through the harmonic subspace (n = (p + 1)^2 rows): the
// M2L of FP64 plans and of FP32 plans in the plain mode, and of small FP32
// batches in the 16-bit modes.
//
// Reference: apply_static_m2l_plan / apply_scaled_m2l_rows_kernel
// (src/static_operators.cpp:16-102, src/cuda_fmm.cu:142-189), regrouped by the
// integer offset o = t - s as in m2l_mfma.hip:
//   Lcc[t] = sum over the offsets o of t's coordinate parity C_o Mc[t - o].
// A wave owns the columns (target box, state) of one parity class, 16 CT of
// them, and all n rows, and walks its share of the parity's 189 offsets; the
// waves of a workgroup share the columns and split the offsets, and their sums
// meet in LDS, so a level of a few boxes still runs hundreds of short chains.
//
// What bounds it: the products, and on small levels the chain of offsets.
//   * Operands go from L2 and L1 to registers, one offset's next 16 depth
//     values loaded during the products of the current ones; nothing is staged
//     in LDS and no barrier is passed before the end.
//   * The class matrices lie in fragment order (matrix_fragments): one 16-byte
//     (FP64: 32-byte) load per lane feeds four products.
//   * The compressed basis puts degree 0 last.  Dipoles have no monopole, so
//     the last depth value is left out, and where n = 16 r + 1 (p = 6 and 8)
//     the last row is summed on the vector ALUs from the fragments at hand, an
//     eighth of what a row tile for it would cost.
//   * Sources and targets in boxes without points are left out where the plan
//     has the bits for it (DevicePlan::source_bits).
//   * A source's Morton index is formed in dilated coordinates: three
//     subtractions under masks; an index outside the grid carries into higher
//     bits, so one compare tells.
//   * block b -> parity b % 8, so each XCD keeps its parity's class matrices in
//     its own L2.
//
// Measured (M2L alone; in brackets the form before it, one workgroup walking
// all 189 offsets through LDS on the vector ALUs): FP32, one state, 37449 boxes,
// p = 6 0.40 ms (1.24), 64 boxes, p = 4 16 us (159); FP64, one state, 4681
// boxes, p = 8 0.35 ms (3.03), p = 4 49 us (1050).
#include "bf16_split.hpp"
#include "common.hpp"

#include <type_traits>

namespace hipfmm {

namespace {

constexpr uint32_t kX = 0x09249249u, kY = kX << 1, kZ = kX << 2;  // Morton bits of x, y, z
constexpr int kOffsets = 189;

template <class S>
struct Mma;
template <>
struct Mma<float> {
  typedef float Acc __attribute__((ext_vector_type(4)));
  __device__ __forceinline__ static Acc mul(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static int row(int q, int r) { return 4 * q + r; }
};
template <>
struct Mma<double> {
  typedef double Acc __attribute__((ext_vector_type(4)));
  __device__ __forceinline__ static Acc mul(double a, double b, Acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static int row(int q, int r) { return 4 * r + q; }
};

// Tiling of n rows and n - 1 depth values.  Depth group s < groups - 1 holds
// depth 16 s + 4 q + j for lane quarter q and product j = 0..3, the last one
// depth 16 s + last * q + j for j < last.
struct Tiling {
  int n;
  constexpr bool extra() const { return n % 16 == 1; }  // the last row on the vector ALUs
  constexpr int row_tiles() const { return extra() ? n / 16 : (n + 15) / 16; }
  constexpr int groups() const { return (n - 1 + 15) / 16; }
  constexpr int last() const { return (n - 1 - 16 * (groups() - 1) + 3) / 4; }
  constexpr int depth(int s, int q, int j) const { return 16 * s + (s + 1 < groups() ? 4 : last()) * q + j; }
  // Scalars of one depth group of one class: the row tiles' fragments
  // [tile][lane][4], then the last row's [quarter][4].
  constexpr int group_size() const { return row_tiles() * 256 + (extra() ? 16 : 0); }
};

struct FullLevels {
  int count;
  int level[kMaxLevels];
  int begin[kMaxLevels + 1];  // first workgroup
};

// W consecutive scalars at any alignment of a scalar.
template <class S, int W>
struct __attribute__((packed, aligned(sizeof(S)))) Run {
  S v[W];
};

// One workgroup: kWavesMax or fewer waves on 16 CT columns.  kRuns: the
// coefficients lie [state][coefficient], so that a column's depth values are
// contiguous ([coefficient][state] otherwise).
template <class S, int N, int CT, bool kRuns, int kWavesMax>
__global__ void __launch_bounds__(64 * kWavesMax) m2l_full_kernel(const DevicePlan d, const FullLevels lv, int K,
                                                                  const S* __restrict__ fragments,
                                                                  const int4* __restrict__ steps,
                                                                  const S* __restrict__ zeros) {
  constexpr Tiling t{N};
  constexpr int RT = t.row_tiles(), NS = t.groups(), ML = t.last(), GS = t.group_size();
  static_assert(t.depth(NS - 1, 3, ML - 1) <= N - 1, "depth values stay within a box");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using M = Mma<S>;
  const int waves = int(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  int li = lv.count - 1;
  while (li > 0 && int(blockIdx.x) < lv.begin[li]) --li;
  const int level = lv.level[li], lb = int(blockIdx.x) - lv.begin[li];
  const int parity = lb & 7;
  const int64_t cols = (int64_t(1) << (3 * (level - 1))) * K;
  const uint32_t boxes = uint32_t(1) << (3 * level);
  const int64_t box_size = int64_t(N) * K;
  const int64_t lvl0 = level_offset(level);
  const S* Mc = static_cast<const S*>(d.M) + lvl0 * box_size;
  // Targets: dilated coordinates, state, and the index limit of a source in
  // the grid (0 for a column past the end: no source passes).
  uint32_t tx[CT], ty[CT], tz[CT], limit[CT];
  int state[CT];
  bool alive = false;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int64_t col = (int64_t(lb >> 3) * CT + c) * 16 + i;
    const uint32_t parent = uint32_t((col < cols ? col : 0) / K), m = parent * 8 + uint32_t(parity);
    state[c] = int(col < cols ? col - int64_t(parent) * K : 0);
    tx[c] = m & kX, ty[c] = m & kY, tz[c] = m & kZ;
    limit[c] = col < cols && (d.target_bits == nullptr || bit_of(d.target_bits, lvl0 + m)) ? boxes : 0u;
    alive |= limit[c] != 0;
  }
  typename M::Acc acc[RT][CT];
  S xs[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    xs[c] = S(0);
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][c] = typename M::Acc{};
  }
  const int o_end = __any(alive) ? (wave + 1) * kOffsets / waves : 0;  // nothing for columns without targets
  const int4* step = steps + parity * kOffsets;
  // The next offset from `o` on with a source for some column: its operands.
  const S* src[CT];
  const S* frag = nullptr;
  auto find = [&](int& o) {
    for (; o < o_end; ++o) {
      const int4 st = step[o];
      bool any = false;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const uint32_t s = ((tx[c] - uint32_t(st.x)) & kX) | ((ty[c] - uint32_t(st.y)) & kY) |
                           ((tz[c] - uint32_t(st.z)) & kZ);
        bool ok = s < limit[c];
        if (d.source_bits != nullptr) ok = ok && bit_of(d.source_bits, lvl0 + s);
        any |= ok;
        src[c] = (ok ? Mc + int64_t(s) * box_size : zeros) + state[c] * (kRuns ? N : 1);
      }
      if (__any(any)) {
        frag = fragments + int64_t(__builtin_amdgcn_readfirstlane(st.w)) * (NS * GS);
        return true;
      }
    }
    return false;
  };
  struct Operands {
    S a[RT][4], x[4], b[CT][4];
  };
  auto load = [&](Operands& f, int s) {
    const S* a = frag + s * GS;
    const int steps_here = s + 1 < NS ? 4 : ML;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const auto v = *reinterpret_cast<const Run<S, 4>*>(__builtin_assume_aligned(a + (r * 64 + lane) * 4, 16));
#pragma unroll
      for (int j = 0; j < 4; ++j) f.a[r][j] = v.v[j];
    }
    if constexpr (t.extra()) {
      const auto v = *reinterpret_cast<const Run<S, 4>*>(__builtin_assume_aligned(a + RT * 256 + q * 4, 16));
#pragma unroll
      for (int j = 0; j < 4; ++j) f.x[j] = v.v[j];
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      if constexpr (kRuns) {
        if (s + 1 < NS) {
          const auto v = *reinterpret_cast<const Run<S, 4>*>(src[c] + 16 * s + 4 * q);
#pragma unroll
          for (int j = 0; j < 4; ++j) f.b[c][j] = v.v[j];
        } else {
          const auto v = *reinterpret_cast<const Run<S, ML>*>(src[c] + 16 * s + ML * q);
#pragma unroll
          for (int j = 0; j < ML; ++j) f.b[c][j] = v.v[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < steps_here) f.b[c][j] = src[c][int64_t(16 * s + steps_here * q + j) * K];
      }
    }
  };
  Operands f;
  int o = wave * kOffsets / waves;
  bool have = find(o);
  if (have) load(f, 0);
  while (have) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      Operands next;
      if (s + 1 < NS) {
        load(next, s + 1);
      } else {
        ++o;
        have = find(o);
        if (have) load(next, 0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= (s + 1 < NS ? 4 : ML)) continue;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[r][c] = M::mul(f.a[r][j], f.b[c][j], acc[r][c]);
        if constexpr (t.extra())
#pragma unroll
          for (int c = 0; c < CT; ++c) xs[c] = fma(f.x[j], f.b[c][j], xs[c]);
      }
      f = next;
    }
  }
  if constexpr (t.extra())
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      xs[c] += __shfl_xor(xs[c], 16);
      xs[c] += __shfl_xor(xs[c], 32);
    }
  // The waves' sums, pairwise: wave w takes wave w + half's.
  constexpr int kPerWave = (RT * 4 + (t.extra() ? 1 : 0)) * CT * 64;
  S* part = reinterpret_cast<S*>(smem_raw);
  for (int half = waves >> 1; half >= 1; half >>= 1) {
    if (wave >= half && wave < 2 * half) {
      S* w = part + (wave - half) * kPerWave + lane;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) w[((c * RT + r) * 4 + e) * 64] = acc[r][c][e];
        if constexpr (t.extra()) w[(CT * RT * 4 + c) * 64] = xs[c];
      }
    }
    __syncthreads();
    if (wave < half) {
      const S* w = part + wave * kPerWave + lane;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][c][e] += w[((c * RT + r) * 4 + e) * 64];
        if constexpr (t.extra()) xs[c] += w[(CT * RT * 4 + c) * 64];
      }
    }
    __syncthreads();
  }
  if (wave != 0) return;
  S* Lc = static_cast<S*>(d.Lc) + lvl0 * box_size;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    if (limit[c] == 0) continue;
    S* out = Lc + int64_t(tx[c] | ty[c] | tz[c]) * box_size + state[c] * (kRuns ? N : 1);
    const int64_t row_step = kRuns ? 1 : K;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * r + M::row(q, e);
        if (row < N) out[row * row_step] = acc[r][c][e];
      }
    if (t.extra() && q == 0) out[(N - 1) * row_step] = xs[c];
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// The same walk in the bf16 mode's arithmetic (x = hi + lo, hi hi + hi lo +
// lo hi on v_mfma_f32_32x32x16_bf16, FP32 accumulation), for batches too small
// for the workgroups of m2l_mfma.hip: class matrices in that kernel's layout
// (T_hi / T_lo, [class][16-deep step][row tile of 32][lane][8]), the sources
// split in registers as they arrive, so no split pass runs.  A wave owns 32 CT
// columns; coefficients lie [state][coefficient].
template <int N, int CT, int kWavesMax>
__global__ void __launch_bounds__(64 * kWavesMax) m2l_bf16_direct_kernel(const DevicePlan d, const FullLevels lv, int K,
                                                                         const int4* __restrict__ steps,
                                                                         const float* __restrict__ zeros) {
  constexpr int MT = (N + 31) / 32, KS = (N + 15) / 16, KD = (N - 1 + 15) / 16;  // row tiles; steps held, multiplied
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int waves = int(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int i = lane & 31, g = lane >> 5;
  int li = lv.count - 1;
  while (li > 0 && int(blockIdx.x) < lv.begin[li]) --li;
  const int level = lv.level[li], lb = int(blockIdx.x) - lv.begin[li];
  const int parity = lb & 7;
  const int64_t cols = (int64_t(1) << (3 * (level - 1))) * K;
  const uint32_t boxes = uint32_t(1) << (3 * level);
  const int64_t box_size = int64_t(N) * K;
  const int64_t lvl0 = level_offset(level);
  const float* Mc = static_cast<const float*>(d.M) + lvl0 * box_size;
  uint32_t tx[CT], ty[CT], tz[CT], limit[CT];
  int state[CT];
  bool alive = false;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int64_t col = (int64_t(lb >> 3) * CT + c) * 32 + i;
    const uint32_t parent = uint32_t((col < cols ? col : 0) / K), m = parent * 8 + uint32_t(parity);
    state[c] = int(col < cols ? col - int64_t(parent) * K : 0);
    tx[c] = m & kX, ty[c] = m & kY, tz[c] = m & kZ;
    limit[c] = col < cols && (d.target_bits == nullptr || bit_of(d.target_bits, lvl0 + m)) ? boxes : 0u;
    alive |= limit[c] != 0;
  }
  f32x16 acc[MT][CT];
#pragma unroll
  for (int r = 0; r < MT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = f32x16{};
  const int o_end = __any(alive) ? (wave + 1) * kOffsets / waves : 0;  // nothing for columns without targets
  const int4* step = steps + parity * kOffsets;
  const float* src[CT];
  const uint4 *hi = nullptr, *lo = nullptr;
  auto find = [&](int& o) {
    for (; o < o_end; ++o) {
      const int4 st = step[o];
      bool any = false;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const uint32_t s = ((tx[c] - uint32_t(st.x)) & kX) | ((ty[c] - uint32_t(st.y)) & kY) |
                           ((tz[c] - uint32_t(st.z)) & kZ);
        bool ok = s < limit[c];
        if (d.source_bits != nullptr) ok = ok && bit_of(d.source_bits, lvl0 + s);
        any |= ok;
        src[c] = (ok ? Mc + int64_t(s) * box_size : zeros) + state[c] * N;
      }
      if (__any(any)) {
        const int64_t at = int64_t(__builtin_amdgcn_readfirstlane(st.w)) * (KS * MT * 64);
        hi = static_cast<const uint4*>(d.T_hi) + at;
        lo = static_cast<const uint4*>(d.T_lo) + at;
        return true;
      }
    }
    return false;
  };
  struct Operands {
    uint4 a[MT][2];
    float b[CT][8];
  };
  auto load = [&](Operands& f, int s) {
#pragma unroll
    for (int r = 0; r < MT; ++r) {
      f.a[r][0] = hi[(s * MT + r) * 64 + lane];
      f.a[r][1] = lo[(s * MT + r) * 64 + lane];
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      if (16 * s + 16 <= N) {
        const auto v = *reinterpret_cast<const Run<float, 8>*>(src[c] + 16 * s + 8 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) f.b[c][e] = v.v[e];
      } else {  // the last step reaches past the box's coefficients
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int at = 16 * s + 8 * g + e;
          const float v = src[c][min(at, N - 1)];
          f.b[c][e] = at < N ? v : 0.0f;
        }
      }
    }
  };
  Operands f;
  int o = wave * kOffsets / waves;
  bool have = find(o);
  if (have) load(f, 0);
  while (have) {
#pragma unroll
    for (int s = 0; s < KD; ++s) {
      Operands next;
      if (s + 1 < KD) {
        load(next, s + 1);
      } else {
        ++o;
        have = find(o);
        if (have) load(next, 0);
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        uint32_t h[4], l[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float x0 = f.b[c][2 * w], x1 = f.b[c][2 * w + 1];
          h[w] = pack_bf16(x0, x1);
          l[w] = pack_bf16(x0 - bf16_low(h[w]), x1 - bf16_high(h[w]));
        }
        const bf16x8 bh = __builtin_bit_cast(bf16x8, uint4{h[0], h[1], h[2], h[3]});
        const bf16x8 bl = __builtin_bit_cast(bf16x8, uint4{l[0], l[1], l[2], l[3]});
#pragma unroll
        for (int r = 0; r < MT; ++r) {
          const bf16x8 ah = __builtin_bit_cast(bf16x8, f.a[r][0]), al = __builtin_bit_cast(bf16x8, f.a[r][1]);
          acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc[r][c], 0, 0, 0);
          acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc[r][c], 0, 0, 0);
          acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc[r][c], 0, 0, 0);
        }
      }
      f = next;
    }
  }
  constexpr int kPerWave = MT * CT * 16 * 64;
  float* part = reinterpret_cast<float*>(smem_raw);
  for (int half = waves >> 1; half >= 1; half >>= 1) {
    if (wave >= half && wave < 2 * half) {
      float* w = part + (wave - half) * kPerWave + lane;
#pragma unroll
      for (int r = 0; r < MT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e) w[((r * CT + c) * 16 + e) * 64] = acc[r][c][e];
    }
    __syncthreads();
    if (wave < half) {
      const float* w = part + wave * kPerWave + lane;
#pragma unroll
      for (int r = 0; r < MT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[r][c][e] += w[((r * CT + c) * 16 + e) * 64];
    }
    __syncthreads();
  }
  if (wave != 0) return;
  float* Lc = static_cast<float*>(d.Lc) + lvl0 * box_size;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    if (limit[c] == 0) continue;
    float* out = Lc + int64_t(tx[c] | ty[c] | tz[c]) * box_size + state[c] * N;
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 32 * r + 8 * (e >> 2) + 4 * g + (e & 3);
        if (row < N) out[row] = acc[r][c][e];
      }
  }
}

// Workgroups of the launch, the last level first (its workgroups fill the
// chip, the smaller levels its tail), `width` columns each.
FullLevels full_levels(const DevicePlan& d, int K, int width) {
  FullLevels lv{};
  lv.count = d.L - 1;
  int begin = 0;
  for (int e = 0; e < lv.count; ++e) {
    const int level = d.L - e;
    const int64_t cols = (int64_t(1) << (3 * (level - 1))) * K;
    lv.level[e] = level;
    lv.begin[e] = begin;
    begin += int(8 * ((cols + width - 1) / width));
  }
  lv.begin[lv.count] = begin;
  return lv;
}

// Launch shape: two column tiles per wave where that gives 256 or more
// workgroups (one per CU), with the offsets split over 4, 2 or 1 waves so that
// the launch has about four waves per SIMD; below, one column tile and the
// most waves whose sums LDS holds.
template <class S, int N>
void launch_full(const DevicePlan& d, int K, hipStream_t s) {
  constexpr Tiling t{N};
  constexpr int many = sizeof(S) == 4 ? 16 : 8;  // waves of a small launch
  FullLevels lv = full_levels(d, K, 32);
  const int groups2 = lv.begin[lv.count];
  const bool wide = groups2 >= 256 && t.row_tiles() <= 5;
  if (!wide) lv = full_levels(d, K, 16);
  const int blocks = lv.begin[lv.count];
  const int waves = wide ? (blocks >= 4096 ? 1 : blocks >= 2048 ? 2 : 4) : blocks >= 2048 ? 2 : blocks >= 1024 ? 4 : many;
  const int ct = wide ? 2 : 1;
  const size_t lds = size_t(waves / 2) * (t.row_tiles() * 4 + (t.extra() ? 1 : 0)) * ct * 64 * sizeof(S);
  const S* fragments = static_cast<const S*>(d.m2l_fragments);
  const S* zeros = static_cast<const S*>(d.m2l_zero_box);
  auto go = [&](auto tiles, auto runs, auto most) {
    m2l_full_kernel<S, N, decltype(tiles)::value, decltype(runs)::value, decltype(most)::value>
        <<<unsigned(blocks), unsigned(64 * waves), lds, s>>>(d, lv, K, fragments, d.m2l_steps, zeros);
  };
  if (wide && d.state_major) go(std::integral_constant<int, 2>{}, std::true_type{}, std::integral_constant<int, 4>{});
  else if (wide) go(std::integral_constant<int, 2>{}, std::false_type{}, std::integral_constant<int, 4>{});
  else if (d.state_major) go(std::integral_constant<int, 1>{}, std::true_type{}, std::integral_constant<int, many>{});
  else go(std::integral_constant<int, 1>{}, std::false_type{}, std::integral_constant<int, many>{});
  HIPFMM_CHECK(hipGetLastError());
}

template <int N>
void launch_bf16_direct(const DevicePlan& d, int K, hipStream_t s) {
  constexpr int MT = (N + 31) / 32;
  FullLevels lv = full_levels(d, K, 64);
  const bool wide = lv.begin[lv.count] >= 512 && MT <= 3;
  if (!wide) lv = full_levels(d, K, 32);
  const int blocks = lv.begin[lv.count];
  const int waves = blocks >= 4096 ? 1 : blocks >= 2048 ? 2 : blocks >= 256 || MT > 2 ? 4 : 8;
  const size_t lds = size_t(waves / 2) * MT * (wide ? 2 : 1) * 16 * 64 * sizeof(float);
  const float* zeros = static_cast<const float*>(d.m2l_zero_box);
  if (wide)
    m2l_bf16_direct_kernel<N, MT <= 3 ? 2 : 1, 4><<<unsigned(blocks), unsigned(64 * waves), lds, s>>>(d, lv, K, d.m2l_steps, zeros);
  else
    m2l_bf16_direct_kernel<N, 1, 8><<<unsigned(blocks), unsigned(64 * waves), lds, s>>>(d, lv, K, d.m2l_steps, zeros);
  HIPFMM_CHECK(hipGetLastError());
}

template <class S>
std::vector<S> fragments_of(int n, const std::vector<double>& C, int classes) {
  const Tiling t{n};
  const size_t per_class = size_t(t.groups()) * t.group_size();
  std::vector<S> out(per_class * std::max(classes, 1), S(0));
  for (int c = 0; c < classes; ++c)
    for (int s = 0; s < t.groups(); ++s) {
      S* g = out.data() + size_t(c) * per_class + size_t(s) * t.group_size();
      const double* T = C.data() + size_t(c) * n * n;  // T[row + n * depth]
      const int steps = s + 1 < t.groups() ? 4 : t.last();
      for (int q = 0; q < 4; ++q)
        for (int j = 0; j < steps; ++j) {
          const int depth = t.depth(s, q, j);
          if (depth >= n - 1) continue;
          for (int r = 0; r < t.row_tiles(); ++r)
            for (int i = 0; i < 16; ++i)
              if (16 * r + i < n) g[(r * 64 + 16 * q + i) * 4 + j] = S(T[16 * r + i + size_t(n) * depth]);
          if (t.extra()) g[t.row_tiles() * 256 + 4 * q + j] = S(T[n - 1 + size_t(n) * depth]);
        }
    }
  return out;
}

}  // namespace

std::vector<float> m2l_fragments_f32(int n, const std::vector<double>& C, int classes) {
  return fragments_of<float>(n, C, classes);
}
std::vector<double> m2l_fragments_f64(int n, const std::vector<double>& C, int classes) {
  return fragments_of<double>(n, C, classes);
}

// (ox, oy, oz) as dilated values whose subtraction under the masks moves a
// target's Morton coordinates to the source's; w the class.
int4 m2l_step(int ox, int oy, int oz, int cls) {
  return int4{int(spread3(uint32_t(ox) & 0x3ffu)), int(spread3(uint32_t(oy) & 0x3ffu) << 1),
              int(spread3(uint32_t(oz) & 0x3ffu) << 2), cls};
}

template <class S>
void launch_m2l_full(const DevicePlan& d, int K, hipStream_t s) {
  if (d.L < 2) return;
  switch (d.n) {
    case 4: launch_full<S, 4>(d, K, s); break;
    case 9: launch_full<S, 9>(d, K, s); break;
    case 16: launch_full<S, 16>(d, K, s); break;
    case 25: launch_full<S, 25>(d, K, s); break;
    case 36: launch_full<S, 36>(d, K, s); break;
    case 49: launch_full<S, 49>(d, K, s); break;
    case 64: launch_full<S, 64>(d, K, s); break;
    case 81: launch_full<S, 81>(d, K, s); break;
    case 100: launch_full<S, 100>(d, K, s); break;
    case 121: launch_full<S, 121>(d, K, s); break;
    default: throw invalid_argument("harmonic M2L of an unsupported expansion order");
  }
}
void launch_m2l_bf16_direct(const DevicePlan& d, int K, hipStream_t s) {
  if (d.L < 2) return;
  if (!d.state_major || d.T_hi == nullptr) throw invalid_argument("the direct bf16 M2L takes state-major coefficients");
  switch (d.n) {
    case 4: launch_bf16_direct<4>(d, K, s); break;
    case 9: launch_bf16_direct<9>(d, K, s); break;
    case 16: launch_bf16_direct<16>(d, K, s); break;
    case 25: launch_bf16_direct<25>(d, K, s); break;
    case 36: launch_bf16_direct<36>(d, K, s); break;
    case 49: launch_bf16_direct<49>(d, K, s); break;
    case 64: launch_bf16_direct<64>(d, K, s); break;
    case 81: launch_bf16_direct<81>(d, K, s); break;
    case 100: launch_bf16_direct<100>(d, K, s); break;
    case 121: launch_bf16_direct<121>(d, K, s); break;
    default: throw invalid_argument("harmonic M2L of an unsupported expansion order");
  }
}

template void launch_m2l_full<float>(const DevicePlan&, int, hipStream_t);
template void launch_m2l_full<double>(const DevicePlan&, int, hipStream_t);

}  // namespace hipfmm
