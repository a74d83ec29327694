// List-1 near field on the vector ALUs: fields, fields with potentials, and
// field gradients, FP32 and FP64, any number of moment states.  It serves
// FP64 plans, FP32 plans below the state counts where the matrix cores pay,
// and near-field variant 1.
//
// Reference: the list-1 pair set of src/uniform_fmm.cpp:678-710 (every source
// of the clipped 3x3x3 leaf neighbourhood of the target's leaf, the identity
// pair skipped, coincident non-identity pairs giving NaN:
// src/static_operators.cpp:435-446), the point-dipole tensor
// D = (3 r r^T/|r|^5 - I/|r|^3)/(4 pi) of src/cuboid.cpp:293-307 and the
// potential (m.r)/(4 pi |r|^3) of src/static_operators.cpp:455-463.
//
// What bounds it: the pair arithmetic, 23 vector instructions per pair and 10
// per state up to three states, 26 and 9 at more (one more per state with the
// potential).  So the
// lanes of a wave are sources and its targets are wave-uniform: a lane keeps
// one source and its moments in registers for T targets of one leaf, whose
// coordinates sit in scalar registers, and nothing is staged in LDS.  A batch
// is eight 8-source blocks of the neighbourhood's block list (nbr_blk), so a
// leaf pads to 8 sources, and a leaf's last targets cost only themselves
// (the targets past its end are skipped by a uniform branch).  The lanes'
// sums meet in one butterfly per T targets.
//
// A wave's targets come from the list of 16-target tiles, so a leaf of many
// targets is many waves: with a workgroup per leaf clustered points waited for
// the fullest leaves (100,000 points in blobs, depth 5, K = 8: 1.16 ms, now
// .36) and small trees left the chip idle (20,000 points, 512 leaves, K = 1
// .06, now .034).
//
// Measured (near field alone, ms; in brackets the form before it, a workgroup
// of 32 target slots per pass that staged each neighbour leaf's sources in LDS
// and formed a pair's geometry once per 1, 4 or 8 states): 2^20 points, 32 per
// leaf, FP32: K = 1 .88 (1.77), 2 1.08 (2.70), 4 1.87 (4.61), 8 3.06 (8.01);
// fields and potentials K = 4 2.08 (4.72); gradients K = 1 1.25 (2.05).
// 512 per leaf, 2^18 points: K = 8 6.5.  FP64, 2^18 points, 64 per leaf:
// K = 1 .60 (1.43).  Whole evaluates of 2^20 points, p = 4, K = 8 with the
// tensor's 3 and the potential's u.m once per pair 4.04, with potentials 4.79
// (2% and 10% more with both once per state).  Taking the 3 as sqrt(3) in both
// factors would save two instructions per pair (3.99 and 4.72) for more error:
// 8 sources, 50,000 targets, K = 8, against FP64, median relative error and mean
// of the signed errors 1.7e-7 and -0.3e-7; with 1 / (4 pi) rounded into each pair
// 1.8e-7 and -0.7e-7, with sqrt(3) besides 2.0e-7 and -1.0e-7.
#include "common.hpp"

namespace hipfmm {

namespace {

constexpr int kWaves = 4;  // waves per workgroup, each with T targets of a 16-target tile

enum NearOutput { kField = 0, kFieldAndPotential = 1, kGradient = 2 };

// Rows of the output per target and state.
constexpr int near_rows(int what) { return what == kGradient ? 6 : what == kFieldAndPotential ? 4 : 3; }

// Targets per wave: T x rows x states accumulators per lane are held to 96
// FP32 (48 FP64) values, which keeps two or more waves per SIMD.  Fewer
// targets per wave cost more than the occupancy gives (K = 8, 256 points per
// leaf: T = 4 19.0 ms, T = 2 26.8 ms; K = 7: 4.6 against 6.3 ms).
template <class S>
constexpr int near_targets(int states, int what) {
  const int most = sizeof(S) == 4 ? 96 : 48;
  int t = 8;
  while (t > 2 && t * near_rows(what) * states > most) t /= 2;
  return t;
}

__device__ __forceinline__ float near_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }  // 1 ulp
// The hardware's 24 bits y and one third-order step from e = 1 - x y^2:
// x^-1/2 = y (1 - e)^-1/2 = y (1 + e/2 + 3 e^2/8 + O(e^3)), within 0.75 ulp; the
// library's 1 / sqrt(x) is within 1 ulp in three times the instructions.
// x = 0 gives NaN.
__device__ __forceinline__ double near_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// A sum of pairs times 4 / pi, to within its rounding.
__device__ __forceinline__ float near_scale(float x) {
  return fmaf(x, 1.2732395447351626862f, x * float(1.2732395447351626862 - double(1.2732395447351626862f)));
}
__device__ __forceinline__ double near_scale(double x) { return x * 1.2732395447351626862; }

// A wave-uniform value moved to scalar registers.
__device__ __forceinline__ float uniform(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ double uniform(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(u))));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(u >> 32))));
  return __builtin_bit_cast(double, uint64_t(lo) | (uint64_t(hi) << 32));
}

// A point: FP32 plans hold hi + lo float parts of the FP64 coordinates, so
// r = (t_hi - s_hi) + (t_lo - s_lo) keeps FP32 relative accuracy for pairs
// far closer than a leaf width.
template <class S>
struct Point;
template <>
struct Point<float> {
  float h[3], l[3];
  __device__ __forceinline__ static Point load(const void* pos, int count, int i) {
    const float4* p = static_cast<const float4*>(pos);
    const float4 a = p[i], b = p[int64_t(count) + i];
    return {{a.x, a.y, a.z}, {b.x, b.y, b.z}};
  }
  __device__ __forceinline__ static float far() { return 1e18f; }
  __device__ __forceinline__ float minus(const Point& s, int c) const { return (h[c] - s.h[c]) + (l[c] - s.l[c]); }
};
template <>
struct Point<double> {
  double h[3];
  __device__ __forceinline__ static Point load(const void* pos, int, int i) {
    const double4 a = static_cast<const double4*>(pos)[i];
    return {{a.x, a.y, a.z}};
  }
  __device__ __forceinline__ static double far() { return 1e150; }
  __device__ __forceinline__ double minus(const Point& s, int c) const { return h[c] - s.h[c]; }
};

// v[0 .. N) summed over the lanes of the wave, lane bits kBit, kBit / 2, .. 1.
// Where the count is even a step halves it: each lane keeps one half's sums
// and hands the other half to its partner.  Afterwards v[0 .. totals_left(N))
// of a lane are the totals of entries first .. (first is per lane).
constexpr int totals_left(int n, int bit = 32) {
  return bit == 0 ? n : totals_left(n % 2 == 0 ? n / 2 : n, bit / 2);
}
template <int N, int kBit, int V, class S>
__device__ __forceinline__ void wave_totals(S (&v)[V], int lane, int& first) {
  if constexpr (kBit >= 1) {
    if constexpr (N % 2 == 0) {
      const bool upper = (lane & kBit) != 0;
#pragma unroll
      for (int i = 0; i < N / 2; ++i) {
        const S send = upper ? v[i] : v[i + N / 2];
        const S keep = upper ? v[i + N / 2] : v[i];
        v[i] = keep + __shfl_xor(send, kBit);
      }
      first += upper ? N / 2 : 0;
      wave_totals<N / 2, kBit / 2>(v, lane, first);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] += __shfl_xor(v[i], kBit);
      wave_totals<N, kBit / 2>(v, lane, first);
    }
  }
}

// KS consecutive scalars of one row, any alignment of a scalar: one or two
// wide loads.
template <class S, int KS>
struct __attribute__((packed, aligned(sizeof(S)))) States {
  S v[KS];
};

// A wave has T targets of one leaf and KS <= K states (blockIdx.y; the last
// group of states ends at K and may repeat some of the one before, which
// stores them).
template <class S, int KS, int kWhat>
__global__ void __launch_bounds__(64 * kWaves) near_lanes_kernel(const DevicePlan d, int K) {
  constexpr int T = near_targets<S>(KS, kWhat), C = near_rows(kWhat), V = T * C * KS;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  // The tile list's 16 targets in groups of T: a leaf of many targets is as
  // many waves, whatever the other leaves hold.
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kWaves + wave;
  if (item >= d.p2p_tile16_count * (16 / T)) return;
  const int2 tile = d.p2p_tiles16[item / (16 / T)];
  const int leaf = tile.x;
  const int2 range = d.leaf_tgt[leaf];
  const int t0 = range.x + tile.y + item % (16 / T) * T, cnt = min(T, range.y - t0);
  if (cnt <= 0) return;
  const int k_first = int(blockIdx.y) * KS, k0 = min(k_first, K - KS);
  const int q0 = d.nbr_blk_start[leaf], q1 = d.nbr_blk_start[leaf + 1];
  const S* sm = static_cast<const S*>(d.sm);
  const int group = lane >> 3, e = lane & 7;  // block of the batch, source of the block
  Point<S> tp[T];
  int self[T];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int t = i < cnt ? t0 + i : t0;
    tp[i] = Point<S>::load(d.tgt_pos, d.nt, t);
    self[i] = __builtin_amdgcn_readfirstlane(d.self[t]);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      tp[i].h[c] = uniform(tp[i].h[c]);
      if constexpr (sizeof(S) == 4) tp[i].l[c] = uniform(tp[i].l[c]);
    }
  }
  S acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = S(0);
  int2 blk = int2{0, 0};  // first source and count of this lane's block
  auto block_of = [&](int q) {
    return q + group < q1 ? d.blk8_src[d.nbr_blk[q + group]] : int2{0, 0};
  };
  if (q0 < q1) blk = block_of(q0);
  for (int q = q0; q < q1; q += 8) {
    // A lane without a source takes one out of reach with no moment: its
    // |r|^-1 is tiny and every term of it zero.
    const bool have = e < blk.y;
    const int s = have ? blk.x + e : -2;
    Point<S> sp;
    S m[3][KS];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      sp.h[c] = Point<S>::far();
      if constexpr (sizeof(S) == 4) sp.l[c] = S(0);
#pragma unroll
      for (int k = 0; k < KS; ++k) m[c][k] = S(0);
    }
    if (have) {
      sp = Point<S>::load(d.src_pos, d.ns, s);
      const S* ms = sm + int64_t(s) * 3 * K + k0;
      if (KS == K) {  // one contiguous row
        const auto row = *reinterpret_cast<const States<S, 3 * KS>*>(ms);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int k = 0; k < KS; ++k) m[c][k] = row.v[c * KS + k];
      } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const auto row = *reinterpret_cast<const States<S, KS>*>(ms + c * K);
#pragma unroll
          for (int k = 0; k < KS; ++k) m[c][k] = row.v[k];
        }
      }
    }
    if (q + 8 < q1) blk = block_of(q + 8);
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if (i >= cnt || s == self[i]) continue;
      const S rx = tp[i].minus(sp, 0), ry = tp[i].minus(sp, 1), rz = tp[i].minus(sp, 2);
      const S r2 = rx * rx + ry * ry + rz * rz;
      const S rinv = near_rsqrt(r2);
      S* a = acc + i * C * KS;
      if constexpr (kWhat == kGradient) {
        // dH_c/dx_j, 3/(4 pi |r|^4) (delta_cj w + u_c m_j + m_c u_j - 5 u_c u_j w), w = u.m.
        const S ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
        const S g = S(0.23873241463784300365332564505877154) * rinv * rinv * rinv * rinv;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const S mx = m[0][k], my = m[1][k], mz = m[2][k];
          const S w = ux * mx + uy * my + uz * mz;
          const S w5 = S(5) * w;
          a[0 * KS + k] += g * (w + S(2) * ux * mx - w5 * ux * ux);
          a[1 * KS + k] += g * (ux * my + mx * uy - w5 * ux * uy);
          a[2 * KS + k] += g * (ux * mz + mx * uz - w5 * ux * uz);
          a[3 * KS + k] += g * (w + S(2) * uy * my - w5 * uy * uy);
          a[4 * KS + k] += g * (uy * mz + my * uz - w5 * uy * uz);
          a[5 * KS + k] += g * (w + S(2) * uz * mz - w5 * uz * uz);
        }
      } else {
        // f (3 (u.m) u - m) with f = |r|^-3 / (4 pi): no |r|^-5, which overflows
        // for close pairs in FP32.  The 3 is multiplied exactly, once per pair
        // (three instructions; up to three states, once with each u.m); as
        // sqrt(3) in both factors it would be 3 (1 - 3.6e-8) in FP32, an error of
        // one sign in every pair.  The potential f r.m is |r|^-2 / (4 pi) u.m.
        // Likewise 1 / (4 pi), which is 4e-8 short in FP32: a pair carries 1 / 16
        // of it, the sums 4 / pi (near_scale).
        constexpr bool kWithState = KS <= 3;
        const S ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
        const S fp = rinv * rinv * S(0.0625), f = fp * rinv;
        const S tx = kWithState ? ux : S(3) * ux, ty = kWithState ? uy : S(3) * uy, tz = kWithState ? uz : S(3) * uz;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const S mx = m[0][k], my = m[1][k], mz = m[2][k];
          const S w = ux * mx + uy * my + uz * mz, v = kWithState ? S(3) * w : w;
          a[0 * KS + k] += f * (v * tx - mx);
          a[1 * KS + k] += f * (v * ty - my);
          a[2 * KS + k] += f * (v * tz - mz);
          if constexpr (kWhat == kFieldAndPotential) a[3 * KS + k] += fp * w;
        }
      }
    }
  }
  int first = 0;
  wave_totals<V, 32>(acc, lane, first);
#pragma unroll
  for (int v = 0; v < totals_left(V); ++v) {
    const int at = first + v, i = at / (C * KS), c = at / KS % C, k = k0 + at % KS;
    if (i >= cnt || k < k_first) continue;
    const int64_t t = t0 + i;
    if constexpr (kWhat == kGradient)
      static_cast<S*>(d.Gn)[(t * 6 + c) * K + k] = acc[v];
    else if (c < 3)
      static_cast<S*>(d.Hn)[(t * 3 + c) * K + k] = near_scale(acc[v]);
    else
      static_cast<S*>(d.Pn)[t * K + k] = near_scale(acc[v]);
  }
}

template <class S, int kWhat>
void launch_near(const DevicePlan& d, int K, hipStream_t s) {
  // States per workgroup: K cut into as few equal parts as the registers
  // allow (8 FP32 or 4 FP64 states; half of that for gradients).
  constexpr int most = (sizeof(S) == 4 ? 8 : 4) / (kWhat == kGradient ? 2 : 1);
  const int parts = (K + most - 1) / most, ks = (K + parts - 1) / parts;
  auto go = [&](auto count) {
    constexpr int KS = decltype(count)::value;
    if constexpr (KS <= most) {
      const int64_t items = int64_t(d.p2p_tile16_count) * (16 / near_targets<S>(KS, kWhat));
      const dim3 grid(unsigned((items + kWaves - 1) / kWaves), unsigned(parts));
      if (items > 0) near_lanes_kernel<S, KS, kWhat><<<grid, 64 * kWaves, 0, s>>>(d, K);
    }
  };
  switch (ks) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{}); break;
  }
  HIPFMM_CHECK(hipGetLastError());
}

}  // namespace

template <class S>
void launch_p2p_lanes(const DevicePlan& d, int K, bool potential, hipStream_t s) {
  if (potential)
    launch_near<S, kFieldAndPotential>(d, K, s);
  else
    launch_near<S, kField>(d, K, s);
}
template <class S>
void launch_p2p_grad_lanes(const DevicePlan& d, int K, hipStream_t s) {
  launch_near<S, kGradient>(d, K, s);
}
template void launch_p2p_lanes<float>(const DevicePlan&, int, bool, hipStream_t);
template void launch_p2p_lanes<double>(const DevicePlan&, int, bool, hipStream_t);
template void launch_p2p_grad_lanes<float>(const DevicePlan&, int, hipStream_t);
template void launch_p2p_grad_lanes<double>(const DevicePlan&, int, hipStream_t);

}  // namespace hipfmm
