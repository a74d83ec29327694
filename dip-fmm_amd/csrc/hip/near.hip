// List-1 P2P (near field) on the matrix cores, and the FP64 direct sum; the
// vector-ALU near field is near_lanes.hip.
//
// Reference: the list-1 pair set of src/uniform_fmm.cpp:678-710 (every
// source of the clipped 3x3x3 leaf neighbourhood of the target's leaf, the
// identity pair skipped, coincident non-identity pairs giving NaN:
// src/static_operators.cpp:435-446) with the point-dipole tensor
// D = (3 r r^T/|r|^5 - I/|r|^3)/(4 pi) of src/cuboid.cpp:293-307.  The
// reference stores one tensor per pair (37 GB at 2^20 points); here the
// tensor is evaluated on the fly and reused for all K moment states.
//
// FP32 plans carry positions as hi+lo float pairs of the FP64 operator-frame
// coordinates, so r = (t_hi - s_hi) + (t_lo - s_lo) keeps FP32 relative
// accuracy even for pairs far closer than a leaf width.
#include "common.hpp"
#include "bf16_split.hpp"

#include <type_traits>

namespace hipfmm {

namespace {

constexpr int kThreads = 256;

template <class S>
struct PairPos;

template <>
struct PairPos<float> {
  float4 hi, lo;
  __device__ static PairPos load(const void* pos, int count, int i) {
    const float4* p = static_cast<const float4*>(pos);
    return {p[i], p[count + i]};
  }
  __device__ inline void diff(const PairPos& s, float& x, float& y, float& z) const {
    x = (hi.x - s.hi.x) + (lo.x - s.lo.x);
    y = (hi.y - s.hi.y) + (lo.y - s.lo.y);
    z = (hi.z - s.hi.z) + (lo.z - s.lo.z);
  }
};

__device__ inline float inv_sqrt(float x) { return __frsqrt_rn(x); }

// FP64 direct field, one thread per target, sources staged through LDS.
// validation.cpp:71-111 / operators.cpp:178-220; model kernel
// src/cuda_fmm.cu:518-569.
__global__ void __launch_bounds__(kThreads) direct_kernel(const double* __restrict__ tgt, int nt,
                                                          const double* __restrict__ src, int ns,
                                                          const double* __restrict__ mom, const int* __restrict__ self,
                                                          double* __restrict__ out) {
  __shared__ double s_pos[kThreads * 3];
  __shared__ double s_mom[kThreads * 3];
  const int t = blockIdx.x * kThreads + threadIdx.x;
  const bool active = t < nt;
  const double tx = active ? tgt[3 * t] : 0.0, ty = active ? tgt[3 * t + 1] : 0.0, tz = active ? tgt[3 * t + 2] : 0.0;
  const int me = active && self ? self[t] : -1;
  const double c = 0.079577471545947667884441881686257181;
  double hx = 0.0, hy = 0.0, hz = 0.0;
  for (int j0 = 0; j0 < ns; j0 += kThreads) {
    const int cnt = min(kThreads, ns - j0);
    __syncthreads();
    for (int w = threadIdx.x; w < 3 * cnt; w += kThreads) {
      s_pos[w] = src[3 * j0 + w];
      s_mom[w] = mom[3 * j0 + w];
    }
    __syncthreads();
    if (!active) continue;
    for (int j = 0; j < cnt; ++j) {
      if (j0 + j == me) continue;
      const double rx = tx - s_pos[3 * j], ry = ty - s_pos[3 * j + 1], rz = tz - s_pos[3 * j + 2];
      const double r2 = rx * rx + ry * ry + rz * rz;
      const double rinv = 1.0 / sqrt(r2);
      const double rinv3 = rinv * rinv * rinv;
      const double rinv5 = rinv3 * rinv * rinv;
      const double mx = s_mom[3 * j], my = s_mom[3 * j + 1], mz = s_mom[3 * j + 2];
      const double mdr = mx * rx + my * ry + mz * rz;
      hx += (rx * (3.0 * mdr * rinv5) - mx * rinv3) * c;
      hy += (ry * (3.0 * mdr * rinv5) - my * rinv3) * c;
      hz += (rz * (3.0 * mdr * rinv5) - mz * rinv3) * c;
    }
  }
  if (active) {
    out[3 * t] = hx;
    out[3 * t + 1] = hy;
    out[3 * t + 2] = hz;
  }
}

}  // namespace

typedef float f32x16 __attribute__((ext_vector_type(16)));

// List-1 P2P on the matrix cores (v_mfma_f32_32x32x2_f32, FP32 products and
// accumulation), for FP32 plans with K a multiple of 32.  For 32 moment
// states the near field of a leaf is one GEMM:
//   H[(t,c)][k] = sum_{(s,c')} D_{cc'}(t,s) m[s][c'][k],
// rows (target, component) packed 3 per target (row = 3*t_local + c), depth
// (source, component), columns k.  With the potential (kRows = 4) a fourth
// row per target carries phi = sum_{c'} f r_{c'} m[s][c'][k].  One wave owns
// a 32-row tile: each lane
// forms the pair tensor entries D_{c,0..2}(t,s) of its row's target and one
// of the two sources of a step (A operand, lane i: row i%32, depth i/32) and
// loads m[s][c'][k] (B operand, lane i: column i%32, depth i/32); the
// identity pair and padding rows/sources contribute zero, coincident pairs
// NaN as in the vector path.  Waves are independent: no LDS, no barriers.
constexpr int kP2PWaves = 4;

template <int kRows>
__global__ void __launch_bounds__(64 * kP2PWaves) p2p_mfma_kernel(const DevicePlan d, const int2* __restrict__ tiles,
                                                                   int tile_count, int K) {
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kP2PWaves + wave;
  if (item >= tile_count) return;
  const int2 tile = tiles[item];
  const int leaf = tile.x;
  const int2 trange = d.leaf_tgt[leaf];
  const int rows = kRows * (trange.y - trange.x);
  const int col = lane & 31, g = lane >> 5;
  const int row = tile.y + col;  // A-operand row of this lane
  const bool row_ok = row < rows;
  const int t = trange.x + (row_ok ? row / kRows : 0);
  const int c = row_ok ? row % kRows : 0;
  const bool pot = kRows == 4 && c == 3;  // potential row
  const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
  const int self = row_ok ? d.self[t] : -2;
  const int k = int(blockIdx.y) * 32 + col;  // B / C column of this lane
  const float c4pi = 0.079577471545947667884441881686257181f;
  const float* sm = static_cast<const float*>(d.sm);
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  const int nb = 1 << d.L;
  int lx, ly, lz;
  demorton3(uint32_t(leaf), d.L, lx, ly, lz);
  for (int dz = -1; dz <= 1; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        const int x = lx + dx, y = ly + dy, z = lz + dz;
        if (x < 0 || y < 0 || z < 0 || x >= nb || y >= nb || z >= nb) continue;
        const int2 sr = d.leaf_src[morton3(uint32_t(x), uint32_t(y), uint32_t(z), d.L)];
        // Blocked summation: every block of up to 32 sources accumulates into
        // a fresh chain, added to the total once (fewer additions into one
        // large sum).
        for (int jb = sr.x; jb < sr.y; jb += 32) {
        const int je = min(sr.y, jb + 32);
        f32x16 part;
#pragma unroll
        for (int r = 0; r < 16; ++r) part[r] = 0.0f;
#pragma unroll 4
        for (int j0 = jb; j0 < je; j0 += 2) {
          const int s = j0 + g;
          const bool src_ok = s < je;
          const int sl = src_ok ? s : sr.x;
          float rx, ry, rz;
          tp.diff(PairPos<float>::load(d.src_pos, d.ns, sl), rx, ry, rz);
          const float r2 = rx * rx + ry * ry + rz * rz;
          const float rinv = inv_sqrt(r2);
          const float f = rinv * rinv * rinv * c4pi;
          const float ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
          const float uc = c == 0 ? ux : (c == 1 ? uy : uz);
          const float f3uc = 3.0f * f * uc;
          const bool use = row_ok & src_ok & (s != self);
          float a0 = f3uc * ux - (c == 0 ? f : 0.0f);
          float a1 = f3uc * uy - (c == 1 ? f : 0.0f);
          float a2 = f3uc * uz - (c == 2 ? f : 0.0f);
          if constexpr (kRows == 4) {
            a0 = pot ? f * rx : a0;
            a1 = pot ? f * ry : a1;
            a2 = pot ? f * rz : a2;
          }
          a0 = use ? a0 : 0.0f;
          a1 = use ? a1 : 0.0f;
          a2 = use ? a2 : 0.0f;
          const float* ms = sm + int64_t(sl) * 3 * K + k;
          const float b0 = src_ok ? ms[0] : 0.0f;
          const float b1 = src_ok ? ms[K] : 0.0f;
          const float b2 = src_ok ? ms[2 * K] : 0.0f;
          part = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, part, 0, 0, 0);
          part = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, part, 0, 0, 0);
          part = __builtin_amdgcn_mfma_f32_32x32x2f32(a2, b2, part, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += part[r];
        }
      }
  // acc[r]: row 8*(r/4) + 4*g + r%4 of the tile, column col.
  float* Hn = static_cast<float*>(d.Hn);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int orow = tile.y + 8 * (r >> 2) + 4 * g + (r & 3);
    if (orow >= rows) continue;
    if constexpr (kRows == 3) {
      Hn[(int64_t(trange.x) * 3 + orow) * K + k] = acc[r];
    } else {
      const int64_t ot = trange.x + orow / 4;
      const int oc = orow % 4;
      if (oc < 3)
        Hn[(ot * 3 + oc) * K + k] = acc[r];
      else
        static_cast<float*>(d.Pn)[ot * K + k] = acc[r];
    }
  }
}

// List-1 P2P on the matrix cores with targets as rows
// (v_mfma_f32_16x16x4_f32), for FP32 plans with K a multiple of 32.  One
// wave owns 16 targets of one leaf and 32 states; the depth of a step is 4
// sources.  Lane l forms the pair (target l%16, source l/16) once -- r, |r|,
// the 6 entries of the symmetric D = f (3 u u^T - I) and, for the potential,
// f r -- and the products run per output component c as separate 16 x 16
// accumulator tiles over 2 column halves:
//   H_c[t][k] += sum_{c'} D_{c c'}(t, s) m[s][c'][k],
// 9 products per 4 sources and 16 states (12 with the potential row).  Lane
// layout (CDNA3/4 16x16x4 f32): A[i][k] in lane i + 16k, B[k][j] in lane
// j + 16k, D[i][j] in lane j + 16 floor(i/4), register i % 4.  Identity pair
// and padding contribute zero; coincident pairs give NaN (r = 0).  Blocked
// summation per 32 sources as in the 32 x 32 kernel.  |r|^-1 is the hardware
// reciprocal square root (1 ulp).
// One step of the targets-as-rows kernel for this lane's pair (row target,
// source s), in two stages so that several steps' loads are in flight
// before their products: the raw loads (source position, moments m[s][c'][k]
// of both 16-state halves), then the operands -- the 6 distinct entries of
// D (d00 d01 d02 d11 d12 d22) and the potential row f r.  Loads address the
// neighbour leaf's sources from wave-uniform bases with a 32-bit lane
// offset; a slot past the leaf's end reads its first source.  Padding slots
// and the identity pair get |r|^-1 = 0, so their D and f r entries are 0 and
// the moments they meet need no masking (a finite moment times 0).
struct P2PSources {
  const float4* hi;  // hi and lo blocks of the leaf's first source position
  const float4* lo;
  const float* m;    // m[first][0][kc0]
};

struct P2PRaw {
  PairPos<float> sp;
  float b[3][2];
  int s;
};

struct P2POperands {
  float d[6];
  float p[3];
};

__device__ __forceinline__ P2PRaw p2p_load(const P2PSources& src, int s, int first, int end, int K, int col) {
  P2PRaw r;
  const uint32_t j = s < end ? uint32_t(s - first) : 0u;
  r.sp.hi = src.hi[j];
  r.sp.lo = src.lo[j];
  const uint32_t off = j * uint32_t(3 * K) + uint32_t(col);
#pragma unroll
  for (int cp = 0; cp < 3; ++cp)
#pragma unroll
    for (int h = 0; h < 2; ++h) r.b[cp][h] = src.m[off + uint32_t(cp * K + 16 * h)];
  r.s = s;
  return r;
}

template <int kComps>
__device__ __forceinline__ P2POperands p2p_finish(const P2PRaw& r, const PairPos<float>& tp, bool row_ok, int self,
                                                  int end) {
  P2POperands o;
  float rx, ry, rz;
  tp.diff(r.sp, rx, ry, rz);
  const float r2 = rx * rx + ry * ry + rz * rz;
  const bool use = row_ok & (r.s < end) & (r.s != self);
  // v_rsq_f32 (1 ulp); a coincident pair (r = 0) that is used gives inf,
  // hence NaN entries below.
  const float rinv = use ? __builtin_amdgcn_rsqf(r2) : 0.0f;
  const float f = rinv * rinv * rinv * 0.079577471545947667884441881686257181f;
  const float ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
  const float f3 = 3.0f * f;
  o.d[0] = f3 * ux * ux - f;
  o.d[1] = f3 * ux * uy;
  o.d[2] = f3 * ux * uz;
  o.d[3] = f3 * uy * uy - f;
  o.d[4] = f3 * uy * uz;
  o.d[5] = f3 * uz * uz - f;
  if constexpr (kComps == 4) {
    o.p[0] = f * rx;
    o.p[1] = f * ry;
    o.p[2] = f * rz;
  } else {
    o.p[0] = o.p[1] = o.p[2] = 0.0f;
  }
  return o;
}

// kU steps of 4 sources from j00: all loads, then geometry and products.
template <int kComps, int kU>
__device__ __forceinline__ void p2p_steps(const P2PSources& src, int j00, int q, int end, int first, int K, int col,
                                          const PairPos<float>& tp, bool row_ok, int self,
                                          f32x4 (&part)[kComps][2]) {
  P2PRaw raw[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) raw[u] = p2p_load(src, j00 + 4 * u + q, first, end, K, col);
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const P2POperands cur = p2p_finish<kComps>(raw[u], tp, row_ok, self, end);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      part[0][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[0], raw[u].b[0][h], part[0][h], 0, 0, 0);
      part[1][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[1], raw[u].b[0][h], part[1][h], 0, 0, 0);
      part[2][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[2], raw[u].b[0][h], part[2][h], 0, 0, 0);
      part[0][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[1], raw[u].b[1][h], part[0][h], 0, 0, 0);
      part[1][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[3], raw[u].b[1][h], part[1][h], 0, 0, 0);
      part[2][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[4], raw[u].b[1][h], part[2][h], 0, 0, 0);
      part[0][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[2], raw[u].b[2][h], part[0][h], 0, 0, 0);
      part[1][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[4], raw[u].b[2][h], part[1][h], 0, 0, 0);
      part[2][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.d[5], raw[u].b[2][h], part[2][h], 0, 0, 0);
      if constexpr (kComps == 4) {
        part[3][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.p[0], raw[u].b[0][h], part[3][h], 0, 0, 0);
        part[3][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.p[1], raw[u].b[1][h], part[3][h], 0, 0, 0);
        part[3][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.p[2], raw[u].b[2][h], part[3][h], 0, 0, 0);
      }
    }
  }
}

template <int kComps>
__global__ void __launch_bounds__(64 * kP2PWaves) p2p_mfma16_kernel(const DevicePlan d, const int2* __restrict__ tiles,
                                                                     int tile_count, int K) {
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kP2PWaves + wave;
  if (item >= tile_count) return;
  const int2 tile = tiles[item];
  const int leaf = tile.x;
  const int2 trange = d.leaf_tgt[leaf];
  const int col = lane & 15, q = lane >> 4;  // A row / B and D column; depth slot
  const bool row_ok = trange.x + tile.y + col < trange.y;
  const int t = row_ok ? trange.x + tile.y + col : trange.x;
  const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
  const int self = row_ok ? d.self[t] : -2;
  const int kc0 = int(blockIdx.y) * 32;
  const float* sm = static_cast<const float*>(d.sm);
  f32x4 acc[kComps][2];
#pragma unroll
  for (int c = 0; c < kComps; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[c][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int nb = 1 << d.L;
  int lx, ly, lz;
  demorton3(uint32_t(leaf), d.L, lx, ly, lz);
  for (int dz = -1; dz <= 1; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        const int x = lx + dx, y = ly + dy, z = lz + dz;
        if (x < 0 || y < 0 || z < 0 || x >= nb || y >= nb || z >= nb) continue;
        const int2 sr = d.leaf_src[morton3(uint32_t(x), uint32_t(y), uint32_t(z), d.L)];
        const P2PSources src{static_cast<const float4*>(d.src_pos) + sr.x,
                             static_cast<const float4*>(d.src_pos) + d.ns + sr.x, sm + int64_t(sr.x) * 3 * K + kc0};
        for (int jb = sr.x; jb < sr.y; jb += 32) {
          const int je = min(sr.y, jb + 32);
          f32x4 part[kComps][2];
#pragma unroll
          for (int c = 0; c < kComps; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) part[c][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          // Two steps (8 sources) per iteration, both steps' loads issued
          // before either's pair geometry and products; a block's last 1-4
          // sources take one step.
          for (int j00 = jb; j00 < je; j00 += 8) {
            if (je - j00 > 4)
              p2p_steps<kComps, 2>(src, j00, q, je, sr.x, K, col, tp, row_ok, self, part);
            else
              p2p_steps<kComps, 1>(src, j00, q, je, sr.x, K, col, tp, row_ok, self, part);
          }
#pragma unroll
          for (int c = 0; c < kComps; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[c][h] += part[c][h];
        }
      }
  // acc[c][h][i]: target tile.y + 4q + i, state kc0 + 16h + col.
  float* Hn = static_cast<float*>(d.Hn);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t ot = int64_t(trange.x) + tile.y + 4 * q + i;
    if (ot >= trange.y) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = kc0 + 16 * h + col;
#pragma unroll
      for (int c = 0; c < 3; ++c) Hn[(ot * 3 + c) * K + k] = acc[c][h][i];
      if constexpr (kComps == 4) static_cast<float*>(d.Pn)[ot * K + k] = acc[3][h][i];
    }
  }
}

// The sorted moments as B operands of p2p_bf16_kernel: per block of 8
// sources of one leaf and tile of 32 states,
// smb[block][state tile][c'][piece][32][8] (pieces hi, mid, lo of
// m[s][c'][k]), zero past the leaf's last source and past the last state; a
// wave's 18 operand loads of one block then sit at fixed offsets from one
// address.  Thread = (block, state of the KP = 32-padded tiles); reads are
// coalesced over the states, writes are 16-byte rows.
// The low pieces of a value x reach down to 2^-23 |x|, and below 2^-126 they
// lose bits.  So in batches that are no multiple of 32, whose sums are repaired
// where they are not finite (p2p_repair), the moments of a block and state
// that are all below 2^-100 (not all zero) enter as NaN: the sums they take part
// in are formed again in FP32, one pair at a time.  A block with a larger
// moment loses at most 2^-26 of it.
constexpr float kSmallestSplitMoment = 0x1p-100f;

__global__ void __launch_bounds__(256) split_moments_kernel(const DevicePlan d, int K, int KP) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(d.blk8_count) * KP) return;
  const int b = int(i / KP), k = int(i % KP);
  const int2 bs = d.blk8_src[b];
  const float* sm = static_cast<const float*>(d.sm);
  uint4* out = static_cast<uint4*>(d.smb) + ((int64_t(b) * (KP / 32) + k / 32) * 9) * 32 + k % 32;
  float x[3][8], most = 0.0f;
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[c][e] = e < bs.y && k < K ? sm[(int64_t(bs.x + e) * 3 + c) * K + k] : 0.0f;
      most = fmaxf(most, fabsf(x[c][e]));
    }
  if (K != KP && most > 0.0f && most < kSmallestSplitMoment) x[0][0] = __builtin_nanf("");
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    uint4 h, m, l;
    split3_bf16(x[c], h, m, l);
    out[(3 * c) * 32] = h;
    out[(3 * c + 1) * 32] = m;
    out[(3 * c + 2) * 32] = l;
  }
}

// part[h] += D_ab m_b for the kH 16-state halves from the pieces of D_ab (A
// operands) and of m_b (B operands): the six products of pieces whose orders
// sum to at most 2, smallest first.  The halves' chains alternate, so that
// consecutive products are independent.
template <int kH>
__device__ __forceinline__ void p2p_bf16_products(f32x4 (&part)[kH], const uint4& ah, const uint4& am, const uint4& al,
                                                  const uint4 (&b)[3][kH]) {
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(am, b[1][h], part[h]);
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(al, b[0][h], part[h]);
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(ah, b[2][h], part[h]);
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(am, b[0][h], part[h]);
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(ah, b[1][h], part[h]);
#pragma unroll
  for (int h = 0; h < kH; ++h) part[h] = mfma_bf16(ah, b[0][h], part[h]);
}

// A tile's sums in batches that are no multiple of 32 states, where one of
// them is not finite (rare): those of that lane's target and state again, one
// pair at a time.  In the products a source that is left out (a target's own,
// a padding slot) has weight zero, and zero times a moment that is not finite
// is NaN; here it is left out.  Pairs closer than 3e-8 of the box, whose |r|^-5
// overflows in the products, and moments too small for the products' pieces
// (split_moments_kernel) come here too.  kRows: 3 the field, 4 with the potential, 6 the
// gradient; acc[c][h][i] is row c of state k0 + 16 h, target t0 + i.
template <int kRows, int kH>
__device__ __forceinline__ void p2p_repair(const DevicePlan& d, f32x4 (&acc)[kRows][kH], int leaf, int t0, int cnt,
                                           int k0, int K) {
  bool bad = false;
#pragma unroll
  for (int c = 0; c < kRows; ++c)
#pragma unroll
    for (int h = 0; h < kH; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) bad |= !__builtin_isfinite(acc[c][h][i]);
  if (__any(bad) == 0) return;
  const int q0 = d.nbr_blk_start[leaf], q1 = d.nbr_blk_start[leaf + 1];
  const float* sm = static_cast<const float*>(d.sm);
#pragma unroll 1
  for (int j = 0; j < 4 * kH; ++j) {
    const int h = j >> 2, i = j & 3, k = k0 + 16 * h;
    if (i >= cnt || k >= K) continue;
    const int t = t0 + i, self = d.self[t];
    const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
    float sum[kRows];
#pragma unroll
    for (int c = 0; c < kRows; ++c) sum[c] = 0.0f;
#pragma unroll 1
    for (int q = q0; q < q1; ++q) {
      const int2 bs = d.blk8_src[d.nbr_blk[q]];
#pragma unroll 1
      for (int s = bs.x; s < bs.x + bs.y; ++s) {
        if (s == self) continue;
        float rx, ry, rz;
        tp.diff(PairPos<float>::load(d.src_pos, d.ns, s), rx, ry, rz);
        const float rinv = __builtin_amdgcn_rsqf(rx * rx + ry * ry + rz * rz);
        const float ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
        const float* ms = sm + int64_t(s) * 3 * K + k;
        const float mx = ms[0], my = ms[K], mz = ms[2 * K], w = ux * mx + uy * my + uz * mz;
        if constexpr (kRows == 6) {
          const float g = 0.23873241463784300365332564505877154f * rinv * rinv * rinv * rinv, w5 = 5.0f * w;
          sum[0] += g * (w + 2.0f * ux * mx - w5 * ux * ux);
          sum[1] += g * (ux * my + mx * uy - w5 * ux * uy);
          sum[2] += g * (ux * mz + mx * uz - w5 * ux * uz);
          sum[3] += g * (w + 2.0f * uy * my - w5 * uy * uy);
          sum[4] += g * (uy * mz + my * uz - w5 * uy * uz);
          sum[5] += g * (w + 2.0f * uz * mz - w5 * uz * uz);
        } else {
          const float f = rinv * rinv * rinv * 0.079577471545947667884441881686257181f;
          sum[0] += f * (3.0f * w * ux - mx);
          sum[1] += f * (3.0f * w * uy - my);
          sum[2] += f * (3.0f * w * uz - mz);
          if constexpr (kRows == 4) sum[3] += f * (rx * mx + ry * my + rz * mz);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kRows; ++c)
#pragma unroll
      for (int hh = 0; hh < kH; ++hh)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          if (4 * hh + ii == j && !__builtin_isfinite(acc[c][hh][ii])) acc[c][hh][ii] = sum[c];
  }
}

// List-1 P2P on the matrix cores with bf16 operands
// (v_mfma_f32_16x16x32_bf16), for FP32 plans: the default with K a multiple of
// 32, and other batches as near_on_matrix_cores says.  Both operands are split in three bf16 pieces (hi + mid +
// lo, 24 significant bits) and the six piece products whose orders sum to at
// most 2 are kept, D m ~ Dh mh + Dh mm + Dm mh + Dh ml + Dl mh + Dm mm: the
// dropped ones are below 2^-26 |D m|, under the rounding of FP32 operands.
// Against the FP32 matrix-core product (16x16x4, 32 cycles for 2048 flops)
// the six bf16 products issue 2.7x fewer matrix-core cycles per pair.
//
// One wave owns 16 targets of one leaf and 32 states; the depth of a product
// is four blocks of 8 sources from the list of the neighbourhood's blocks,
// and lane (row i, group g) forms the pairs of target i with the 8 sources of
// block g: their offsets r, then the 6 distinct entries
// D_ab = 3 f r_a r_b / |r|^2 - delta_ab f with f = |r|^-3 / (4 pi), each
// split into pieces for the products of both components it couples.  With
// the potential (kPot) a fourth accumulator row takes phi += f r . m from the
// entries f r_c'.  Lane layout (CDNA4 16x16x32 bf16): A[i][k] in lane
// i + 16 (k / 8), element k % 8; B[k][j] in lane j + 16 (k / 8), element
// k % 8; D[i][j] in lane j + 16 (i / 4), register i % 4.  The moments' pieces
// come from split_moments_kernel in 8-source blocks, so a lane's B operand is
// one 16-byte load; a group past the list's end reads the product's first
// block, and its pairs, padding pairs and the identity pair have |r|^-1 = 0
// and so zero entries.  Coincident pairs give NaN.  Blocked summation per
// product (32 source slots) as in the FP32 kernels.
//
// Fields are capped at 168 registers, three waves per SIMD (4.7 ms at 1M
// points, p = 8, depth 5, K = 32, against 7.4 ms for the FP32 kernel); the
// potential form runs at two, where the cap would spill; with one half of
// states (kH = 1) each has one more.
// kH: 16-state halves of a state tile (one where at most 16 states are left);
// tile0: its first state tile; kRagged: K is no multiple of 32.
template <bool kPot, int kH, bool kRagged>
__global__ void __launch_bounds__(64 * kP2PWaves) __attribute__((amdgpu_waves_per_eu(kPot ? (kH == 1 ? 3 : 2) : (kH == 1 ? 4 : 3))))
p2p_bf16_kernel(const DevicePlan d, const int2* __restrict__ tiles, int tile_count, int K, int tile0) {
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kP2PWaves + wave;
  if (item >= tile_count) return;
  const int2 tile = tiles[item];
  const int leaf = tile.x;
  const int2 trange = d.leaf_tgt[leaf];
  const int col = lane & 15, g = lane >> 4;  // A row / B and D column; source group
  const bool row_ok = trange.x + tile.y + col < trange.y;
  const int t = row_ok ? trange.x + tile.y + col : trange.x;
  const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
  const int self = row_ok ? d.self[t] : -2;
  const int kc0 = (tile0 + int(blockIdx.y)) * 32, KT = (K + 31) / 32;
  const uint4* mb = static_cast<const uint4*>(d.smb);
  constexpr int kRows = kPot ? 4 : 3;  // field components, then the potential
  f32x4 acc[kRows][kH];
#pragma unroll
  for (int c = 0; c < kRows; ++c)
#pragma unroll
    for (int h = 0; h < kH; ++h) acc[c][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // The neighbourhood's 8-source blocks in one list, four per product (one
  // per lane group): a leaf pads to 8 sources rather than to 32.
  const int q0 = d.nbr_blk_start[leaf], q1 = d.nbr_blk_start[leaf + 1];
  const float4* shi = static_cast<const float4*>(d.src_pos);
  const float4* slo = shi + d.ns;
  for (int q = q0; q < q1; q += 4) {
    const bool grp_ok = q + g < q1;
    const int blk = d.nbr_blk[grp_ok ? q + g : q];
    const int2 bs = d.blk8_src[blk];
    const int cnt = grp_ok ? bs.y : 0;
    const uint4* bp = mb + ((int64_t(blk) * KT + (kc0 >> 5)) * 9) * 32 + col;
    uint4 b[3][3][kH];  // [component][piece][state half]
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int pc = 0; pc < 3; ++pc)
#pragma unroll
        for (int h = 0; h < kH; ++h) b[c][pc][h] = bp[(3 * c + pc) * 32 + 16 * h];
    float r[3][8], f[8], gf[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int sidx = bs.x + (e < cnt ? e : 0);
      const PairPos<float> sp{shi[sidx], slo[sidx]};
      tp.diff(sp, r[0][e], r[1][e], r[2][e]);
      const float r2 = r[0][e] * r[0][e] + r[1][e] * r[1][e] + r[2][e] * r[2][e];
      const bool use = row_ok & (e < cnt) & (bs.x + e != self);
      const float rinv = use ? __builtin_amdgcn_rsqf(r2) : 0.0f;
      const float ri2 = rinv * rinv;
      f[e] = ri2 * rinv * 0.079577471545947667884441881686257181f;
      gf[e] = 3.0f * f[e] * ri2;
    }
    f32x4 part[kRows][kH];
#pragma unroll
    for (int c = 0; c < kRows; ++c)
#pragma unroll
      for (int h = 0; h < kH; ++h) part[c][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int bc = a; bc < 3; ++bc) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gf[e] * r[a][e] * r[bc][e] - (a == bc ? f[e] : 0.0f);
        uint4 ph, pm, pl;
        split3_bf16(v, ph, pm, pl);
        uint4 bb[3][kH];
#pragma unroll
        for (int pc = 0; pc < 3; ++pc)
#pragma unroll
          for (int h = 0; h < kH; ++h) bb[pc][h] = b[bc][pc][h];
        p2p_bf16_products(part[a], ph, pm, pl, bb);
        if (a != bc) {
          uint4 ba[3][kH];
#pragma unroll
          for (int pc = 0; pc < 3; ++pc)
#pragma unroll
            for (int h = 0; h < kH; ++h) ba[pc][h] = b[a][pc][h];
          p2p_bf16_products(part[bc], ph, pm, pl, ba);
        }
      }
    if constexpr (kPot) {
      // phi += f (r . m): the entries f r_c' against the moments' component c'.
#pragma unroll
      for (int cp = 0; cp < 3; ++cp) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = f[e] * r[cp][e];
        uint4 ph, pm, pl;
        split3_bf16(v, ph, pm, pl);
        uint4 bb[3][kH];
#pragma unroll
        for (int pc = 0; pc < 3; ++pc)
#pragma unroll
          for (int h = 0; h < kH; ++h) bb[pc][h] = b[cp][pc][h];
        p2p_bf16_products(part[3], ph, pm, pl, bb);
      }
    }
#pragma unroll
    for (int c = 0; c < kRows; ++c)
#pragma unroll
      for (int h = 0; h < kH; ++h) acc[c][h] += part[c][h];
  }
  // acc[c][h][i]: target tile.y + 4g + i, state kc0 + 16h + col.
  if constexpr (kRagged) {
    const int t0 = trange.x + tile.y + 4 * g;
    p2p_repair<kRows, kH>(d, acc, leaf, t0, trange.y - t0, kc0 + col, K);
  }
  float* Hn = static_cast<float*>(d.Hn);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t ot = int64_t(trange.x) + tile.y + 4 * g + i;
    if (ot >= trange.y) continue;
#pragma unroll
    for (int h = 0; h < kH; ++h) {
      const int k = kc0 + 16 * h + col;
      if (kRagged && k >= K) continue;
#pragma unroll
      for (int c = 0; c < 3; ++c) Hn[(ot * 3 + c) * K + k] = acc[c][h][i];
      if constexpr (kPot) static_cast<float*>(d.Pn)[ot * K + k] = acc[3][h][i];
    }
  }
}

// State tiles of 32, and a last one of 16 where at most 16 states are left:
// launch(halves, first tile, tiles).
template <class F>
void for_state_tiles(int K, F&& launch) {
  const int rest = K % 32, whole = K / 32 + (rest > 16 ? 1 : 0);
  if (whole > 0) launch(std::integral_constant<int, 2>{}, 0, whole);
  if (rest > 0 && rest <= 16) launch(std::integral_constant<int, 1>{}, K / 32, 1);
  HIPFMM_CHECK(hipGetLastError());
}

// Batches that are no multiple of 32 take the bf16 kernels where a 32-state
// (or 16-state) tile costs less than the vector ALUs' passes per group of states
// (the near-field variants choose among the kernels of the multiples of 32).
//   * From 9 states on (gradients: 7).  Near field alone, ms, vector ALUs / bf16
//     tiles: fields, 2^20 points, 32 per leaf: K = 8 2.59 / 3.00, 9 3.92 / 3.04,
//     16 5.51 / 3.19, 31 12.6 / 4.8; fields and potentials: K = 8 3.20 / 3.68,
//     9 4.12 / 3.69; gradients: K = 6 5.6 / 5.2, 7 6.19 / 4.88.
//   * On trees of 64 leaves and fewer, where the tiles fill the chip: a
//     neighbourhood there is a good part of all points, so a wave of 16 targets
//     and 32 states is one long chain, a launch of few takes a wave's time
//     however many states it holds, and the vector ALUs' shorter waves end
//     sooner.  The line is at target tiles x states per launch (33 to 48 states
//     are two).  Whole evaluates, 64 leaves, p = 6, bf16 M2L, ms, vector ALUs /
//     bf16 tiles, fields: 154 tiles K = 9 .101 / .123, 30 .126 / .166, 40
//     .145 / .275; 508 tiles K = 9 .157 / .282, 30 .315 / .372, 50 .552 / .425;
//     1033 tiles K = 20 .614 / .673, 30 .906 / .689.  p = 4 to 8, 10 to 250 points
//     per leaf, 7 to 63 states: the line is within .3% of the faster kernel on
//     average, bf16 tiles alone 18 to 25%.  With 512 leaves and more the tiles
//     alone are within .7% (9728 points, 871 tiles: K = 9 .151 / .145, 30
//     .406 / .326).  On 8 leaves and one, whose vector-ALU waves read every
//     source, the line is lower: 8 leaves, p = 4, fields: 303 tiles K = 30
//     .400 / .574, 50 .740 / .617, 1005 tiles K = 12 1.16 / 1.41, 20 2.10 / 1.86;
//     with potentials 303 tiles K = 16 .280 / .431, 30 .668 / .514; gradients 303
//     tiles K = 20 .449 / .742, 1005 K = 7 1.56 / 1.51, 9 1.90 / 1.51.
// rows: outputs per target and state (3, with the potential 4, gradient 6).
static bool near_on_matrix_cores(const DevicePlan& d, int K, int rows) {
  if (K < (rows == 6 ? kNearGradBf16States : kNearBf16States)) return false;
  if (d.leaves > 64) return true;
  int launches = 0;
  for_state_tiles(K, [&](auto, int, int) { ++launches; });
  const bool few = d.leaves <= 8;
  const int64_t line = rows == 3 ? (few ? 15000 : 25000) : rows == 4 ? (few ? 5500 : 13000) : few ? 7000 : 14000;
  return int64_t(d.p2p_tile16_count) * K >= line * launches;
}

// The moments' bf16 pieces for the near-field kernels on bf16 operands.
void launch_split_moments(const DevicePlan& d, int K, hipStream_t s) {
  if (d.smb == nullptr || d.smb_blocks < d.blk8_count)
    throw invalid_argument("bf16 near-field moment buffer is not allocated");
  if (d.blk8_count == 0) return;  // without sources the near-field kernels write zeros
  const int KP = (K + 31) / 32 * 32;
  const int64_t threads = int64_t(d.blk8_count) * KP;
  split_moments_kernel<<<unsigned((threads + 255) / 256), 256, 0, s>>>(d, K, KP);
  HIPFMM_CHECK(hipGetLastError());
}

void launch_p2p_bf16(const DevicePlan& d, int K, bool potential, hipStream_t s) {
  const int count = d.p2p_tile16_count;
  if (count == 0) return;
  launch_split_moments(d, K, s);
  const bool ragged = K % 32 != 0;
  for_state_tiles(K, [&](auto halves, int tile0, int tiles) {
    constexpr int H = decltype(halves)::value;
    const dim3 grid(unsigned((count + kP2PWaves - 1) / kP2PWaves), unsigned(tiles));
    if (potential && ragged)
      p2p_bf16_kernel<true, H, true><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
    else if (ragged)
      p2p_bf16_kernel<false, H, true><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
    else if constexpr (H == 2) {
      if (potential)
        p2p_bf16_kernel<true, 2, false><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
      else
        p2p_bf16_kernel<false, 2, false><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
    }
  });
}

template <class S>
void launch_p2p(const DevicePlan& d, int K, bool potential, hipStream_t s) {
  if (d.leaves == 0 || d.nt == 0) return;
  if (potential && d.Pn == nullptr) throw invalid_argument("near-field potential buffer is not allocated");
  if constexpr (sizeof(S) == 4) {
    if (K % 32 == 0 ? d.p2p_variant == 4 || d.p2p_variant == 0 : near_on_matrix_cores(d, K, potential ? 4 : 3)) {
      launch_p2p_bf16(d, K, potential, s);
      return;
    }
    if (K % 32 == 0 && d.p2p_variant != 1 && d.p2p_variant != 2) {
      const int count = d.p2p_tile16_count;
      if (count == 0) return;
      const dim3 grid(unsigned((count + kP2PWaves - 1) / kP2PWaves), unsigned(K / 32));
      if (potential)
        p2p_mfma16_kernel<4><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K);
      else
        p2p_mfma16_kernel<3><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K);
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
    if (K % 32 == 0 && d.p2p_variant == 2) {
      const int count = potential ? d.p2p_tile4_count : d.p2p_tile_count;
      if (count == 0) return;
      const dim3 grid(unsigned((count + kP2PWaves - 1) / kP2PWaves), unsigned(K / 32));
      if (potential)
        p2p_mfma_kernel<4><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles4, count, K);
      else
        p2p_mfma_kernel<3><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles, count, K);
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_p2p_lanes<S>(d, K, potential, s);
}
template void launch_p2p<float>(const DevicePlan&, int, bool, hipStream_t);
template void launch_p2p<double>(const DevicePlan&, int, bool, hipStream_t);

// acc[E] += W m_D over both state halves, for one entry of W (its pieces)
// and the moments' component D.
template <int E, int D, int kH>
__device__ __forceinline__ void grad_bf16_products(f32x4 (&acc)[6][kH], const uint4& ph, const uint4& pm,
                                                   const uint4& pl, const uint4 (&b)[3][3][kH]) {
  p2p_bf16_products(acc[E], ph, pm, pl, b[D]);
}

// Near-field gradient on bf16 three-piece operands (FP32 plans: the default
// with K a multiple of 32, other batches as near_on_matrix_cores says): the tiles, the neighbourhood's block list and
// the operand layout of p2p_bf16_kernel, with the 10 distinct entries of the
// symmetric 3-tensor W_cjd = g (delta_cj u_d + delta_jd u_c + delta_cd u_j -
// 5 u_c u_j u_d), g = 3/(4 pi |r|^4), each split once and multiplied by the
// moments' components it meets in G_cj += sum_d W_cjd m_d: 18 (output,
// component) pairs of six bf16 products per state half.  Two waves per SIMD;
// accumulation straight into the totals, as in the FP32 gradient kernel.
// Padding pairs and the identity pair have |r|^-1 = 0; coincident pairs give
// NaN.  Writes Gn[t][6][K] (xx xy xz yy yz zz).
template <int kH, bool kRagged>
__global__ void __launch_bounds__(64 * kP2PWaves) __attribute__((amdgpu_waves_per_eu(2)))
p2p_grad_bf16_kernel(const DevicePlan d, const int2* __restrict__ tiles, int tile_count, int K, int tile0) {
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kP2PWaves + wave;
  if (item >= tile_count) return;
  const int2 tile = tiles[item];
  const int leaf = tile.x;
  const int2 trange = d.leaf_tgt[leaf];
  const int col = lane & 15, g = lane >> 4;
  const bool row_ok = trange.x + tile.y + col < trange.y;
  const int t = row_ok ? trange.x + tile.y + col : trange.x;
  const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
  const int self = row_ok ? d.self[t] : -2;
  const int kc0 = (tile0 + int(blockIdx.y)) * 32, KT = (K + 31) / 32;
  const uint4* mb = static_cast<const uint4*>(d.smb);
  f32x4 acc[6][kH];
#pragma unroll
  for (int e = 0; e < 6; ++e)
#pragma unroll
    for (int h = 0; h < kH; ++h) acc[e][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const float c34pi = 0.23873241463784300365332564505877154f;  // 3/(4 pi)
  const int q0 = d.nbr_blk_start[leaf], q1 = d.nbr_blk_start[leaf + 1];
  const float4* shi = static_cast<const float4*>(d.src_pos);
  const float4* slo = shi + d.ns;
  for (int q = q0; q < q1; q += 4) {
    const bool grp_ok = q + g < q1;
    const int blk = d.nbr_blk[grp_ok ? q + g : q];
    const int2 bs = d.blk8_src[blk];
    const int cnt = grp_ok ? bs.y : 0;
    const uint4* bp = mb + ((int64_t(blk) * KT + (kc0 >> 5)) * 9) * 32 + col;
    uint4 b[3][3][kH];  // [component][piece][state half]
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int pc = 0; pc < 3; ++pc)
#pragma unroll
        for (int h = 0; h < kH; ++h) b[c][pc][h] = bp[(3 * c + pc) * 32 + 16 * h];
    float ux[8], uy[8], uz[8], gg[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int sidx = bs.x + (e < cnt ? e : 0);
      const PairPos<float> sp{shi[sidx], slo[sidx]};
      float rx, ry, rz;
      tp.diff(sp, rx, ry, rz);
      const float r2 = rx * rx + ry * ry + rz * rz;
      const bool use = row_ok & (e < cnt) & (bs.x + e != self);
      const float rinv = use ? __builtin_amdgcn_rsqf(r2) : 0.0f;
      ux[e] = rx * rinv;
      uy[e] = ry * rinv;
      uz[e] = rz * rinv;
      gg[e] = c34pi * rinv * rinv * rinv * rinv;
    }
    uint4 ph, pm, pl;
    float v[8];
    // W_cjd with sorted indices 000 001 002 011 012 022 111 112 122 222, and
    // the (output cj, component d) pairs each one serves.
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gg[e] * ux[e] * (3.0f - 5.0f * ux[e] * ux[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<0, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = uy[e] * gg[e] * (1.0f - 5.0f * ux[e] * ux[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<0, 1>(acc, ph, pm, pl, b);
    grad_bf16_products<1, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = uz[e] * gg[e] * (1.0f - 5.0f * ux[e] * ux[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<0, 2>(acc, ph, pm, pl, b);
    grad_bf16_products<2, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = ux[e] * gg[e] * (1.0f - 5.0f * uy[e] * uy[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<1, 1>(acc, ph, pm, pl, b);
    grad_bf16_products<3, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = -5.0f * gg[e] * ux[e] * uy[e] * uz[e];
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<1, 2>(acc, ph, pm, pl, b);
    grad_bf16_products<2, 1>(acc, ph, pm, pl, b);
    grad_bf16_products<4, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = ux[e] * gg[e] * (1.0f - 5.0f * uz[e] * uz[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<2, 2>(acc, ph, pm, pl, b);
    grad_bf16_products<5, 0>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gg[e] * uy[e] * (3.0f - 5.0f * uy[e] * uy[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<3, 1>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = uz[e] * gg[e] * (1.0f - 5.0f * uy[e] * uy[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<3, 2>(acc, ph, pm, pl, b);
    grad_bf16_products<4, 1>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = uy[e] * gg[e] * (1.0f - 5.0f * uz[e] * uz[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<4, 2>(acc, ph, pm, pl, b);
    grad_bf16_products<5, 1>(acc, ph, pm, pl, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gg[e] * uz[e] * (3.0f - 5.0f * uz[e] * uz[e]);
    split3_bf16(v, ph, pm, pl);
    grad_bf16_products<5, 2>(acc, ph, pm, pl, b);
  }
  // acc[e][h][i]: target tile.y + 4g + i, state kc0 + 16h + col.
  if constexpr (kRagged) {
    const int t0 = trange.x + tile.y + 4 * g;
    p2p_repair<6, kH>(d, acc, leaf, t0, trange.y - t0, kc0 + col, K);
  }
  float* Gn = static_cast<float*>(d.Gn);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t ot = int64_t(trange.x) + tile.y + 4 * g + i;
    if (ot >= trange.y) continue;
#pragma unroll
    for (int h = 0; h < kH; ++h) {
      const int k = kc0 + 16 * h + col;
      if (kRagged && k >= K) continue;
#pragma unroll
      for (int e = 0; e < 6; ++e) Gn[(ot * 6 + e) * K + k] = acc[e][h][i];
    }
  }
}

// Near-field gradient on the matrix cores (FP32 plans, K a multiple of 32),
// targets as rows like p2p_mfma16_kernel: with g = 3/(4 pi |r|^4) the
// derivative of the pair tensor is the fully symmetric 3-tensor
//   W_cjd = g (delta_cj u_d + delta_jd u_c + delta_cd u_j - 5 u_c u_j u_d),
// 10 distinct entries, and G_cj += sum_d W_cjd m_d: 18 products per 4
// sources and 16 states, six 16 x 16 accumulator tiles per column half.
// Padding slots and the identity pair get |r|^-1 = 0.  Writes Gn[t][6][K]
// (xx xy xz yy yz zz) for the far-field gradient kernel to complete.
__global__ void __launch_bounds__(64 * kP2PWaves) p2p_grad_mfma16_kernel(const DevicePlan d,
                                                                        const int2* __restrict__ tiles,
                                                                        int tile_count, int K) {
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * kP2PWaves + wave;
  if (item >= tile_count) return;
  const int2 tile = tiles[item];
  const int leaf = tile.x;
  const int2 trange = d.leaf_tgt[leaf];
  const int col = lane & 15, q = lane >> 4;
  const bool row_ok = trange.x + tile.y + col < trange.y;
  const int t = row_ok ? trange.x + tile.y + col : trange.x;
  const PairPos<float> tp = PairPos<float>::load(d.tgt_pos, d.nt, t);
  const int self = row_ok ? d.self[t] : -2;
  const int kc0 = int(blockIdx.y) * 32;
  const float* sm = static_cast<const float*>(d.sm);
  f32x4 acc[6][2];
#pragma unroll
  for (int e = 0; e < 6; ++e) acc[e][0] = acc[e][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int nb = 1 << d.L;
  int lx, ly, lz;
  demorton3(uint32_t(leaf), d.L, lx, ly, lz);
  const float c34pi = 0.23873241463784300365332564505877154f;  // 3/(4 pi)
  for (int dz = -1; dz <= 1; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        const int x = lx + dx, y = ly + dy, z = lz + dz;
        if (x < 0 || y < 0 || z < 0 || x >= nb || y >= nb || z >= nb) continue;
        const int2 sr = d.leaf_src[morton3(uint32_t(x), uint32_t(y), uint32_t(z), d.L)];
        if (sr.x == sr.y) continue;
        const P2PSources src{static_cast<const float4*>(d.src_pos) + sr.x,
                             static_cast<const float4*>(d.src_pos) + d.ns + sr.x, sm + int64_t(sr.x) * 3 * K + kc0};
        for (int j00 = sr.x; j00 < sr.y; j00 += 8) {
          P2PRaw raw[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) raw[u] = p2p_load(src, j00 + 4 * u + q, sr.x, sr.y, K, col);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float rx, ry, rz;
            tp.diff(raw[u].sp, rx, ry, rz);
            const float r2 = rx * rx + ry * ry + rz * rz;
            const bool use = row_ok & (raw[u].s < sr.y) & (raw[u].s != self);
            // A coincident pair that is used gives inf, hence NaN entries.
            const float rinv = use ? __builtin_amdgcn_rsqf(r2) : 0.0f;
            const float g = c34pi * rinv * rinv * rinv * rinv;
            const float ux = rx * rinv, uy = ry * rinv, uz = rz * rinv;
            const float g5 = 5.0f * g;
            // W_cjd with sorted indices 000 001 002 011 012 022 111 112 122 222.
            const float w000 = g * ux * (3.0f - 5.0f * ux * ux);
            const float w001 = uy * (g - g5 * ux * ux);
            const float w002 = uz * (g - g5 * ux * ux);
            const float w011 = ux * (g - g5 * uy * uy);
            const float w012 = -g5 * ux * uy * uz;
            const float w022 = ux * (g - g5 * uz * uz);
            const float w111 = g * uy * (3.0f - 5.0f * uy * uy);
            const float w112 = uz * (g - g5 * uy * uy);
            const float w122 = uy * (g - g5 * uz * uz);
            const float w222 = g * uz * (3.0f - 5.0f * uz * uz);
            const float W[6][3] = {{w000, w001, w002}, {w001, w011, w012}, {w002, w012, w022},
                                   {w011, w111, w112}, {w012, w112, w122}, {w022, w122, w222}};
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int dd = 0; dd < 3; ++dd)
#pragma unroll
                for (int e = 0; e < 6; ++e)
                  acc[e][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(W[e][dd], raw[u].b[dd][h], acc[e][h], 0, 0, 0);
          }
        }
      }
  // acc[e][h][i]: target tile.y + 4q + i, state kc0 + 16h + col.
  float* Gn = static_cast<float*>(d.Gn);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t ot = int64_t(trange.x) + tile.y + 4 * q + i;
    if (ot >= trange.y) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 6; ++e) Gn[(ot * 6 + e) * K + kc0 + 16 * h + col] = acc[e][h][i];
  }
}

template <class S>
void launch_p2p_grad(const DevicePlan& d, int K, hipStream_t s) {
  if (d.leaves == 0 || d.nt == 0) return;
  if (d.Gn == nullptr) throw invalid_argument("near-field gradient buffer is not allocated");
  if constexpr (sizeof(S) == 4) {
    const int count = d.p2p_tile16_count;
    const unsigned blocks = unsigned((count + kP2PWaves - 1) / kP2PWaves);
    if (count > 0 && (K % 32 == 0 ? d.p2p_variant == 0 || d.p2p_variant == 4 : near_on_matrix_cores(d, K, 6))) {
      launch_split_moments(d, K, s);
      for_state_tiles(K, [&](auto halves, int tile0, int tiles) {
        constexpr int H = decltype(halves)::value;
        const dim3 grid(blocks, unsigned(tiles));
        if (K % 32 != 0)
          p2p_grad_bf16_kernel<H, true><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
        else if constexpr (H == 2)
          p2p_grad_bf16_kernel<2, false><<<grid, 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K, tile0);
      });
      return;
    }
    if (count > 0 && K % 32 == 0) {
      p2p_grad_mfma16_kernel<<<dim3(blocks, unsigned(K / 32)), 64 * kP2PWaves, 0, s>>>(d, d.p2p_tiles16, count, K);
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_p2p_grad_lanes<S>(d, K, s);
}
template void launch_p2p_grad<float>(const DevicePlan&, int, hipStream_t);
template void launch_p2p_grad<double>(const DevicePlan&, int, hipStream_t);

void direct_field_fp64(const double* targets, int nt, const double* sources, int ns, const double* moments,
                       const int* self, double* fields) {
  if (nt == 0) return;
  direct_kernel<<<unsigned((nt + kThreads - 1) / kThreads), kThreads, 0, nullptr>>>(targets, nt, sources, ns,
                                                                                      moments, self, fields);
  HIPFMM_CHECK(hipGetLastError());
}

}  // namespace hipfmm
