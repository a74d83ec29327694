// Far-field kernels of the HipFull path on the matrix cores for FP32 plans with
// a multiple of 32 moment states: leaf P2M, level-wise M2M and L2L, the
// harmonic compression and expansion, and leaf L2P with the near-field
// combine; the moment gather and the unsorts; and the dispatch between these
// and the kernels of columns.hip, which serve every other number of states and
// FP64.  One workgroup owns one box (P2M, L2P) or one parent box (M2M, L2L),
// reads its inputs once and writes its outputs once, with no atomics.
//
// Reference operations restated here:
//   permute_moments / prepare_moments_float   src/cuda_fmm.cu:56-64, src/far_field.cpp:334-365
//   P2M   M_a = (-1)^|a| sum_j sum_{c: a_c>0} m_jc d_j^(a-e_c)/(a-e_c)!
//         src/static_operators.cpp:186-220, src/operators.cpp:16-52
//   M2M / L2L  shared per-(level, class) shift operators
//         src/static_operators.cpp:257-298, src/far_field.cpp:395-446, :555-574
//   L2P   H_c = -sum_{b: b_c>0} L_b dx^(b-e_c)/(b-e_c)!
//         src/static_operators.cpp:300-335
//   combine + unsort  src/cuda_fmm.cu:503-516, src/uniform_fmm.cpp:1439-1452
#include "common.hpp"
#include "bf16_split.hpp"

namespace hipfmm {

namespace {

constexpr int kThreads = 256;

__host__ __device__ inline int round_up(int x, int m) { return (x + m - 1) / m * m; }
// Moments from the user layout [k][user][3] into the sorted state layout
// sm[sorted][3][K], times the frame factor.  A workgroup owns `points`
// consecutive user points: it reads their rows of every state (3 * points
// contiguous scalars per state) into LDS and writes each point's 3K scalars
// contiguously at its sorted slot, so both sides move whole cache lines.
// kVec: FP32, full tiles of 64 points, 16-byte aligned rows (N and K
// multiples of 4): both sides move float4s.
template <class S, bool kVec>
__global__ void __launch_bounds__(kThreads) gather_kernel(const S* __restrict__ mu, const int* __restrict__ inv,
                                                          S scale, int ns, int K, int points, S* __restrict__ sm) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  S* tile = reinterpret_cast<S*>(smem_raw);  // [point][3K + 4]
  const int row = 3 * K + 4, width = 3 * K;
  const int u0 = blockIdx.x * points;
  if constexpr (kVec) {
    constexpr int kRow4 = 3 * 64 / 4;  // float4s of one state's row of the tile
    const float4* src = reinterpret_cast<const float4*>(mu);
    for (int e = threadIdx.x; e < K * kRow4; e += kThreads) {
      const int k = e / kRow4, q = e - k * kRow4;
      const float4 v = src[(int64_t(k) * ns + u0) * 3 / 4 + q];
      const float w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * q + i, u = r / 3, c = r - 3 * u;
        tile[u * row + c * K + k] = w[i];
      }
    }
    __syncthreads();
    const int w4 = width / 4;
    for (int e = threadIdx.x; e < 64 * w4; e += kThreads) {
      const int u = e / w4, q = e - u * w4;
      float4 v = *reinterpret_cast<const float4*>(tile + u * row + 4 * q);
      v.x *= scale;
      v.y *= scale;
      v.z *= scale;
      v.w *= scale;
      reinterpret_cast<float4*>(sm + int64_t(inv[u0 + u]) * width)[q] = v;
    }
  } else {
    const int cnt = min(points, ns - u0);
    const int span = 3 * cnt;
    for (int e = threadIdx.x; e < span * K; e += kThreads) {
      const int k = e / span, r = e - k * span;
      const int u = r / 3, c = r - 3 * u;
      tile[u * row + c * K + k] = mu[(int64_t(k) * ns + u0) * 3 + r];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < cnt * width; e += kThreads) {
      const int u = e / width, r = e - u * width;
      sm[int64_t(inv[u0 + u]) * width + r] = tile[u * row + r] * scale;
    }
  }
}

// The inverse of gather_kernel for the fields: sorted totals Hn[t][3][K] to
// the user layout out[k][user][3].  A workgroup owns 64 consecutive user
// points: it reads each point's 3K values contiguously from its sorted slot
// into LDS, then writes the 64 points' 192 contiguous values of every
// state.  FP32, N and K multiples of 64 and 4, 16-byte aligned output.
__global__ void __launch_bounds__(kThreads) scatter_fields_kernel(const float* __restrict__ hs,
                                                                  const int* __restrict__ inv, int nt, int K,
                                                                  float* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* tile = reinterpret_cast<float*>(smem_raw);  // [point][3K + 4]
  const int row = 3 * K + 4, w4 = 3 * K / 4;
  const int u0 = blockIdx.x * 64;
  for (int e = threadIdx.x; e < 64 * w4; e += kThreads) {
    const int u = e / w4, q = e - u * w4;
    *reinterpret_cast<float4*>(tile + u * row + 4 * q) =
        reinterpret_cast<const float4*>(hs + int64_t(inv[u0 + u]) * 3 * K)[q];
  }
  __syncthreads();
  constexpr int kRow4 = 3 * 64 / 4;
  float4* dst = reinterpret_cast<float4*>(out);
  for (int e = threadIdx.x; e < K * kRow4; e += kThreads) {
    const int k = e / kRow4, q = e - k * kRow4;
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * q + i, u = r / 3, c = r - 3 * u;
      w[i] = tile[u * row + c * K + k];
    }
    dst[(int64_t(k) * nt + u0) * 3 / 4 + q] = float4{w[0], w[1], w[2], w[3]};
  }
}

// The same for the potentials: sorted Pn[t][K] to pot[k][user].  A
// workgroup owns 64 consecutive user points: each point's K values are one
// contiguous read, and each state's 64 values one contiguous write.
__global__ void __launch_bounds__(kThreads) scatter_potentials_kernel(const float* __restrict__ ps,
                                                                      const int* __restrict__ inv, int nt, int K,
                                                                      float* __restrict__ pot) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* tile = reinterpret_cast<float*>(smem_raw);  // [point][K + 4]
  const int row = K + 4, k4 = K / 4;
  const int u0 = blockIdx.x * 64;
  for (int e = threadIdx.x; e < 64 * k4; e += kThreads) {
    const int u = e / k4, q = e - u * k4;
    *reinterpret_cast<float4*>(tile + u * row + 4 * q) =
        reinterpret_cast<const float4*>(ps + int64_t(inv[u0 + u]) * K)[q];
  }
  __syncthreads();
  float4* dst = reinterpret_cast<float4*>(pot);
  for (int e = threadIdx.x; e < K * 16; e += kThreads) {
    const int k = e >> 4, q = e & 15;
    dst[(int64_t(k) * nt + u0) / 4 + q] = float4{tile[(4 * q) * row + k], tile[(4 * q + 1) * row + k],
                                                 tile[(4 * q + 2) * row + k], tile[(4 * q + 3) * row + k]};
  }
}

// Dense transposed shift operators: T[(level*8 + class)][col][NP], row
// (output coefficient) contiguous, rows n..NP-1 zero.
template <class S>
__device__ __forceinline__ const S* shift_operator(const void* dense, int level, int cls, int n, int NP) {
  return static_cast<const S*>(dense) + (size_t(level) * 8 + cls) * size_t(n) * NP;
}

template <class S>
__global__ void zero_kernel(S* p, size_t count) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += size_t(gridDim.x) * blockDim.x)
    p[i] = S(0);
}

// P2M on the matrix cores (FP32 plans, K a multiple of 32).  With
// g = alpha - e_c the multipoles of a leaf are
//   M[alpha][k] = (-1)^|alpha| sum_{c: alpha_c > 0} C_c[alpha - e_c][k],
//   C_c[g][k]   = sum_s mono_g(d_s) m[s][c][k]        (|g| < p)
// (src/static_operators.cpp:186-220); the C_c are v_mfma_f32_16x16x4_f32
// products with the monomials as rows (A, shared by the three components),
// 4 sources of depth per step and kH 16-state column tiles.  One workgroup
// (4 waves) per leaf and 16 kH states; wave w owns monomial row tiles w,
// w+4, ... (kTW of them).  Sources go through LDS 64 at a time as
// axis-power tables; the C_c meet in LDS, where the sign-and-shift
// combination writes M.
template <int kTW, int kH>
__global__ void __launch_bounds__(256) p2m_mfma_kernel(const DevicePlan d, int K) {
  constexpr int kCols = 16 * kH;  // states of this workgroup
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = d.n, nm = d.nm, PW = d.p;  // axis powers 0..p-1
  const int NT = (nm + 15) / 16, NMP = NT * 16;
  float* pw = reinterpret_cast<float*>(smem_raw);  // [64][3][PW]
  float* Cl = pw + 64 * 3 * PW;                      // [3][NMP][kCols]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, q = lane >> 4;
  const int leaf = blockIdx.x, kc0 = int(blockIdx.y) * kCols;
  const int2 range = d.leaf_src[leaf];
  const int64_t node = level_offset(d.L) + leaf;
  if (range.x == range.y) {
    float* o = static_cast<float*>(d.M) + node * int64_t(n) * K + kc0;
    for (int w = tid; w < n * kCols; w += 256) o[int64_t(w / kCols) * K + w % kCols] = 0.0f;
    return;
  }
  const auto* rel = static_cast<const float4*>(d.src_rel);
  const float* sm = static_cast<const float*>(d.sm);
  int4 ex[kTW];
  bool row_ok[kTW];
#pragma unroll
  for (int j = 0; j < kTW; ++j) {
    const int g = (wave + 4 * j) * 16 + col;
    row_ok[j] = g < nm;
    ex[j] = row_ok[j] ? d.p2m_tab[n + g] : int4{0, 0, 0, 0};
  }
  f32x4 acc[kTW][3][kH];
#pragma unroll
  for (int j = 0; j < kTW; ++j)
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int h = 0; h < kH; ++h) acc[j][c][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int j0 = range.x; j0 < range.y; j0 += 64) {
    const int cnt = min(64, range.y - j0);
    __syncthreads();  // the previous chunk's tables are no longer read
    if (tid < 192) {
      const int sj = tid / 3, a = tid % 3;
      float x = 0.0f;
      if (sj < cnt) {
        const float4 r = rel[j0 + sj];
        x = a == 0 ? r.x : (a == 1 ? r.y : r.z);
      }
      float v = 1.0f;
      float* row = pw + tid * PW;
      row[0] = 1.0f;
      for (int i = 1; i < PW; ++i) {
        v = v * x / float(i);
        row[i] = v;
      }
    }
    __syncthreads();
    // Four steps (16 sources) per iteration: all four steps' loads are
    // issued before any product, so a leaf of up to 32 sources waits on
    // memory twice.  Loads are unconditional (clamped index) and masked
    // afterwards, so they do not become branches that each wait.
    constexpr int kSteps = 4;
    for (int s00 = 0; s00 < cnt; s00 += 4 * kSteps) {
      float b[kSteps][3][kH];
      bool okv[kSteps];
      int sjv[kSteps];
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const int sj = s00 + 4 * u + q;
        okv[u] = sj < cnt;
        sjv[u] = okv[u] ? sj : 0;
        const float* ms = sm + int64_t(j0 + sjv[u]) * 3 * K + kc0 + col;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int h = 0; h < kH; ++h) b[u][c][h] = ms[c * K + 16 * h];
      }
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const float* ps = pw + sjv[u] * 3 * PW;
        // A tile past the last monomial row has row_ok false and multiplies
        // zeros; its products are never stored.
#pragma unroll
        for (int j = 0; j < kTW; ++j) {
          const float a = (okv[u] && row_ok[j]) ? ps[ex[j].x] * ps[PW + ex[j].y] * ps[2 * PW + ex[j].z] : 0.0f;
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int h = 0; h < kH; ++h)
              acc[j][c][h] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(a, okv[u] ? b[u][c][h] : 0.0f, acc[j][c][h], 0, 0, 0);
        }
      }
    }
  }
  // C_c[g][k] to LDS: acc[j][c][h][r] is row (wave + 4j)*16 + 4q + r, state 16h + col.
#pragma unroll
  for (int j = 0; j < kTW; ++j) {
    if (wave + 4 * j >= NT) break;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int h = 0; h < kH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          Cl[(c * NMP + (wave + 4 * j) * 16 + 4 * q + r) * kCols + 16 * h + col] = acc[j][c][h][r];
  }
  __syncthreads();
  float* M = static_cast<float*>(d.M) + node * int64_t(n) * K + kc0;
  for (int w = tid; w < n * kCols; w += 256) {
    const int b = w / kCols, k = w % kCols;
    const int4 t = d.p2m_tab[b];
    float v = 0.0f;
    if (t.x >= 0) v += Cl[(0 * NMP + t.x) * kCols + k];
    if (t.y >= 0) v += Cl[(1 * NMP + t.y) * kCols + k];
    if (t.z >= 0) v += Cl[(2 * NMP + t.z) * kCols + k];
    M[int64_t(b) * K + k] = t.w > 0 ? v : -v;
  }
}

// L2P on the matrix cores (FP32 plans, K a multiple of 32): for 16 targets
// of one leaf and 32 states,
//   H_c[t][k] = Hn[t][c][k] - sum_g mono_g(t) L[g + e_c][k]      (|g| < p)
//   phi[t][k] = W (Pn[t][k] + sum_b mono_b(t) L[b][k])           (|b| <= p)
// with mono_g(t) = d_t^g / g! (src/static_operators.cpp:300-335), as
// v_mfma_f32_16x16x4_f32 products: A = monomials (rows = targets, depth = 4
// monomials), B = rows of the leaf local, one accumulator tile per output
// component and 16-state half; the monomial operand is shared by the three
// components.  One wave per 16-target tile (the near-field tiles), four per
// workgroup; per wave LDS holds the axis powers x^i / i!, and each step forms
// its monomial as the product of three of them (a monomial table in LDS kept
// the kernel at 3 waves per SIMD).  Writes out[k][user target][3] (and pot[k][user target]), or
// with kSorted the total fields over the near field in sorted order
// Hn[t][3][K], for scatter_fields_kernel to unsort.
template <bool kPot, bool kSorted>
__global__ void __launch_bounds__(256) l2p_mfma_kernel(const DevicePlan d, float* __restrict__ out,
                                                       float* __restrict__ pot, int K) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = d.n, p = d.p, NM = kPot ? d.n : d.nm, PW = p + 1;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  float* pw = reinterpret_cast<float*>(smem_raw) + wave * (48 * PW);       // [t][axis][i]
  // Basis tables shared by the workgroup: exponents of the NM monomials and
  // the raising table g -> g + e_c (so no step waits on a table load).
  int4* ex_l = reinterpret_cast<int4*>(reinterpret_cast<float*>(smem_raw) + 4 * 48 * PW);
  int4* up_l = ex_l + NM;
  for (int i = threadIdx.x; i < NM; i += 256) ex_l[i] = d.p2m_tab[n + i];
  for (int i = threadIdx.x; i < d.nm; i += 256) up_l[i] = d.l2p_up[i];
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * 4 + wave;
  const bool valid = item < d.p2p_tile16_count;
  const int2 tile = valid ? d.p2p_tiles16[item] : int2{0, 0};
  const int2 trange = valid ? d.leaf_tgt[tile.x] : int2{0, 0};
  const int t0 = trange.x + tile.y;
  const int cnt = valid ? min(16, trange.y - t0) : 0;
  const auto* rel = static_cast<const float4*>(d.tgt_rel);
  if (lane < 48) {
    const int t = lane / 3, a = lane % 3;
    float x = 0.0f;
    if (t < cnt) {
      const float4 r = rel[t0 + t];
      x = a == 0 ? r.x : (a == 1 ? r.y : r.z);
    }
    float v = 1.0f;
    pw[lane * PW] = 1.0f;
    for (int i = 1; i < PW; ++i) {
      v = v * x / float(i);
      pw[lane * PW + i] = v;
    }
  }
  __syncthreads();  // axis powers and basis tables in LDS
  if (!valid) return;
  const int col = lane & 15, q = lane >> 4;
  const float* pt = pw + col * 3 * PW;  // this lane's target
  auto mono = [&](int g) {
    const int4 e = ex_l[g];
    return pt[e.x] * pt[PW + e.y] * pt[2 * PW + e.z];
  };
  const int kc0 = int(blockIdx.y) * 32;
  const int64_t node = level_offset(d.L) + tile.x;
  const float* Lb = static_cast<const float*>(d.Lc) + node * int64_t(n) * K + kc0 + col;
  // The near field this tile adds to (Hn, Pn) is loaded before the products
  // so that its loads are in flight meanwhile; the far field is summed apart
  // and added once at the end (H = Hn - sum, phi = W (Pn + sum)), which
  // keeps the small far-field terms from rounding at the near field's
  // magnitude.  near[c][h][r], acc[c][h][r]: target t0 + 4q + r, state
  // kc0 + 16h + col.
  const float* Hn = static_cast<const float*>(d.Hn);
  const bool fields = !kPot || out != nullptr;
  f32x4 acc[3][2], accp[2], near[kPot ? 4 : 3][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t ts = 4 * q + r < cnt ? t0 + 4 * q + r : t0;
      const int k = kc0 + 16 * h + col;
      const float* hn = Hn + ts * 3 * K + k;
#pragma unroll
      for (int c = 0; c < 3; ++c) near[c][h][r] = fields ? hn[c * K] : 0.0f;
      if constexpr (kPot) near[3][h][r] = static_cast<const float*>(d.Pn)[ts * K + k];
    }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    acc[0][h] = acc[1][h] = acc[2][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    accp[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const int nm = d.nm;
  // Loads are unconditional (past-the-end monomials read row 0 and are
  // masked afterwards), so they do not become branches that each wait; eight
  // steps' loads are in flight together (4 waits per wave at p = 8).
  constexpr int kSteps = 8;
  for (int g00 = 0; g00 < nm; g00 += 4 * kSteps) {
    float av[kSteps], bv[kSteps][3][2];
    bool okv[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int g = g00 + 4 * u + q;
      okv[u] = g < nm;
      const int gl = okv[u] ? g : 0;
      av[u] = okv[u] ? mono(gl) : 0.0f;
      const int4 up = up_l[gl];
      const int rows[3] = {up.x, up.y, up.z};
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) bv[u][c][h] = Lb[int64_t(rows[c]) * K + 16 * h];
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], okv[u] ? bv[u][c][h] : 0.0f, acc[c][h], 0, 0, 0);
  }
  if constexpr (kPot) {
#pragma unroll 4
    for (int b0 = 0; b0 < n; b0 += 4) {
      const int b = b0 + q;
      const bool ok = b < n;
      const int bl = ok ? b : 0;
      const float a = ok ? mono(bl) : 0.0f;
      float bv[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) bv[h] = Lb[int64_t(bl) * K + 16 * h];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        accp[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, ok ? bv[h] : 0.0f, accp[h], 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int tl = 4 * q + r;
    if (tl >= cnt) continue;
    const int ts = t0 + tl;
    const int user = kSorted ? 0 : d.tgt_perm[ts];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = kc0 + 16 * h + col;
      if constexpr (kSorted) {
        // The total overwrites the near field in sorted order; the unsort
        // follows as its own coalesced pass.
        if (fields) {
          float* hn = const_cast<float*>(Hn) + int64_t(ts) * 3 * K + k;
          hn[0] = near[0][h][r] - acc[0][h][r];
          hn[K] = near[1][h][r] - acc[1][h][r];
          hn[2 * K] = near[2][h][r] - acc[2][h][r];
        }
      } else if (fields) {
        float* o = out + (int64_t(k) * d.nt + user) * 3;
        o[0] = near[0][h][r] - acc[0][h][r];
        o[1] = near[1][h][r] - acc[1][h][r];
        o[2] = near[2][h][r] - acc[2][h][r];
      }
      if constexpr (kPot) {
        const float phi = float(d.potential_scale) * (near[3][h][r] + accp[h][r]);
        if constexpr (kSorted)
          static_cast<float*>(d.Pn)[int64_t(ts) * K + k] = phi;  // unsorted by scatter_potentials_kernel
        else
          pot[int64_t(k) * d.nt + user] = phi;
      }
    }
  }
}

}  // namespace

template <class S>
void launch_gather(const DevicePlan& d, const S* user_moments, S scale, int K, hipStream_t s) {
  const int64_t work = int64_t(d.ns) * K;
  if (work == 0) return;
  int points = 64;  // within 64 KiB of LDS
  while (points > 8 && size_t(points) * (3 * K + 4) * sizeof(S) > 65536) points /= 2;
  const size_t lds = size_t(points) * (3 * K + 4) * sizeof(S);
  const unsigned blocks = unsigned((d.ns + points - 1) / points);
  const bool vec = sizeof(S) == 4 && points == 64 && d.ns % 64 == 0 && K % 4 == 0 &&
                   reinterpret_cast<uintptr_t>(user_moments) % 16 == 0;
  if (vec)
    gather_kernel<S, true><<<blocks, kThreads, lds, s>>>(user_moments, d.src_inv, scale, d.ns, K, points,
                                                         static_cast<S*>(d.sm));
  else
    gather_kernel<S, false><<<blocks, kThreads, lds, s>>>(user_moments, d.src_inv, scale, d.ns, K, points,
                                                          static_cast<S*>(d.sm));
  HIPFMM_CHECK(hipGetLastError());
}

template <class S>
void launch_p2m(const DevicePlan& d, int K, hipStream_t s) {
  if (d.leaves == 0) return;
  if constexpr (sizeof(S) == 4) {
    const int NT = (d.nm + 15) / 16, TW = (NT + 3) / 4;
    // 16 states per workgroup: the C_c tiles in LDS stay small enough for
    // several workgroups per CU to hide each other's memory latency.
    const size_t lds = (size_t(64) * 3 * std::max(d.p, 1) + size_t(3) * NT * 16 * 16) * sizeof(float);
    if (K % 32 == 0 && d.p >= 1 && TW <= 4 && lds <= 65536) {
      const dim3 grid(unsigned(d.leaves), unsigned(K / 16));
      switch (TW) {
        case 1: p2m_mfma_kernel<1, 1><<<grid, 256, lds, s>>>(d, K); break;
        case 2: p2m_mfma_kernel<2, 1><<<grid, 256, lds, s>>>(d, K); break;
        case 3: p2m_mfma_kernel<3, 1><<<grid, 256, lds, s>>>(d, K); break;
        default: p2m_mfma_kernel<4, 1><<<grid, 256, lds, s>>>(d, K); break;
      }
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_p2m_columns<S>(d, K, s);
}

// Far-field gradient on the matrix cores (FP32 plans, K a multiple of 32),
// laid out like l2p_mfma_kernel: for 16 targets of one leaf and 32 states,
//   G_e[t][k] = Gn[t][e][k] - sum_g mono_g(t) L[g + e_c + e_j][k]
// over the monomials g of degree <= p - 2 (the A operand, 4 per step) and
// the six (c, j) = xx xy xz yy yz zz (a second raising table), as six 16 x 16
// accumulator tiles per 16-state half; times the frame factor 1/W, written
// to out[k][user target][6].  One wave per 16-target tile, four per
// workgroup; four steps' loads are in flight together.  Each step forms its
// monomial from three LDS axis powers, as the field's L2P does.
__global__ void __launch_bounds__(256) l2p_grad_mfma_kernel(const DevicePlan d, float* __restrict__ out, int K,
                                                           int nm2, float scale) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = d.n, PW = max(d.p - 1, 1);  // axis powers 0..p-2
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  float* pw = reinterpret_cast<float*>(smem_raw) + wave * (48 * PW);                 // [t][axis][i]
  int4* ex_l = reinterpret_cast<int4*>(reinterpret_cast<float*>(smem_raw) + 4 * 48 * PW);
  int* up_l = reinterpret_cast<int*>(ex_l + nm2);  // [g][8]
  for (int i = threadIdx.x; i < nm2; i += 256) ex_l[i] = d.p2m_tab[n + i];
  for (int i = threadIdx.x; i < nm2 * 8; i += 256) up_l[i] = d.grad_up[i];
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * 4 + wave;
  const bool valid = item < d.p2p_tile16_count;
  const int2 tile = valid ? d.p2p_tiles16[item] : int2{0, 0};
  const int2 trange = valid ? d.leaf_tgt[tile.x] : int2{0, 0};
  const int t0 = trange.x + tile.y;
  const int cnt = valid ? min(16, trange.y - t0) : 0;
  const auto* rel = static_cast<const float4*>(d.tgt_rel);
  if (lane < 48) {
    const int t = lane / 3, a = lane % 3;
    float x = 0.0f;
    if (t < cnt) {
      const float4 r = rel[t0 + t];
      x = a == 0 ? r.x : (a == 1 ? r.y : r.z);
    }
    float v = 1.0f;
    pw[lane * PW] = 1.0f;
    for (int i = 1; i < PW; ++i) {
      v = v * x / float(i);
      pw[lane * PW + i] = v;
    }
  }
  __syncthreads();  // axis powers and tables in LDS
  if (!valid) return;
  const int col = lane & 15, q = lane >> 4;
  const float* pt = pw + col * 3 * PW;  // this lane's target
  auto mono = [&](int g) {
    const int4 e = ex_l[g];
    return pt[e.x] * pt[PW + e.y] * pt[2 * PW + e.z];
  };
  const int kc0 = int(blockIdx.y) * 32;
  const int64_t node = level_offset(d.L) + tile.x;
  const float* Lb = static_cast<const float*>(d.Lc) + node * int64_t(n) * K + kc0 + col;
  f32x4 acc[6][2];
#pragma unroll
  for (int e = 0; e < 6; ++e) acc[e][0] = acc[e][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int kSteps = 4;
  for (int g00 = 0; g00 < nm2; g00 += 4 * kSteps) {
    float av[kSteps], bv[kSteps][6][2];
    bool okv[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int g = g00 + 4 * u + q;
      okv[u] = g < nm2;
      const int gl = okv[u] ? g : 0;
      av[u] = okv[u] ? mono(gl) : 0.0f;
#pragma unroll
      for (int e = 0; e < 6; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) bv[u][e][h] = Lb[int64_t(up_l[gl * 8 + e]) * K + 16 * h];
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int e = 0; e < 6; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          acc[e][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], okv[u] ? bv[u][e][h] : 0.0f, acc[e][h], 0, 0, 0);
  }
  // acc[e][h][r]: target t0 + 4q + r, state kc0 + 16h + col.
  const float* Gn = static_cast<const float*>(d.Gn);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int tl = 4 * q + r;
    if (tl >= cnt) continue;
    const int ts = t0 + tl;
    const int user = d.tgt_perm[ts];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = kc0 + 16 * h + col;
      float* o = out + (int64_t(k) * d.nt + user) * 6;
      const float* gn = Gn + int64_t(ts) * 6 * K + k;
#pragma unroll
      for (int e = 0; e < 6; ++e) o[e] = scale * (gn[int64_t(e) * K] - acc[e][h][r]);
    }
  }
}

template <class S>
void launch_l2p_grad_unsort(const DevicePlan& d, S* gradients, int K, hipStream_t s) {
  if (d.leaves == 0 || d.nt == 0) return;
  if (d.Gn == nullptr) throw invalid_argument("field-gradient buffers are not allocated");
  const int nm2 = d.p >= 2 ? coefficient_count(d.p - 2) : 0;
  if constexpr (sizeof(S) == 4) {
    const size_t lds_m = size_t(4) * 48 * std::max(d.p - 1, 1) * sizeof(float) + size_t(nm2) * sizeof(int4) +
                         size_t(nm2) * 8 * sizeof(int);
    if (K % 32 == 0 && nm2 > 0 && d.grad_up != nullptr && d.p2p_tile16_count > 0 && lds_m <= 65536) {
      const dim3 grid(unsigned((d.p2p_tile16_count + 3) / 4), unsigned(K / 32));
      l2p_grad_mfma_kernel<<<grid, 256, lds_m, s>>>(d, gradients, K, nm2, float(1.0 / d.potential_scale));
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_l2p_grad_columns<S>(d, gradients, K, s);
}

// Box GEMMs on the matrix cores (FP32 plans, K a multiple of 32): M2M, L2L,
// harmonic compression and expansion are products
//   out[r][k] (+)= sum_{dd < D} A[dd * lda + r] in[dd][k],   r < R,
// of a per-level operator A (depth-major, output row contiguous; rows
// lda..R-1 read as zero) with a box's coefficient block.  One workgroup per
// box (or parent) and 32 states: the block is staged in LDS as B[dd][48]
// (rows >= D zero; the 48-float stride keeps the four depth rows of a
// v_mfma_f32_16x16x4_f32 B fragment on distinct banks), and wave w owns the
// row tiles w + 4t for both 16-state column tiles, so each operator value it
// loads feeds two products.  Depth steps of 4 go in batches of 7 (21 and 42
// steps at p = 8), each batch's operand loads issued before its products, so
// a wave waits on the operator's L2 latency once per 28 depth rows; clamped
// unconditional loads, zero-selected past D and lda.
constexpr int kBoxLd = 48;

__device__ __forceinline__ void stage_box_mfma(float* __restrict__ Bl, const float* __restrict__ in, int D, int D4,
                                               int K) {
  for (int w = threadIdx.x; w < D4 * 8; w += 256) {
    const int dd = w >> 3, v = w & 7;
    float4 x = float4{0.0f, 0.0f, 0.0f, 0.0f};
    if (dd < D) x = *reinterpret_cast<const float4*>(in + int64_t(dd) * K + 4 * v);
    *reinterpret_cast<float4*>(Bl + dd * kBoxLd + 4 * v) = x;
  }
}

template <int RTW>
__device__ __forceinline__ void box_mfma_tiles(const float* __restrict__ A, int lda, int D, int RT,
                                               const float* __restrict__ Bl, int wave, int lane,
                                               f32x4 (&acc)[RTW][2]) {
  const int i = lane & 15, q = lane >> 4;
  constexpr int kBatch = 7;
  const int steps = (D + 3) / 4;
  for (int s0 = 0; s0 < steps; s0 += kBatch) {
    float a[kBatch][RTW], b[kBatch][2];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int dd = 4 * (s0 + u) + q;
      const bool dok = dd < D;
      const int ddc = dok ? dd : D - 1;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float v = Bl[(dok ? dd : 0) * kBoxLd + 16 * c + i];
        b[u][c] = dok ? v : 0.0f;
      }
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        const int row = (wave + 4 * t) * 16 + i;
        const bool ok = row < lda;
        const float v = A[int64_t(ddc) * lda + (ok ? row : 0)];
        a[u][t] = ok ? v : 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int t = 0; t < RTW; ++t)
        if (wave + 4 * t < RT)
#pragma unroll
          for (int c = 0; c < 2; ++c)
            acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][t], b[u][c], acc[t][c], 0, 0, 0);
  }
}

template <int RTW>
__device__ __forceinline__ void box_mfma_zero(f32x4 (&acc)[RTW][2]) {
#pragma unroll
  for (int t = 0; t < RTW; ++t) acc[t][0] = acc[t][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}

// The wave's accumulator tiles loaded from in[row][K] (rows [R), zero
// past R; in offset to the first state): the layout box_mfma_store writes.
template <int RTW>
__device__ __forceinline__ void box_mfma_load(const float* __restrict__ in, int R, int RT, int K, int wave, int lane,
                                              f32x4 (&acc)[RTW][2]) {
  const int i = lane & 15, q = lane >> 4;
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (wave + 4 * t) * 16 + 4 * q + r;
      const bool ok = wave + 4 * t < RT && row < R;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float v = in[int64_t(ok ? row : 0) * K + 16 * c + i];
        acc[t][c][r] = ok ? v : 0.0f;
      }
    }
  }
}

// Rows [R) of the wave's tiles to out[row][K] (out offset to the first state).
template <int RTW, bool kAdd>
__device__ __forceinline__ void box_mfma_store(float* __restrict__ out, int R, int RT, int K, int wave, int lane,
                                               const f32x4 (&acc)[RTW][2]) {
  const int i = lane & 15, q = lane >> 4;
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    if (wave + 4 * t >= RT) break;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (wave + 4 * t) * 16 + 4 * q + r;
      if (row >= R) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float* o = out + int64_t(row) * K + 16 * c + i;
        if constexpr (kAdd)
          *o += acc[t][c][r];
        else
          *o = acc[t][c][r];
      }
    }
  }
}

// The same products on three-piece bf16 operands (FP32 harmonic plans):
// v_mfma_f32_16x16x32_bf16, six piece products per term (see
// bf16_split.hpp), 32 depth rows per step.  The operator comes pre-split
// (box_x3_elems layout: a lane's A fragment is 8 consecutive depth values of
// one row, one 16-byte load per piece).  The box's block is split while it
// is staged, as Bx[piece][state column][x3_ld(S)] with the depth
// contiguous; rows past D are zero.
__host__ __device__ inline int x3_ld(int steps) { return steps * 32 + 8; }  // +8: fragment rows spread over the banks

// A block of S steps is S * 128 items of 8 depth values.  Held in registers
// (M2M, where the depth is the row count and so at most 192 rows, 6 steps),
// that is at most 3 items per thread.
constexpr int kStageItems = 3;
constexpr int kStageSteps = kStageItems * 2;

// The thread's items of one block in[depth][K] (depth rows [D), zero past
// D, S <= kStageSteps), held in registers so that the loads can be in flight
// during products.
__device__ __forceinline__ void load_box_x3(float (&x)[kStageItems][8], const float* __restrict__ in, int D, int S,
                                            int K) {
#pragma unroll
  for (int u = 0; u < kStageItems; ++u) {
    const int w = int(threadIdx.x) + 256 * u;
    if (w >= S * 128) break;
    const int col = w & 31, d8 = w >> 5;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int dd = 8 * d8 + e;
      x[u][e] = dd < D ? in[int64_t(dd) * K + col] : 0.0f;
    }
  }
}

// The items split and written as Bx[piece][state column][x3_ld(S)].
__device__ __forceinline__ void store_box_x3(uint16_t* __restrict__ Bx, const float (&x)[kStageItems][8], int S) {
  const int ld = x3_ld(S);
#pragma unroll
  for (int u = 0; u < kStageItems; ++u) {
    const int w = int(threadIdx.x) + 256 * u;
    if (w >= S * 128) break;
    const int col = w & 31, d8 = w >> 5;
    uint4 h, m, l;
    split3_bf16(x[u], h, m, l);
    uint16_t* o = Bx + col * ld + 8 * d8;
    *reinterpret_cast<uint4*>(o) = h;
    *reinterpret_cast<uint4*>(o + 32 * ld) = m;
    *reinterpret_cast<uint4*>(o + 64 * ld) = l;
  }
}

// Any depth: the items loaded, split and written in turn.
__device__ __forceinline__ void stage_box_x3(uint16_t* __restrict__ Bx, const float* __restrict__ in, int D, int S,
                                             int K) {
  const int ld = x3_ld(S);
  for (int w = threadIdx.x; w < S * 4 * 32; w += 256) {
    const int col = w & 31, d8 = w >> 5;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int dd = 8 * d8 + e;
      x[e] = dd < D ? in[int64_t(dd) * K + col] : 0.0f;
    }
    uint4 h, m, l;
    split3_bf16(x, h, m, l);
    uint16_t* o = Bx + col * ld + 8 * d8;
    *reinterpret_cast<uint4*>(o) = h;
    *reinterpret_cast<uint4*>(o + 32 * ld) = m;
    *reinterpret_cast<uint4*>(o + 64 * ld) = l;
  }
}

// The wave's A fragments of step s (row tiles wave + 4t, three pieces).
template <int RTW>
__device__ __forceinline__ void box_x3_load_a(const uint16_t* __restrict__ A, int s, int RP, int RT, int64_t piece,
                                              int wave, int i, int kq, uint4 (&a)[RTW][3]) {
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    if (wave + 4 * t >= RT) break;
    const uint16_t* a0 = A + (int64_t(s) * RP + (wave + 4 * t) * 16 + i) * 32 + 8 * kq;
#pragma unroll
    for (int p = 0; p < 3; ++p) a[t][p] = *reinterpret_cast<const uint4*>(a0 + p * piece);
  }
}

template <int RTW>
__device__ __forceinline__ void box_x3_step(const uint16_t* __restrict__ Bx, int s, int ld, int RT, int wave, int i,
                                            int kq, const uint4 (&a)[RTW][3], f32x4 (&acc)[RTW][2]) {
  uint4 b[3][2];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      b[p][c] = *reinterpret_cast<const uint4*>(Bx + (p * 32 + 16 * c + i) * ld + 32 * s + 8 * kq);
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    if (wave + 4 * t >= RT) break;
    // The six piece products whose orders sum to at most 2, smallest first.
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc[t][c] = mfma_bf16(a[t][1], b[1][c], acc[t][c]);
      acc[t][c] = mfma_bf16(a[t][2], b[0][c], acc[t][c]);
      acc[t][c] = mfma_bf16(a[t][0], b[2][c], acc[t][c]);
      acc[t][c] = mfma_bf16(a[t][1], b[0][c], acc[t][c]);
      acc[t][c] = mfma_bf16(a[t][0], b[1][c], acc[t][c]);
      acc[t][c] = mfma_bf16(a[t][0], b[0][c], acc[t][c]);
    }
  }
}

// With at most two row tiles per wave the operator's fragments of step
// s + 1 are loaded before the products of step s, so their latency is hidden
// where few workgroups run (the upper M2M and L2L levels: 0.07 -> 0.03 ms at
// p = 8, K = 32); three tiles keep one set, whose registers would otherwise
// cost the launch occupancy.
template <int RTW>
__device__ __forceinline__ void box_x3_tiles(const uint16_t* __restrict__ A, int R, int D, const uint16_t* __restrict__ Bx,
                                             int wave, int lane, f32x4 (&acc)[RTW][2]) {
  const int i = lane & 15, kq = lane >> 4, S = (D + 31) / 32, RP = (R + 15) / 16 * 16, RT = RP / 16, ld = x3_ld(S);
  const int64_t piece = int64_t(S) * RP * 32;
  if constexpr (RTW <= 2) {
    uint4 a[RTW][3];
    box_x3_load_a<RTW>(A, 0, RP, RT, piece, wave, i, kq, a);
#pragma unroll 1
    for (int s = 0; s < S; ++s) {
      uint4 an[RTW][3];
      const bool more = s + 1 < S;
      if (more) box_x3_load_a<RTW>(A, s + 1, RP, RT, piece, wave, i, kq, an);
      box_x3_step<RTW>(Bx, s, ld, RT, wave, i, kq, a, acc);
      if (!more) break;
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        if (wave + 4 * t >= RT) break;
#pragma unroll
        for (int p = 0; p < 3; ++p) a[t][p] = an[t][p];
      }
    }
  } else {
    // One tile's fragments at a time.
    for (int s = 0; s < S; ++s) {
      uint4 b[3][2];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          b[p][c] = *reinterpret_cast<const uint4*>(Bx + (p * 32 + 16 * c + i) * ld + 32 * s + 8 * kq);
#pragma unroll
      for (int t = 0; t < RTW; ++t) {
        if (wave + 4 * t >= RT) break;
        const uint16_t* a0 = A + (int64_t(s) * RP + (wave + 4 * t) * 16 + i) * 32 + 8 * kq;
        const uint4 ah = *reinterpret_cast<const uint4*>(a0);
        const uint4 am = *reinterpret_cast<const uint4*>(a0 + piece);
        const uint4 al = *reinterpret_cast<const uint4*>(a0 + 2 * piece);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          acc[t][c] = mfma_bf16(am, b[1][c], acc[t][c]);
          acc[t][c] = mfma_bf16(al, b[0][c], acc[t][c]);
          acc[t][c] = mfma_bf16(ah, b[2][c], acc[t][c]);
          acc[t][c] = mfma_bf16(am, b[0][c], acc[t][c]);
          acc[t][c] = mfma_bf16(ah, b[1][c], acc[t][c]);
          acc[t][c] = mfma_bf16(ah, b[0][c], acc[t][c]);
        }
      }
    }
  }
}

// Single-box products (harmonic compression, expansion): out = A in.
template <int RTW, bool kX3>
__global__ void __launch_bounds__(256)
box_mfma_kernel(const void* __restrict__ A, int lda, int R, int D,
                                                       const float* __restrict__ in, int64_t in_stride,
                                                       float* __restrict__ out, int64_t out_stride, int K,
                                                       const uint32_t* __restrict__ bits, int64_t node0, bool zeros) {
  extern __shared__ __align__(16) float box_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  // A box without points: its compressed multipole is zero, its local unread
  // (2^20 points in blobs, depth 6, 32 states: with the P2M, L2L and operand
  // split alike 66.3 -> 61.7 ms per evaluate).
  if (bits != nullptr && !bit_of(bits, node0 + blockIdx.x)) {
    float* o = out + int64_t(blockIdx.x) * out_stride + int(blockIdx.y) * 32;
    if (zeros)
      for (int w = threadIdx.x; w < R * 32; w += 256) o[int64_t(w >> 5) * K + (w & 31)] = 0.0f;
    return;
  }
  const int kc0 = int(blockIdx.y) * 32, D4 = (D + 3) / 4 * 4, RT = (R + 15) / 16;
  f32x4 acc[RTW][2];
  box_mfma_zero<RTW>(acc);
  if constexpr (kX3) {
    uint16_t* Bx = reinterpret_cast<uint16_t*>(box_lds);
    stage_box_x3(Bx, in + int64_t(blockIdx.x) * in_stride + kc0, D, (D + 31) / 32, K);
    __syncthreads();
    box_x3_tiles<RTW>(static_cast<const uint16_t*>(A), R, D, Bx, wave, lane, acc);
  } else {
    stage_box_mfma(box_lds, in + int64_t(blockIdx.x) * in_stride + kc0, D, D4, K);
    __syncthreads();
    box_mfma_tiles<RTW>(static_cast<const float*>(A), lda, D, RT, box_lds, wave, lane, acc);
  }
  box_mfma_store<RTW, false>(out + int64_t(blockIdx.x) * out_stride + kc0, R, RT, K, wave, lane, acc);
}

// M2M: parent (n coefficients) = sum over its 8 children c of T_c child.
template <int RTW, bool kX3>
__global__ void __launch_bounds__(256)
m2m_mfma_kernel(const DevicePlan d, int level, int K) {
  extern __shared__ __align__(16) float box_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int n = d.n, NP = round_up(n, 8), D4 = (n + 3) / 4 * 4, RT = (n + 15) / 16;
  const int kc0 = int(blockIdx.y) * 32;
  const int64_t parent = blockIdx.x, cnode0 = level_offset(level + 1) + parent * 8;
  const float* M = static_cast<const float*>(d.M) + kc0;
  f32x4 acc[RTW][2];
  box_mfma_zero<RTW>(acc);
  if constexpr (kX3) {
    // The next child's block is loaded into registers during this child's
    // products, and split into LDS after them.
    uint16_t* Bx = reinterpret_cast<uint16_t*>(box_lds);
    const int S = (n + 31) / 32;
    float x[kStageItems][8];
    load_box_x3(x, M + cnode0 * int64_t(n) * K, n, S, K);
    for (int c = 0; c < 8; ++c) {
      __syncthreads();
      store_box_x3(Bx, x, S);
      if (c + 1 < 8) load_box_x3(x, M + (cnode0 + c + 1) * int64_t(n) * K, n, S, K);
      __syncthreads();
      const uint16_t* A = static_cast<const uint16_t*>(d.m2m_x3) + ((level + 1) * 8 + c) * box_x3_elems(n, n);
      box_x3_tiles<RTW>(A, n, n, Bx, wave, lane, acc);
    }
  } else {
    for (int c = 0; c < 8; ++c) {
      __syncthreads();
      stage_box_mfma(box_lds, M + (cnode0 + c) * int64_t(n) * K, n, D4, K);
      __syncthreads();
      box_mfma_tiles<RTW>(shift_operator<float>(d.m2m_dense, level + 1, c, n, NP), NP, n, RT, box_lds, wave, lane,
                          acc);
    }
  }
  box_mfma_store<RTW, false>(static_cast<float*>(d.M) + (level_offset(level) + parent) * int64_t(n) * K + kc0, n, RT,
                             K, wave, lane, acc);
}

// L2L: child c += T_c parent, for the 8 children of one parent.
template <int RTW, bool kX3>
__global__ void __launch_bounds__(256)
l2l_mfma_kernel(const DevicePlan d, int child_level, int K) {
  extern __shared__ __align__(16) float box_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int n = d.n, NP = round_up(n, 8), D4 = (n + 3) / 4 * 4, RT = (n + 15) / 16;
  const int kc0 = int(blockIdx.y) * 32;
  const int64_t parent = blockIdx.x, child0 = level_offset(child_level) + parent * 8;
  uint32_t wanted = 0xffu;  // the children with targets
  if (d.target_bits != nullptr) {
    wanted = 0;
    for (int c = 0; c < 8; ++c) wanted |= uint32_t(bit_of(d.target_bits, child0 + c)) << c;
    if (wanted == 0) return;
  }
  float* Lc = static_cast<float*>(d.Lc) + kc0;
  uint16_t* Bx = reinterpret_cast<uint16_t*>(box_lds);
  if constexpr (kX3)
    stage_box_x3(Bx, Lc + (level_offset(child_level - 1) + parent) * int64_t(n) * K, n, (n + 31) / 32, K);
  else
    stage_box_mfma(box_lds, Lc + (level_offset(child_level - 1) + parent) * int64_t(n) * K, n, D4, K);
  __syncthreads();
  // The child's own local (from the M2L) is the accumulators' start, and the
  // next child's is loaded during this child's products.
  f32x4 next[RTW][2];
  box_mfma_load<RTW>(Lc + child0 * int64_t(n) * K, n, RT, K, wave, lane, next);
  for (int c = 0; c < 8; ++c) {
    const int64_t child = child0 + c;
    f32x4 acc[RTW][2];
#pragma unroll
    for (int t = 0; t < RTW; ++t) acc[t][0] = next[t][0], acc[t][1] = next[t][1];
    if (c + 1 < 8) box_mfma_load<RTW>(Lc + (child + 1) * int64_t(n) * K, n, RT, K, wave, lane, next);
    if (((wanted >> c) & 1u) == 0) continue;
    if constexpr (kX3)
      box_x3_tiles<RTW>(static_cast<const uint16_t*>(d.l2l_x3) + (child_level * 8 + c) * box_x3_elems(n, n), n, n,
                        Bx, wave, lane, acc);
    else
      box_mfma_tiles<RTW>(shift_operator<float>(d.l2l_dense, child_level, c, n, NP), NP, n, RT, box_lds, wave, lane,
                          acc);
    box_mfma_store<RTW, false>(Lc + child * int64_t(n) * K, n, RT, K, wave, lane, acc);
  }
}

// Row tiles per wave of the box products (at most 12 row tiles), or 0
// where they do not apply.
inline int box_mfma_rtw(int R, int D, int K) {
  const int rtw = ((R + 15) / 16 + 3) / 4;
  if (K % 32 != 0 || rtw > 3 || size_t((D + 3) / 4 * 4) * kBoxLd * sizeof(float) > 65536) return 0;
  return rtw;
}

// LDS bytes of a box staged for the three-piece products (depth D).
inline size_t box_x3_lds_bytes(int D) { return size_t(3) * 32 * x3_ld((D + 31) / 32) * sizeof(uint16_t); }

#define HIPFMM_BOX_RTW(rtw, launch) \
  switch (rtw) {                    \
    case 1: launch(1); break;       \
    case 2: launch(2); break;       \
    default: launch(3); break;      \
  }

template <class S>
void launch_m2m(const DevicePlan& d, int parent_level, int K, hipStream_t s) {
  if constexpr (sizeof(S) == 4) {
    if (const int rtw = box_mfma_rtw(d.n, d.n, K)) {
      const dim3 grid(unsigned(int64_t(1) << (3 * parent_level)), unsigned(K / 32));
      if (d.m2m_x3 != nullptr) {
        // The kernel holds a child's block in registers: n <= 192 rows
        // (rtw <= 3) is at most kStageSteps steps of depth.
        if ((d.n + 31) / 32 > kStageSteps) throw invalid_argument("M2M block deeper than its register staging");
        const size_t lds = box_x3_lds_bytes(d.n);
#define HIPFMM_M2M(R) m2m_mfma_kernel<R, true><<<grid, 256, lds, s>>>(d, parent_level, K)
        HIPFMM_BOX_RTW(rtw, HIPFMM_M2M)
#undef HIPFMM_M2M
      } else {
        const size_t lds = size_t((d.n + 3) / 4 * 4) * kBoxLd * sizeof(float);
#define HIPFMM_M2M(R) m2m_mfma_kernel<R, false><<<grid, 256, lds, s>>>(d, parent_level, K)
        HIPFMM_BOX_RTW(rtw, HIPFMM_M2M)
#undef HIPFMM_M2M
      }
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_m2m_columns<S>(d, parent_level, K, s);
}

template <class S>
void launch_l2l(const DevicePlan& d, int child_level, int K, hipStream_t s) {
  if constexpr (sizeof(S) == 4) {
    if (const int rtw = box_mfma_rtw(d.n, d.n, K)) {
      const dim3 grid(unsigned(int64_t(1) << (3 * (child_level - 1))), unsigned(K / 32));
      if (d.l2l_x3 != nullptr) {
        const size_t lds = box_x3_lds_bytes(d.n);
#define HIPFMM_L2L(R) l2l_mfma_kernel<R, true><<<grid, 256, lds, s>>>(d, child_level, K)
        HIPFMM_BOX_RTW(rtw, HIPFMM_L2L)
#undef HIPFMM_L2L
      } else {
        const size_t lds = size_t((d.n + 3) / 4 * 4) * kBoxLd * sizeof(float);
#define HIPFMM_L2L(R) l2l_mfma_kernel<R, false><<<grid, 256, lds, s>>>(d, child_level, K)
        HIPFMM_BOX_RTW(rtw, HIPFMM_L2L)
#undef HIPFMM_L2L
      }
      HIPFMM_CHECK(hipGetLastError());
      return;
    }
  }
  launch_l2l_columns<S>(d, child_level, K, s);
}

template <class S>
void launch_l2p_unsort(const DevicePlan& d, S* fields, S* potentials, int K, hipStream_t s) {
  if (d.leaves == 0 || d.nt == 0) return;
  const bool pot = potentials != nullptr;
  if (!pot && fields == nullptr) throw invalid_argument("no output requested");
  if (pot && d.Pn == nullptr) throw invalid_argument("near-field potential buffer is not allocated");
  if constexpr (sizeof(S) == 4) {
    const int NM = pot ? d.n : d.nm;
    const size_t lds = size_t(4) * 48 * (d.p + 1) * sizeof(float) + size_t(NM + d.nm) * sizeof(int4);
    if (K % 32 == 0 && d.l2p_up != nullptr && d.p2p_tile16_count > 0 && lds <= 65536) {
      const dim3 grid(unsigned((d.p2p_tile16_count + 3) / 4), unsigned(K / 32));
      // Fields only, whole 64-point tiles: the totals stay sorted and one
      // coalesced pass unsorts them (a direct unsort writes 12-byte pieces
      // of 32 rows per target).
      const bool sorted = d.nt % 64 == 0 && reinterpret_cast<uintptr_t>(fields) % 16 == 0 &&
                          reinterpret_cast<uintptr_t>(potentials) % 16 == 0 &&
                          size_t(64) * (3 * K + 4) * sizeof(float) <= 65536;
      if (pot && sorted)
        l2p_mfma_kernel<true, true><<<grid, 256, lds, s>>>(d, fields, potentials, K);
      else if (pot)
        l2p_mfma_kernel<true, false><<<grid, 256, lds, s>>>(d, fields, potentials, K);
      else if (sorted)
        l2p_mfma_kernel<false, true><<<grid, 256, lds, s>>>(d, fields, nullptr, K);
      else
        l2p_mfma_kernel<false, false><<<grid, 256, lds, s>>>(d, fields, nullptr, K);
      HIPFMM_CHECK(hipGetLastError());
      if (sorted && fields != nullptr) {
        scatter_fields_kernel<<<unsigned(d.nt / 64), kThreads, size_t(64) * (3 * K + 4) * sizeof(float), s>>>(
            static_cast<const float*>(d.Hn), d.tgt_inv, d.nt, K, fields);
        HIPFMM_CHECK(hipGetLastError());
      }
      if (sorted && pot) {
        scatter_potentials_kernel<<<unsigned(d.nt / 64), kThreads, size_t(64) * (K + 4) * sizeof(float), s>>>(
            static_cast<const float*>(d.Pn), d.tgt_inv, d.nt, K, potentials);
        HIPFMM_CHECK(hipGetLastError());
      }
      return;
    }
  }
  launch_l2p_columns<S>(d, fields, potentials, K, s);
}

template <class S>
void launch_m2l_compress(const DevicePlan& d, int K, int first_level, hipStream_t s) {
  for (int level = std::max(first_level, 2); level <= d.L; ++level) {
    if constexpr (sizeof(S) == 4) {
      if (const int rtw = box_mfma_rtw(d.nc, d.n, K)) {
        const dim3 g2(unsigned(int64_t(1) << (3 * level)), unsigned(K / 32));
        const int64_t node0 = level_offset(level);
        const float* in = static_cast<const float*>(d.M) + node0 * d.n * K;
        float* out = static_cast<float*>(d.Mc) + node0 * d.nc * K;
        if (d.cmp_x3 != nullptr) {
          const size_t l2 = box_x3_lds_bytes(d.n);
          const uint16_t* A = static_cast<const uint16_t*>(d.cmp_x3) + level * box_x3_elems(d.nc, d.n);
#define HIPFMM_CMP(R) box_mfma_kernel<R, true><<<g2, 256, l2, s>>>(A, 0, d.nc, d.n, in, int64_t(d.n) * K, out, \
                                                                    int64_t(d.nc) * K, K, d.source_bits, node0, true)
          HIPFMM_BOX_RTW(rtw, HIPFMM_CMP)
#undef HIPFMM_CMP
        } else {
          const size_t l2 = size_t((d.n + 3) / 4 * 4) * kBoxLd * sizeof(float);
          const int NPc = round_up(d.nc, 16);
          const float* A = static_cast<const float*>(d.cmp_op) + size_t(level) * d.n * NPc;
#define HIPFMM_CMP(R) box_mfma_kernel<R, false><<<g2, 256, l2, s>>>(A, NPc, d.nc, d.n, in, int64_t(d.n) * K, out, \
                                                                     int64_t(d.nc) * K, K, d.source_bits, node0, true)
          HIPFMM_BOX_RTW(rtw, HIPFMM_CMP)
#undef HIPFMM_CMP
        }
        HIPFMM_CHECK(hipGetLastError());
        continue;
      }
    }
    launch_compress_columns<S>(d, level, K, s);
  }
}

template <class S>
void launch_m2l_expand(const DevicePlan& d, int K, int first_level, hipStream_t s) {
  for (int level = std::max(first_level, 2); level <= d.L; ++level) {
    if constexpr (sizeof(S) == 4) {
      if (const int rtw = box_mfma_rtw(d.n, d.nc, K)) {
        const dim3 g2(unsigned(int64_t(1) << (3 * level)), unsigned(K / 32));
        const int64_t node0 = level_offset(level);
        const float* in = static_cast<const float*>(d.Lcc) + node0 * d.nc * K;
        float* out = static_cast<float*>(d.Lc) + node0 * d.n * K;
        if (d.exp_x3 != nullptr) {
          const size_t l2 = box_x3_lds_bytes(d.nc);
          const uint16_t* A = static_cast<const uint16_t*>(d.exp_x3) + level * box_x3_elems(d.n, d.nc);
#define HIPFMM_EXP(R) box_mfma_kernel<R, true><<<g2, 256, l2, s>>>(A, 0, d.n, d.nc, in, int64_t(d.nc) * K, out, \
                                                                    int64_t(d.n) * K, K, d.target_bits, node0, false)
          HIPFMM_BOX_RTW(rtw, HIPFMM_EXP)
#undef HIPFMM_EXP
        } else {
          const size_t l2 = size_t((d.nc + 3) / 4 * 4) * kBoxLd * sizeof(float);
          const int NP = round_up(d.n, 8);
          const float* A = static_cast<const float*>(d.exp_op) + size_t(level) * d.nc * NP;
#define HIPFMM_EXP(R) box_mfma_kernel<R, false><<<g2, 256, l2, s>>>(A, NP, d.n, d.nc, in, int64_t(d.nc) * K, out, \
                                                                     int64_t(d.n) * K, K, d.target_bits, node0, false)
          HIPFMM_BOX_RTW(rtw, HIPFMM_EXP)
#undef HIPFMM_EXP
        }
        HIPFMM_CHECK(hipGetLastError());
        continue;
      }
    }
    launch_expand_columns<S>(d, level, K, s);
  }
}

template <class S>
void launch_zero(S* ptr, size_t count, hipStream_t s) {
  if (count == 0) return;
  const unsigned blocks = unsigned(std::min<size_t>((count + kThreads - 1) / kThreads, 65536));
  zero_kernel<S><<<blocks, kThreads, 0, s>>>(ptr, count);
  HIPFMM_CHECK(hipGetLastError());
}

#define HIPFMM_INSTANTIATE(S)                                                       \
  template void launch_gather<S>(const DevicePlan&, const S*, S, int, hipStream_t); \
  template void launch_p2m<S>(const DevicePlan&, int, hipStream_t);                \
  template void launch_m2m<S>(const DevicePlan&, int, int, hipStream_t);           \
  template void launch_l2l<S>(const DevicePlan&, int, int, hipStream_t);           \
  template void launch_l2p_unsort<S>(const DevicePlan&, S*, S*, int, hipStream_t);     \
  template void launch_l2p_grad_unsort<S>(const DevicePlan&, S*, int, hipStream_t);    \
  template void launch_m2l_compress<S>(const DevicePlan&, int, int, hipStream_t); \
  template void launch_m2l_expand<S>(const DevicePlan&, int, int, hipStream_t);    \
  template void launch_zero<S>(S*, size_t, hipStream_t);
HIPFMM_INSTANTIATE(float)
HIPFMM_INSTANTIATE(double)
#undef HIPFMM_INSTANTIATE

}  // namespace hipfmm
