// Far-field box kernels for any number of moment states, FP32 and FP64: P2M,
// the shift and transform products (M2M, L2L, harmonic compression and
// expansion) and L2P (fields, potentials, field gradients), on the
// full-precision matrix instructions (v_mfma_f32_16x16x4_f32 and
// v_mfma_f64_16x16x4_f64: FMA chains in the type's own precision).  They serve
// FP64 plans, and FP32 plans whose state count is no multiple of 32 (those
// take the three-piece bf16 kernels of far.hip).
//
// A product's 16 columns are whatever shares the operator: the (box, state)
// pairs of a level for the shift and transform products, the (component,
// state) pairs of a leaf for P2M and L2P.  So one state fills the columns as
// well as 32 do.  What bounds them is latency: the products are a few us of
// matrix-core time per level.
//
// Measured (us; in brackets the forms before them on the vector ALUs, one
// workgroup per box): FP32, 2^20 points, p = 6, depth 5, one state, P2M 100
// (1400, both beside the near field), L2P 88 (390), M2M and L2L levels 6-19
// (62-167), compression 40 (199), expansion 19 (97); FP64, 2^18 points, p = 8,
// depth 4, L2P 59 (682), L2L 16-18 (320).  131,075 points, p = 8, 20 states:
// P2M 103 (1870), L2P and unsort 102 (353).
// Where many boxes hold no points, workgroups of empty boxes end at once
// (262,144 points of a slab, p = 6, one state: compression 18 -> 8, the pass of
// four evaluates 1218 -> 1136).
//
// Reference operations restated here:
//   P2M   M_a = (-1)^|a| sum_j sum_{c: a_c>0} m_jc d_j^(a-e_c)/(a-e_c)!
//         src/static_operators.cpp:186-220, src/operators.cpp:16-52
//   M2M / L2L  shared per-(level, class) shift operators
//         src/static_operators.cpp:257-298, src/far_field.cpp:395-446, :555-574
//   L2P   H_c = -sum_{b: b_c>0} L_b dx^(b-e_c)/(b-e_c)!
//         src/static_operators.cpp:300-335
//   combine + unsort  src/cuda_fmm.cu:503-516, src/uniform_fmm.cpp:1439-1452
#include "common.hpp"

#include <type_traits>

namespace hipfmm {

namespace {

// 16 x 16 += (16 x 4)(4 x 16).  Lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; register r of the accumulator holds column l % 16 of
// row row(l / 16, r).
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

// How a box's coefficients lie: rows row values apart, states state apart.
struct Strides {
  uint32_t row, state;
};
// [coefficient][K], or (state_major) [K][count].
inline Strides strides(bool state_major, int K, int count) {
  return state_major ? Strides{1u, uint32_t(count)} : Strides{uint32_t(K), 1u};
}

// out[row][col] (+)= sum over segments g and depth d of A_g[d][row] in_g[d][col]
// with the columns col = (box, state): in_g[d][col] = in[box * in_box +
// g * in_seg + d * in_at.row + state * in_at.state], out likewise,
// A_g = A + g * a_seg.  blockIdx.z offsets A and out by a_z and out_z (the 8
// children of the L2L).
template <class S>
struct Product {
  const S* A;
  int64_t a_seg, a_z;
  int lda, R, D, segments;
  const S* in;
  int64_t in_box, in_seg;
  Strides in_at;
  S* out;
  int64_t out_box, out_z;
  Strides out_at;
  int K;
  int64_t cols;
  // Where bits is set, a workgroup none of whose boxes has a point (node bit0 +
  // box bit_box + blockIdx.z) stores zeros, or nothing (idle_stores).
  const uint32_t* bits;
  int64_t bit0;
  int bit_box;
  bool idle_stores;
  int row_waves;  // waves side by side over the rows; blockDim / 64 / row_waves groups share the segments
  bool add;
};

// base[bytes / sizeof(S)] as a uniform base plus a 32-bit lane offset.
template <class S>
__device__ __forceinline__ S load_at(const S* base, uint32_t bytes) {
  return *reinterpret_cast<const S*>(reinterpret_cast<const unsigned char*>(base) + bytes);
}

// One wave: RTW row tiles x CT column tiles.  The operator comes from L2 (a
// 64 B row piece per depth value), the columns straight from memory through
// L1; a batch of kU steps' loads is issued before its products.  The groups'
// sums over their segments meet in LDS.
template <class S, int RTW, int CT>
__global__ void __launch_bounds__(1024) product_kernel(const Product<S> p) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using M = Mma<S>;
  constexpr int kU = 7;  // steps per batch: 1, 2, 3 and 6 batches for 25, 49 to 56, 81 to 84 and 165 coefficients
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const int rw = wave % p.row_waves, group = wave / p.row_waves, groups = int(blockDim.x >> 6) / p.row_waves;
  // Columns relative to the workgroup's first box, so that every address is
  // a uniform base plus a 32-bit lane offset.
  const int64_t first = int64_t(blockIdx.x) * (16 * CT), box0 = first / p.K;
  const uint32_t K = uint32_t(p.K), rem = uint32_t(first - box0 * p.K);
  const uint32_t left = uint32_t(min(p.cols - first, int64_t(16 * CT)));  // columns of this workgroup
  bool idle = false;  // the same for every wave
  if (p.bits != nullptr) {
    const uint32_t last = (rem + left - 1) / K;  // at most 16 CT boxes
    idle = __any(uint32_t(lane) <= last &&
                 bit_of(p.bits, p.bit0 + (box0 + lane) * p.bit_box + int64_t(blockIdx.z))) == 0;
    if (idle && !p.idle_stores) return;
  }
  const S* in = p.in + box0 * p.in_box;
  S* out = p.out + box0 * p.out_box + int64_t(blockIdx.z) * p.out_z;
  uint32_t in_at[CT], out_at[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const uint32_t x = rem + min(uint32_t(16 * c + i), left - 1), box = x / K, k = x - box * K;
    in_at[c] = (box * uint32_t(p.in_box) + k * p.in_at.state) * uint32_t(sizeof(S));
    out_at[c] = box * uint32_t(p.out_box) + k * p.out_at.state;
  }
  const uint32_t a_step = uint32_t(p.lda) * uint32_t(sizeof(S)), b_step = p.in_at.row * uint32_t(sizeof(S));  // per depth value
  uint32_t row[RTW];
#pragma unroll
  for (int t = 0; t < RTW; ++t)
    row[t] = uint32_t(min((rw * RTW + t) * 16 + i, p.lda - 1)) * uint32_t(sizeof(S));
  typename M::Acc acc[RTW][CT];
#pragma unroll
  for (int t = 0; t < RTW; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = typename M::Acc{};
  const int per_group = p.segments / groups;
  const int batches = idle ? 0 : (p.D + 4 * kU - 1) / (4 * kU);
  for (int g = group * per_group; g < (group + 1) * per_group; ++g) {
    const S* A = p.A + int64_t(blockIdx.z) * p.a_z + g * p.a_seg;
    const int64_t seg = g * p.in_seg;
    for (int n = 0; n < batches; ++n) {
      const int d0 = 4 * kU * n;
      S a[kU][RTW], b[kU][CT];
      if (n + 1 < batches) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
#pragma unroll
          for (int t = 0; t < RTW; ++t) a[u][t] = load_at(A + int64_t(d0 + 4 * u) * p.lda, uint32_t(q) * a_step + row[t]);
#pragma unroll
          for (int c = 0; c < CT; ++c)
            b[u][c] = load_at(in + seg + int64_t(d0 + 4 * u) * p.in_at.row, uint32_t(q) * b_step + in_at[c]);
        }
      } else {  // the last batch: depth values past D read the last one, times zero
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int d = d0 + 4 * u + q, dc = min(d, p.D - 1);
#pragma unroll
          for (int t = 0; t < RTW; ++t) a[u][t] = load_at(A, uint32_t(dc) * a_step + row[t]);
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            const S v = load_at(in + seg, uint32_t(dc) * b_step + in_at[c]);
            b[u][c] = d < p.D ? v : S(0);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int t = 0; t < RTW; ++t)
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[t][c] = M::mul(a[u][t], b[u][c], acc[t][c]);
    }
  }
  if (groups > 1) {  // [group - 1][row wave][t][c][r][lane]
    S* part = reinterpret_cast<S*>(smem_raw);
    constexpr int per_wave = RTW * CT * 4 * 64;
    if (group > 0) {
      S* o = part + int64_t((group - 1) * p.row_waves + rw) * per_wave + lane;
#pragma unroll
      for (int t = 0; t < RTW; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[((t * CT + c) * 4 + r) * 64] = acc[t][c][r];
    }
    __syncthreads();
    if (group > 0) return;
    for (int g = 1; g < groups; ++g) {
      const S* o = part + int64_t((g - 1) * p.row_waves + rw) * per_wave + lane;
#pragma unroll
      for (int t = 0; t < RTW; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][c][r] += o[((t * CT + c) * 4 + r) * 64];
    }
  }
#pragma unroll
  for (int t = 0; t < RTW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int orow = (rw * RTW + t) * 16 + M::row(q, r);
      if (orow >= p.R) continue;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (uint32_t(16 * c + i) >= left) continue;
        S* o = out + uint32_t(orow) * p.out_at.row + out_at[c];
        *o = p.add ? *o + acc[t][c][r] : acc[t][c][r];
      }
    }
}

// Launch shape: one row tile per wave up to 12 row tiles (p <= 8), two above;
// two column tiles per wave where that still leaves two workgroups per CU,
// one below; on a small level the segments (M2M children) are shared by as
// many groups as 16 waves allow, which cuts its serial chain to an eighth to a
// half.  Above 64 workgroups the chain no longer counts, and workgroups of 16
// waves wait for room beside the near field (level 4 at one state: 0.66 ms).
template <class S>
void launch_product(Product<S> p, int z, hipStream_t s) {
  if (p.cols <= 0 || p.R <= 0) return;
  const int tiles = (p.R + 15) / 16, rtw = tiles <= 12 ? 1 : 2;
  p.row_waves = (tiles + rtw - 1) / rtw;
  int groups = 1;
  if (p.cols <= 1024)
    while (groups * 2 <= p.segments && groups * 2 * p.row_waves <= 16) groups *= 2;
  const bool wide = rtw == 1 && (p.cols + 31) / 32 * z >= 512;
  const int ct = wide ? 2 : 1;
  const dim3 grid(unsigned((p.cols + 16 * ct - 1) / (16 * ct)), 1, unsigned(z));
  const unsigned threads = unsigned(64 * p.row_waves * groups);
  const size_t lds = size_t(groups - 1) * p.row_waves * rtw * ct * 256 * sizeof(S);
  if (wide)
    product_kernel<S, 1, 2><<<grid, threads, lds, s>>>(p);
  else if (rtw == 1)
    product_kernel<S, 1, 1><<<grid, threads, lds, s>>>(p);
  else
    product_kernel<S, 2, 1><<<grid, threads, lds, s>>>(p);
  HIPFMM_CHECK(hipGetLastError());
}

inline int round_to(int x, int m) { return (x + m - 1) / m * m; }

// P2M.  With g = alpha - e_c,
//   M[alpha][k] = (-1)^|alpha| sum_{c: alpha_c > 0} C_c[alpha - e_c][k],
//   C_c[g][k]   = sum_s mono_g(d_s) m[s][c][k]        (|g| < p),
// one workgroup (4 waves) per leaf and KC states: rows g, columns (c, state),
// depth the leaf's sources.  Wave w owns row tiles w, w + 4, ..; a lane forms
// its monomial from three axis powers in LDS for all CT column tiles.  The
// C_c meet in LDS, where the sign-and-shift combination writes M.
constexpr int kChunk = 64;  // sources whose axis powers are in LDS at a time

template <class S, int RTW, int CT>
__global__ void __launch_bounds__(256) p2m_columns_kernel(const DevicePlan d, int K, int KC) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using M = Mma<S>;
  const int n = d.n, nm = d.nm, PW = d.p;
  const int NMP = (nm + 15) / 16 * 16;
  S* pw = reinterpret_cast<S*>(smem_raw);  // [source][axis][power]
  S* Cl = pw + kChunk * 3 * PW;            // [(c, state)][g]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i = lane & 15, q = lane >> 4;
  const int leaf = blockIdx.x, k0 = int(blockIdx.y) * KC, KCn = min(KC, K - k0);
  const int2 range = d.leaf_src[leaf];
  S* Mout = static_cast<S*>(d.M) + (level_offset(d.L) + leaf) * int64_t(n) * K + k0;
  if (range.x == range.y) {
    for (int w = tid; w < n * KCn; w += 256) Mout[int64_t(w / KCn) * K + w % KCn] = S(0);
    return;
  }
  const auto* rel = static_cast<const typename Vec4<S>::type*>(d.src_rel);
  const S* sm = static_cast<const S*>(d.sm);
  int4 ex[RTW];
  bool row_ok[RTW];
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    const int g = (wave + 4 * t) * 16 + i;
    row_ok[t] = g < nm;
    ex[t] = row_ok[t] ? d.p2m_tab[n + g] : int4{0, 0, 0, 0};
  }
  int off[CT];  // of this lane's columns in a source's row of 3K moments
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int col = min(16 * c + i, 3 * KCn - 1);
    off[c] = col / KCn * K + k0 + col % KCn;
  }
  typename M::Acc acc[RTW][CT];
#pragma unroll
  for (int t = 0; t < RTW; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = typename M::Acc{};
  for (int j0 = range.x; j0 < range.y; j0 += kChunk) {
    const int cnt = min(kChunk, range.y - j0);
    __syncthreads();  // the previous chunk's powers are no longer read
    for (int w = tid; w < 3 * cnt; w += 256) {
      const int j = w / 3, a = w - 3 * j;
      const auto r = rel[j0 + j];
      const S x = a == 0 ? r.x : (a == 1 ? r.y : r.z);
      S v = S(1);
      S* o = pw + w * PW;
      o[0] = v;
      for (int e = 1; e < PW; ++e) {
        v = v * x / S(e);
        o[e] = v;
      }
    }
    __syncthreads();
    constexpr int kSteps = 4;  // 16 sources' loads before their products
    for (int s0 = 0; s0 < cnt; s0 += 4 * kSteps) {
      S b[kSteps][CT];
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const int j = s0 + 4 * u + q;
        const S* ms = sm + int64_t(j0 + min(j, cnt - 1)) * 3 * K;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const S v = ms[off[c]];
          b[u][c] = j < cnt ? v : S(0);
        }
      }
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const S* ps = pw + min(s0 + 4 * u + q, cnt - 1) * 3 * PW;
#pragma unroll
        for (int t = 0; t < RTW; ++t) {
          const S a = ps[ex[t].x] * ps[PW + ex[t].y] * ps[2 * PW + ex[t].z];
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[t][c] = M::mul(a, b[u][c], acc[t][c]);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < RTW; ++t) {
    if ((wave + 4 * t) * 16 >= nm) break;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) Cl[(16 * c + i) * NMP + (wave + 4 * t) * 16 + M::row(q, r)] = acc[t][c][r];
  }
  __syncthreads();
  for (int w = tid; w < n * KCn; w += 256) {
    const int a = w / KCn, k = w - a * KCn;
    const int4 e = d.p2m_tab[a];
    S v = S(0);
    if (e.x >= 0) v += Cl[k * NMP + e.x];
    if (e.y >= 0) v += Cl[(KCn + k) * NMP + e.y];
    if (e.z >= 0) v += Cl[(2 * KCn + k) * NMP + e.z];
    Mout[int64_t(a) * K + k] = e.w > 0 ? v : -v;
  }
}

enum L2pOutput { kField = 0, kFieldAndPotential = 1, kGradient = 2 };
constexpr int l2p_rows(int what) { return what == kGradient ? 6 : what == kFieldAndPotential ? 4 : 3; }

// L2P.  For 16 targets of one leaf (rows) and the columns (output row e,
// state): the sums over the monomials g of
//   mono_g(d_t) L[g + e_c][k]          (|g| < p)       fields
//   mono_b(d_t) L[b][k]                (|b| <= p)      potential
//   mono_g(d_t) L[g + e_c + e_j][k]    (|g| <= p - 2)  field gradient
// A lane's column fixes which raised row of the leaf local it reads (a table
// in LDS), so one operand of monomials serves every output.  One wave per
// tile, four per workgroup.  The totals H = Hn - sum, phi = W (Pn + sum),
// G = (Gn - sum) / W go to user order directly, or (kSorted) over the near
// field in sorted order for scatter_kernel.
template <class S, int kWhat, int CT>
__global__ void __launch_bounds__(256) l2p_columns_kernel(const DevicePlan d, S* __restrict__ out, S* __restrict__ pot,
                                                         int K, int KC, int NM, int PW, S scale, bool sorted) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using M = Mma<S>;
  constexpr int C = l2p_rows(kWhat), TW = kWhat == kGradient ? 8 : 4;  // outputs; table width
  const int n = d.n;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  int4* ex = reinterpret_cast<int4*>(smem_raw);       // exponents of the NM monomials
  int* up = reinterpret_cast<int*>(ex + NM);          // [g][TW] raised rows, -1: none
  S* pw = reinterpret_cast<S*>(up + NM * TW) + wave * (48 * PW);  // [target][axis][power]
  for (int w = threadIdx.x; w < NM; w += 256) ex[w] = d.p2m_tab[n + w];
  for (int w = threadIdx.x; w < NM * TW; w += 256) {
    const int g = w / TW, c = w % TW;
    if constexpr (kWhat == kGradient)
      up[w] = d.grad_up[w];
    else
      up[w] = c == 3 ? g : g < d.nm ? (c == 0 ? d.l2p_up[g].x : c == 1 ? d.l2p_up[g].y : d.l2p_up[g].z) : -1;
  }
  const int item = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x)) * 4 + wave;
  const bool valid = item < d.p2p_tile16_count;
  const int2 tile = valid ? d.p2p_tiles16[item] : int2{0, 0};
  const int2 range = valid ? d.leaf_tgt[tile.x] : int2{0, 0};
  const int t0 = range.x + tile.y, cnt = valid ? min(16, range.y - t0) : 0;
  const auto* rel = static_cast<const typename Vec4<S>::type*>(d.tgt_rel);
  if (lane < 48) {
    const int t = lane / 3, a = lane % 3;
    S x = S(0);
    if (t < cnt) {
      const auto r = rel[t0 + t];
      x = a == 0 ? r.x : (a == 1 ? r.y : r.z);
    }
    S v = S(1);
    pw[lane * PW] = v;
    for (int e = 1; e < PW; ++e) {
      v = v * x / S(e);
      pw[lane * PW + e] = v;
    }
  }
  __syncthreads();
  if (!valid) return;
  const S* pt = pw + i * 3 * PW;
  const int k0 = int(blockIdx.y) * KC, KCn = min(KC, K - k0);
  const S* L = static_cast<const S*>(d.Lc) + (level_offset(d.L) + tile.x) * int64_t(n) * K + k0;
  int comp[CT], state[CT];
  bool col_ok[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int col = 16 * c + i;
    col_ok[c] = col < C * KCn;
    const int cc = col_ok[c] ? col : 0;
    comp[c] = cc / KCn;
    state[c] = cc - comp[c] * KCn;
  }
  typename M::Acc acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = typename M::Acc{};
  constexpr int kSteps = 8;
  for (int g0 = 0; g0 < NM; g0 += 4 * kSteps) {
    S a[kSteps], b[kSteps][CT];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int g = g0 + 4 * u + q, gc = min(g, NM - 1);
      const int4 e = ex[gc];
      a[u] = pt[e.x] * pt[PW + e.y] * pt[2 * PW + e.z];
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int row = up[gc * TW + comp[c]];
        const S v = L[int64_t(max(row, 0)) * K + state[c]];
        b[u][c] = g < NM && row >= 0 ? v : S(0);
      }
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[c] = M::mul(a[u], b[u][c], acc[c]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int tl = M::row(q, r);
    if (tl >= cnt) continue;
    const int64_t t = t0 + tl;
    const int64_t user = sorted ? 0 : d.tgt_perm[t];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      if (!col_ok[c]) continue;
      const int e = comp[c];
      const int64_t k = k0 + state[c];
      if (kWhat == kFieldAndPotential && e == 3) {
        S* pn = static_cast<S*>(d.Pn) + t * K + k;
        const S v = scale * (*pn + acc[c][r]);
        if (sorted)
          *pn = v;
        else
          pot[k * d.nt + user] = v;
        continue;
      }
      if (kWhat == kFieldAndPotential && out == nullptr) continue;
      S* near = static_cast<S*>(kWhat == kGradient ? d.Gn : d.Hn) + (t * (kWhat == kGradient ? 6 : 3) + e) * K + k;
      const S v = kWhat == kGradient ? scale * (*near - acc[c][r]) : *near - acc[c][r];
      if (sorted)
        *near = v;
      else
        out[(k * d.nt + user) * (kWhat == kGradient ? 6 : 3) + e] = v;
    }
  }
}

// Sorted rows in[t][C][K] to the user layout out[k][user][C].  A workgroup
// owns `points` consecutive user points: each point's C K values are one
// contiguous read from its sorted slot into LDS, and each state's C * points
// values one contiguous write.
template <class S>
__global__ void __launch_bounds__(256) scatter_kernel(const S* __restrict__ in, const int* __restrict__ inv, int nt,
                                                      int K, int C, int points, S* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  S* tile = reinterpret_cast<S*>(smem_raw);  // [point][C K + 1]
  const int width = C * K, row = width + 1;
  const int u0 = blockIdx.x * points, cnt = min(points, nt - u0);
  for (int w = threadIdx.x; w < cnt * width; w += 256) {
    const int u = w / width, r = w - u * width;
    tile[u * row + r] = in[int64_t(inv[u0 + u]) * width + r];
  }
  __syncthreads();
  const int span = C * cnt;
  for (int w = threadIdx.x; w < span * K; w += 256) {
    const int k = w / span, r = w - k * span;
    const int u = r / C, c = r - u * C;
    out[(int64_t(k) * nt + u0) * C + r] = tile[u * row + c * K + k];
  }
}

template <class S>
void launch_scatter(const S* in, const DevicePlan& d, int K, int C, S* out, hipStream_t s) {
  int points = 64;
  while (points > 4 && size_t(points) * (C * K + 1) * sizeof(S) > 32768) points /= 2;
  scatter_kernel<S><<<unsigned((d.nt + points - 1) / points), 256, size_t(points) * (C * K + 1) * sizeof(S), s>>>(
      in, d.tgt_inv, d.nt, K, C, points, out);
  HIPFMM_CHECK(hipGetLastError());
}

// From this many states on, writing the totals in sorted order and unsorting
// them in a pass of whole lines beats single values scattered from the L2P.
constexpr int kScatterStates = 4;

template <class S, int kWhat>
void launch_l2p(const DevicePlan& d, S* out, S* pot, int K, S scale, hipStream_t s) {
  constexpr int C = l2p_rows(kWhat), TW = kWhat == kGradient ? 8 : 4;
  if (d.p2p_tile16_count == 0) return;
  const int NM = kWhat == kFieldAndPotential ? d.n : kWhat == kField ? d.nm : d.p >= 2 ? coefficient_count(d.p - 2) : 0;
  const int PW = std::max(kWhat == kFieldAndPotential ? d.p + 1 : kWhat == kField ? d.p : d.p - 1, 1);
  constexpr int most = 64 / C;  // states of four column tiles
  const int parts = (K + most - 1) / most, KC = (K + parts - 1) / parts;
  const bool sorted = K >= kScatterStates;
  const size_t lds = size_t(NM) * (sizeof(int4) + TW * sizeof(int)) + size_t(4) * 48 * PW * sizeof(S);
  const dim3 grid(unsigned((d.p2p_tile16_count + 3) / 4), unsigned((K + KC - 1) / KC));
  auto go = [&](auto ct) {
    l2p_columns_kernel<S, kWhat, decltype(ct)::value><<<grid, 256, lds, s>>>(d, out, pot, K, KC, NM, PW, scale, sorted);
  };
  switch ((C * KC + 15) / 16) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    default: go(std::integral_constant<int, 4>{}); break;
  }
  HIPFMM_CHECK(hipGetLastError());
  if (!sorted) return;
  if (kWhat == kGradient)
    launch_scatter<S>(static_cast<const S*>(d.Gn), d, K, 6, out, s);
  else if (out != nullptr)
    launch_scatter<S>(static_cast<const S*>(d.Hn), d, K, 3, out, s);
  if (kWhat == kFieldAndPotential) launch_scatter<S>(static_cast<const S*>(d.Pn), d, K, 1, pot, s);
}

}  // namespace

template <class S>
void launch_p2m_columns(const DevicePlan& d, int K, hipStream_t s) {
  const int tiles = (d.nm + 15) / 16, rtw = std::max((tiles + 3) / 4, 1);
  // States per workgroup: at most four column tiles, and the C_c in 32 KiB.
  const int per_state = 3 * std::max(tiles, 1) * 16 * int(sizeof(S));
  const int most = std::max(1, std::min(21, 32768 / per_state));
  const int parts = (K + most - 1) / most, KC = (K + parts - 1) / parts;
  const int ct = (3 * KC + 15) / 16;
  const size_t lds = (size_t(kChunk) * 3 * std::max(d.p, 1) + size_t(16 * ct) * tiles * 16) * sizeof(S);
  const dim3 grid(unsigned(d.leaves), unsigned((K + KC - 1) / KC));
  auto go = [&](auto rt, auto c) {
    p2m_columns_kernel<S, decltype(rt)::value, decltype(c)::value><<<grid, 256, lds, s>>>(d, K, KC);
  };
  auto rows = [&](auto c) {
    switch (rtw) {
      case 1: go(std::integral_constant<int, 1>{}, c); break;
      case 2: go(std::integral_constant<int, 2>{}, c); break;
      case 3: go(std::integral_constant<int, 3>{}, c); break;
      default: go(std::integral_constant<int, 4>{}, c); break;
    }
  };
  switch (ct) {
    case 1: rows(std::integral_constant<int, 1>{}); break;
    case 2: rows(std::integral_constant<int, 2>{}); break;
    case 3: rows(std::integral_constant<int, 3>{}); break;
    default: rows(std::integral_constant<int, 4>{}); break;
  }
  HIPFMM_CHECK(hipGetLastError());
}

template <class S>
void launch_m2m_columns(const DevicePlan& d, int parent_level, int K, hipStream_t s) {
  const int n = d.n, NP = round_to(n, 8);
  const int64_t box = int64_t(n) * K, parents = int64_t(1) << (3 * parent_level);
  S* M = static_cast<S*>(d.M);
  Product<S> p{};
  p.A = static_cast<const S*>(d.m2m_dense) + size_t(parent_level + 1) * 8 * n * NP;
  p.a_seg = int64_t(n) * NP;
  p.lda = NP, p.R = n, p.D = n, p.segments = 8;
  p.in = M + level_offset(parent_level + 1) * box;
  p.in_box = 8 * box, p.in_seg = box;
  p.out = M + level_offset(parent_level) * box;
  p.out_box = box;
  p.in_at = p.out_at = strides(d.state_major, K, n);
  p.K = K, p.cols = parents * K;
  p.bits = d.source_bits, p.bit0 = level_offset(parent_level), p.bit_box = 1, p.idle_stores = true;
  launch_product<S>(p, 1, s);
}

template <class S>
void launch_l2l_columns(const DevicePlan& d, int child_level, int K, hipStream_t s) {
  const int n = d.n, NP = round_to(n, 8);
  const int64_t box = int64_t(n) * K, parents = int64_t(1) << (3 * (child_level - 1));
  S* L = static_cast<S*>(d.Lc);
  Product<S> p{};
  p.A = static_cast<const S*>(d.l2l_dense) + size_t(child_level) * 8 * n * NP;
  p.a_z = int64_t(n) * NP;
  p.lda = NP, p.R = n, p.D = n, p.segments = 1;
  p.in = L + level_offset(child_level - 1) * box;
  p.in_box = box;
  p.out = L + level_offset(child_level) * box;
  p.out_box = 8 * box, p.out_z = box;
  p.in_at = p.out_at = strides(d.state_major, K, n);
  p.K = K, p.cols = parents * K;
  p.add = true;
  p.bits = d.target_bits, p.bit0 = level_offset(child_level), p.bit_box = 8;
  launch_product<S>(p, 8, s);
}

template <class S>
void launch_compress_columns(const DevicePlan& d, int level, int K, hipStream_t s) {
  const int NPc = round_to(d.nc, 16);
  const int64_t node0 = level_offset(level), boxes = int64_t(1) << (3 * level);
  Product<S> p{};
  p.A = static_cast<const S*>(d.cmp_op) + size_t(level) * d.n * NPc;
  p.lda = NPc, p.R = d.nc, p.D = d.n, p.segments = 1;
  p.in_box = int64_t(d.n) * K, p.out_box = int64_t(d.nc) * K;
  p.in = static_cast<const S*>(d.M) + node0 * p.in_box;
  p.out = static_cast<S*>(d.Mc) + node0 * p.out_box;
  p.in_at = strides(false, K, d.n), p.out_at = strides(d.compressed_state_major, K, d.nc);
  p.K = K, p.cols = boxes * K;
  p.bits = d.source_bits, p.bit0 = node0, p.bit_box = 1, p.idle_stores = true;
  launch_product<S>(p, 1, s);
}

template <class S>
void launch_expand_columns(const DevicePlan& d, int level, int K, hipStream_t s) {
  const int NP = round_to(d.n, 8);
  const int64_t node0 = level_offset(level), boxes = int64_t(1) << (3 * level);
  Product<S> p{};
  p.A = static_cast<const S*>(d.exp_op) + size_t(level) * d.nc * NP;
  p.lda = NP, p.R = d.n, p.D = d.nc, p.segments = 1;
  p.in_box = int64_t(d.nc) * K, p.out_box = int64_t(d.n) * K;
  p.in = static_cast<const S*>(d.Lcc) + node0 * p.in_box;
  p.out = static_cast<S*>(d.Lc) + node0 * p.out_box;
  p.in_at = strides(d.compressed_state_major, K, d.nc), p.out_at = strides(false, K, d.n);
  p.K = K, p.cols = boxes * K;
  p.bits = d.target_bits, p.bit0 = node0, p.bit_box = 1;
  launch_product<S>(p, 1, s);
}

template <class S>
void launch_l2p_columns(const DevicePlan& d, S* fields, S* potentials, int K, hipStream_t s) {
  if (potentials != nullptr)
    launch_l2p<S, kFieldAndPotential>(d, fields, potentials, K, S(d.potential_scale), s);
  else
    launch_l2p<S, kField>(d, fields, nullptr, K, S(1), s);
}

template <class S>
void launch_l2p_grad_columns(const DevicePlan& d, S* gradients, int K, hipStream_t s) {
  launch_l2p<S, kGradient>(d, gradients, nullptr, K, S(1.0 / d.potential_scale), s);
}

#define HIPFMM_INSTANTIATE(S)                                                      \
  template void launch_p2m_columns<S>(const DevicePlan&, int, hipStream_t);        \
  template void launch_m2m_columns<S>(const DevicePlan&, int, int, hipStream_t);   \
  template void launch_l2l_columns<S>(const DevicePlan&, int, int, hipStream_t);   \
  template void launch_compress_columns<S>(const DevicePlan&, int, int, hipStream_t); \
  template void launch_expand_columns<S>(const DevicePlan&, int, int, hipStream_t); \
  template void launch_l2p_columns<S>(const DevicePlan&, S*, S*, int, hipStream_t); \
  template void launch_l2p_grad_columns<S>(const DevicePlan&, S*, int, hipStream_t);
HIPFMM_INSTANTIATE(float)
HIPFMM_INSTANTIATE(double)
#undef HIPFMM_INSTANTIATE

}  // namespace hipfmm
