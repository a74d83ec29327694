// HipFull device plan: C-ABI implementation (include/hipfmm.h).
//
// Replaces the reference's CudaFullPlan (src/cuda_fmm_plan.hpp:95-114,
// src/cuda_fmm.cu:2636-3665).  Static data is uploaded once at create; each
// evaluate enqueues
//   far field, on the caller's stream (host operands, groups: a stream of the
//   plan's): gather -> P2M -> M2M (levels L-1..2) -> M2L (levels 2..L) -> L2L
//   (levels 3..L) -> [wait near] -> L2P + combine + unsort
//   near field, on a stream of the plan's: [wait gather] -> list-1 P2P
// and, for host operands, exactly one H2D (moments) and one D2H (fields),
// matching the reference's transfer contract (tests/test_cuda_backend.cpp:
// 102-105 there).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../../include/hipfmm.h"
#include "common.hpp"

#include <atomic>

namespace hipfmm {

std::atomic<int> g_inject_error{0};
std::atomic<int> g_inject_countdown{0};

hipError_t injected_error(hipError_t actual) {
  if (actual != hipSuccess || g_inject_error.load(std::memory_order_relaxed) == 0) return actual;
  if (g_inject_countdown.fetch_sub(1) != 0) return actual;
  const int error = g_inject_error.exchange(0);
  return error != 0 ? hipError_t(error) : actual;
}

}  // namespace hipfmm

using hipfmm::DevicePlan;

static_assert(HIPFMM_NOALLOC_MAX_POINTS == hipfmm::kNoAllocMaxPoints, "one limit for the header and the library");

namespace {

thread_local std::string g_last_error;

enum Ev {
  kEvH2D0,
  kEvH2D1,
  kEvGather,
  kEvP2M,
  kEvM2M,
  kEvM2L,
  kEvL2L,
  kEvL2P,
  kEvCaptured,
  kEvNear1,
  kEvD2H0,
  kEvD2H1,
  kEvCount
};

}  // namespace

// The M2L kernels: in the type's own precision on the vector ALUs or the matrix
// cores, in bf16 without split operands, and in tiles of split operands.
enum M2lPath { kVectorM2l, kFullM2l, kDirectM2l, kTileM2l };

// Tile order of the M2L over the boxes that hold points (DevicePlan::sparse_order).
struct SparseBoxes {
  std::vector<int> order;
  int base[hipfmm::kMaxLevels] = {};
  int len[hipfmm::kMaxLevels] = {};
};

struct hipfmm_plan {
  DevicePlan d;
  int device = 0;
  std::vector<void*> persistent;
  std::vector<void*> state;
  hipStream_t s_far = nullptr, s_near = nullptr;  // s_far: see far_stream
  bool done_recorded = false;         // ev[kEvL2P] marks the end of the last evaluate outside a capture
  int last_done = 0;                  // event at the end of the last evaluate
  unsigned long long capture_id = 0;  // of the last captured evaluate, which ends at ev[kEvCaptured]
  hipEvent_t ev[kEvCount] = {};
  void* pinned_in = nullptr;
  void* pinned_out = nullptr;
  size_t pinned_in_bytes = 0, pinned_out_bytes = 0;
  std::vector<int> fixed_self;
  bool identity_initialised = false;
  // Role-exchanged view used by the adjoint: near-field items over source
  // leaves and the inverse identity map (sorted source -> sorted target).
  int2* adj_tiles = nullptr;
  int adj_tile_count = 0;
  int2* adj_tiles16 = nullptr;
  int adj_tile16_count = 0;
  int* adj_blk8_start = nullptr;
  int2* adj_blk8_src = nullptr;
  int adj_blk8_count = 0;
  int* adj_nbr_blk_start = nullptr;
  int* adj_nbr_blk = nullptr;
  int* adj_self = nullptr;
  SparseBoxes adj_sparse;  // bases and lengths; the order itself is adj_sparse_order
  const int* adj_sparse_order = nullptr;
  bool adj_self_valid = true;  // false when two targets share one source
  bool potential_used = false;  // keep the near-field potential buffers in the state
  bool gradient_used = false;   // keep the field-gradient buffers in the state
  void* pinned_grad = nullptr;
  size_t pinned_grad_bytes = 0;
  void* pinned_pot = nullptr;
  size_t pinned_pot_bytes = 0;
  double device_moment_scale = 1.0;
  int m2l_mode = HIPFMM_M2L_VALU;
  bool mfma_ready = false;
  hipfmm_stats stats{};
  hipfmm_timings timings{};
  bool timings_pending = false;
  // Ring of per-launch M2L kernel events: evaluates never wait on the host
  // for earlier ones; a slot is read back when it is reused or when the
  // timings are asked for.
  static constexpr int kRing = 64;
  hipEvent_t m2l_ring[kRing][2] = {};
  bool m2l_ring_pending[kRing] = {};
  int last_ring_slot = 0;         // of the last evaluate
  M2lPath last_path = kFullM2l;   // what it ran, for complete_locals
  int last_mode = 0;
  bool last_adjoint = false;
  bool locals_complete = false;   // complete_locals has run since
  bool last_m2l_expands = false;  // its M2L ends at kEvM2L, after its kernel
  uint64_t m2l_launch_count = 0;
  double m2l_total_seconds = 0.0;
  uint64_t m2l_total_launches = 0;
  bool last_host = false;
  int last_K = 0;
  size_t persistent_bytes = 0;
  size_t state_bytes = 0;
};

namespace {

struct DeviceGuard {
  int previous = -1;
  explicit DeviceGuard(int device) {
    HIPFMM_CHECK(hipGetDevice(&previous));
    if (previous != device) HIPFMM_CHECK(hipSetDevice(device));
  }
  ~DeviceGuard() {
    int now = -1;
    if (hipGetDevice(&now) == hipSuccess && now != previous && previous >= 0) (void)hipSetDevice(previous);
  }
};

template <class F>
int guarded(F&& f) {
  try {
    f();
    return HIPFMM_OK;
  } catch (const hipfmm::invalid_argument& e) {
    g_last_error = e.what();
    return HIPFMM_ERROR_INVALID_ARGUMENT;
  } catch (const std::invalid_argument& e) {
    g_last_error = e.what();
    return HIPFMM_ERROR_INVALID_ARGUMENT;
  } catch (const std::bad_alloc&) {
    g_last_error = "host allocation failed";
    return HIPFMM_ERROR_RUNTIME;
  } catch (const std::exception& e) {
    g_last_error = e.what();
    return HIPFMM_ERROR_RUNTIME;
  }
}

void require(bool ok, const char* what) {
  if (!ok) throw hipfmm::invalid_argument(what);
}

void* device_alloc(hipfmm_plan* P, size_t bytes, std::vector<void*>& list, size_t& counter) {
  if (bytes == 0) bytes = 16;
  void* ptr = nullptr;
  HIPFMM_CHECK(hipMalloc(&ptr, bytes));
  list.push_back(ptr);
  counter += bytes;
  return ptr;
}

template <class T>
T* upload(hipfmm_plan* P, const T* host, size_t count) {
  const size_t bytes = count * sizeof(T);
  T* ptr = static_cast<T*>(device_alloc(P, bytes, P->persistent, P->persistent_bytes));
  if (count && host) HIPFMM_CHECK(hipMemcpy(ptr, host, bytes, hipMemcpyHostToDevice));
  if (count && !host) HIPFMM_CHECK(hipMemset(ptr, 0, bytes));  // empty population placeholder
  P->stats.setup_h2d_bytes += bytes;
  return ptr;
}

int gfx950_devices() {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return count;
}

bool device_is_gfx950(int device) {
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return false;
  return std::strncmp(prop.gcnArchName, "gfx950", 6) == 0;
}

// Basis tables: entry a -> (index(a-e_x), index(a-e_y), index(a-e_z), sign);
// entry n+a -> (ax, ay, az, |a|).  include/cdfmm/multi_index.hpp:62-71.
std::vector<int4> basis_tables(int p) {
  std::vector<int4> exps;
  for (int d = 0; d <= p; ++d)
    for (int ax = 0; ax <= d; ++ax)
      for (int ay = 0; ay <= d - ax; ++ay) exps.push_back(int4{ax, ay, d - ax - ay, d});
  const int n = int(exps.size());
  auto index_of = [&](int ax, int ay, int az) {
    if (ax < 0 || ay < 0 || az < 0) return -1;
    for (int i = 0; i < n; ++i)
      if (exps[i].x == ax && exps[i].y == ay && exps[i].z == az) return i;
    return -1;
  };
  std::vector<int4> tab(2 * size_t(n));
  for (int a = 0; a < n; ++a) {
    const int4 e = exps[a];
    tab[a] = int4{index_of(e.x - 1, e.y, e.z), index_of(e.x, e.y - 1, e.z), index_of(e.x, e.y, e.z - 1),
                  e.w % 2 == 0 ? 1 : -1};
    tab[n + a] = e;
  }
  return tab;
}

template <class S>
hipfmm::ShiftCsr shift_csr(hipfmm_plan* P, const double* dense, int L, int n) {
  // Union sparsity pattern over levels 1..L and the 8 classes.
  std::vector<char> nz(size_t(n) * n, 0);
  for (int l = 1; l <= L; ++l)
    for (int c = 0; c < 8; ++c) {
      const double* m = dense + (size_t(l - 1) * 8 + c) * n * n;
      for (size_t i = 0; i < size_t(n) * n; ++i)
        if (m[i] != 0.0) nz[i] = 1;
    }
  std::vector<int> off(n + 1, 0), col;
  for (int r = 0; r < n; ++r) {
    for (int cidx = 0; cidx < n; ++cidx)
      if (nz[size_t(r) * n + cidx]) col.push_back(cidx);
    off[r + 1] = int(col.size());
  }
  const int nnz = int(col.size());
  std::vector<S> vals(size_t(L + 1) * 8 * std::max(nnz, 1), S(0));
  for (int l = 1; l <= L; ++l)
    for (int c = 0; c < 8; ++c) {
      const double* m = dense + (size_t(l - 1) * 8 + c) * n * n;
      S* v = vals.data() + (size_t(l) * 8 + c) * nnz;
      for (int r = 0; r < n; ++r)
        for (int e = off[r]; e < off[r + 1]; ++e) v[e] = S(m[size_t(r) * n + col[e]]);
    }
  hipfmm::ShiftCsr out;
  out.nnz = nnz;
  out.row_offsets = upload(P, off.data(), off.size());
  out.columns = upload(P, col.data(), std::max<size_t>(col.size(), 1));
  out.values = upload(P, vals.data(), vals.size());
  return out;
}

// Dense transposed copy of a shift operator family for the box-GEMM kernels:
// bf16 of an FP32 value, rounded to nearest even (the rounding of the
// device's v_cvt_pk_bf16_f32); NaN stays NaN.
uint16_t bf16_rne(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return uint16_t((u >> 16) | ((u & 0xffffu) != 0 ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}
float bf16_value(uint16_t h) {
  const uint32_t u = uint32_t(h) << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

// `count` box operators, op[o][dd * lda + row] (R rows, depth D, `stride`
// values apart), as FP32 values split in three bf16 pieces x = hi + mid + lo
// (each rounded to nearest, as split3_bf16 does on the device), laid out as
// the A fragments of the box products: per operator
// [piece][dd / 32][row, padded to 16][dd % 32], zeros in the padding.
template <class T>
std::vector<uint16_t> box_operators_x3(const T* op, int count, size_t stride, int lda, int R, int D) {
  const int RP = (R + 15) / 16 * 16;
  const int64_t per = hipfmm::box_x3_elems(R, D), piece = per / 3;
  std::vector<uint16_t> out(size_t(count) * size_t(per), 0);
  for (int o = 0; o < count; ++o)
    for (int dd = 0; dd < D; ++dd)
      for (int row = 0; row < R; ++row) {
        const float x = float(op[size_t(o) * stride + size_t(dd) * lda + row]);
        const uint16_t h = bf16_rne(x);
        const float r1 = x - bf16_value(h);
        const uint16_t m = bf16_rne(r1);
        const uint16_t l = bf16_rne(r1 - bf16_value(m));
        const size_t at = size_t(o) * size_t(per) + (size_t(dd / 32) * RP + row) * 32 + dd % 32;
        out[at] = h;
        out[at + size_t(piece)] = m;
        out[at + 2 * size_t(piece)] = l;
      }
  return out;
}

// out[(l*8 + c)][col][NP] = op_l,c[row][col], rows padded to NP = round8(n).
template <class S>
void* shift_dense_transposed(hipfmm_plan* P, const double* dense, int L, int n) {
  const int NP = (n + 7) / 8 * 8;
  std::vector<S> out(size_t(L + 1) * 8 * n * NP, S(0));
  for (int l = 1; l <= L; ++l)
    for (int c = 0; c < 8; ++c) {
      const double* m = dense + (size_t(l - 1) * 8 + c) * n * n;
      S* o = out.data() + (size_t(l) * 8 + c) * n * NP;
      for (int r = 0; r < n; ++r)
        for (int col = 0; col < n; ++col) o[size_t(col) * NP + r] = S(m[size_t(r) * n + col]);
    }
  return upload(P, out.data(), out.size());
}

// Inverse of the fixed identity map for the adjoint (sorted source ->
// sorted target, or -1).  A map with two targets on one source has no
// inverse; the adjoint then refuses to run.
void refresh_adjoint_self(hipfmm_plan* P) {
  const DevicePlan& d = P->d;
  std::vector<int> inv(std::max(d.ns, 1), -1);
  P->adj_self_valid = true;
  for (int t = 0; t < int(P->fixed_self.size()); ++t) {
    const int s = P->fixed_self[t];
    if (s < 0) continue;
    if (inv[s] >= 0) P->adj_self_valid = false;
    inv[s] = t;
  }
  if (P->adj_self && d.ns) HIPFMM_CHECK(hipMemcpy(P->adj_self, inv.data(), size_t(d.ns) * sizeof(int), hipMemcpyHostToDevice));
}

// List-2 pairs of the levels 2..L: of the grid, and with points on both sides
// (of all levels and of the last).
template <class F>
void count_m2l_pairs(int L, F&& occupied, uint64_t& grid, uint64_t& pairs, uint64_t& leaf_pairs) {
  for (int level = 2; level <= L; ++level) {
    const int nb = 1 << level;
    for (int64_t m = 0; m < (int64_t(1) << (3 * level)); ++m) {
      int x, y, z;
      hipfmm::demorton3(uint32_t(m), level, x, y, z);
      auto inside = [&](int c, int reach) {  // sources within reach boxes of the target's parent, or of the target
        const int lo = reach == 1 ? c - 1 : (c & ~1) - 2, hi = reach == 1 ? c + 1 : (c & ~1) + 3;
        return uint64_t(std::min(hi, nb - 1) - std::max(lo, 0) + 1);
      };
      grid += inside(x, 2) * inside(y, 2) * inside(z, 2) - inside(x, 1) * inside(y, 1) * inside(z, 1);
      if (!occupied(level, m, false)) continue;
      for (int ox = (x & 1) - 3; ox <= (x & 1) + 2; ++ox)
        for (int oy = (y & 1) - 3; oy <= (y & 1) + 2; ++oy)
          for (int oz = (z & 1) - 3; oz <= (z & 1) + 2; ++oz) {
            if (std::max({std::abs(ox), std::abs(oy), std::abs(oz)}) <= 1) continue;
            const int sx = x - ox, sy = y - oy, sz = z - oz;
            if (sx < 0 || sy < 0 || sz < 0 || sx >= nb || sy >= nb || sz >= nb) continue;
            if (occupied(level, int64_t(hipfmm::morton3(sx, sy, sz, level)), true)) {
              ++pairs;
              if (level == L) ++leaf_pairs;
            }
          }
    }
  }
}

// The parents of a level's boxes in the order of the M2L's tiles, a list per
// boundary class (one in Morton order below level 4).
std::vector<std::vector<int>> boundary_classes(int level) {
  const int bits = level - 1, np = 1 << bits;
  const int64_t parents = int64_t(1) << (3 * bits);
  if (level < 4) {
    std::vector<int> all(static_cast<size_t>(parents));
    for (int64_t q = 0; q < parents; ++q) all[size_t(q)] = int(q);
    return {all};
  }
  // Within a class the parents follow the Morton order of their coordinates
  // relative to the class's own region (inner axes from 1, boundary axes
  // fixed), so a workgroup's parents are whole aligned octants of the inner
  // region (14 = 2 x 7 per axis at level 5) or compact patches of a face.
  std::vector<std::vector<std::pair<uint32_t, int>>> cls(27);
  auto axis_class = [&](int c) { return c == 0 ? 0 : (c == np - 1 ? 2 : 1); };
  auto rel = [&](int c) { return uint32_t(axis_class(c) == 1 ? c - 1 : 0); };
  for (int64_t q = 0; q < parents; ++q) {
    int x, y, z;
    hipfmm::demorton3(uint32_t(q), bits, x, y, z);
    cls[(axis_class(x) * 3 + axis_class(y)) * 3 + axis_class(z)].push_back(
        {hipfmm::morton3(rel(x), rel(y), rel(z), bits), int(q)});
  }
  // Classes in the order inner, faces, edges, corners: the inner class (most
  // of the work, every offset active) first, so that its equal-length
  // workgroups start together and walk the offsets in step, reading one
  // shifted region of sources that L2 holds; the shorter boundary workgroups
  // follow and fill the tail.
  auto boundary_axes = [](int k) { return int(k / 9 != 1) + int(k / 3 % 3 != 1) + int(k % 3 != 1); };
  std::vector<int> class_order(27);
  for (int k = 0; k < 27; ++k) class_order[k] = k;
  std::stable_sort(class_order.begin(), class_order.end(),
                   [&](int a, int b) { return boundary_axes(a) < boundary_axes(b); });
  std::vector<std::vector<int>> out;
  for (const int k : class_order) {
    auto& c = cls[k];
    std::stable_sort(c.begin(), c.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    out.emplace_back();
    for (const auto& e : c) out.back().push_back(e.second);
  }
  return out;
}

// The tile order of the M2L over the boxes of a level that `holds` names: per
// parity the parents of its boxes, each class padded to whole workgroups and
// the parities to one length.
template <class F>
void add_sparse_level(SparseBoxes& b, int level, const std::vector<std::vector<int>>& classes, F&& holds) {
  std::vector<int> lists[8];
  size_t most = 0;
  for (int parity = 0; parity < 8; ++parity) {
    auto& l = lists[parity];
    for (const auto& c : classes) {
      for (const int q : c)
        if (holds(int64_t(q) * 8 + parity)) l.push_back(q);
      l.resize((l.size() + hipfmm::kM2LSparseTiles - 1) / hipfmm::kM2LSparseTiles * hipfmm::kM2LSparseTiles, -1);
    }
    most = std::max(most, l.size());
  }
  b.base[level] = int(b.order.size());
  b.len[level] = int(most);
  for (auto& l : lists) {
    l.resize(most, -1);
    b.order.insert(b.order.end(), l.begin(), l.end());
  }
}

template <class S>
void create_impl(hipfmm_plan* P, const hipfmm_plan_desc& desc) {
  DevicePlan& d = P->d;
  const int p = desc.order, L = desc.max_level, n = hipfmm::coefficient_count(p);
  d.precision = desc.precision;
  d.p = p;
  d.n = n;
  d.nm = p >= 1 ? hipfmm::coefficient_count(p - 1) : 0;
  d.L = L;
  d.ns = desc.source_count;
  d.nt = desc.target_count;
  d.nodes = hipfmm::level_offset(L + 1);
  d.leaves = int64_t(1) << (3 * L);
  const int64_t leaf0 = hipfmm::level_offset(L);
  const int64_t* ranges = desc.node_ranges;
  // Geometry.
  using V4 = typename hipfmm::Vec4<S>::type;
  auto pack = [&](const double* pos, int count, void*& abs_out, void*& rel_out, bool is_src) {
    std::vector<V4> rel(std::max(count, 1));
    std::vector<int> leaf_of(std::max(count, 1), -1);
    for (int64_t leaf = 0; leaf < d.leaves; ++leaf) {
      const int64_t* r = ranges + 4 * (leaf0 + leaf) + (is_src ? 0 : 2);
      require(r[0] >= 0 && r[1] >= r[0] && r[1] <= count, "node ranges are inconsistent with the point count");
      for (int64_t i = r[0]; i < r[1]; ++i) leaf_of[size_t(i)] = int(leaf);
    }
    for (int i = 0; i < count; ++i) {
      require(leaf_of[i] >= 0, "leaf ranges do not cover every point");
      const double* c = desc.node_centres + 3 * (leaf0 + leaf_of[i]);
      const double* x = pos + 3 * size_t(i);
      rel[i] = V4{S(x[0] - c[0]), S(x[1] - c[1]), S(x[2] - c[2]), S(0)};
    }
    if constexpr (sizeof(S) == 4) {
      std::vector<float4> hl(2 * size_t(std::max(count, 1)));
      for (int i = 0; i < count; ++i) {
        const double* x = pos + 3 * size_t(i);
        const float hx = float(x[0]), hy = float(x[1]), hz = float(x[2]);
        hl[i] = float4{hx, hy, hz, 0.0f};
        hl[size_t(count) + i] =
            float4{float(x[0] - double(hx)), float(x[1] - double(hy)), float(x[2] - double(hz)), 0.0f};
      }
      abs_out = upload(P, hl.data(), hl.size());
    } else {
      std::vector<double4> a(std::max(count, 1));
      for (int i = 0; i < count; ++i) {
        const double* x = pos + 3 * size_t(i);
        a[i] = double4{x[0], x[1], x[2], 0.0};
      }
      abs_out = upload(P, a.data(), a.size());
    }
    rel_out = upload(P, rel.data(), rel.size());
  };
  pack(desc.sorted_sources, d.ns, d.src_pos, d.src_rel, true);
  pack(desc.sorted_targets, d.nt, d.tgt_pos, d.tgt_rel, false);
  d.src_perm = upload(P, desc.source_permutation, std::max(d.ns, 1));
  d.tgt_perm = upload(P, desc.target_permutation, std::max(d.nt, 1));
  // The index arrays below are built on the device from the leaf ranges
  // (lists.hip), on the far stream; each builder returns once its arrays
  // are complete.
  const auto index_t0 = std::chrono::steady_clock::now();
  const hipStream_t sb = P->s_near;
  const hipfmm::DeviceAllocator persistent = [P](size_t bytes) {
    return device_alloc(P, bytes, P->persistent, P->persistent_bytes);
  };
  auto inverse = [&](const int* perm, int count, const char* what) {
    int* inv = static_cast<int*>(persistent(size_t(std::max(count, 1)) * sizeof(int)));
    if (count == 0) HIPFMM_CHECK(hipMemsetAsync(inv, 0xff, sizeof(int), sb));  // the placeholder entry, -1
    require(hipfmm::device_inverse(perm, count, inv, sb), what);
    return inv;
  };
  d.src_inv = inverse(d.src_perm, d.ns, "source_permutation is not a permutation");
  d.tgt_inv = inverse(d.tgt_perm, d.nt, "target_permutation is not a permutation");
  std::vector<int2> ls(d.leaves), lt(d.leaves);
  for (int64_t leaf = 0; leaf < d.leaves; ++leaf) {
    const int64_t* r = ranges + 4 * (leaf0 + leaf);
    ls[leaf] = int2{int(r[0]), int(r[1])};
    lt[leaf] = int2{int(r[2]), int(r[3])};
  }
  d.leaf_src = upload(P, ls.data(), ls.size());
  d.leaf_tgt = upload(P, lt.data(), lt.size());
  // Near-field row tiles of the matrix-core P2P: 32 rows of (target,
  // component) pairs of one leaf each (4 rows per target with the
  // potential); the adjoint's tiles run over the source leaves.
  d.p2p_tile_count = hipfmm::device_tiles(d.leaf_tgt, d.leaves, 3, 32, &d.p2p_tiles, persistent, sb);
  d.p2p_tile4_count = hipfmm::device_tiles(d.leaf_tgt, d.leaves, 4, 32, &d.p2p_tiles4, persistent, sb);
  P->adj_tile_count = hipfmm::device_tiles(d.leaf_src, d.leaves, 3, 32, &P->adj_tiles, persistent, sb);
  d.potential_scale = desc.potential_scale > 0.0 ? desc.potential_scale : 1.0;
  // 16-target tiles of the bf16 and FP32 matrix-core kernels.
  d.p2p_tile16_count = hipfmm::device_tiles(d.leaf_tgt, d.leaves, 1, 16, &d.p2p_tiles16, persistent, sb);
  P->adj_tile16_count = hipfmm::device_tiles(d.leaf_src, d.leaves, 1, 16, &P->adj_tiles16, persistent, sb);
  // Source blocks of 8 of the bf16 three-piece near field, per source leaf
  // (the adjoint's source leaves are the target leaves), and per target leaf
  // the blocks of its 3x3x3 neighbourhood in one list (neighbours in the
  // order dz, dy, dx from -1 to 1, each leaf's blocks in source order).
  hipfmm::device_blocks8(d.leaf_src, d.L, d.leaves, &d.blk8_start, &d.blk8_src, &d.blk8_count, &d.nbr_blk_start,
                         &d.nbr_blk, persistent, sb);
  hipfmm::device_blocks8(d.leaf_tgt, d.L, d.leaves, &P->adj_blk8_start, &P->adj_blk8_src, &P->adj_blk8_count,
                         &P->adj_nbr_blk_start, &P->adj_nbr_blk, persistent, sb);
  P->adj_self = static_cast<int*>(persistent(size_t(std::max(d.ns, 1)) * sizeof(int)));
  HIPFMM_CHECK(hipMemsetAsync(P->adj_self, 0xff, size_t(std::max(d.ns, 1)) * sizeof(int), sb));  // -1
  HIPFMM_CHECK(hipStreamSynchronize(sb));
  P->stats.setup_index_seconds =
      std::chrono::duration<double>(std::chrono::steady_clock::now() - index_t0).count();
  std::vector<int> self(std::max(d.nt, 1), -1);
  if (desc.fixed_self_indices) {
    for (int t = 0; t < d.nt; ++t) {
      require(desc.fixed_self_indices[t] >= -1 && desc.fixed_self_indices[t] < d.ns,
              "fixed identity map contains an invalid index");
      self[t] = desc.fixed_self_indices[t];
    }
    P->fixed_self.assign(self.begin(), self.begin() + d.nt);
    P->identity_initialised = true;
    refresh_adjoint_self(P);
  }
  d.self = upload(P, self.data(), self.size());
  const auto tab = basis_tables(p);
  d.p2m_tab = upload(P, tab.data(), tab.size());
  // Raising table of the matrix-core L2P: g (degree < p) -> g + e_c.
  {
    std::vector<int4> up(std::max(d.nm, 1), int4{0, 0, 0, 0});
    for (int g = 0; g < d.nm; ++g) {
      const int4 e = tab[n + g];
      int idx[3] = {-1, -1, -1};
      for (int b = 0; b < n; ++b) {
        const int4 f = tab[n + b];
        if (f.x == e.x + 1 && f.y == e.y && f.z == e.z) idx[0] = b;
        if (f.x == e.x && f.y == e.y + 1 && f.z == e.z) idx[1] = b;
        if (f.x == e.x && f.y == e.y && f.z == e.z + 1) idx[2] = b;
      }
      if (idx[0] < 0 || idx[1] < 0 || idx[2] < 0) throw std::logic_error("basis raising table");
      up[g] = int4{idx[0], idx[1], idx[2], 0};
    }
    d.l2p_up = upload(P, up.data(), up.size());
  }
  // Raising table of the matrix-core field gradient: g (degree <= p - 2) ->
  // g + e_c + e_j for (c, j) = xx xy xz yy yz zz, as two int4 per g.
  if (p >= 2) {
    const int nm2 = hipfmm::coefficient_count(p - 2);
    const int cj[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    std::vector<int> up2(size_t(nm2) * 8, 0);
    for (int g = 0; g < nm2; ++g) {
      const int4 e = tab[n + g];
      for (int q = 0; q < 6; ++q) {
        int x[3] = {e.x, e.y, e.z};
        ++x[cj[q][0]];
        ++x[cj[q][1]];
        int idx = -1;
        for (int b = 0; b < n; ++b) {
          const int4 f = tab[n + b];
          if (f.x == x[0] && f.y == x[1] && f.z == x[2]) idx = b;
        }
        if (idx < 0) throw std::logic_error("basis second raising table");
        up2[size_t(g) * 8 + q] = idx;
      }
    }
    d.grad_up = upload(P, up2.data(), up2.size());
  }
  // M2L class matrices keyed by offset slot.
  std::vector<int> slot(hipfmm::kOffsetSlots, -1), slot_of_class(std::max(desc.m2l_class_count, 1), -1);
  for (int c = 0; c < desc.m2l_class_count; ++c) {
    const int* o = desc.m2l_class_offsets + 3 * c;
    require(std::abs(o[0]) <= 3 && std::abs(o[1]) <= 3 && std::abs(o[2]) <= 3, "M2L class offset out of range");
    const int s = hipfmm::offset_slot(o[0], o[1], o[2]);
    slot[s] = c;
    slot_of_class[c] = s;
  }
  if (L >= 2) {
    for (int x = -3; x <= 3; ++x)
      for (int y = -3; y <= 3; ++y)
        for (int z = -3; z <= 3; ++z)
          if (std::max({std::abs(x), std::abs(y), std::abs(z)}) >= 2)
            require(slot[hipfmm::offset_slot(x, y, z)] >= 0, "an M2L class matrix for a list-2 offset is missing");
  }
  const size_t nn = size_t(n) * n;
  // Harmonic-subspace form of the M2L (T_o = Q C_o P): class matrices of
  // size nc x nc and the level scalings folded into P and Q.
  hipfmm::HarmonicBasis hb;
  if (L >= 2 && desc.m2l_class_count > 0) hb = hipfmm::harmonic_m2l_basis(p, desc.m2l_matrices, desc.m2l_class_count);
  if (hb.nc > 0) {
    const int nc = hb.nc, NPc = (nc + 15) / 16 * 16, NP = (n + 7) / 8 * 8;
    d.nc = nc;
    std::vector<S> cmp(size_t(L + 1) * n * NPc, S(0)), expd(size_t(L + 1) * nc * NP, S(0));
    for (int l = 0; l <= L; ++l)
      for (int r = 0; r < nc; ++r) {
        for (int a = 0; a < n; ++a)
          cmp[(size_t(l) * n + a) * NPc + r] = S(hb.P[size_t(r) * n + a] * desc.m2l_multipole_scaling[size_t(l) * n + a]);
        for (int b = 0; b < n; ++b)
          expd[(size_t(l) * nc + r) * NP + b] = S(desc.m2l_local_scaling[size_t(l) * n + b] * hb.Q[size_t(b) * nc + r]);
      }
    d.cmp_op = upload(P, cmp.data(), cmp.size());
    d.exp_op = upload(P, expd.data(), expd.size());
    if (sizeof(S) == 4) {
      const auto c3 = box_operators_x3(cmp.data(), L + 1, size_t(n) * NPc, NPc, nc, n);
      const auto e3 = box_operators_x3(expd.data(), L + 1, size_t(nc) * NP, NP, n, nc);
      d.cmp_x3 = upload(P, c3.data(), c3.size());
      d.exp_x3 = upload(P, e3.data(), e3.size());
    }
    if constexpr (sizeof(S) == 4) {
      const auto f = hipfmm::m2l_fragments_f32(nc, hb.C, desc.m2l_class_count);
      d.m2l_fragments = upload(P, f.data(), f.size());
    } else {
      const auto f = hipfmm::m2l_fragments_f64(nc, hb.C, desc.m2l_class_count);
      d.m2l_fragments = upload(P, f.data(), f.size());
    }
    const std::vector<S> zero_box(size_t(nc) * hipfmm::kMaxBatch, S(0));
    d.m2l_zero_box = upload(P, zero_box.data(), zero_box.size());
    P->stats.m2l_reconstruction_error = hb.max_reconstruction_error;
    // FP32 plans run the upward and downward passes in the harmonic subspace
    // too.  A multipole with no harmonic part has no field, and neither has
    // its translate, so P M2M = A P with A = P ms_p S ms_c^-1 P^T; the Taylor
    // polynomial of a harmonic local stays harmonic under L2L, so
    // L2L Q = Q B with B = Q^T ls_c^-1 S ls_p Q (ms/ls per-degree, commuting
    // with the block-diagonal bases).  Both identities are checked on every
    // operator; if one fails the passes stay on the full coefficients.
    if (sizeof(S) == 4 && L >= 3 && desc.m2m_operators && desc.l2l_operators) {
      const int NPc8 = (nc + 7) / 8 * 8;
      std::vector<S> am(size_t(L + 1) * 8 * nc * NPc8, S(0)), bl(am.size(), S(0));
      std::vector<double> X(size_t(nc) * n), Y(size_t(n) * nc);
      double leak = 0.0;
      for (int l = 1; l <= L; ++l)
        for (int c = 0; c < 8; ++c) {
          const double* Sm = desc.m2m_operators + (size_t(l - 1) * 8 + c) * n * n;  // row-major out x in
          const double* Sl = desc.l2l_operators + (size_t(l - 1) * 8 + c) * n * n;
          const double* msp = desc.m2l_multipole_scaling + size_t(l - 1) * n;
          const double* msc = desc.m2l_multipole_scaling + size_t(l) * n;
          const double* lsp = desc.m2l_local_scaling + size_t(l - 1) * n;
          const double* lsc = desc.m2l_local_scaling + size_t(l) * n;
          // X = P ms_p S ms_c^-1 (nc x n), then A = X P^T; leak = X (I - P^T P).
          for (int r = 0; r < nc; ++r)
            for (int b = 0; b < n; ++b) {
              double acc = 0.0;
              for (int a = 0; a < n; ++a) acc += hb.P[size_t(r) * n + a] * msp[a] * Sm[size_t(a) * n + b];
              X[size_t(r) * n + b] = acc / msc[b];
            }
          // Y = ls_c^-1 S ls_p Q (n x nc), then B = Q^T Y; leak = (I - Q Q^T) Y.
          for (int a = 0; a < n; ++a)
            for (int r = 0; r < nc; ++r) {
              double acc = 0.0;
              for (int b = 0; b < n; ++b) acc += Sl[size_t(a) * n + b] * lsp[b] * hb.Q[size_t(b) * nc + r];
              Y[size_t(a) * nc + r] = acc / lsc[a];
            }
          double xmax = 0.0, ymax = 0.0, xl = 0.0, yl = 0.0;
          S* ao = am.data() + (size_t(l) * 8 + c) * nc * NPc8;
          S* bo = bl.data() + (size_t(l) * 8 + c) * nc * NPc8;
          std::vector<double> A(size_t(nc) * nc), B(size_t(nc) * nc);
          for (int r = 0; r < nc; ++r)
            for (int q = 0; q < nc; ++q) {
              double av = 0.0, bv = 0.0;
              for (int a = 0; a < n; ++a) {
                av += X[size_t(r) * n + a] * hb.P[size_t(q) * n + a];
                bv += hb.Q[size_t(a) * nc + r] * Y[size_t(a) * nc + q];
              }
              A[size_t(r) * nc + q] = av;
              B[size_t(r) * nc + q] = bv;
              ao[size_t(q) * NPc8 + r] = S(av);  // transposed: [column q][row r]
              bo[size_t(q) * NPc8 + r] = S(bv);
            }
          // Leaks: X - A P and Y - Q B.
          for (int r = 0; r < nc; ++r)
            for (int b = 0; b < n; ++b) {
              double proj = 0.0;
              for (int q = 0; q < nc; ++q) proj += A[size_t(r) * nc + q] * hb.P[size_t(q) * n + b];
              xmax = std::max(xmax, std::fabs(X[size_t(r) * n + b]));
              xl = std::max(xl, std::fabs(X[size_t(r) * n + b] - proj));
            }
          for (int a = 0; a < n; ++a)
            for (int r = 0; r < nc; ++r) {
              double proj = 0.0;
              for (int q = 0; q < nc; ++q) proj += hb.Q[size_t(a) * nc + q] * B[size_t(q) * nc + r];
              ymax = std::max(ymax, std::fabs(Y[size_t(a) * nc + r]));
              yl = std::max(yl, std::fabs(Y[size_t(a) * nc + r] - proj));
            }
          if (xmax > 0.0) leak = std::max(leak, xl / xmax);
          if (ymax > 0.0) leak = std::max(leak, yl / ymax);
        }
      if (leak <= 1e-10) {
        d.m2m_dense_c = upload(P, am.data(), am.size());
        d.l2l_dense_c = upload(P, bl.data(), bl.size());
        const auto m3 = box_operators_x3(am.data(), (L + 1) * 8, size_t(nc) * NPc8, NPc8, nc, nc);
        const auto l3 = box_operators_x3(bl.data(), (L + 1) * 8, size_t(nc) * NPc8, NPc8, nc, nc);
        d.m2m_x3_c = upload(P, m3.data(), m3.size());
        d.l2l_x3_c = upload(P, l3.data(), l3.size());
      }
      P->stats.harmonic_pass_leak = leak;
    }
  }
  if (hb.nc == 0) {
    std::vector<S> T(std::max<size_t>(size_t(desc.m2l_class_count) * nn, 1));
    for (size_t i = 0; i < size_t(desc.m2l_class_count) * nn; ++i) T[i] = S(desc.m2l_matrices[i]);
    d.m2l_T = upload(P, T.data(), T.size());
  }
  d.m2l_slot = upload(P, slot.data(), slot.size());
  // The 189 list-2 offsets of each parity class (target coordinate parity
  // q per axis: offsets in [q-3, q+2] minus the near cube), ordered by the
  // offset's own coordinate parity: within one such group the sources of
  // same-parity targets are shared between consecutive offsets.
  std::vector<int4> parity_offsets(8 * 189, int4{0, 0, 0, 0});
  if (L >= 2) {
    for (int parity = 0; parity < 8; ++parity) {
      const int q[3] = {parity & 1, (parity >> 1) & 1, (parity >> 2) & 1};
      int k = 0;
      for (int group = 0; group < 8; ++group)
        for (int ox = q[0] - 3; ox <= q[0] + 2; ++ox)
          for (int oy = q[1] - 3; oy <= q[1] + 2; ++oy)
            for (int oz = q[2] - 3; oz <= q[2] + 2; ++oz) {
              if (std::max({std::abs(ox), std::abs(oy), std::abs(oz)}) <= 1) continue;
              if (((ox & 1) | ((oy & 1) << 1) | ((oz & 1) << 2)) != group) continue;
              parity_offsets[parity * 189 + k++] = int4{ox, oy, oz, slot[hipfmm::offset_slot(ox, oy, oz)]};
            }
      if (k != 189) throw std::logic_error("list-2 offset enumeration");
    }
  }
  d.parity_offsets = upload(P, parity_offsets.data(), parity_offsets.size());
  std::vector<int4> parity_steps(parity_offsets.size());
  for (size_t i = 0; i < parity_steps.size(); ++i) {
    const int4 o = parity_offsets[i];
    parity_steps[i] = hipfmm::m2l_step(o.x, o.y, o.z, o.w);
  }
  d.m2l_steps = upload(P, parity_steps.data(), parity_steps.size());
  // Tile order of the matrix-core M2L.  A workgroup applies every offset
  // that any of its boxes uses, so a box whose list 2 is cut by the grid
  // boundary multiplies zeros for the offsets it lacks.  Along each axis only
  // the first and the last parent layer lose offsets, so from level 4 on the
  // parents are grouped by their boundary class per axis (first, inner, last;
  // Morton order within a class) and each class is padded to whole
  // workgroups: at 1M points, depth 5, the products beyond the list-2 pairs
  // fall from 17% to 3%.  Levels 2 and 3 keep the Morton order, which pads
  // less there.
  // Where a tenth or more of the list-2 pairs have a box without points, the
  // M2L takes boxes with targets only, and sources with points only: 2^20
  // points in blobs, depth 6, 32 states (63% of the pairs), M2L 52.6 -> 35.9
  // ms; 262,144 points of a slab seen from a plane, depth 5, one state (all but
  // a few), 296 -> 46 us.  The line keeps trees of uniform points on the full
  // order: at 5 points per leaf under 2% of their pairs have an empty side, in
  // boxes scattered singly, which saves no tile and few steps.
  const auto occupied = [&](int level, int64_t m, bool sources) {
    const int64_t* r = ranges + 4 * (hipfmm::level_offset(level) + m) + (sources ? 0 : 2);
    return r[1] > r[0];
  };
  uint64_t grid_pairs = 0, m2l_pairs = 0, leaf_pairs = 0;
  count_m2l_pairs(L, occupied, grid_pairs, m2l_pairs, leaf_pairs);
  const bool sparse = 10 * m2l_pairs <= 9 * grid_pairs && grid_pairs > 0;
  if (L >= 2 && L < hipfmm::kMaxLevels) {
    std::vector<int> order;
    SparseBoxes boxes[2];  // of targets, and of sources (the adjoint's targets)
    for (int level = 2; level <= L; ++level) {
      const auto classes = boundary_classes(level);
      for (int g = 0; g < 5; ++g) {
        const int G = hipfmm::kM2LGroupTiles[g];
        d.m2l_order_base[g][level] = int(order.size());
        for (const auto& c : classes) {
          order.insert(order.end(), c.begin(), c.end());
          if (level >= 4) order.insert(order.end(), (G - int(c.size()) % G) % G, -1);
        }
        d.m2l_order_len[g][level] = int(order.size()) - d.m2l_order_base[g][level];
      }
      if (sparse)
        for (int side = 0; side < 2; ++side)
          add_sparse_level(boxes[side], level, classes, [&](int64_t m) { return occupied(level, m, side == 1); });
    }
    d.m2l_order = upload(P, order.data(), order.size());
    if (sparse) {
      std::vector<uint32_t> bits[2];
      for (int side = 0; side < 2; ++side) {
        bits[side].assign(size_t(d.nodes + 31) / 32, 0u);
        for (int level = 0; level <= L; ++level)
          for (int64_t m = 0; m < (int64_t(1) << (3 * level)); ++m) {
            const int64_t node = hipfmm::level_offset(level) + m;
            if (occupied(level, m, side == 1)) bits[side][size_t(node >> 5)] |= 1u << (node & 31);
          }
      }
      d.target_bits = upload(P, bits[0].data(), bits[0].size());
      const bool same = bits[0] == bits[1];
      d.source_bits = same ? d.target_bits : upload(P, bits[1].data(), bits[1].size());
      d.sparse_order = upload(P, boxes[0].order.data(), boxes[0].order.size());
      P->adj_sparse = boxes[1];
      P->adj_sparse_order = same ? d.sparse_order : upload(P, boxes[1].order.data(), boxes[1].order.size());
      std::copy(boxes[0].base, boxes[0].base + hipfmm::kMaxLevels, d.sparse_base);
      std::copy(boxes[0].len, boxes[0].len + hipfmm::kMaxLevels, d.sparse_len);
      P->adj_sparse.order.clear();
      P->adj_sparse.order.shrink_to_fit();
    }
  }
  std::vector<S> ms(size_t(L + 1) * n), lsc(size_t(L + 1) * n);
  for (size_t i = 0; i < ms.size(); ++i) {
    ms[i] = S(desc.m2l_multipole_scaling[i]);
    lsc[i] = S(desc.m2l_local_scaling[i]);
  }
  d.ms = upload(P, ms.data(), ms.size());
  d.ls = upload(P, lsc.data(), lsc.size());
  if (L >= 1) {
    d.m2m = shift_csr<S>(P, desc.m2m_operators, L, n);
    d.l2l = shift_csr<S>(P, desc.l2l_operators, L, n);
    d.m2m_dense = shift_dense_transposed<S>(P, desc.m2m_operators, L, n);
    d.l2l_dense = shift_dense_transposed<S>(P, desc.l2l_operators, L, n);
  }
  P->stats.scalar_bytes = sizeof(S);
  P->stats.m2m_unique_matrix_count = uint64_t(L) * 8;
  P->stats.m2m_matrix_bytes = uint64_t(L) * 8 * d.m2m.nnz * sizeof(S);
  P->stats.l2l_unique_matrix_count = uint64_t(L) * 8;
  P->stats.l2l_matrix_bytes = uint64_t(L) * 8 * d.l2l.nnz * sizeof(S);
  P->stats.m2l_unique_matrix_count = uint64_t(desc.m2l_class_count);
  P->stats.m2l_matrix_bytes = uint64_t(desc.m2l_class_count) * nn * sizeof(S);
  // Interaction counts of the canonical plan (non-empty pairs only).
  uint64_t p2p_pairs = 0;
  {
    const int nb = 1 << L;
    for (int64_t m = 0; m < d.leaves; ++m) {
      const int64_t tc = lt[m].y - lt[m].x;
      if (tc == 0) continue;
      int x, y, z;
      hipfmm::demorton3(uint32_t(m), L, x, y, z);
      int64_t sc = 0;
      for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy)
          for (int dx = -1; dx <= 1; ++dx) {
            const int a = x + dx, b = y + dy, c = z + dz;
            if (a < 0 || b < 0 || c < 0 || a >= nb || b >= nb || c >= nb) continue;
            const int2 r = ls[hipfmm::morton3(a, b, c, L)];
            sc += r.y - r.x;
          }
      p2p_pairs += uint64_t(tc * sc);
    }
  }
  P->stats.m2l_interaction_count = m2l_pairs;
  P->stats.m2l_leaf_interaction_count = leaf_pairs;
  P->stats.m2l_operand_size = uint64_t(d.nc > 0 ? d.nc : n);
  P->stats.p2p_interaction_count = p2p_pairs;
  if constexpr (sizeof(S) == 4) {
    if (L >= 2 && desc.m2l_class_count > 0) {
      size_t bytes = 0;
      if (d.nc > 0) {
        const std::vector<double> ones(size_t(L + 1) * d.nc, 1.0);
        hipfmm::prepare_mfma_operators(d, d.nc, hb.C, desc.m2l_class_count, ones, P->persistent, bytes);
        hipfmm::prepare_mfma_fp16_operators(d, d.nc, hb.C, desc.m2l_class_count, p, P->persistent, bytes);
        // The last compressed multipole (degree 0) is zero for dipole
        // sources: the depth stops before it.
        d.mfma_depth_steps = (d.nc - 1 + 15) / 16;
      } else {
        std::vector<double> mats(desc.m2l_matrices, desc.m2l_matrices + size_t(desc.m2l_class_count) * nn);
        std::vector<double> lsd(desc.m2l_local_scaling, desc.m2l_local_scaling + size_t(L + 1) * n);
        hipfmm::prepare_mfma_operators(d, n, mats, desc.m2l_class_count, lsd, P->persistent, bytes);
      }
      P->persistent_bytes += bytes;
      P->stats.setup_h2d_bytes += bytes;
      P->mfma_ready = true;
    }
  }
}

void free_state(hipfmm_plan* P) {
  for (void* ptr : P->state) (void)hipFree(ptr);
  P->state.clear();
  P->state_bytes = 0;
  P->d.kcap = 0;
}

// Earlier evaluates may still be running on the callers' and the plan's streams.
void wait_for_evaluates(hipfmm_plan* P) {
  if (P->done_recorded) HIPFMM_CHECK(hipEventSynchronize(P->ev[kEvL2P]));
  if (P->s_far) HIPFMM_CHECK(hipStreamSynchronize(P->s_far));
  HIPFMM_CHECK(hipStreamSynchronize(P->s_near));
}

// The plan's own stream of the far field, for evaluates without a stream of
// the caller's: created with the first of them, since streams share the
// process's few hardware queues.
hipStream_t far_stream(hipfmm_plan* P) {
  if (!P->s_far) HIPFMM_CHECK(hipStreamCreateWithFlags(&P->s_far, hipStreamNonBlocking));
  return P->s_far;
}

template <class S>
void ensure_capacity(hipfmm_plan* P, int K, bool potential, bool gradient = false) {
  DevicePlan& d = P->d;
  if ((potential && !P->potential_used) || (gradient && !P->gradient_used)) {
    P->potential_used = P->potential_used || potential;
    P->gradient_used = P->gradient_used || gradient;
    wait_for_evaluates(P);
    free_state(P);  // reallocated below with the extra buffers
  }
  if (K <= d.kcap) return;
  wait_for_evaluates(P);
  free_state(P);
  const int cap = std::min(hipfmm::kMaxBatch, std::max(K, 1));
  const size_t cs = size_t(d.nodes) * d.n * cap;
  auto alloc = [&](size_t count, size_t elem) {
    return device_alloc(P, count * elem, P->state, P->state_bytes);
  };
  // Point-sized buffers hold max(N_s, N_t) so that the adjoint (roles
  // exchanged) runs on the same state.
  const size_t points = size_t(std::max({d.ns, d.nt, 1}));
  d.moments_in = alloc(points * 3 * cap, sizeof(S));
  d.fields_out = alloc(points * 3 * cap, sizeof(S));
  d.sm = alloc(points * 3 * cap, sizeof(S));
  d.Hn = alloc(points * 3 * cap, sizeof(S));
  d.smb = nullptr;
  d.smb_blocks = 0;
  if (sizeof(S) == 4 && cap >= hipfmm::kNearGradBf16States) {  // bf16 moments in tiles of 32 states
    d.smb_blocks = std::max({d.blk8_count, P->adj_blk8_count, 1});
    d.smb = alloc(size_t(d.smb_blocks) * 9 * 8 * ((cap + 31) / 32 * 32), 2);
  }
  d.Pn = nullptr;
  d.potentials_out = nullptr;
  if (P->potential_used) {
    d.Pn = alloc(points * cap, sizeof(S));
    d.potentials_out = alloc(points * cap, sizeof(S));
  }
  d.Gn = nullptr;
  d.gradients_out = nullptr;
  if (P->gradient_used) {
    d.Gn = alloc(points * 6 * cap, sizeof(S));
    d.gradients_out = alloc(points * 6 * cap, sizeof(S));
  }
  d.M = alloc(cs, sizeof(S));
  d.Lc = alloc(cs, sizeof(S));
  HIPFMM_CHECK(hipMemset(d.M, 0, cs * sizeof(S)));
  HIPFMM_CHECK(hipMemset(d.Lc, 0, cs * sizeof(S)));
  if (d.nc > 0) {
    const size_t cc = size_t(d.nodes) * d.nc * cap;
    d.Mc = alloc(cc, sizeof(S));
    d.Lcc = alloc(cc, sizeof(S));
    HIPFMM_CHECK(hipMemset(d.Mc, 0, cc * sizeof(S)));
    HIPFMM_CHECK(hipMemset(d.Lcc, 0, cc * sizeof(S)));
  }
  if (sizeof(S) == 4 && P->mfma_ready) {
    const size_t ms = size_t(d.nodes) * hipfmm::m2l_operand_capacity(d, cap) * d.apad;
    // Each half is followed by a 1 KiB zero block (the operand of sources
    // outside the grid); zeroed once here.
    d.mt_zero_offset = int64_t(ms) * 2;
    d.mt_hi = alloc(ms + 512, 2);
    d.mt_lo = alloc(ms + 512, 2);
    HIPFMM_CHECK(hipMemset(d.mt_hi, 0, (ms + 512) * 2));
    HIPFMM_CHECK(hipMemset(d.mt_lo, 0, (ms + 512) * 2));
  }
  d.kcap = cap;
  P->stats.batch_capacity = uint64_t(cap);
}

float elapsed(hipEvent_t a, hipEvent_t b) {
  float ms = 0.0f;
  if (hipEventElapsedTime(&ms, a, b) != hipSuccess) {
    (void)hipGetLastError();
    return 0.0f;
  }
  return ms;
}

// Read back one ring slot of M2L kernel events (waits for it).
void drain_m2l_slot(hipfmm_plan* P, int slot) {
  if (!P->m2l_ring_pending[slot]) return;
  HIPFMM_CHECK(hipEventSynchronize(P->m2l_ring[slot][1]));
  P->m2l_total_seconds += 1e-3 * elapsed(P->m2l_ring[slot][0], P->m2l_ring[slot][1]);
  P->m2l_total_launches += 1;
  P->m2l_ring_pending[slot] = false;
}

void finalize_timings(hipfmm_plan* P) {
  if (!P->timings_pending) return;
  HIPFMM_CHECK(hipEventSynchronize(P->ev[kEvL2P]));
  if (P->last_host) HIPFMM_CHECK(hipEventSynchronize(P->ev[kEvD2H1]));
  hipfmm_timings& t = P->timings;
  hipEvent_t* e = P->ev;
  // A record between two kernels costs about 6 us, so no point of the stream
  // has two: without a copy the kernels start where the call does, the near
  // field starts at the gather's end, and the M2L ends with its kernel unless
  // an expansion follows.
  const hipEvent_t kernels0 = P->last_host ? e[kEvH2D1] : e[kEvH2D0];
  const hipEvent_t* m2l_kernel = P->m2l_ring[P->last_ring_slot];
  const hipEvent_t m2l_end = P->last_m2l_expands ? e[kEvM2L] : m2l_kernel[1];
  t.h2d_seconds = P->last_host ? 1e-3 * elapsed(e[kEvH2D0], e[kEvH2D1]) : 0.0;
  t.p2m_seconds = 1e-3 * elapsed(kernels0, e[kEvP2M]);
  t.m2m_seconds = 1e-3 * elapsed(e[kEvP2M], e[kEvM2M]);
  t.m2l_seconds = 1e-3 * elapsed(e[kEvM2M], m2l_end);
  t.l2l_seconds = 1e-3 * elapsed(m2l_end, e[kEvL2L]);
  t.l2p_seconds = 1e-3 * elapsed(e[kEvL2L], e[kEvL2P]);
  t.p2p_seconds = 1e-3 * elapsed(e[kEvGather], e[kEvNear1]);
  t.kernel_seconds = 1e-3 * elapsed(kernels0, e[kEvL2P]);
  t.d2h_seconds = P->last_host ? 1e-3 * elapsed(e[kEvD2H0], e[kEvD2H1]) : 0.0;
  t.total_seconds = 1e-3 * elapsed(e[kEvH2D0], P->last_host ? e[kEvD2H1] : e[kEvL2P]);
  t.m2l_kernel_seconds = P->d.L >= 2 ? 1e-3 * elapsed(m2l_kernel[0], m2l_kernel[1]) : 0.0;
  P->timings_pending = false;
}

// The plan seen with the roles of sources and targets exchanged: the
// adjoint runs every kernel of the forward evaluate on this view.
DevicePlan role_exchanged(const hipfmm_plan* P) {
  DevicePlan a = P->d;
  std::swap(a.ns, a.nt);
  std::swap(a.src_pos, a.tgt_pos);
  std::swap(a.src_rel, a.tgt_rel);
  std::swap(a.src_perm, a.tgt_perm);
  std::swap(a.src_inv, a.tgt_inv);
  std::swap(a.leaf_src, a.leaf_tgt);
  a.self = P->adj_self;
  a.p2p_tiles = P->adj_tiles;
  a.p2p_tile_count = P->adj_tile_count;
  a.p2p_tiles16 = P->adj_tiles16;
  a.p2p_tile16_count = P->adj_tile16_count;
  a.blk8_start = P->adj_blk8_start;
  a.blk8_src = P->adj_blk8_src;
  a.blk8_count = P->adj_blk8_count;
  a.nbr_blk_start = P->adj_nbr_blk_start;
  a.nbr_blk = P->adj_nbr_blk;
  std::swap(a.source_bits, a.target_bits);
  a.sparse_order = P->adj_sparse_order;
  std::copy(P->adj_sparse.base, P->adj_sparse.base + hipfmm::kMaxLevels, a.sparse_base);
  std::copy(P->adj_sparse.len, P->adj_sparse.len + hipfmm::kMaxLevels, a.sparse_len);
  return a;
}

// Identity map: fixed with the plan on first use (src/cuda_fmm.cu:3470-3486);
// null keeps the plan's map.
void install_identity(hipfmm_plan* P, const int* self) {
  if (self == nullptr) return;
  const hipfmm::DevicePlan& f = P->d;
  if (!P->identity_initialised) {
    for (int t = 0; t < f.nt; ++t) require(self[t] >= -1 && self[t] < f.ns, "identity map contains an invalid index");
    P->fixed_self.assign(self, self + f.nt);
    if (f.nt) HIPFMM_CHECK(hipMemcpy(f.self, self, size_t(f.nt) * sizeof(int), hipMemcpyHostToDevice));
    P->stats.setup_h2d_bytes += size_t(f.nt) * sizeof(int);
    P->identity_initialised = true;
    refresh_adjoint_self(P);
  } else if (!std::equal(self, self + f.nt, P->fixed_self.begin())) {
    throw hipfmm::invalid_argument("HipFull identity map changed; rebuild the static plan");
  }
}

// The plan in harmonic-subspace form, where it has one: the operands are the
// compressed multipoles and locals (the level scalings are in the transforms).
DevicePlan compressed_view(const DevicePlan& d) {
  DevicePlan c = d;
  if (d.nc == 0 || d.L < 2) return c;
  c.n = d.nc;
  c.M = d.Mc;
  c.Lc = d.Lcc;
  c.state_major = d.compressed_state_major;
  c.m2m_dense = d.m2m_dense_c;
  c.l2l_dense = d.l2l_dense_c;
  c.m2m_x3 = d.m2m_x3_c;
  c.l2l_x3 = d.l2l_x3_c;
  return c;
}
bool harmonic_passes(const DevicePlan& d) { return d.m2m_dense_c != nullptr && d.nc > 0 && d.L >= 3; }
// Layout of the compressed coefficients (DevicePlan::compressed_state_major).
template <class S>
bool state_major(const DevicePlan& d, int K) {
  return d.nc > 0 && (sizeof(S) == 8 || K % 32 != 0);
}

// The M2L kernel of a batch of K states.
//
// The 16-bit modes split the multipoles in a pass of their own and run in
// workgroups of 256 columns whose chain of up to 189 offsets takes 0.23-0.6
// ms however few there are.  A small batch runs on the direct kernels
// instead, whose waves share the offsets and which need no split: the bf16
// mode in its own arithmetic, the FP16 mode in full FP32 (24 bits per
// operand against 22, and no pass over the level maxima).  The line is at
// the batch's size in boxes x states x coefficients.  Whole evaluates (ms,
// workgroups of 256 / direct), bf16: p = 8, 4681 boxes 0.92 / 0.49 at K = 1,
// 1.24 / 1.06 at 6, 1.32 / 1.26 at 8 (3.0e6); 37449 boxes 2.07 / 1.96 at
// K = 1 (3.0e6), 2.92 / 3.04 at 2; p = 6 1.49 / 1.40 at 1, 2.03 / 2.00 at 2
// (3.7e6), 2.58 / 2.80 at 3.  FP16: p = 8, 4681 boxes 1.12 / 1.06 at K = 4,
// 1.24 / 1.36 at 6 (2.3e6); p = 6 0.82 / 0.76 at 6, 0.86 / 0.89 at 8 (1.8e6).
// From 9 states on the operands are padded to whole 32-column boxes (see
// m2l_operand_states) and the line is lower: bf16 p = 6, 585 boxes
// 0.48 / 0.45 at K = 24 (6.9e5), 0.55 / 0.58 at 31.
template <class S>
M2lPath m2l_path(const hipfmm_plan* P, int K) {
  const DevicePlan& d = P->d;
  const bool sixteen = sizeof(S) == 4 && P->m2l_mode != HIPFMM_M2L_VALU && P->mfma_ready;
  const bool bf16 = P->m2l_mode == HIPFMM_M2L_MFMA_BF16X3;
  const int64_t size = d.nodes * K * d.nc;
  const bool small = d.nc > 0 && K % 32 != 0 && size <= (K < 9 ? (bf16 ? 3500000 : 1800000) : 700000);
  if (sixteen && !small) return kTileM2l;
  if (sixteen && bf16) return kDirectM2l;
  return d.nc > 0 ? kFullM2l : kVectorM2l;
}

template <class S>
void launch_m2l(const DevicePlan& compressed, M2lPath path, int mode, int K, hipStream_t s) {
  switch (path) {
    case kTileM2l: hipfmm::launch_m2l_mfma(compressed, K, mode, s); break;
    case kDirectM2l: hipfmm::launch_m2l_bf16_direct(compressed, K, s); break;
    case kFullM2l: hipfmm::launch_m2l_full<S>(compressed, K, s); break;
    case kVectorM2l: hipfmm::launch_m2l_valu<S>(compressed, K, s); break;
  }
}
// L2L, and the leaf level's expansion where the passes are harmonic.
template <class S>
void launch_downward(const DevicePlan& d, const DevicePlan& compressed, int K, hipStream_t s) {
  const bool harmonic = harmonic_passes(d);
  for (int level = 3; level <= d.L; ++level) hipfmm::launch_l2l<S>(harmonic ? compressed : d, level, K, s);
  if (harmonic) hipfmm::launch_m2l_expand<S>(d, K, d.L, s);
}

// The last evaluate's locals of a box that its M2L left out (DevicePlan::
// target_bits): the M2L and the downward pass again, over every box, once per
// evaluate.  (A captured evaluate's replays change the locals unseen: after a
// capture they are formed on every read.)
template <class S>
void complete_locals(hipfmm_plan* P, int node) {
  DevicePlan d = P->last_adjoint ? role_exchanged(P) : P->d;
  if (d.target_bits == nullptr) return;
  uint32_t word = 0;
  HIPFMM_CHECK(hipMemcpy(&word, d.target_bits + (node >> 5), sizeof(word), hipMemcpyDeviceToHost));
  if ((word >> (node & 31)) & 1u) return;
  if (P->locals_complete) return;
  d.target_bits = nullptr;
  d.sparse_order = nullptr;
  d.compressed_state_major = state_major<S>(d, P->last_K);
  const DevicePlan c = compressed_view(d);
  launch_m2l<S>(c, P->last_path, P->last_mode, P->last_K, P->s_near);
  if (d.nc > 0 && !harmonic_passes(d)) hipfmm::launch_m2l_expand<S>(d, P->last_K, 2, P->s_near);
  launch_downward<S>(d, c, P->last_K, P->s_near);
  HIPFMM_CHECK(hipStreamSynchronize(P->s_near));
  P->locals_complete = P->capture_id == 0;
}

// Kernels of an evaluate that failed half-way, which no event marks: they end
// before the error is reported, so that the next evaluate finds the plan's
// buffers free whatever stream it runs on.  (Not within a capture, where nothing
// runs yet.)
struct SettleOnFailure {
  hipStream_t far, near;
  bool armed;
  ~SettleOnFailure() {
    if (!armed) return;
    (void)hipStreamSynchronize(far);
    (void)hipStreamSynchronize(near);
    (void)hipGetLastError();
  }
};

// One evaluate.  The near field runs on a stream of the plan's.  The rest of a
// device-resident evaluate runs on the caller's stream `user`, which then needs
// no fork and no join (1,000 points, p = 4, depth 2: 97 us per evaluate, with
// both 117).
// `fork`: when set, the far field runs on the plan's own stream after this
// event (recorded by the caller on `user`), and the wait of `user` on the
// plan's last stage is left to the caller.  Evaluates of one plan run in the
// order of their calls, whatever their streams.
template <class S>
void evaluate_impl(hipfmm_plan* P, const void* moments, void* fields, void* potentials, int K, const int* self,
                   int memspace, hipStream_t user, bool adjoint, void* field_gradients = nullptr,
                   hipEvent_t fork = nullptr) {
  const bool want_pot = potentials != nullptr;
  const bool want_grad = field_gradients != nullptr;
  {
    const DevicePlan& f = P->d;
    const int n_in = adjoint ? f.nt : f.ns, n_out = adjoint ? f.ns : f.nt;
    require(K >= 1 && K <= hipfmm::kMaxBatch, "batch must be between 1 and 64 moment states");
    require(moments != nullptr || n_in == 0, adjoint ? "cotangents pointer is null" : "moments pointer is null");
    require(!adjoint || potentials == nullptr, "the adjoint is of the field map only");
    require(!want_grad || (fields == nullptr && potentials == nullptr),
            "the field gradient is evaluated on its own");
    require(want_pot || want_grad || fields != nullptr || n_out == 0,
            adjoint ? "gradients pointer is null" : "fields pointer is null");
    require(memspace == HIPFMM_HOST || memspace == HIPFMM_DEVICE, "unknown memory space");
    install_identity(P, self);
    require(!adjoint || P->adj_self_valid,
            "the identity map pairs two targets with one source; the adjoint has no transposed form of it");
  }
  // No wait on earlier evaluates here: their stage events are read back
  // only when timings are asked for, so the host can enqueue ahead.
  (void)hipGetLastError();
  ensure_capacity<S>(P, K, want_pot, want_grad);
  DevicePlan d = adjoint ? role_exchanged(P) : P->d;
  d.compressed_state_major = state_major<S>(d, K);
  const bool host = memspace == HIPFMM_HOST;
  const hipStream_t s = host || fork != nullptr ? far_stream(P) : user;
  hipEvent_t* e = P->ev;
  // The plan's buffers are free once its last evaluate is done.  On a stream
  // under capture an event is recorded into the graph and marks nothing outside
  // it, so a captured evaluate ends at an event of its own and follows only those
  // of the same capture (a graph's replays are the caller's to order).
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  unsigned long long capture_id = 0;
  HIPFMM_CHECK(hipStreamGetCaptureInfo(host ? s : user, &capture, &capture_id));
  const bool captured = capture != hipStreamCaptureStatusNone;
  if (captured ? P->capture_id == capture_id : P->done_recorded)
    HIPFMM_CHECK(hipStreamWaitEvent(s, e[captured ? kEvCaptured : kEvL2P], 0));
  SettleOnFailure settle{s, P->s_near, !captured};
  P->locals_complete = false;
  auto mark = [&](int ev, hipStream_t on) {
    HIPFMM_CHECK(hipEventRecord(e[ev], on));
  };
  const S* mu = nullptr;
  S* out = nullptr;
  S* pot = nullptr;
  S* grad = nullptr;
  S scale = S(1);
  const size_t in_bytes = size_t(K) * d.ns * 3 * sizeof(S);
  const size_t out_bytes = fields != nullptr ? size_t(K) * d.nt * 3 * sizeof(S) : 0;
  const size_t pot_bytes = want_pot ? size_t(K) * d.nt * sizeof(S) : 0;
  const size_t grad_bytes = want_grad ? size_t(K) * d.nt * 6 * sizeof(S) : 0;
  if (host) {
    if (P->pinned_grad_bytes < grad_bytes) {
      if (P->pinned_grad) (void)hipHostFree(P->pinned_grad);
      P->pinned_grad = nullptr;
      HIPFMM_CHECK(hipHostMalloc(&P->pinned_grad, std::max<size_t>(grad_bytes, 16)));
      P->pinned_grad_bytes = grad_bytes;
    }
    if (P->pinned_pot_bytes < pot_bytes) {
      if (P->pinned_pot) (void)hipHostFree(P->pinned_pot);
      P->pinned_pot = nullptr;
      HIPFMM_CHECK(hipHostMalloc(&P->pinned_pot, std::max<size_t>(pot_bytes, 16)));
      P->pinned_pot_bytes = pot_bytes;
    }
    if (P->pinned_in_bytes < in_bytes) {
      if (P->pinned_in) (void)hipHostFree(P->pinned_in);
      P->pinned_in = nullptr;
      HIPFMM_CHECK(hipHostMalloc(&P->pinned_in, std::max<size_t>(in_bytes, 16)));
      P->pinned_in_bytes = in_bytes;
    }
    if (P->pinned_out_bytes < out_bytes) {
      if (P->pinned_out) (void)hipHostFree(P->pinned_out);
      P->pinned_out = nullptr;
      HIPFMM_CHECK(hipHostMalloc(&P->pinned_out, std::max<size_t>(out_bytes, 16)));
      P->pinned_out_bytes = out_bytes;
    }
    if (in_bytes) std::memcpy(P->pinned_in, moments, in_bytes);
    mark(kEvH2D0, s);
    if (in_bytes) HIPFMM_CHECK(hipMemcpyAsync(d.moments_in, P->pinned_in, in_bytes, hipMemcpyHostToDevice, s));
    mark(kEvH2D1, s);
    mu = static_cast<const S*>(d.moments_in);
    out = fields != nullptr ? static_cast<S*>(d.fields_out) : nullptr;
    pot = want_pot ? static_cast<S*>(d.potentials_out) : nullptr;
    grad = want_grad ? static_cast<S*>(d.gradients_out) : nullptr;
    P->stats.evaluation_h2d_bytes = in_bytes;
    P->stats.evaluation_d2h_bytes = out_bytes + pot_bytes + grad_bytes;
    P->stats.evaluation_h2d_calls += 1;
    P->stats.evaluation_d2h_calls += 1;
  } else {
    if (fork != nullptr) HIPFMM_CHECK(hipStreamWaitEvent(s, fork, 0));
    mark(kEvH2D0, s);
    mu = static_cast<const S*>(moments);
    out = static_cast<S*>(fields);
    pot = static_cast<S*>(potentials);
    grad = static_cast<S*>(field_gradients);
    scale = S(P->device_moment_scale);
    P->stats.evaluation_h2d_bytes = 0;
    P->stats.evaluation_d2h_bytes = 0;
  }
  hipfmm::launch_gather<S>(d, mu, scale, K, s);
  HIPFMM_CHECK(hipEventRecord(e[kEvGather], s));
  HIPFMM_CHECK(hipStreamWaitEvent(P->s_near, e[kEvGather], 0));
  if (want_grad)
    hipfmm::launch_p2p_grad<S>(d, K, P->s_near);
  else
    hipfmm::launch_p2p<S>(d, K, want_pot, P->s_near);
  HIPFMM_CHECK(hipEventRecord(e[kEvNear1], P->s_near));
  hipfmm::launch_p2m<S>(d, K, s);
  mark(kEvP2M, s);
  // Harmonic passes: leaf multipoles compressed once, M2M and (below) L2L on
  // the compressed coefficients, the expansion at the leaf level only.
  const bool harmonic = harmonic_passes(d);
  const DevicePlan dc = compressed_view(d);
  if (harmonic) {
    hipfmm::launch_m2l_compress<S>(d, K, d.L, s);
    for (int level = d.L - 1; level >= 2; --level) hipfmm::launch_m2m<S>(dc, level, K, s);
  } else {
    for (int level = d.L - 1; level >= 2; --level) hipfmm::launch_m2m<S>(d, level, K, s);
  }
  // Levels 0 and 1 hold no list-2 work: their coefficients are zero
  // (hipfmm_plan_coefficients), and only a tree without deeper levels reads
  // them here.
  if (d.L < 2) hipfmm::launch_zero<S>(static_cast<S*>(d.Lc), size_t(d.nodes) * d.n * K, s);
  mark(kEvM2M, s);
  const M2lPath path = m2l_path<S>(P, K);
  const bool mfma = path == kTileM2l;
  if (d.nc > 0 && d.L >= 2) {
    if (!harmonic) hipfmm::launch_m2l_compress<S>(d, K, 2, s);
    if (mfma && P->m2l_mode == HIPFMM_M2L_MFMA_FP16X3)
      hipfmm::launch_m2l_fp16_split(d, K, s);
    else if (mfma)
      hipfmm::launch_m2l_bf16_split(d, K, s);
  } else if (mfma) {
    hipfmm::launch_m2l_split(d, K, P->m2l_mode, s);
  }
  // Which M2L starts once the near field is done, and which beside it (whole
  // evaluates, ms, after / beside; the upward pass before this point always runs
  // beside the near field).
  //   * The tiles from K = 32 on, after: both kernels then fill the chip and are
  //     bound by instruction issue, one after the other takes as long (2^20
  //     points, depth 5, K = 32: p = 8 14.48 / 14.49, p = 4 6.88 / 7.07), and the
  //     M2L runs alone.  A smaller batch is too few workgroups to fill it, beside
  //     (131,072 points, depth 4, p = 4: K = 12 .678 / .630, 31 1.009 / .935).
  //   * The direct and the full-precision kernels on a small tree (585 boxes and
  //     fewer), beside: 1024 points, depth 2, p = 4: K = 1 .076 / .067, 20
  //     .136 / .109; 32,768 points, depth 3: p = 4 K = 1 .123 / .101, FP64 K = 4
  //     .223 / .191, p = 8 K = 20 .760 / .661; nowhere slower with fewer than 32
  //     states.
  //   * On a larger one, after.  Beside it most gain (131,072 points, depth 4,
  //     p = 4, bf16: K = 4 .405 / .322, 8 .565 / .493; K = 1 and 2 0 to 2%), but
  //     where a launch is one to three workgroups per CU those placed around the
  //     near field's last ones crowd some CUs: 65,536 points, K = 7, p = 7 bf16
  //     .537 / .643, FP32 .880 / .938; 180,000 points, p = 8, bf16 K = 3
  //     .576 / .661, 4 .781 / .837.
  const bool after_near = K >= 32 || (!mfma && d.nodes > hipfmm::level_offset(4));
  if (after_near) HIPFMM_CHECK(hipStreamWaitEvent(s, e[kEvNear1], 0));
  const int ring_slot = int(P->m2l_launch_count % hipfmm_plan::kRing);
  drain_m2l_slot(P, ring_slot);
  HIPFMM_CHECK(hipEventRecord(P->m2l_ring[ring_slot][0], s));
  P->last_path = path;
  P->last_mode = P->m2l_mode;
  P->last_adjoint = adjoint;
  launch_m2l<S>(dc, path, P->last_mode, K, s);
  HIPFMM_CHECK(hipEventRecord(P->m2l_ring[ring_slot][1], s));
  P->m2l_ring_pending[ring_slot] = true;
  P->last_ring_slot = ring_slot;
  ++P->m2l_launch_count;
  P->last_m2l_expands = d.nc > 0 && d.L >= 2 && !harmonic;
  if (P->last_m2l_expands) {
    hipfmm::launch_m2l_expand<S>(d, K, 2, s);
    mark(kEvM2L, s);
  }
  launch_downward<S>(d, dc, K, s);
  mark(kEvL2L, s);
  if (!after_near) HIPFMM_CHECK(hipStreamWaitEvent(s, e[kEvNear1], 0));
  if (want_grad)
    hipfmm::launch_l2p_grad_unsort<S>(d, grad, K, s);
  else
    hipfmm::launch_l2p_unsort<S>(d, out, pot, K, s);
  P->last_done = captured ? kEvCaptured : kEvL2P;
  HIPFMM_CHECK(hipEventRecord(e[P->last_done], s));
  if (captured)
    P->capture_id = capture_id;
  else
    P->done_recorded = true;
  P->last_K = K;
  P->last_host = host;
  P->timings_pending = true;
  if (host) {
    HIPFMM_CHECK(hipEventRecord(e[kEvD2H0], s));
    if (out_bytes) HIPFMM_CHECK(hipMemcpyAsync(P->pinned_out, d.fields_out, out_bytes, hipMemcpyDeviceToHost, s));
    if (pot_bytes) HIPFMM_CHECK(hipMemcpyAsync(P->pinned_pot, d.potentials_out, pot_bytes, hipMemcpyDeviceToHost, s));
    if (grad_bytes)
      HIPFMM_CHECK(hipMemcpyAsync(P->pinned_grad, d.gradients_out, grad_bytes, hipMemcpyDeviceToHost, s));
    HIPFMM_CHECK(hipEventRecord(e[kEvD2H1], s));
    HIPFMM_CHECK(hipStreamSynchronize(s));
    if (out_bytes) std::memcpy(fields, P->pinned_out, out_bytes);
    if (pot_bytes) std::memcpy(potentials, P->pinned_pot, pot_bytes);
    if (grad_bytes) std::memcpy(field_gradients, P->pinned_grad, grad_bytes);
    finalize_timings(P);
  }
  settle.armed = false;
}

}  // namespace

extern "C" {

const char* hipfmm_last_error(void) { return g_last_error.c_str(); }

int hipfmm_debug_inject_error(int error, int skip) {
  return guarded([&] {
    require(error >= 0 && skip >= 0, "error and skip must not be negative");
    hipfmm::g_inject_countdown.store(skip);
    hipfmm::g_inject_error.store(error);
  });
}

int hipfmm_debug_plan_index_array(const hipfmm_plan* plan, const char* name, int* out, int64_t capacity,
                                  int64_t* count) {
  return guarded([&] {
    require(plan != nullptr && name != nullptr && count != nullptr, "plan, name and count must not be null");
    const DevicePlan& d = plan->d;
    const std::string n(name);
    const int64_t leaves = d.leaves;
    auto last = [&](const int* start) {
      int v = 0;
      HIPFMM_CHECK(hipMemcpy(&v, start + leaves, sizeof(int), hipMemcpyDeviceToHost));
      return int64_t(v);
    };
    const void* src = nullptr;
    int64_t elems = 0;
    if (n == "src_inv") src = d.src_inv, elems = d.ns;
    else if (n == "tgt_inv") src = d.tgt_inv, elems = d.nt;
    else if (n == "adj_self") src = plan->adj_self, elems = d.ns;
    else if (n == "p2p_tiles") src = d.p2p_tiles, elems = 2 * int64_t(d.p2p_tile_count);
    else if (n == "p2p_tiles4") src = d.p2p_tiles4, elems = 2 * int64_t(d.p2p_tile4_count);
    else if (n == "p2p_tiles16") src = d.p2p_tiles16, elems = 2 * int64_t(d.p2p_tile16_count);
    else if (n == "adj_tiles") src = plan->adj_tiles, elems = 2 * int64_t(plan->adj_tile_count);
    else if (n == "adj_tiles16") src = plan->adj_tiles16, elems = 2 * int64_t(plan->adj_tile16_count);
    else if (n == "blk8_start") src = d.blk8_start, elems = leaves + 1;
    else if (n == "blk8_src") src = d.blk8_src, elems = 2 * int64_t(d.blk8_count);
    else if (n == "nbr_blk_start") src = d.nbr_blk_start, elems = leaves + 1;
    else if (n == "nbr_blk") src = d.nbr_blk, elems = last(d.nbr_blk_start);
    else if (n == "adj_blk8_start") src = plan->adj_blk8_start, elems = leaves + 1;
    else if (n == "adj_blk8_src") src = plan->adj_blk8_src, elems = 2 * int64_t(plan->adj_blk8_count);
    else if (n == "adj_nbr_blk_start") src = plan->adj_nbr_blk_start, elems = leaves + 1;
    else if (n == "adj_nbr_blk") src = plan->adj_nbr_blk, elems = last(plan->adj_nbr_blk_start);
    else throw hipfmm::invalid_argument("unknown index array");
    *count = elems;
    if (out != nullptr && elems > 0) {
      require(capacity >= elems, "output capacity is smaller than the array");
      HIPFMM_CHECK(hipMemcpy(out, src, size_t(elems) * sizeof(int), hipMemcpyDeviceToHost));
    }
  });
}

int hipfmm_runtime_available(void) {
  try {
    const int count = gfx950_devices();
    for (int i = 0; i < count; ++i)
      if (device_is_gfx950(i)) return 1;
  } catch (...) {
  }
  return 0;
}

int hipfmm_device_description(char* buffer, size_t length) {
  return guarded([&] {
    require(buffer != nullptr && length > 0, "buffer is empty");
    std::string text;
    const int count = gfx950_devices();
    if (count == 0) {
      text = "no HIP device is available";
    } else {
      int dev = 0;
      HIPFMM_CHECK(hipGetDevice(&dev));
      hipDeviceProp_t prop;
      HIPFMM_CHECK(hipGetDeviceProperties(&prop, dev));
      text = std::string(prop.name) + " (" + prop.gcnArchName + "), " + std::to_string(prop.multiProcessorCount) +
             " CUs, " + std::to_string(prop.totalGlobalMem >> 20) + " MiB";
    }
    std::strncpy(buffer, text.c_str(), length - 1);
    buffer[length - 1] = '\0';
  });
}

int hipfmm_plan_create(const hipfmm_plan_desc* desc, hipfmm_plan** plan) {
  return guarded([&] {
    require(desc != nullptr && plan != nullptr, "descriptor and output must not be null");
    *plan = nullptr;
    require(desc->precision == 32 || desc->precision == 64, "precision must be 32 or 64");
    require(desc->order >= 0 && desc->order <= hipfmm::kMaxOrder, "expansion order must be in [0, 10]");
    require(desc->max_level >= 0 && desc->max_level <= 9, "max_level must be in [0, 9]");
    require(desc->source_count >= 0 && desc->target_count >= 0, "point counts must be non-negative");
    require((desc->source_count == 0 || desc->sorted_sources) && (desc->target_count == 0 || desc->sorted_targets),
            "positions must not be null");
    require(desc->node_ranges && desc->node_centres, "node ranges and centres must not be null");
    require((desc->source_count == 0 || desc->source_permutation) &&
                (desc->target_count == 0 || desc->target_permutation),
            "permutations must not be null");
    require(desc->m2l_class_count >= 0 && (desc->m2l_class_count == 0 || (desc->m2l_class_offsets && desc->m2l_matrices)),
            "M2L classes are inconsistent");
    require(desc->m2l_multipole_scaling && desc->m2l_local_scaling, "M2L scalings must not be null");
    require(desc->max_level == 0 || (desc->m2m_operators && desc->l2l_operators), "shift operators must not be null");
    require(desc->m2l_mode >= HIPFMM_M2L_VALU && desc->m2l_mode <= HIPFMM_M2L_MFMA_FP16X3, "unknown M2L mode");
    require(desc->precision == 32 || desc->m2l_mode == HIPFMM_M2L_VALU, "MFMA M2L modes need an FP32 plan");
    if (gfx950_devices() == 0) {
      g_last_error = "HipFull is unavailable: no HIP device";
      throw std::runtime_error(g_last_error);
    }
    auto P = std::make_unique<hipfmm_plan>();
    HIPFMM_CHECK(hipGetDevice(&P->device));
    HIPFMM_CHECK(hipStreamCreateWithFlags(&P->s_near, hipStreamNonBlocking));
    // The events between stages order kernels of this device and are read for
    // their times, so they release at device scope; the default's release to
    // the system took 3-4 us at each (1,000 points, p = 4: 95 us per evaluate,
    // now 74).  The ends of an evaluate keep it.
    for (int i = 0; i < kEvCount; ++i)
      HIPFMM_CHECK(hipEventCreateWithFlags(
          &P->ev[i], i == kEvL2P || i == kEvCaptured || i == kEvD2H1 ? hipEventDefault : hipEventDisableSystemFence));
    for (auto& pair : P->m2l_ring)
      for (auto& ev : pair) HIPFMM_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableSystemFence));
    P->device_moment_scale = desc->device_moment_scale;
    P->m2l_mode = desc->m2l_mode;
    try {
      if (desc->precision == 32)
        create_impl<float>(P.get(), *desc);
      else
        create_impl<double>(P.get(), *desc);
      require(P->m2l_mode != HIPFMM_M2L_MFMA_FP16X3 || P->d.T16_hi != nullptr,
              "the FP16 M2L mode needs M2L class matrices of harmonic form (max_level >= 2)");
    } catch (...) {
      hipfmm_plan_destroy(P.release());
      throw;
    }
    P->stats.plan_generation_count = 1;
    P->stats.static_upload_count = 1;
    *plan = P.release();
  });
}

int hipfmm_plan_evaluate(hipfmm_plan* plan, const void* moments, void* fields, int batch,
                         const int* sorted_self_indices, int memspace, void* stream) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    DeviceGuard guard(plan->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    if (plan->d.precision == 32)
      evaluate_impl<float>(plan, moments, fields, nullptr, batch, sorted_self_indices, memspace, user, false);
    else
      evaluate_impl<double>(plan, moments, fields, nullptr, batch, sorted_self_indices, memspace, user, false);
  });
}

int hipfmm_plan_evaluate_potential(hipfmm_plan* plan, const void* moments, void* fields, void* potentials, int batch,
                                   const int* sorted_self_indices, int memspace, void* stream) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    require(potentials != nullptr || plan->d.nt == 0, "potentials pointer is null");
    if (potentials == nullptr && fields == nullptr) return;  // no targets, nothing asked for
    DeviceGuard guard(plan->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    if (plan->d.precision == 32)
      evaluate_impl<float>(plan, moments, fields, potentials, batch, sorted_self_indices, memspace, user, false);
    else
      evaluate_impl<double>(plan, moments, fields, potentials, batch, sorted_self_indices, memspace, user, false);
  });
}

int hipfmm_plan_evaluate_field_gradient(hipfmm_plan* plan, const void* moments, void* gradients, int batch,
                                        const int* sorted_self_indices, int memspace, void* stream) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    require(gradients != nullptr || plan->d.nt == 0, "gradients pointer is null");
    if (gradients == nullptr) return;
    DeviceGuard guard(plan->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    if (plan->d.precision == 32)
      evaluate_impl<float>(plan, moments, nullptr, nullptr, batch, sorted_self_indices, memspace, user, false,
                           gradients);
    else
      evaluate_impl<double>(plan, moments, nullptr, nullptr, batch, sorted_self_indices, memspace, user, false,
                            gradients);
  });
}

int hipfmm_plan_evaluate_field_gradient_adjoint(hipfmm_plan* plan, const void* cotangents, void* gradients,
                                                int batch, int memspace, void* stream) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    require(gradients != nullptr || plan->d.ns == 0, "gradients pointer is null");
    if (gradients == nullptr) return;
    DeviceGuard guard(plan->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    if (plan->d.precision == 32)
      evaluate_impl<float>(plan, cotangents, nullptr, nullptr, batch, nullptr, memspace, user, true, gradients);
    else
      evaluate_impl<double>(plan, cotangents, nullptr, nullptr, batch, nullptr, memspace, user, true, gradients);
  });
}

int hipfmm_plan_evaluate_adjoint(hipfmm_plan* plan, const void* cotangents, void* gradients, int batch,
                                 int memspace, void* stream) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    DeviceGuard guard(plan->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    if (plan->d.precision == 32)
      evaluate_impl<float>(plan, cotangents, gradients, nullptr, batch, nullptr, memspace, user, true);
    else
      evaluate_impl<double>(plan, cotangents, gradients, nullptr, batch, nullptr, memspace, user, true);
  });
}

int hipfmm_plan_set_m2l_mode(hipfmm_plan* plan, int mode) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    require(mode >= HIPFMM_M2L_VALU && mode <= HIPFMM_M2L_MFMA_FP16X3, "unknown M2L mode");
    require(mode == HIPFMM_M2L_VALU || plan->d.precision == 32, "MFMA M2L modes need an FP32 plan");
    require(mode != HIPFMM_M2L_MFMA_FP16X3 || plan->d.T16_hi != nullptr,
            "the FP16 M2L mode needs M2L class matrices of harmonic form (max_level >= 2)");
    plan->m2l_mode = mode;
  });
}

int hipfmm_plan_autotune(hipfmm_plan* plan, int batch) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    require(batch >= 1 && batch <= hipfmm::kMaxBatch, "batch must be between 1 and 64 moment states");
    DeviceGuard guard(plan->device);
    const auto t0 = std::chrono::steady_clock::now();
    hipfmm_plan* P = plan;
    auto run = [&]() {
      // Device evaluate on the plan's own staging buffers (contents are
      // irrelevant to the timing).
      if (P->d.precision == 32)
        evaluate_impl<float>(P, P->d.moments_in, P->d.fields_out, nullptr, batch, nullptr, HIPFMM_DEVICE, nullptr,
                             false);
      else
        evaluate_impl<double>(P, P->d.moments_in, P->d.fields_out, nullptr, batch, nullptr, HIPFMM_DEVICE, nullptr,
                              false);
      finalize_timings(P);
    };
    // Allocate the state and zero the staging input the timed runs read.
    if (P->timings_pending) finalize_timings(P);
    if (P->d.precision == 32)
      ensure_capacity<float>(P, batch, false);
    else
      ensure_capacity<double>(P, batch, false);
    HIPFMM_CHECK(hipMemset(P->d.moments_in, 0, size_t(std::max({P->d.ns, P->d.nt, 1})) * 3 * P->d.kcap *
                                                  (P->d.precision == 32 ? 4 : 8)));
    auto best_of = [&](auto&& set, const std::vector<int>& choices, auto&& measure) {
      int best = choices.front();
      double best_t = 1e300;
      for (int c : choices) {
        set(c);
        run();  // warm
        double t = 1e300;
        for (int r = 0; r < 3; ++r) {
          run();
          t = std::min(t, measure());
        }
        if (t < best_t) {
          best_t = t;
          best = c;
        }
      }
      set(best);
      return best;
    };
    // The tile shapes matter where this batch runs on them.
    const bool tiles = P->d.precision == 32 && m2l_path<float>(P, batch) == kTileM2l;
    if (tiles && P->d.bpad / 32 <= 3) {
      std::vector<int> shapes(std::begin(hipfmm::kM2LShapes), std::end(hipfmm::kM2LShapes));
      best_of([&](int c) { P->d.m2l_shape = c; }, shapes, [&] { return P->timings.m2l_kernel_seconds; });
    }
    if (P->d.precision == 32 && batch % 32 == 0)
      // The near field overlaps the far chain and both compete for the CUs:
      // a candidate is judged by the whole evaluate, not by its own span.
      best_of([&](int c) { P->d.p2p_variant = c; }, {4, 3, 2, 1}, [&] { return P->timings.kernel_seconds; });
    P->stats.m2l_tile_shape = uint64_t(P->d.m2l_shape);
    P->stats.p2p_kernel_variant = uint64_t(P->d.p2p_variant);
    P->stats.autotune_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  });
}

int hipfmm_plan_set_launch_choices(hipfmm_plan* plan, int m2l_tile_shape, int p2p_kernel_variant) {
  return guarded([&] {
    require(plan != nullptr, "plan is null");
    const bool shape_ok = m2l_tile_shape == 0 || std::find(std::begin(hipfmm::kM2LShapes), std::end(hipfmm::kM2LShapes),
                                                           m2l_tile_shape) != std::end(hipfmm::kM2LShapes);
    require(shape_ok, "unknown M2L tile shape code");
    require(p2p_kernel_variant >= 0 && p2p_kernel_variant <= 4, "unknown near-field kernel variant");
    plan->d.m2l_shape = m2l_tile_shape;
    plan->d.p2p_variant = p2p_kernel_variant;
    plan->stats.m2l_tile_shape = uint64_t(m2l_tile_shape);
    plan->stats.p2p_kernel_variant = uint64_t(p2p_kernel_variant);
  });
}

int hipfmm_plan_statistics(const hipfmm_plan* plan, hipfmm_stats* out) {
  return guarded([&] {
    require(plan != nullptr && out != nullptr, "plan and output must not be null");
    *out = plan->stats;
    out->persistent_device_bytes = plan->persistent_bytes + plan->state_bytes;
  });
}

int hipfmm_plan_timings(const hipfmm_plan* plan, hipfmm_timings* out) {
  return guarded([&] {
    require(plan != nullptr && out != nullptr, "plan and output must not be null");
    auto* P = const_cast<hipfmm_plan*>(plan);
    DeviceGuard guard(P->device);
    finalize_timings(P);
    for (int slot = 0; slot < hipfmm_plan::kRing; ++slot) drain_m2l_slot(P, slot);
    *out = P->timings;
    out->m2l_kernel_total_seconds = P->m2l_total_seconds;
    out->m2l_kernel_launches = P->m2l_total_launches;
  });
}

int hipfmm_plan_coefficients(hipfmm_plan* plan, int which, int node, int state, double* out) {
  return guarded([&] {
    require(plan != nullptr && out != nullptr, "plan and output must not be null");
    const DevicePlan& d = plan->d;
    require(plan->last_K > 0, "no evaluation has run");
    require(node >= 0 && node < d.nodes && state >= 0 && state < plan->last_K, "node or state out of range");
    require(d.m2m_dense_c == nullptr || node >= hipfmm::level_offset(d.L),
            "this plan forms the expansions above the leaf level in harmonic-subspace form only");
    DeviceGuard guard(plan->device);
    wait_for_evaluates(plan);
    const int K = plan->last_K;
    const size_t elem = d.precision == 32 ? 4 : 8;
    if (node < 9) {  // levels 0 and 1
      std::fill(out, out + d.n, 0.0);
      return;
    }
    if (which != 0 && d.precision == 32) complete_locals<float>(plan, node);
    if (which != 0 && d.precision != 32) complete_locals<double>(plan, node);
    std::vector<unsigned char> buf(size_t(d.n) * K * elem);
    const void* base = which == 0 ? d.M : d.Lc;
    HIPFMM_CHECK(hipMemcpy(buf.data(), static_cast<const unsigned char*>(base) + size_t(node) * d.n * K * elem,
                           buf.size(), hipMemcpyDeviceToHost));
    for (int a = 0; a < d.n; ++a) {
      const size_t i = size_t(a) * K + state;
      out[a] = d.precision == 32 ? double(reinterpret_cast<const float*>(buf.data())[i])
                                 : reinterpret_cast<const double*>(buf.data())[i];
    }
  });
}

void hipfmm_plan_destroy(hipfmm_plan* plan) {
  if (plan == nullptr) return;
  int prev = -1;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(plan->device);
  if (plan->done_recorded) (void)hipEventSynchronize(plan->ev[kEvL2P]);
  if (plan->s_far) (void)hipStreamSynchronize(plan->s_far);
  if (plan->s_near) (void)hipStreamSynchronize(plan->s_near);
  free_state(plan);
  for (void* ptr : plan->persistent) (void)hipFree(ptr);
  plan->persistent.clear();
  if (plan->pinned_in) (void)hipHostFree(plan->pinned_in);
  if (plan->pinned_out) (void)hipHostFree(plan->pinned_out);
  if (plan->pinned_pot) (void)hipHostFree(plan->pinned_pot);
  if (plan->pinned_grad) (void)hipHostFree(plan->pinned_grad);
  for (auto& ev : plan->ev)
    if (ev) (void)hipEventDestroy(ev);
  for (auto& pair : plan->m2l_ring)
    for (auto& ev : pair)
      if (ev) (void)hipEventDestroy(ev);
  if (plan->s_far) (void)hipStreamDestroy(plan->s_far);
  if (plan->s_near) (void)hipStreamDestroy(plan->s_near);
  if (prev >= 0) (void)hipSetDevice(prev);
  delete plan;
}

int hipfmm_tree_leaf_order(const double* positions, int count, const double* root_centre, double root_half_width,
                           int max_level, int memspace, int* permutation, int64_t* leaf_ranges, void* stream) {
  return guarded([&] {
    require(count >= 0, "point count must be non-negative");
    require(root_centre != nullptr && leaf_ranges != nullptr && (count == 0 || (positions && permutation)),
            "arrays must not be null");
    require(memspace == HIPFMM_HOST || memspace == HIPFMM_DEVICE, "unknown memory space");
    if (gfx950_devices() == 0) throw std::runtime_error("no HIP device is available");
    const int64_t leaves = max_level >= 0 && max_level <= 9 ? int64_t(1) << (3 * max_level) : 0;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (memspace == HIPFMM_DEVICE) {
      hipfmm::device_leaf_order(positions, count, root_centre, root_half_width, max_level, permutation, leaf_ranges,
                                s);
      return;
    }
    struct Free {
      std::vector<void*> ptrs;
      ~Free() {
        for (void* p : ptrs) (void)hipFree(p);
      }
    } cleanup;
    double* pos = nullptr;
    int* perm = nullptr;
    int64_t* ranges = nullptr;
    HIPFMM_CHECK(hipMalloc(&pos, std::max<size_t>(size_t(count) * 3 * sizeof(double), 16)));
    cleanup.ptrs.push_back(pos);
    HIPFMM_CHECK(hipMalloc(&perm, std::max<size_t>(size_t(count) * sizeof(int), 16)));
    cleanup.ptrs.push_back(perm);
    HIPFMM_CHECK(hipMalloc(&ranges, std::max<size_t>(size_t(2 * leaves) * sizeof(int64_t), 16)));
    cleanup.ptrs.push_back(ranges);
    if (count) HIPFMM_CHECK(hipMemcpy(pos, positions, size_t(count) * 3 * sizeof(double), hipMemcpyHostToDevice));
    hipfmm::device_leaf_order(pos, count, root_centre, root_half_width, max_level, perm, ranges, s);
    if (count) HIPFMM_CHECK(hipMemcpy(permutation, perm, size_t(count) * sizeof(int), hipMemcpyDeviceToHost));
    HIPFMM_CHECK(hipMemcpy(leaf_ranges, ranges, size_t(2 * leaves) * sizeof(int64_t), hipMemcpyDeviceToHost));
  });
}

int hipfmm_tree_leaf_order_noalloc(const double* positions, int count, const double* root_centre,
                                   double root_half_width, int max_level, int* permutation, int64_t* leaf_ranges,
                                   void* stream) {
  return guarded([&] {
    require(count >= 0, "point count must be non-negative");
    require(root_centre != nullptr && leaf_ranges != nullptr && (count == 0 || (positions && permutation)),
            "arrays must not be null");
    require(count <= hipfmm::kNoAllocMaxPoints,
            "point count exceeds HIPFMM_NOALLOC_MAX_POINTS, the allocation-free leaf order's limit");
    if (gfx950_devices() == 0) throw std::runtime_error("no HIP device is available");
    hipfmm::device_leaf_order_noalloc(positions, count, root_centre, root_half_width, max_level, permutation,
                                      leaf_ranges, static_cast<hipStream_t>(stream));
  });
}

int hipfmm_direct_field(const double* targets, int nt, const double* sources, int ns, const double* moments,
                        const int* self_indices, double* fields) {
  return guarded([&] {
    require(nt >= 0 && ns >= 0, "counts must be non-negative");
    require((nt == 0 || (targets && fields)) && (ns == 0 || (sources && moments)), "arrays must not be null");
    if (gfx950_devices() == 0) throw std::runtime_error("no HIP device is available");
    double *t = nullptr, *s = nullptr, *m = nullptr, *f = nullptr;
    int* id = nullptr;
    struct Free {
      std::vector<void*> ptrs;
      ~Free() {
        for (void* p : ptrs) (void)hipFree(p);
      }
    } cleanup;
    auto dev = [&](auto*& ptr, const void* host, size_t bytes) {
      HIPFMM_CHECK(hipMalloc(reinterpret_cast<void**>(&ptr), std::max<size_t>(bytes, 16)));
      cleanup.ptrs.push_back(ptr);
      if (host && bytes) HIPFMM_CHECK(hipMemcpy(ptr, host, bytes, hipMemcpyHostToDevice));
    };
    dev(t, targets, size_t(nt) * 3 * sizeof(double));
    dev(s, sources, size_t(ns) * 3 * sizeof(double));
    dev(m, moments, size_t(ns) * 3 * sizeof(double));
    dev(f, nullptr, size_t(nt) * 3 * sizeof(double));
    if (self_indices) dev(id, self_indices, size_t(nt) * sizeof(int));
    hipfmm::direct_field_fp64(t, nt, s, ns, m, id, f);
    HIPFMM_CHECK(hipDeviceSynchronize());
    if (nt) HIPFMM_CHECK(hipMemcpy(fields, f, size_t(nt) * 3 * sizeof(double), hipMemcpyDeviceToHost));
  });
}

struct hipfmm_group {
  std::vector<hipfmm_plan*> plans;
  std::vector<const void*> moments;
  std::vector<void*> fields;
  std::vector<int> batches;
  hipEvent_t fork = nullptr;
  int device = 0;
};

int hipfmm_group_create(hipfmm_plan* const* plans, int count, const void* const* moments, void* const* fields,
                        const int* batches, const int* const* sorted_self_indices, hipfmm_group** group) {
  return guarded([&] {
    require(group != nullptr, "group output is null");
    *group = nullptr;
    require(count >= 1 && plans != nullptr && moments != nullptr && fields != nullptr && batches != nullptr,
            "a group needs at least one plan with operands");
    for (int i = 0; i < count; ++i) {
      require(plans[i] != nullptr, "plan is null");
      for (int j = 0; j < i; ++j) require(plans[j] != plans[i], "a plan may appear once in a group");
      require(plans[i]->device == plans[0]->device, "the plans of a group share one device");
      require(batches[i] >= 1 && batches[i] <= hipfmm::kMaxBatch, "batch must be between 1 and 64 moment states");
      const hipfmm::DevicePlan& d = plans[i]->d;
      require(moments[i] != nullptr || d.ns == 0, "moments pointer is null");
      require(fields[i] != nullptr || d.nt == 0, "fields pointer is null");
    }
    DeviceGuard guard(plans[0]->device);
    auto G = std::make_unique<hipfmm_group>();
    G->device = plans[0]->device;
    G->plans.assign(plans, plans + count);
    G->moments.assign(moments, moments + count);
    G->fields.assign(fields, fields + count);
    G->batches.assign(batches, batches + count);
    // Everything that allocates or waits happens here, not at launch.
    for (int i = 0; i < count; ++i) {
      hipfmm_plan* P = plans[i];
      if (sorted_self_indices != nullptr) install_identity(P, sorted_self_indices[i]);
      if (P->timings_pending) finalize_timings(P);
      far_stream(P);
      if (P->d.precision == 32)
        ensure_capacity<float>(P, batches[i], false);
      else
        ensure_capacity<double>(P, batches[i], false);
    }
    HIPFMM_CHECK(hipEventCreateWithFlags(&G->fork, hipEventDisableTiming));
    *group = G.release();
  });
}

int hipfmm_group_launch(hipfmm_group* group, void* stream) {
  return guarded([&] {
    require(group != nullptr, "group is null");
    DeviceGuard guard(group->device);
    const hipStream_t user = static_cast<hipStream_t>(stream);
    // One fork point for every plan, then one join per plan: the plans' own
    // streams run concurrently between them.
    HIPFMM_CHECK(hipEventRecord(group->fork, user));
    for (size_t i = 0; i < group->plans.size(); ++i) {
      hipfmm_plan* P = group->plans[i];
      if (P->d.precision == 32)
        evaluate_impl<float>(P, group->moments[i], group->fields[i], nullptr, group->batches[i], nullptr,
                             HIPFMM_DEVICE, user, false, nullptr, group->fork);
      else
        evaluate_impl<double>(P, group->moments[i], group->fields[i], nullptr, group->batches[i], nullptr,
                              HIPFMM_DEVICE, user, false, nullptr, group->fork);
    }
    for (hipfmm_plan* P : group->plans) HIPFMM_CHECK(hipStreamWaitEvent(user, P->ev[P->last_done], 0));
  });
}

void hipfmm_group_destroy(hipfmm_group* group) {
  if (group == nullptr) return;
  int prev = -1;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(group->device);
  if (group->fork) (void)hipEventDestroy(group->fork);
  if (prev >= 0) (void)hipSetDevice(prev);
  delete group;
}

}  // extern "C"
