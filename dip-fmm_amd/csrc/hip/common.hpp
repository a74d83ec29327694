// Internal declarations shared by the HipFull device translation units.
//
// Device data layout (HBM), for a plan of order p (n coefficients), leaf
// level L, N_s sources, N_t targets, batch K moment states:
//   positions     sorted, split as float4 hi + float4 lo (FP32 plans) or
//                 double4 (FP64 plans); plus leaf-relative offsets (float4 /
//                 double4) rounded once from FP64 on the host
//   moments       sm[source][3][K]        (sorted, k fastest)
//   multipoles    M[node][n][K]           (node-major, level by level)
//   locals        Lc[node][n][K]
//   near field    Hn[target][3][K]        (sorted)
//   fields out    out[k][user target][3]
// Boxes of one level are addressed by their Morton index; a child's node is
// level_offset(l+1) + 8*parent_morton + class, so the 8 children of a parent
// are contiguous and the list-1/list-2 neighbourhoods are enumerated from
// integer box offsets instead of stored lists.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <stdexcept>
#include <string>
#include <vector>

namespace hipfmm {

constexpr int kMaxBatch = 64;
constexpr int kMaxLevels = 11;  // tree levels 0..10 of a plan
// bf16 values of one three-piece box operator of R rows and depth D.
__host__ __device__ inline int64_t box_x3_elems(int R, int D) {
  return int64_t(3) * ((D + 31) / 32) * ((R + 15) / 16 * 16) * 32;
}
// Tiles per workgroup of the matrix-core M2L shapes (4 waves x 1..5 tiles).
constexpr int kM2LGroupTiles[5] = {4, 8, 12, 16, 20};
constexpr int kM2LSparseTiles = 8;
constexpr int kMaxOrder = 10;
constexpr int kOffsetSlots = 343;  // (dx,dy,dz) in [-3,3]^3

struct hip_error : std::runtime_error {
  using std::runtime_error::runtime_error;
};
struct invalid_argument : std::invalid_argument {
  using std::invalid_argument::invalid_argument;
};

// `actual`, or the error armed by hipfmm_debug_inject_error once its
// countdown of successful checked calls runs out.
hipError_t injected_error(hipError_t actual);

#define HIPFMM_CHECK(expr)                                                                   \
  do {                                                                                       \
    const hipError_t hipfmm_err_ = ::hipfmm::injected_error(expr);                           \
    if (hipfmm_err_ != hipSuccess) {                                                         \
      (void)hipGetLastError(); /* clear the sticky copy so later checks see fresh state */   \
      throw ::hipfmm::hip_error(std::string(#expr) + ": " + hipGetErrorString(hipfmm_err_)); \
    }                                                                                        \
  } while (0)

__host__ __device__ inline int coefficient_count(int p) { return (p + 1) * (p + 2) * (p + 3) / 6; }
__host__ __device__ inline int64_t level_offset(int level) { return ((int64_t(1) << (3 * level)) - 1) / 7; }
__host__ __device__ inline int offset_slot(int dx, int dy, int dz) { return (dx + 3) * 49 + (dy + 3) * 7 + (dz + 3); }

// Spread the low 10 bits of v to every third bit (bit b -> bit 3b).
__host__ __device__ inline uint32_t spread3(uint32_t v) {
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}
// Morton index of box (x, y, z) at a level of `bits` bits per axis (<= 10):
// bit b of x, y, z goes to bit 3b, 3b+1, 3b+2.
__host__ __device__ inline uint32_t morton3(uint32_t x, uint32_t y, uint32_t z, int bits) {
  const uint32_t mask = bits >= 10 ? 0x3ffu : (1u << bits) - 1u;
  return spread3(x & mask) | (spread3(y & mask) << 1) | (spread3(z & mask) << 2);
}
// Inverse of spread3: gather every third bit (bit 3b -> bit b).
__host__ __device__ inline uint32_t compact3(uint32_t v) {
  v &= 0x09249249u;
  v = (v ^ (v >> 2)) & 0x030c30c3u;
  v = (v ^ (v >> 4)) & 0x0300f00fu;
  v = (v ^ (v >> 8)) & 0x030000ffu;
  v = (v ^ (v >> 16)) & 0x3ffu;
  return v;
}
__host__ __device__ inline void demorton3(uint32_t m, int bits, int& x, int& y, int& z) {
  const uint32_t mask = bits >= 10 ? 0x3ffu : (1u << bits) - 1u;
  x = int(compact3(m) & mask);
  y = int(compact3(m >> 1) & mask);
  z = int(compact3(m >> 2) & mask);
}

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b on XCD
// b % 8), and each XCD has its own L2.  This bijection of [0, blocks) hands
// XCD x one contiguous range of logical blocks instead of every 8th one, so
// work items that share inputs (the near-field tiles of neighbouring leaves,
// the tiles of one leaf) read them through one L2.
__device__ inline int xcd_contiguous_block(int b, int blocks) {
  const int q = blocks >> 3, r = blocks & 7, x = b & 7, i = b >> 3;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

template <class S>
struct Vec4;
template <>
struct Vec4<float> {
  using type = float4;
};
template <>
struct Vec4<double> {
  using type = double4;
};

// Sparse shift operator (M2M or L2L) shared by all levels and child classes:
// CSR over output coefficients, values per (level, class).
struct ShiftCsr {
  int nnz = 0;
  int* row_offsets = nullptr;  // n+1
  int* columns = nullptr;      // nnz
  void* values = nullptr;      // (L+1) x 8 x nnz scalars (levels 1..L used)
};

__host__ __device__ inline bool bit_of(const uint32_t* bits, int64_t node) { return (bits[node >> 5] >> (node & 31)) & 1u; }

// Everything the kernels read, with device pointers.
struct DevicePlan {
  int precision = 32;
  int p = 0, n = 0, nm = 0;  // nm: coefficients of order p-1 (monomials used by P2M/L2P)
  int L = 0;
  int ns = 0, nt = 0;
  int64_t nodes = 0, leaves = 0;
  // geometry
  void* src_pos = nullptr;  // FP32: 2*ns float4 (hi block then lo block); FP64: ns double4
  void* tgt_pos = nullptr;
  void* src_rel = nullptr;  // ns float4/double4 leaf-relative offsets
  void* tgt_rel = nullptr;
  int* src_perm = nullptr;  // sorted index -> user index
  int* tgt_perm = nullptr;
  int* src_inv = nullptr;   // user index -> sorted index
  int* tgt_inv = nullptr;
  int* self = nullptr;      // nt sorted self indices (-1 none)
  int2* leaf_src = nullptr; // per leaf [begin, end)
  int2* leaf_tgt = nullptr;
  int2* p2p_tiles = nullptr; // (leaf, first row) of each 32-row near-field tile; row = 3*target + component
  int p2p_tile_count = 0;
  int2* p2p_tiles4 = nullptr; // the same with the potential: row = 4*target + (component or 3 = potential)
  int p2p_tile4_count = 0;
  int2* p2p_tiles16 = nullptr; // (leaf, first target) of each 16-target tile (targets-as-rows kernel)
  int p2p_tile16_count = 0;
  // Moments of the bf16 three-piece near field, in blocks of 8 sources of
  // one leaf: leaf l's sources fill blocks [blk8_start[l], blk8_start[l+1]);
  // blk8_src[b] = (first source, sources in the block).
  int* blk8_start = nullptr;
  int2* blk8_src = nullptr;
  int blk8_count = 0;
  int* nbr_blk_start = nullptr;  // per target leaf: its neighbourhood's blocks are
  int* nbr_blk = nullptr;        // nbr_blk[nbr_blk_start[l] .. nbr_blk_start[l+1])
  void* smb = nullptr;         // bf16 [block][3 components][3 pieces][K][8 sources]
  int smb_blocks = 0;          // blocks smb holds (both roles)
  // basis tables
  int4* p2m_tab = nullptr;  // per alpha: index(alpha-e_c) or -1 for c=0..2, w = sign (+1/-1)
  int4* l2p_up = nullptr;   // per g of degree < p: index(g + e_c) for c = 0..2
  // operators
  void* m2l_T = nullptr;     // FP32/FP64 class matrices, column-major [class][alpha][beta] (plans without harmonic form)
  // Harmonic form: the class matrices C_o in fragment order (m2l_full.hip), the
  // 189 offsets of each parity as dilated Morton steps (x, y, z, class), and a
  // box of zeros at the largest batch (the source of columns without one).
  void* m2l_fragments = nullptr;
  int4* m2l_steps = nullptr;
  void* m2l_zero_box = nullptr;
  int* m2l_slot = nullptr;   // 343 slot -> class index or -1
  int4* parity_offsets = nullptr;  // [8 parities][189] (ox, oy, oz, class) list-2 offsets
  // Order of the target parents over the tiles of the matrix-core M2L (one
  // box per tile), per workgroup tile count kM2LGroupTiles[g] and level:
  // m2l_order[m2l_order_base[g][level] + i] is the Morton index of the
  // parent of tile i, or -1 for a padding tile; m2l_order_len[g][level]
  // tiles.  Parents are grouped by boundary class so that the boxes of one
  // workgroup have the same list-2 offsets inside the grid.
  int* m2l_order = nullptr;
  int m2l_order_base[5][kMaxLevels] = {};
  int m2l_order_len[5][kMaxLevels] = {};
  // Where many boxes hold no points (null otherwise; plan.hip gives the line):
  // a bit per node that holds sources and one per node that holds targets, and
  // the tile order of kM2LSparseTiles tiles per workgroup over the boxes that
  // hold targets: the parent of tile i of a parity is sparse_order[
  // sparse_base[level] + parity * sparse_len[level] + i].  The M2L leaves out
  // sources without moments (zeros), and the locals of boxes without targets,
  // which no target reads.
  const uint32_t* source_bits = nullptr;
  const uint32_t* target_bits = nullptr;
  const int* sparse_order = nullptr;
  int sparse_base[kMaxLevels] = {};
  int sparse_len[kMaxLevels] = {};
  void* ms = nullptr;        // (L+1) x n
  void* ls = nullptr;
  ShiftCsr m2m, l2l;
  // The same operators dense and transposed, [(level*8 + class)][col][NP]
  // with NP = n rounded up to 8 (rows n..NP-1 zero), levels 0..L.
  void* m2m_dense = nullptr;
  void* l2l_dense = nullptr;
  // Harmonic-subspace shift operators (same layout, nc rows/columns, NP =
  // nc rounded up to 8): Mc_parent = sum_c A_c Mc_child and Lcc_child +=
  // B_c Lcc_parent, with the level scalings folded in.  Null: the upward and
  // downward passes run on the full n coefficients.
  void* m2m_dense_c = nullptr;
  void* l2l_dense_c = nullptr;
  // state (capacity K)
  int kcap = 0;
  void* moments_in = nullptr;  // host-path staging: K x ns x 3
  void* fields_out = nullptr;  // host-path staging: K x nt x 3
  void* potentials_out = nullptr;  // host-path staging: K x nt (with the potential buffers)
  void* sm = nullptr;
  void* M = nullptr;
  void* Lc = nullptr;
  void* Hn = nullptr;
  void* Pn = nullptr;          // near-field potential Pn[target][K] (allocated once a potential is asked for)
  void* Gn = nullptr;          // near-field field gradient Gn[target][6][K] (allocated once asked for)
  void* gradients_out = nullptr;  // host-path staging: K x nt x 6
  int* grad_up = nullptr;      // [g][8], g of degree <= p - 2: index of g + e_c + e_j (6 used)
  double potential_scale = 1.0;  // frame factor of the potential (root width W for FP32 plans)
  // Harmonic-subspace M2L: L = Q sum_o C_o P M with the level scalings folded
  // into P and Q (nc = 0: the M2L runs on the full n coefficients).
  int nc = 0;
  void* cmp_op = nullptr;  // [(level)][alpha n][NPc] = P[r][alpha] * ms[level][alpha], NPc = nc rounded up to 16
  void* exp_op = nullptr;  // [(level)][r nc][NP]    = ls[level][beta] * Q[beta][r], NP = n rounded up to 8
  // The box-product operators as three-piece bf16 A fragments of
  // v_mfma_f32_16x16x32_bf16 (FP32 harmonic plans; null otherwise): per
  // operator [piece][32-deep step][row, padded to 16][32], box_x3_elems
  // bf16 values.  cmp/exp per level; m2m/l2l per (level, child class) of the
  // operators this view's box kernels use (the harmonic ones: m2m_x3_c,
  // l2l_x3_c, which plan.hip hands to the compressed view).
  void* cmp_x3 = nullptr;
  void* exp_x3 = nullptr;
  void* m2m_x3 = nullptr;
  void* l2l_x3 = nullptr;
  void* m2m_x3_c = nullptr;
  void* l2l_x3_c = nullptr;
  // Where no kernel of far.hip's K = 32 n forms runs, a node's compressed
  // coefficients lie [K][nc] instead of [nc][K] (compressed_state_major): the
  // depth of the M2L's columns is contiguous at every K.  state_major says the
  // same of M and Lc as this view sees them (the compressed view).
  bool compressed_state_major = false;
  bool state_major = false;
  void* Mc = nullptr;      // compressed multipoles [node][nc][K]
  void* Lcc = nullptr;     // compressed locals [node][nc][K] (M2L output)
  // MFMA operands
  void* mt_hi = nullptr;  // bf16/fp16 [node][K][apad]
  void* mt_lo = nullptr;
  int64_t mt_zero_offset = 0;  // byte offset of the 1 KiB zero block that follows each of mt_hi / mt_lo
  void* T_hi = nullptr;   // [class][bpad][apad] 16-bit, MFMA fragment order
  void* T_lo = nullptr;
  void* ls_pad = nullptr; // (L+1) x bpad float local scaling (0 beyond n)
  // FP16 mode (harmonic form only).  The class matrices enter as
  // rho_j C_o sigma_k (j, k the degrees of row and column, rho and sigma
  // powers of two that centre every degree block high in FP16's range), split
  // into fp16 hi/lo; the compressed multipoles as 2^e_l Mc / sigma_k, with e_l
  // from the level's largest value in the current evaluate; the epilogue
  // multiplies by 2^-e_l / rho_j.
  void* T16_hi = nullptr;
  void* T16_lo = nullptr;
  void* ls16_pad = nullptr;          // (L+1) x bpad float: 1 / rho of each row
  void* col16_scale = nullptr;       // apad float: 1 / sigma of each column (0 beyond nc)
  unsigned* lvl_max_bits = nullptr;  // L+1: largest |Mc / sigma| per level (float bits)
  const void* zero_block = nullptr;  // 1 KiB of zeros: the operand of sources outside the grid
  int apad = 0, bpad = 0;
  int mfma_depth_steps = 0;  // 16-deep steps the MFMA M2L reads (<= apad / 16; 0 = apad / 16)
  // Launch choices (set by the autotuner; 0 = built-in default).
  int m2l_shape = 0;    // MFMA M2L tile shape code (kM2LShapes)
  int p2p_variant = 0;  // near field at K % 32 == 0 (FP32): 1 vector ALU, 2 matrix cores with
                        // (target, component) rows, 3 matrix cores with target rows, 4 (= default)
                        // matrix cores on bf16 three-piece operands
};

// MFMA M2L tile shapes of the harmonic form (<= 3 row tiles): the code is
// 10 * (column tiles per wave) + (ring stages).
constexpr int kM2LShapes[] = {23, 13, 43, 53, 24, 34, 26};

// Kernel launchers (one translation unit each).
template <class S>
void launch_gather(const DevicePlan& d, const S* user_moments, S scale, int K, hipStream_t s);
template <class S>
void launch_p2m(const DevicePlan& d, int K, hipStream_t s);
template <class S>
void launch_m2m(const DevicePlan& d, int parent_level, int K, hipStream_t s);
template <class S>
void launch_l2l(const DevicePlan& d, int child_level, int K, hipStream_t s);
// M2L of all levels 2..L in the type's own precision: on the matrix cores for
// the harmonic form (d seen through the compressed view: n = nc, M = Mc,
// Lc = Lcc), on the vector ALUs otherwise.
template <class S>
void launch_m2l_full(const DevicePlan& d, int K, hipStream_t s);
template <class S>
void launch_m2l_valu(const DevicePlan& d, int K, hipStream_t s);
// The bf16 mode's M2L for small batches (same view, state-major; needs no
// split operands).
void launch_m2l_bf16_direct(const DevicePlan& d, int K, hipStream_t s);
// Operands of launch_m2l_full, built with the plan: class matrices C[row + n * depth]
// in fragment order, and one parity offset with its class.
std::vector<float> m2l_fragments_f32(int n, const std::vector<double>& C, int classes);
std::vector<double> m2l_fragments_f64(int n, const std::vector<double>& C, int classes);
int4 m2l_step(int ox, int oy, int oz, int cls);
template <class S>
void launch_p2p(const DevicePlan& d, int K, bool potential, hipStream_t s);
// State counts from which FP32 batches that are no multiple of 32 may take the
// matrix cores (near.hip gives the whole rule): fields with and without
// potentials, and gradients.
constexpr int kNearBf16States = 9, kNearGradBf16States = 7;
// The vector-ALU near field (near_lanes.hip): any K, FP32 and FP64.
template <class S>
void launch_p2p_lanes(const DevicePlan& d, int K, bool potential, hipStream_t s);
template <class S>
void launch_p2p_grad_lanes(const DevicePlan& d, int K, hipStream_t s);
// Leaf order of `count` points (device arrays; tree.hip): the stable sort by
// leaf Morton index into permutation[sorted] = input index, and leaf_ranges
// [2 * leaf] = {begin, end} (count, count for an empty leaf).
void device_leaf_order(const double* positions, int count, const double* centre, double half_width, int L,
                       int* permutation, int64_t* leaf_ranges, hipStream_t s);
// The same with the scratch in a fixed per-device array instead of device
// allocations, for count <= kNoAllocMaxPoints; calls that overlap on one
// device share that array and race.
constexpr int kNoAllocMaxPoints = 1 << 21;
void device_leaf_order_noalloc(const double* positions, int count, const double* centre, double half_width, int L,
                               int* permutation, int64_t* leaf_ranges, hipStream_t s);
// Near-field index arrays built on the device from the leaf ranges
// (ranges[leaf] = [begin, end) of the sorted points, device memory), into
// arrays from `alloc`; all calls return once the arrays are complete.
using DeviceAllocator = std::function<void*(size_t bytes)>;
// Tiles (leaf, first row) of `step` rows over mult x (end - begin) rows per
// leaf, leaves in order; returns the count.
int device_tiles(const int2* ranges, int64_t leaves, int mult, int step, int2** out, const DeviceAllocator& alloc,
                 hipStream_t s);
// Blocks of 8 sources per leaf (start: leaves + 1 offsets; src: (first,
// count) per block) and per target leaf the blocks of its in-grid 3x3x3
// neighbourhood (nbr_start: leaves + 1 offsets into nbr), neighbours in the
// order dz, dy, dx from -1 to 1.
void device_blocks8(const int2* ranges, int L, int64_t leaves, int** start, int2** src, int* count, int** nbr_start,
                    int** nbr, const DeviceAllocator& alloc, hipStream_t s);
// inv[perm[j]] = j; false when perm (device memory) is not a permutation.
bool device_inverse(const int* perm, int count, int* inv, hipStream_t s);
// Field gradient dH_c/dx_j: near part into Gn, far part from the leaf locals
// plus Gn, unsorted to out[k][user target][6] (xx xy xz yy yz zz).
template <class S>
void launch_p2p_grad(const DevicePlan& d, int K, hipStream_t s);
template <class S>
void launch_l2p_grad_unsort(const DevicePlan& d, S* gradients, int K, hipStream_t s);
// Far field from the leaf locals plus the near field, unsorted to user
// order: fields out[k][target][3] (may be null when potentials are asked
// for) and potentials pot[k][target] (null: fields only).
template <class S>
void launch_l2p_unsort(const DevicePlan& d, S* fields, S* potentials, int K, hipStream_t s);
template <class S>
void launch_zero(S* ptr, size_t count, hipStream_t s);
// The same operations for any number of states, FP32 and FP64 (columns.hip):
// what the launchers above use where the batch is no multiple of 32 FP32
// states.
template <class S>
void launch_p2m_columns(const DevicePlan& d, int K, hipStream_t s);
template <class S>
void launch_m2m_columns(const DevicePlan& d, int parent_level, int K, hipStream_t s);
template <class S>
void launch_l2l_columns(const DevicePlan& d, int child_level, int K, hipStream_t s);
template <class S>
void launch_compress_columns(const DevicePlan& d, int level, int K, hipStream_t s);
template <class S>
void launch_expand_columns(const DevicePlan& d, int level, int K, hipStream_t s);
template <class S>
void launch_l2p_columns(const DevicePlan& d, S* fields, S* potentials, int K, hipStream_t s);
template <class S>
void launch_l2p_grad_columns(const DevicePlan& d, S* gradients, int K, hipStream_t s);

void launch_m2l_split(const DevicePlan& d, int K, int mode, hipStream_t s);  // all levels 2..L
// Harmonic-subspace transforms around the M2L, levels first_level..L (at
// least 2): M -> Mc, and Lcc -> Lc.
template <class S>
void launch_m2l_compress(const DevicePlan& d, int K, int first_level, hipStream_t s);
template <class S>
void launch_m2l_expand(const DevicePlan& d, int K, int first_level, hipStream_t s);
// bf16 hi/lo split of the compressed multipoles (levels 2..L) into the MFMA
// operand layout, for plans whose upper levels are formed in compressed form.
void launch_m2l_bf16_split(const DevicePlan& d, int K, hipStream_t s);
void launch_m2l_mfma(const DevicePlan& d, int K, int mode, hipStream_t s);   // all levels 2..L
// Columns per box of the 16-bit M2L operands at K states, given the mt buffers,
// and of buffers for batches of up to K.
int m2l_operand_states(const DevicePlan& d, int K);
int m2l_operand_capacity(const DevicePlan& d, int K);
void prepare_mfma_operators(DevicePlan& d, int n, const std::vector<double>& matrices, int classes,
                            const std::vector<double>& local_scaling, std::vector<void*>& allocations, size_t& bytes);
// FP16 operators of the harmonic form (n = nc); call after prepare_mfma_operators.
void prepare_mfma_fp16_operators(DevicePlan& d, int n, const std::vector<double>& matrices, int classes, int order,
                                 std::vector<void*>& allocations, size_t& bytes);
// FP16 mode operands: per-level maxima of Mc, then the scaled fp16 split.
void launch_m2l_fp16_split(const DevicePlan& d, int K, hipStream_t s);

// Harmonic subspace factorisation of the M2L class matrices (host, FP64):
// T_o = Q C_o P with orthonormal block-diagonal bases; nc = 0 when the
// matrices are not of that form.
struct HarmonicBasis {
  // Compressed index r holds the harmonic basis function (r + 1) mod nc of
  // the degree-major order (degree j at j^2 .. (j+1)^2 - 1): degree 0 last.
  int nc = 0;              // (p+1)^2, or 0
  std::vector<double> P;   // nc x n row-major: compressed multipole = P * multipole
  std::vector<double> Q;   // n x nc row-major: local = Q * compressed local
  std::vector<double> C;   // classes x nc x nc, column-major C[beta' + nc*alpha']
  double max_reconstruction_error = 0.0;
};
HarmonicBasis harmonic_m2l_basis(int p, const double* T, int classes);

void direct_field_fp64(const double* targets, int nt, const double* sources, int ns, const double* moments,
                       const int* self, double* fields);

}  // namespace hipfmm
