// M2L on the CDNA4 matrix cores (v_mfma_f32_32x32x16_bf16).
//
// Same regrouped contraction as the VALU path (m2l_valu.hip):
//   L[t][b] = ls[l][b] * sum_{o in list2 offsets} sum_a T_o[b][a] * Mt[t-o][a],
//   Mt[s][a] = ms[l][a] * M[s][a]
// written as one GEMM per offset class: A = T_o (rows b, depth a), B = the
// gathered source columns (depth a, columns = target box x moment state).
//
// Work decomposition (one launch covers every level 2..L):
//   * a workgroup holds W waves and owns W*NB tiles of 32 output columns of
//     one parity class at one level; each wave owns NB tiles and every row
//     tile of L for them (n rounded up to 32 rows), so each local is written
//     once and no atomics are needed;
//   * the workgroup walks (depth step ks, offset o) with ks outermost: for a
//     fixed ks the sources of all resident workgroups are one 16-deep slice
//     of the multipoles, which stays in L2 / the last-level cache while the
//     189 offsets of the parity are applied;
//   * offsets are ordered by their coordinate parity (the host table), so
//     consecutive offsets of the same class read sources shifted by one
//     lattice step of the target parity and re-hit L2;
//   * operands of a step (the class matrix slice T_o[ks], hi and lo, shared
//     by the workgroup; each wave's source fragments) are fetched straight
//     into LDS by global_load_lds DMA, kStages - 1 steps ahead, into a ring
//     of kStages slots; one barrier per step
//     publishes a slot to every wave and frees the oldest one;
//   * block b -> parity b % 8, so the 8 XCDs each serve one parity class and
//     keep its class matrices in their own L2; consecutive workgroups of one
//     XCD hold spatially consecutive tiles.
//
// Precision: FP32 operands are split x = hi + lo with hi = bf16(x) and
// lo = bf16(x - hi) (16 significant bits), and each product is formed as
// hi*hi + hi*lo + lo*hi with FP32 accumulation on the matrix cores.
//
// Data layout:
//   T_hi/T_lo  [class][depth step][row tile][lane][8] bf16 -- MFMA A-fragment
//              order (lane i: row i%32, depth 8*(i/32)..+7 of the 16-deep
//              step), so the slice of one step is MT contiguous 1 KiB blocks
//   mt_hi/lo   [node][depth step][state][16] bf16 -- a B fragment (column =
//              lane%32 -> state, depth 8*(i/32)..+7) is one 16-byte load and
//              the 32 columns of a step form one contiguous 1 KiB block
#include <cmath>
#include <cstdlib>
#include <string>

#include "common.hpp"

namespace hipfmm {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4;  // waves per workgroup (one per SIMD)
constexpr int kParityOffsets = 189;

// s_waitcnt immediate (gfx9 encoding): at most `vm` vector-memory operations
// outstanding, every LDS operation complete.
constexpr int wait_vm_lgkm0(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }

// 16 bytes per lane from global memory straight into LDS: lane i writes
// lds_wave_base[i] (M0 holds the wave-uniform LDS address; one wait state
// separates the M0 write from its use).  Issued as inline assembly so the
// compiler's wait insertion does not track it: that tracking loses the ring
// slot a DMA wrote at the step's branches and would then wait for every DMA
// in flight before each LDS read.  Ordering is explicit instead: the
// pre-barrier s_waitcnt of each step.  The compiler keeps no value of its
// own in M0 in this kernel (it uses M0 only for its own LDS DMA and message
// instructions, which the kernel does not contain).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ uint32_t lds_address(const uint4* p) {
  return uint32_t(uintptr_t((const __attribute__((address_space(3))) uint4*)p));
}
// Per-lane 64-bit source address.
__device__ __forceinline__ void lds_dma16(const uint4* src, const uint4* lds_wave_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src),
               "s"(lds_address(lds_wave_base))
               : "memory", "m0");
}
// Wave-uniform base plus a per-lane 32-bit byte offset.  Callers pass a base
// that is the same on every lane; it is moved to an SGPR pair explicitly.
__device__ __forceinline__ void lds_dma16_sbase(const void* base, uint32_t lane_bytes, const uint4* lds_wave_base) {
  const uint64_t b = uint64_t(uintptr_t(base));
  const uint64_t sb = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(b))))) |
                      (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(b >> 32))))) << 32);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(sb),
               "s"(lds_address(lds_wave_base))
               : "memory", "m0");
}
// Array base (a kernel argument: the same on every lane) plus a per-lane
// 32-bit byte offset.
__device__ __forceinline__ void lds_dma16_voff(const void* base, uint32_t lane_bytes, const uint4* lds_wave_base) {
  const uint64_t b = uint64_t(uintptr_t(base));
  const uint64_t sb = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(b))))) |
                      (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(b >> 32))))) << 32);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(sb),
               "s"(lds_address(lds_wave_base))
               : "memory", "m0");
}
#pragma clang diagnostic pop

__host__ __device__ inline uint16_t bf16_bits(float x) {
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  if ((u & 0x7f800000u) == 0x7f800000u) return uint16_t(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);                                   // round to nearest even
  return uint16_t(u >> 16);
}
__host__ __device__ inline float bf16_value(uint16_t h) { return __builtin_bit_cast(float, uint32_t(h) << 16); }

// Power-of-two exponent e of a level's FP16 operand scale: the level's
// largest |Mc / sigma| (float bits) times 2^e lies in [2^14, 2^15), the top
// binade below FP16's largest finite value, so that the lo half of the split
// of every value above 2^-3 is a normal FP16 number; 0 for an empty or
// non-finite maximum.
__host__ __device__ inline int fp16_level_exponent(unsigned max_bits) {
  const int biased = int((max_bits >> 23) & 0xffu);
  if (max_bits == 0u || biased == 0 || biased == 255) return 0;
  return 15 - (biased - 126);
}

__device__ inline int level_of_node(int64_t node) {
  int level = 0;
  while (level_offset(level + 1) <= node) ++level;
  return level;
}

// One workgroup per (box at level >= 2, chunk of kc moment states):
// transpose M[node][a][k] into the fragment layout, scale by ms and split
// into hi/lo bf16 halves; padding depth entries are zero.
__global__ void __launch_bounds__(256) split_kernel(const DevicePlan d, int K, int kc) {
  extern __shared__ float tile[];  // n x kc
  const int n = d.n, AP = d.apad, KS = AP / 16;
  const int k0 = blockIdx.y * kc;
  const int64_t node = level_offset(2) + blockIdx.x;
  const int level = level_of_node(node);
  const float* M = static_cast<const float*>(d.M) + node * int64_t(n) * K;
  for (int w = threadIdx.x; w < n * kc; w += blockDim.x) {
    const int a = w / kc, k = k0 + w % kc;
    tile[w] = k < K ? M[a * K + k] : 0.0f;
  }
  __syncthreads();
  const float* ms = static_cast<const float*>(d.ms) + int64_t(level) * n;
  uint16_t* hi = static_cast<uint16_t*>(d.mt_hi);
  uint16_t* lo = static_cast<uint16_t*>(d.mt_lo);
  const int kn = min(kc, K - k0);
  for (int w = threadIdx.x; w < kn * AP; w += blockDim.x) {
    const int k = w / AP, a = w % AP;  // consecutive threads: consecutive depth
    const float x = a < n ? ms[a] * tile[a * kc + k] : 0.0f;
    const uint16_t h = bf16_bits(x);
    const int64_t at = ((node * KS + a / 16) * K + k0 + k) * 16 + a % 16;
    hi[at] = h;
    lo[at] = bf16_bits(x - bf16_value(h));
  }
}


struct LevelTable {
  int count;  // entries, each a run of blocks of one level
  int states;  // moment states of the output; the operands may hold more columns
  int level[12];
  int block_begin[12];
  int blocks_per_parity[12];
  int tiles[12];  // 32-column tiles per parity
  int cols_per_box[12];
  int kchunks[12];
  // One box per tile: the parent of tile group t is order[order_base + t]
  // (-1: padding); null when tiles follow the Morton order of the parents.
  const int* order;
  int order_base[12];
  int order_stride[12];  // from one parity's order to the next (0: they share one)
};

// Morton index of the parent of tile group bg (-1 for a padding tile).
__device__ __forceinline__ int64_t tile_parent(const LevelTable& lt, int li, int parity, int bg) {
  return lt.order ? int64_t(lt.order[lt.order_base[li] + parity * lt.order_stride[li] + bg]) : int64_t(bg);
}

// False for a source box known to hold no sources: its operands are zeros.
__device__ __forceinline__ bool holds_sources(const DevicePlan& d, int64_t node) {
  return d.source_bits == nullptr || bit_of(d.source_bits, node);
}

// Per-lane view of the columns of the NB tiles one wave owns.  With
// kUniformBox (32 states per box, K a multiple of 32) every column of a tile
// belongs to the same box, so the box coordinates are wave-uniform.
template <int NB>
struct Columns {
  bool valid[NB];
  int tx[NB], ty[NB], tz[NB], kk[NB];
};

template <int NB>
__device__ __forceinline__ bool source_inside(const Columns<NB>& c, int nb, int ox, int oy, int oz, int nbox, int& sx,
                                              int& sy, int& sz) {
  sx = c.tx[nb] - ox;
  sy = c.ty[nb] - oy;
  sz = c.tz[nb] - oz;
  return c.valid[nb] & (sx >= 0) & (sy >= 0) & (sz >= 0) & (sx < nbox) & (sy < nbox) & (sz < nbox);
}

struct StepGeometry {
  int K, KS, KD, level, nbox, nsteps;  // KS: 16-deep slices per box (stride); KD: slices multiplied
  int64_t lvl0;
};

// Per-workgroup step tables of the uniform-box path, built once: for each
// used offset, the byte offset of its class-matrix block in T_hi/T_lo and,
// per tile, the byte offset of the source box's block in mt_hi/mt_lo, or
// kOutside for a source outside the grid.
constexpr uint32_t kOutside = 0xffffffffu;

template <int W, int NB>
struct StepTables {
  uint32_t a[kParityOffsets];
  uint32_t b[kParityOffsets][W * NB];
};

// Fetch the operands of step (ks, offset oi) into one ring slot.  Every step
// issues the same number of DMA operations per wave.  The uniform-box path
// addresses every operand as a fixed array base (SGPR pair) plus a 32-bit
// per-lane byte offset computed on the vector ALUs; sources outside the grid
// read the zero block that follows the multipole arrays.
template <int MT, int NB, int W, bool kUniformBox>
__device__ __forceinline__ void issue_step(int ks, int oi, const uint4* a_slot, const uint4* b_slot,
                                           const int4* offs, const StepTables<W, NB>& tab, const DevicePlan& d,
                                           const Columns<NB>& c, const StepGeometry& sg, int wave, int lane) {
  constexpr int kAChunks = 2 * MT, kAPerWave = (kAChunks + W - 1) / W;
  const int g = lane >> 5, col = lane & 31;
  if constexpr (kUniformBox) {
    const uint32_t ta = tab.a[oi] + uint32_t(ks) * (MT * 1024) + uint32_t(lane) * 16u;
#pragma unroll
    for (int i = 0; i < kAPerWave; ++i) {
      int ch = wave + W * i;
      if (ch >= kAChunks) ch -= kAChunks;  // repeats another wave's chunk: same bytes to the same place
      const int half = ch >= MT ? 1 : 0, m = ch - half * MT;
      lds_dma16_voff(half ? d.T_lo : d.T_hi, ta + uint32_t(m) * 1024u, a_slot + ch * 64);
    }
    const uint32_t kstep = uint32_t(ks) * uint32_t(sg.K) * 32u;
    const uint32_t lane_bytes = uint32_t(col * 2 + g) * 16u;
    const uint32_t zero = uint32_t(d.mt_zero_offset) + lane_bytes;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const uint32_t tb = tab.b[oi][wave * NB + nb];
      const uint32_t off = tb != kOutside ? tb + kstep + lane_bytes : zero;
      const uint4* dst = b_slot + (wave * NB + nb) * 128;
      lds_dma16_voff(d.mt_hi, off, dst);
      lds_dma16_voff(d.mt_lo, off, dst + 64);
    }
  } else {
    const int4 o = offs[oi];
    const int cls = __builtin_amdgcn_readfirstlane(o.w);
    const int64_t tunits = (int64_t(cls) * sg.KS + ks) * MT * 64;  // uint4 units
#pragma unroll
    for (int i = 0; i < kAPerWave; ++i) {
      int ch = wave + W * i;
      if (ch >= kAChunks) ch -= kAChunks;
      const int half = ch >= MT ? 1 : 0, m = ch - half * MT;
      const uint4* base = static_cast<const uint4*>(half ? d.T_lo : d.T_hi) + tunits + int64_t(m) * 64;
      lds_dma16_sbase(base, uint32_t(lane) * 16u, a_slot + ch * 64);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      int sx, sy, sz;
      const bool inside = source_inside(c, nb, o.x, o.y, o.z, sg.nbox, sx, sy, sz);
      const int64_t snode = sg.lvl0 + morton3(uint32_t(sx), uint32_t(sy), uint32_t(sz), sg.level);
      const uint4* dst = b_slot + (wave * NB + nb) * 128;
      const int64_t at = ((snode * sg.KS + ks) * sg.K + c.kk[nb]) * 2 + g;
      const uint4* zero = static_cast<const uint4*>(d.zero_block) + lane;
      lds_dma16(inside ? static_cast<const uint4*>(d.mt_hi) + at : zero, dst);
      lds_dma16(inside ? static_cast<const uint4*>(d.mt_lo) + at : zero, dst + 64);
    }
  }
}

// Operand fragments of one step: the wave's source fragments (hi, lo per
// tile) and the class-matrix row tiles (hi, lo per row tile).
template <int MT, int NB>
struct Fragments {
  uint4 a[MT][2];
  uint4 b[NB][2];
};

template <int MT, int NB>
__device__ __forceinline__ void read_fragments(const uint4* a_slot, const uint4* b_slot, int wave, int lane,
                                               Fragments<MT, NB>& f) {
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const uint4* src = b_slot + (wave * NB + nb) * 128 + lane;
    f.b[nb][0] = src[0];
    f.b[nb][1] = src[64];
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    f.a[m][0] = a_slot[m * 64 + lane];
    f.a[m][1] = a_slot[(MT + m) * 64 + lane];
  }
}

// The 3 * NB products of row tiles [M0, M1) (hi*hi + hi*lo + lo*hi), on
// bf16 or (kF16) fp16 operands.
template <bool kF16>
__device__ __forceinline__ f32x16 mfma_split(uint4 a, uint4 b, f32x16 c) {
  if constexpr (kF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                  0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

template <int MT, int NB, int M0, int M1, bool kF16>
__device__ __forceinline__ void multiply_rows(const uint4 (&a)[MT][2], const uint4 (&b)[NB][2],
                                              f32x16 (&acc)[NB][MT]) {
#pragma unroll
  for (int m = M0; m < M1; ++m) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      acc[nb][m] = mfma_split<kF16>(a[m][0], b[nb][0], acc[nb][m]);
      acc[nb][m] = mfma_split<kF16>(a[m][0], b[nb][1], acc[nb][m]);
      acc[nb][m] = mfma_split<kF16>(a[m][1], b[nb][0], acc[nb][m]);
    }
  }
}

template <int MT, int NB, int W, int kStages, bool kUniformBox, bool kF16>
__global__ void __launch_bounds__(W * 64, 1) m2l_mfma_kernel(const DevicePlan d, const LevelTable lt, int K) {
  static_assert(kStages >= 3, "the ring holds the current step and at least two in flight");
  constexpr int kAUnits = 2 * MT * 64, kBUnits = W * NB * 2 * 64, kSlot = kAUnits + kBUnits;
  constexpr int kAPerWave = (2 * MT + W - 1) / W;
  constexpr int kDmaPerStep = kAPerWave + 2 * NB;
  static_assert((kStages - 2) * kDmaPerStep <= 63, "vmcnt holds at most 63 outstanding operations");
  // Ring slots: the class-matrix slice, then the waves' source fragments.
  __shared__ uint4 ring[kStages * kSlot];
  __shared__ int4 offs[kParityOffsets];  // the offsets some column of this workgroup uses
  // The parity's offsets and the per-wave usage flags are read only by the
  // compaction below, which ends with a barrier before the first DMA writes
  // the ring; they live in the ring's first bytes.
  static_assert(kParityOffsets * (16 + W) <= kStages * kSlot * 16, "compaction scratch fits the ring");
  int4* const offs_all = reinterpret_cast<int4*>(ring);
  unsigned char (*const used)[kParityOffsets] =
      reinterpret_cast<unsigned char (*)[kParityOffsets]>(reinterpret_cast<unsigned char*>(ring) + kParityOffsets * 16);
  __shared__ int active_count;
  __shared__ StepTables<W, NB> tab;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  int li = lt.count - 1;
  while (li > 0 && int(blockIdx.x) < lt.block_begin[li]) --li;
  const int level = lt.level[li];
  const int lb = int(blockIdx.x) - lt.block_begin[li];
  const int parity = lb & 7, wgp = lb >> 3;
  const int px = parity & 1, py = (parity >> 1) & 1, pz = (parity >> 2) & 1;
  const int n = d.n, BP = d.bpad;
  StepGeometry sg;
  sg.K = K;
  sg.KS = d.apad / 16;
  sg.KD = d.mfma_depth_steps > 0 ? d.mfma_depth_steps : sg.KS;
  sg.level = level;
  sg.nbox = 1 << level;
  sg.lvl0 = level_offset(level);
  const int64_t parents = int64_t(1) << (3 * (level - 1));
  const int cpb = lt.cols_per_box[li], kchunks = lt.kchunks[li], tiles = lt.tiles[li];
  const int col = lane & 31, g = lane >> 5;
  Columns<NB> c;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int tile = (wgp * W + wave) * NB + nb;
    const int bg = tile / kchunks, kc = tile % kchunks;
    int64_t q;
    if constexpr (kUniformBox) {
      q = tile < tiles ? tile_parent(lt, li, parity, bg) : -1;  // one box per tile
      c.kk[nb] = kc * 32;
      c.valid[nb] = q >= 0 && q < parents;
    } else {
      q = int64_t(bg) * (32 / cpb) + col / cpb;
      c.kk[nb] = kc * cpb + col % cpb;
      c.valid[nb] = tile < tiles && q < parents && c.kk[nb] < K;
    }
    int x = 0, y = 0, z = 0;
    if (c.valid[nb]) demorton3(uint32_t(q), level - 1, x, y, z);
    c.tx[nb] = 2 * x + px;
    c.ty[nb] = 2 * y + py;
    c.tz[nb] = 2 * z + pz;
  }
  for (int i = threadIdx.x; i < kParityOffsets; i += W * 64) offs_all[i] = d.parity_offsets[parity * kParityOffsets + i];
  __syncthreads();
  // Offsets no column of this workgroup can use (source outside the grid, or
  // without points, for all of them) are dropped from the step sequence.
  if constexpr (kUniformBox) {
    // Every tile is one box: thread i decides offset i for all W*NB tiles.
    for (int i = threadIdx.x; i < kParityOffsets; i += W * 64) {
      const int4 o = offs_all[i];
      bool any = false;
      for (int t = 0; t < W * NB; ++t) {
        const int tile = wgp * W * NB + t;
        if (tile >= tiles) continue;
        const int64_t q = tile_parent(lt, li, parity, tile / kchunks);
        if (q < 0 || q >= parents) continue;
        int x, y, z;
        demorton3(uint32_t(q), level - 1, x, y, z);
        const int sx = 2 * x + px - o.x, sy = 2 * y + py - o.y, sz = 2 * z + pz - o.z;
        any |= sx >= 0 && sy >= 0 && sz >= 0 && sx < sg.nbox && sy < sg.nbox && sz < sg.nbox &&
               holds_sources(d, sg.lvl0 + morton3(uint32_t(sx), uint32_t(sy), uint32_t(sz), level));
      }
      used[0][i] = any ? 1 : 0;
    }
  } else {
  for (int i = 0; i < kParityOffsets; ++i) {
    const int4 o = offs_all[i];
    bool any = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      int sx, sy, sz;
      any |= source_inside(c, nb, o.x, o.y, o.z, sg.nbox, sx, sy, sz);
    }
    const bool wave_any = __any(any) != 0;
    if (lane == 0) used[wave][i] = wave_any ? 1 : 0;
  }
  }
  __syncthreads();
  if (wave == 0) {
    int count = 0;
    for (int i0 = 0; i0 < kParityOffsets; i0 += 64) {
      const int i = i0 + lane;
      bool u = false;
      if (i < kParityOffsets)
#pragma unroll
        for (int w = 0; w < (kUniformBox ? 1 : W); ++w) u |= used[w][i] != 0;
      const unsigned long long mask = __ballot(u);
      if (u) offs[count + __popcll(mask & ((1ull << lane) - 1ull))] = offs_all[i];
      count += __popcll(mask);
    }
    if (lane == 0) active_count = count;
  }
  __syncthreads();
  const int nact = active_count;
  sg.nsteps = sg.KD * nact;
  if constexpr (kUniformBox) {
    // Step tables of the used offsets.
    for (int e = threadIdx.x; e < nact * (W * NB + 1); e += W * 64) {
      const int a = e / (W * NB + 1), t = e - a * (W * NB + 1);
      const int4 o = offs[a];
      if (t == W * NB) {
        tab.a[a] = uint32_t(o.w) * uint32_t(sg.KS * MT * 1024);
        continue;
      }
      const int tile = wgp * W * NB + t;
      const int kc = tile % kchunks;
      const int64_t q = tile < tiles ? tile_parent(lt, li, parity, tile / kchunks) : -1;
      uint32_t off = kOutside;
      if (q >= 0 && q < parents) {
        int x, y, z;
        demorton3(uint32_t(q), level - 1, x, y, z);
        const int sx = 2 * x + px - o.x, sy = 2 * y + py - o.y, sz = 2 * z + pz - o.z;
        if (sx >= 0 && sy >= 0 && sz >= 0 && sx < sg.nbox && sy < sg.nbox && sz < sg.nbox) {
          const uint64_t snode = uint64_t(sg.lvl0 + morton3(uint32_t(sx), uint32_t(sy), uint32_t(sz), level));
          if (holds_sources(d, int64_t(snode)))
            off = uint32_t((snode * uint64_t(sg.KS) * uint64_t(K) + uint64_t(kc) * 32u) * 32u);
        }
      }
      tab.b[a][t] = off;
    }
    __syncthreads();
  }

  f32x16 acc[NB][MT];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[nb][m][r] = 0.0f;

  if (nact > 0) {
    // (ks, oi) of the next step to fetch; past the last step the last step
    // is fetched again into a slot nobody reads.
    int iks = 0, ioi = 0;
    auto advance = [&]() {  // branch-free: selects only
      const bool last = (iks == sg.KD - 1) & (ioi == nact - 1);
      const bool wrap = ioi + 1 == nact;
      const int next_oi = wrap ? 0 : ioi + 1;
      const int next_ks = iks + (wrap ? 1 : 0);
      ioi = last ? ioi : next_oi;
      iks = last ? iks : next_ks;
    };
#pragma unroll
    for (int slot = 0; slot < kStages - 1; ++slot) {
      issue_step<MT, NB, W, kUniformBox>(iks, ioi, ring + slot * kSlot, ring + slot * kSlot + kAUnits, offs, tab, d,
                                         c, sg, wave, lane);
      advance();
    }
    // Step s: wait for this wave's DMA of step s (the kStages - 2 younger
    // steps may stay in flight) and for its LDS reads of step s-1, barrier
    // (every wave's share of slot s is in LDS; slot s-1 is free), read the
    // fragments of slot s, refill slot s-1 with step s + kStages - 1, and
    // multiply; the products overlap the next fetch's address arithmetic.
    // The inline-asm barrier keeps the compiler from moving LDS accesses
    // across it.
    int cur = 0, nxt = kStages - 1;
    for (int s = 0; s < sg.nsteps; ++s) {
      __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((kStages - 2) * kDmaPerStep));
      asm volatile("s_barrier" ::: "memory");
      Fragments<MT, NB> f;
      read_fragments<MT, NB>(ring + cur * kSlot, ring + cur * kSlot + kAUnits, wave, lane, f);
      issue_step<MT, NB, W, kUniformBox>(iks, ioi, ring + nxt * kSlot, ring + nxt * kSlot + kAUnits, offs, tab, d, c,
                                         sg, wave, lane);
      advance();
      multiply_rows<MT, NB, 0, MT, kF16>(f.a, f.b, acc);
      cur = cur + 1 == kStages ? 0 : cur + 1;
      nxt = nxt + 1 == kStages ? 0 : nxt + 1;
    }
    __builtin_amdgcn_s_waitcnt(0);  // the trailing repeat fetches land before the workgroup's LDS is released
  }

  const float* lsp = static_cast<const float*>(kF16 ? d.ls16_pad : d.ls_pad) + int64_t(level) * BP;
  // FP16 operands of this level carry the power-of-two scale 2^e (see
  // fp16_level_exponent); the products are divided by it here.
  const float unscale = kF16 ? ldexpf(1.0f, -fp16_level_exponent(d.lvl_max_bits[level])) : 1.0f;
  float* Lc = static_cast<float*>(d.Lc);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    if (!c.valid[nb]) continue;
    const int64_t tnode = sg.lvl0 + morton3(uint32_t(c.tx[nb]), uint32_t(c.ty[nb]), uint32_t(c.tz[nb]), level);
    const int state = c.kk[nb] + (kUniformBox ? col : 0);
    if (state >= lt.states) continue;  // a column of the padding
    float* out = Lc + tnode * int64_t(n) * lt.states + (d.state_major ? state * n : state);
    const int64_t row_step = d.state_major ? 1 : lt.states;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        if (row < n) out[row * row_step] = (lsp[row] * unscale) * acc[nb][m][r];
      }
  }
}

// One box per 32-column tile, and every operand byte offset within 32 bits.
bool uniform_box(const DevicePlan& d, int K) {
  return K % 32 == 0 && d.mt_zero_offset + 1024 <= int64_t(0xffffffffu);
}

LevelTable level_table(const DevicePlan& d, int states, int K, int nb) {
  LevelTable lt{};
  lt.states = states;
  lt.count = d.L - 1;
  // With one box per tile, tiles follow the plan's boundary-class order of
  // the parents for this workgroup size (kM2LGroupTiles).
  int g = -1;
  for (int i = 0; i < 5; ++i)
    if (kM2LGroupTiles[i] == kWaves * nb) g = i;
  const bool ordered = uniform_box(d, K) && d.m2l_order != nullptr && g >= 0;
  const bool sparse = ordered && d.sparse_order != nullptr && kWaves * nb == kM2LSparseTiles;
  lt.order = sparse ? d.sparse_order : ordered ? d.m2l_order : nullptr;
  int begin = 0;
  for (int i = 0; i < lt.count; ++i) {
    const int level = sparse ? d.L - i : 2 + i;  // the last level first (see inner_class_first)
    lt.level[i] = level;
    int cpb = 1;
    while (cpb < K && cpb < 32) cpb *= 2;
    const int kchunks = (K + cpb - 1) / cpb;
    const int64_t parents = int64_t(1) << (3 * (level - 1));
    const int boxes_per_tile = 32 / cpb;
    const int groups = sparse    ? d.sparse_len[level]
                       : ordered ? d.m2l_order_len[g][level]
                                 : int((parents + boxes_per_tile - 1) / boxes_per_tile);
    lt.order_base[i] = sparse ? d.sparse_base[level] : ordered ? d.m2l_order_base[g][level] : 0;
    lt.order_stride[i] = sparse ? d.sparse_len[level] : 0;
    const int tiles = groups * kchunks;
    const int bpp = (tiles + kWaves * nb - 1) / (kWaves * nb);
    lt.block_begin[i] = begin;
    lt.blocks_per_parity[i] = bpp;
    lt.tiles[i] = tiles;
    lt.cols_per_box[i] = cpb;
    lt.kchunks[i] = kchunks;
    begin += 8 * bpp;
  }
  lt.block_begin[lt.count] = begin;
  return lt;
}

// The last level's inner class (the parents with every list-2 offset in the
// grid; first in the plan's order at levels >= 4, padded to whole
// workgroups) moved to the front of the launch, then levels 2..L-1, then the
// last level's boundary classes.  Dispatched first, the inner class's
// equal-length workgroups start together and walk the offsets in lockstep,
// so each reads the sources its neighbours have just brought into L2, and
// the shorter workgroups behind them fill its tail.  (With the levels in
// order, levels 2..L-1 go first and the inner workgroups start staggered
// behind them: at 1M points, depth 5, the M2L then fetches 29.6 GB against
// 13.7 GB.)
bool inner_class_first(const LevelTable& lt, int L, int G, LevelTable& out) {
  const int last = lt.count - 1;
  if (lt.order == nullptr || L < 4 || last < 0 || lt.level[last] != L || lt.order_stride[last] != 0 || lt.count + 2 > 12)
    return false;
  const int64_t np = int64_t(1) << (L - 1);
  const int inner_groups = int(((np - 2) * (np - 2) * (np - 2) + G - 1) / G * G);
  const int kchunks = lt.kchunks[last], inner_tiles = inner_groups * kchunks;
  if (inner_tiles <= 0 || inner_tiles >= lt.tiles[last]) return false;
  out = lt;
  int e = 0, begin = 0;
  auto put = [&](int level, int tiles, int cpb, int kch, int order_base) {
    out.level[e] = level;
    out.block_begin[e] = begin;
    out.tiles[e] = tiles;
    out.cols_per_box[e] = cpb;
    out.kchunks[e] = kch;
    out.order_base[e] = order_base;
    out.blocks_per_parity[e] = (tiles + G - 1) / G;
    begin += 8 * out.blocks_per_parity[e];
    ++e;
  };
  put(L, inner_tiles, lt.cols_per_box[last], kchunks, lt.order_base[last]);
  for (int i = 0; i < last; ++i) put(lt.level[i], lt.tiles[i], lt.cols_per_box[i], lt.kchunks[i], lt.order_base[i]);
  put(L, lt.tiles[last] - inner_tiles, lt.cols_per_box[last], kchunks, lt.order_base[last] + inner_groups);
  out.count = e;
  out.block_begin[e] = begin;
  return true;
}

template <int MT, int NB, int kStages, bool kF16>
void launch_uniform(const DevicePlan& v, const LevelTable& lt, int K, hipStream_t s) {
  LevelTable t;
  const LevelTable& use = inner_class_first(lt, v.L, kWaves * NB, t) ? t : lt;
  if (use.block_begin[use.count] == 0) return;  // no box holds targets
  m2l_mfma_kernel<MT, NB, kWaves, kStages, true, kF16>
      <<<unsigned(use.block_begin[use.count]), kWaves * 64, 0, s>>>(v, use, K);
}

template <int MT, int NB, int kStages>
void launch_mfma_cfg(const DevicePlan& d, int states, bool f16, hipStream_t s) {
  const int K = m2l_operand_states(d, states);
  const LevelTable lt = level_table(d, states, K, NB);
  const unsigned blocks = unsigned(lt.block_begin[lt.count]);
  const bool uniform = uniform_box(d, K);
  DevicePlan v = d;
  if (f16) {
    v.T_hi = d.T16_hi;
    v.T_lo = d.T16_lo;
  }
  if (uniform && f16)
    launch_uniform<MT, NB, kStages, true>(v, lt, K, s);
  else if (uniform)
    launch_uniform<MT, NB, kStages, false>(v, lt, K, s);
  else if (f16)
    m2l_mfma_kernel<MT, NB, kWaves, kStages, false, true><<<blocks, kWaves * 64, 0, s>>>(v, lt, K);
  else
    m2l_mfma_kernel<MT, NB, kWaves, kStages, false, false><<<blocks, kWaves * 64, 0, s>>>(v, lt, K);
  HIPFMM_CHECK(hipGetLastError());
}

// Tile shape per row-tile count MT: NB 32-column tiles per wave (NB * MT *
// 16 accumulator registers) and the ring depth that fits LDS (160 KiB per
// CU).  At MT <= 3 the default 2 x 3 takes 77 KB, so two workgroups share a
// CU and one's barrier wait overlaps the other's products (81% MFMA-busy,
// against 67% for 5 x 3 at one workgroup per CU).  The shape only regroups
// whole output columns, so every shape gives bitwise the same locals.
// HIPFMM_M2L_MFMA_SHAPE=NBxS (1x3, 2x3, 2x4, 3x4, 4x3, 5x3, 2x6) overrides
// the choice among the compiled shapes, for measurement.
inline int mfma_shape_override() {
  static const int v = [] {
    const char* e = std::getenv("HIPFMM_M2L_MFMA_SHAPE");
    if (!e) return 0;
    if (std::string(e) == "2x4") return 24;
    if (std::string(e) == "3x4") return 34;
    if (std::string(e) == "4x3") return 43;
    if (std::string(e) == "2x6") return 26;
    if (std::string(e) == "5x3") return 53;
    if (std::string(e) == "2x3") return 23;
    if (std::string(e) == "1x3") return 13;
    return 0;
  }();
  return v;
}

template <int MT>
void launch_mfma_t(const DevicePlan& d, int K, bool f16, hipStream_t s) {
  if constexpr (MT <= 3) {
    switch (d.m2l_shape ? d.m2l_shape : mfma_shape_override()) {
      case 24: launch_mfma_cfg<MT, 2, 4>(d, K, f16, s); return;
      case 34: launch_mfma_cfg<MT, 3, 4>(d, K, f16, s); return;
      case 26: launch_mfma_cfg<MT, 2, 6>(d, K, f16, s); return;
      case 43: launch_mfma_cfg<MT, 4, 3>(d, K, f16, s); return;
      case 23: launch_mfma_cfg<MT, 2, 3>(d, K, f16, s); return;
      case 53: launch_mfma_cfg<MT, 5, 3>(d, K, f16, s); return;
      case 13: launch_mfma_cfg<MT, 1, 3>(d, K, f16, s); return;
      default: launch_mfma_cfg<MT, 2, 3>(d, K, f16, s); return;
    }
  } else {
    launch_mfma_cfg<MT, 2, 4>(d, K, f16, s);
  }
}

}  // namespace

void launch_m2l_split(const DevicePlan& d, int K, int mode, hipStream_t s) {
  (void)mode;
  if (d.L < 2) return;
  const unsigned boxes = unsigned(d.nodes - level_offset(2));
  int kc = K;
  while (kc > 1 && size_t(d.n) * kc * sizeof(float) > 32768) kc = (kc + 1) / 2;
  const dim3 grid(boxes, unsigned((K + kc - 1) / kc));
  split_kernel<<<grid, 256, size_t(d.n) * kc * sizeof(float), s>>>(d, K, kc);
  HIPFMM_CHECK(hipGetLastError());
}

void launch_m2l_mfma(const DevicePlan& d, int K, int mode, hipStream_t s) {
  if (d.L < 2) return;
  const bool f16 = mode == 2;  // HIPFMM_M2L_MFMA_FP16X3
  if (f16 && (d.T16_hi == nullptr || d.nc == 0))
    throw invalid_argument("the FP16 M2L mode needs class matrices of harmonic form");
  switch (d.bpad / 32) {
    case 1: launch_mfma_t<1>(d, K, f16, s); break;
    case 2: launch_mfma_t<2>(d, K, f16, s); break;
    case 3: launch_mfma_t<3>(d, K, f16, s); break;
    case 4: launch_mfma_t<4>(d, K, f16, s); break;
    case 5: launch_mfma_t<5>(d, K, f16, s); break;
    case 6: launch_mfma_t<6>(d, K, f16, s); break;
    default: throw invalid_argument("expansion order too large for the MFMA M2L path");
  }
}

namespace {

// Largest |Mc / sigma| of each level (positive float bits compare as
// unsigned; vector atomics).  One workgroup per box at levels >= 2.
__global__ void __launch_bounds__(256) level_max_kernel(const DevicePlan d, int K) {
  __shared__ unsigned red[256];
  const int64_t node = level_offset(2) + blockIdx.x;
  const int level = level_of_node(node);
  const float* Mc = static_cast<const float*>(d.Mc) + node * int64_t(d.nc) * K;
  const float* cs = static_cast<const float*>(d.col16_scale);
  unsigned mx = 0u;
  for (int i = threadIdx.x; i < d.nc * K; i += blockDim.x)
    mx = max(mx, __builtin_bit_cast(unsigned, fabsf(Mc[i] * cs[d.compressed_state_major ? i % d.nc : i / K])));
  red[threadIdx.x] = mx;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(d.lvl_max_bits + level, red[0]);
}

// FP16 hi/lo split of 2^e_l Mc / sigma into the MFMA B layout
// mt[node][ks][KO][16] (KO >= K columns, zeros from K on); each thread packs 8
// consecutive coefficients of one column (16-byte stores).
__global__ void __launch_bounds__(256) split_f16_kernel(const DevicePlan d, int K, int KO, const uint32_t* bits) {
  const int nc = d.nc, AP = d.apad, KS = AP / 16;
  const int64_t node = level_offset(2) + blockIdx.x;
  if (bits != nullptr && !bit_of(bits, node)) return;
  const int level = level_of_node(node);
  const float scale = ldexpf(1.0f, fp16_level_exponent(d.lvl_max_bits[level]));
  const float* Mc = static_cast<const float*>(d.Mc) + node * int64_t(nc) * K;
  const float* cs = static_cast<const float*>(d.col16_scale);
  const int row = d.compressed_state_major ? 1 : K, state = d.compressed_state_major ? nc : 1;
  for (int w = threadIdx.x; w < KO * (AP / 8); w += blockDim.x) {
    const int k = w % KO, a0 = (w / KO) * 8;
    half8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int a = a0 + e;
      const float x = a < nc && k < K ? (scale * cs[a]) * Mc[a * row + k * state] : 0.0f;
      const _Float16 h = _Float16(x);
      hi[e] = h;
      lo[e] = _Float16(x - float(h));
    }
    const int64_t at = ((node * KS + a0 / 16) * KO + k) * 16 + a0 % 16;
    *reinterpret_cast<uint4*>(static_cast<_Float16*>(d.mt_hi) + at) = __builtin_bit_cast(uint4, hi);
    *reinterpret_cast<uint4*>(static_cast<_Float16*>(d.mt_lo) + at) = __builtin_bit_cast(uint4, lo);
  }
}

// bf16 hi/lo split of Mc into the MFMA B layout mt[node][ks][KO][16] (levels
// 2..L, KO as above); each thread packs 8 consecutive coefficients of one
// column.
__global__ void __launch_bounds__(256) split_bf16_kernel(const DevicePlan d, int K, int KO, const uint32_t* bits) {
  const int nc = d.nc, AP = d.apad, KS = AP / 16;
  const int64_t node = level_offset(2) + blockIdx.x;
  if (bits != nullptr && !bit_of(bits, node)) return;
  const float* Mc = static_cast<const float*>(d.Mc) + node * int64_t(nc) * K;
  const int row = d.compressed_state_major ? 1 : K, state = d.compressed_state_major ? nc : 1;
  for (int w = threadIdx.x; w < KO * (AP / 8); w += blockDim.x) {
    const int k = w % KO, a0 = (w / KO) * 8;
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float x0 = a0 + e < nc && k < K ? Mc[(a0 + e) * row + k * state] : 0.0f;
      const float x1 = a0 + e + 1 < nc && k < K ? Mc[(a0 + e + 1) * row + k * state] : 0.0f;
      const uint16_t h0 = bf16_bits(x0), h1 = bf16_bits(x1);
      hi[e / 2] = uint32_t(h0) | (uint32_t(h1) << 16);
      lo[e / 2] = uint32_t(bf16_bits(x0 - bf16_value(h0))) | (uint32_t(bf16_bits(x1 - bf16_value(h1))) << 16);
    }
    const int64_t at = (((node * KS + a0 / 16) * KO + k) * 16 + a0 % 16) / 8;  // uint4 index
    static_cast<uint4*>(d.mt_hi)[at] = uint4{hi[0], hi[1], hi[2], hi[3]};
    static_cast<uint4*>(d.mt_lo)[at] = uint4{lo[0], lo[1], lo[2], lo[3]};
  }
}

}  // namespace

// From 9 states on a box's operand columns are padded with zeros to a multiple
// of 32, so that every 32-column tile is one box and its step runs on the
// uniform-box path: at 4681 boxes of p = 6 a batch of 12 to 31 states takes
// 0.41 ms padded and 0.77-1.38 ms with several boxes per tile; up to 8 states
// (four or more boxes per tile) it takes 0.37 ms.  Not where the padded columns
// would not fit that path's 32-bit offsets (or, for a batch below the capacity,
// the operand buffer): several boxes per tile would then walk the padding too.
static bool padding_fits(const DevicePlan& d, int K, int64_t bytes) {
  return d.nc > 0 && K >= 9 && int64_t(d.nodes) * ((K + 31) / 32 * 32) * d.apad * 2 <= bytes &&
         bytes + 1024 <= int64_t(0xffffffffu);
}
int m2l_operand_states(const DevicePlan& d, int K) {
  return padding_fits(d, K, d.mt_zero_offset) ? (K + 31) / 32 * 32 : K;
}
int m2l_operand_capacity(const DevicePlan& d, int K) {
  const int padded = (K + 31) / 32 * 32;
  return padding_fits(d, K, int64_t(d.nodes) * padded * d.apad * 2) ? padded : K;
}

// The boxes whose operands the tiles read: of one box per tile, those with
// sources (holds_sources); of several, all.
static const uint32_t* split_bits(const DevicePlan& d, int KO) {
  return uniform_box(d, KO) ? d.source_bits : nullptr;
}

void launch_m2l_bf16_split(const DevicePlan& d, int K, hipStream_t s) {
  if (d.L < 2) return;
  const unsigned boxes = unsigned(d.nodes - level_offset(2));
  const int KO = m2l_operand_states(d, K);
  split_bf16_kernel<<<boxes, 256, 0, s>>>(d, K, KO, split_bits(d, KO));
  HIPFMM_CHECK(hipGetLastError());
}

void launch_m2l_fp16_split(const DevicePlan& d, int K, hipStream_t s) {
  if (d.L < 2) return;
  const unsigned boxes = unsigned(d.nodes - level_offset(2));
  launch_zero<float>(reinterpret_cast<float*>(d.lvl_max_bits), size_t(d.L + 1), s);
  level_max_kernel<<<boxes, 256, 0, s>>>(d, K);
  HIPFMM_CHECK(hipGetLastError());
  const int KO = m2l_operand_states(d, K);
  split_f16_kernel<<<boxes, 256, 0, s>>>(d, K, KO, split_bits(d, KO));
  HIPFMM_CHECK(hipGetLastError());
}

void prepare_mfma_fp16_operators(DevicePlan& d, int n, const std::vector<double>& matrices, int classes, int order,
                                 std::vector<void*>& allocations, size_t& bytes) {
  const int MT = d.bpad / 32, KS = d.apad / 16, D = order + 1;
  if (n != D * D) throw invalid_argument("the FP16 M2L mode needs class matrices of harmonic form");
  // Degree of each compressed row/column: index r is harmonic row
  // (r + 1) mod n of the degree-major order (degree 0 last).
  std::vector<int> deg(n);
  for (int j = 0; j < D; ++j)
    for (int r = j * j; r < (j + 1) * (j + 1); ++r) deg[(r + n - 1) % n] = j;
  // log2 of the largest entry of each degree block (j, k) over all classes.
  std::vector<double> lt(size_t(D) * D, 0.0), tab(size_t(D) * D, 0.0);
  for (int c = 0; c < classes; ++c)
    for (int a = 0; a < n; ++a)
      for (int b = 0; b < n; ++b) {
        double& t = tab[size_t(deg[b]) * D + deg[a]];
        t = std::max(t, std::fabs(matrices[size_t(c) * n * n + b + size_t(n) * a]));
      }
  bool all_nonzero = true;
  for (size_t i = 0; i < tab.size(); ++i) {
    all_nonzero = all_nonzero && tab[i] > 0.0;
    lt[i] = tab[i] > 0.0 ? std::log2(tab[i]) : 0.0;
  }
  // Column exponents: the column effect of the two-way least-squares fit
  // log2 tab[j][k] ~ a_j + b_k (column mean minus grand mean), rounded; the
  // block magnitudes of these operators depend on j + k mostly, so the fit
  // leaves every block within a few binades of its row's largest.
  std::vector<int> bexp(D, 0), rexp(D, 0);
  if (all_nonzero) {
    double grand = 0.0;
    for (double v : lt) grand += v;
    grand /= double(lt.size());
    for (int k = 0; k < D; ++k) {
      double col = 0.0;
      for (int j = 0; j < D; ++j) col += lt[size_t(j) * D + k];
      bexp[k] = int(std::lround(col / D - grand));
    }
  }
  // Row exponents: the row's largest scaled block in [2^13, 2^14].
  for (int j = 0; j < D; ++j) {
    double mx = -1e300;
    for (int k = 0; k < D; ++k)
      if (tab[size_t(j) * D + k] > 0.0) mx = std::max(mx, lt[size_t(j) * D + k] - bexp[k]);
    rexp[j] = mx > -1e300 ? 14 - int(std::ceil(mx)) : 0;
  }
  const size_t per_class = size_t(MT) * KS * 64 * 8;
  std::vector<_Float16> hi(per_class * classes), lo(per_class * classes);
  for (int c = 0; c < classes; ++c) {
    const double* T = matrices.data() + size_t(c) * n * n;
    for (int ks = 0; ks < KS; ++ks)
      for (int m = 0; m < MT; ++m)
        for (int lane = 0; lane < 64; ++lane)
          for (int e = 0; e < 8; ++e) {
            const int row = m * 32 + lane % 32;
            const int dep = ks * 16 + 8 * (lane / 32) + e;
            const float v = (row < n && dep < n)
                                ? float(std::ldexp(T[row + size_t(n) * dep], rexp[deg[row]] - bexp[deg[dep]]))
                                : 0.0f;
            const size_t i = size_t(c) * per_class + ((size_t(ks) * MT + m) * 64 + lane) * 8 + e;
            hi[i] = _Float16(v);
            lo[i] = _Float16(v - float(hi[i]));
          }
  }
  const int levels = d.L + 1;
  std::vector<float> lsp(size_t(levels) * d.bpad, 0.0f), csc(d.apad, 0.0f);
  for (int l = 0; l < levels; ++l)
    for (int b = 0; b < n; ++b) lsp[size_t(l) * d.bpad + b] = std::ldexp(1.0f, -rexp[deg[b]]);
  for (int a = 0; a < n; ++a) csc[a] = std::ldexp(1.0f, bexp[deg[a]]);
  auto up = [&](const void* host, size_t count) {
    void* ptr = nullptr;
    HIPFMM_CHECK(hipMalloc(&ptr, std::max<size_t>(count, 16)));
    allocations.push_back(ptr);
    HIPFMM_CHECK(hipMemcpy(ptr, host, count, hipMemcpyHostToDevice));
    bytes += count;
    return ptr;
  };
  d.T16_hi = up(hi.data(), hi.size() * 2);
  d.T16_lo = up(lo.data(), lo.size() * 2);
  d.ls16_pad = up(lsp.data(), lsp.size() * 4);
  d.col16_scale = up(csc.data(), csc.size() * 4);
  const std::vector<unsigned> zeros(levels, 0u);
  d.lvl_max_bits = static_cast<unsigned*>(up(zeros.data(), zeros.size() * sizeof(unsigned)));
}

void prepare_mfma_operators(DevicePlan& d, int n, const std::vector<double>& matrices, int classes,
                            const std::vector<double>& local_scaling, std::vector<void*>& allocations, size_t& bytes) {
  d.apad = ((n + 15) / 16) * 16;
  d.bpad = ((n + 31) / 32) * 32;
  const int MT = d.bpad / 32, KS = d.apad / 16;
  const size_t per_class = size_t(MT) * KS * 64 * 8;
  std::vector<uint16_t> hi(per_class * classes), lo(per_class * classes);
  for (int c = 0; c < classes; ++c) {
    const double* T = matrices.data() + size_t(c) * n * n;  // T[beta + n*alpha]
    for (int ks = 0; ks < KS; ++ks)
      for (int m = 0; m < MT; ++m)
        for (int lane = 0; lane < 64; ++lane)
          for (int e = 0; e < 8; ++e) {
            const int row = m * 32 + lane % 32;
            const int dep = ks * 16 + 8 * (lane / 32) + e;
            const float v = (row < n && dep < n) ? float(T[row + size_t(n) * dep]) : 0.0f;
            const size_t i = size_t(c) * per_class + ((size_t(ks) * MT + m) * 64 + lane) * 8 + e;
            hi[i] = bf16_bits(v);
            lo[i] = bf16_bits(v - bf16_value(hi[i]));
          }
  }
  const int levels = d.L + 1;
  std::vector<float> lsp(size_t(levels) * d.bpad, 0.0f);
  for (int l = 0; l < levels; ++l)
    for (int b = 0; b < n; ++b) lsp[size_t(l) * d.bpad + b] = float(local_scaling[size_t(l) * n + b]);
  auto up = [&](const void* host, size_t count) {
    void* ptr = nullptr;
    HIPFMM_CHECK(hipMalloc(&ptr, std::max<size_t>(count, 16)));
    allocations.push_back(ptr);
    HIPFMM_CHECK(hipMemcpy(ptr, host, count, hipMemcpyHostToDevice));
    bytes += count;
    return ptr;
  };
  const std::vector<uint16_t> zeros(512, 0);
  d.zero_block = up(zeros.data(), zeros.size() * 2);
  d.T_hi = up(hi.data(), hi.size() * 2);
  d.T_lo = up(lo.data(), lo.size() * 2);
  d.ls_pad = up(lsp.data(), lsp.size() * 4);
}

}  // namespace hipfmm
