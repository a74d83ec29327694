/*
 * hipfmm.h -- C-ABI of the HipFull device plan (one MI355X / gfx950 GPU).
 *
 * This is the boundary a host FMM front-end binds to replace the reference's
 * device plan: `cdfmm::CudaFullPlan` (src/cuda_fmm_plan.hpp:95-114, built by
 * `UniformFmm::build_cuda_full_plan`, src/uniform_fmm.cpp:826-1013, and
 * driven by `UniformFmm::evaluate_into[_float32]`, src/uniform_fmm.cpp:1102-
 * 1136 and :1307-1349).  The host keeps building the Morton octree,
 * permutations, identity map, translation operators and M2L class matrices
 * once; `hipfmm_plan_create` uploads them a single time.  Every evaluate then
 * runs P2M, M2M, M2L, L2L, L2P, list-1 P2P and the unsort to user target
 * order on the device.
 *
 * Conventions
 *  - Plain pointers and sizes only; no C++ or framework types.
 *  - Every function returns a status (HIPFMM_OK == 0).  On failure a
 *    thread-local message is available from hipfmm_last_error().  The C++
 *    front-end maps HIPFMM_ERROR_INVALID_ARGUMENT to std::invalid_argument and
 *    every other failure to std::runtime_error, as the reference does
 *    (src/cuda_fmm.cu:32-54, :3462-3486).
 *  - Coefficient order is the reference's total-degree multi-index order
 *    (include/cdfmm/multi_index.hpp:62-71); n = (p+1)(p+2)(p+3)/6.
 *  - Nodes are stored level by level, Morton order within a level
 *    (src/uniform_tree.cpp:100-113); a complete tree has (8^(L+1)-1)/7 nodes.
 *  - One plan is not re-entrant (include/cdfmm/uniform_fmm.hpp:222-229);
 *    separate plans may be used concurrently.
 */
#ifndef HIPFMM_H
#define HIPFMM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct hipfmm_plan hipfmm_plan;

enum hipfmm_status {
  HIPFMM_OK = 0,
  HIPFMM_ERROR_RUNTIME = 1,          /* device or runtime failure */
  HIPFMM_ERROR_INVALID_ARGUMENT = 2, /* dimensions, identity map, options */
  HIPFMM_ERROR_UNAVAILABLE = 3       /* no usable HIP device */
};

enum hipfmm_memspace { HIPFMM_HOST = 0, HIPFMM_DEVICE = 1 };

/* M2L arithmetic.  VALU is the plain path: FMA chains in the plan's own
 * precision, on the full-precision matrix instructions (on the vector ALUs for
 * class matrices that do not factor).  The MFMA modes exist for FP32 plans only: operands are split
 * into two 16-bit halves (hi + lo) and three products are accumulated in FP32
 * on the matrix cores.  A small batch that is no multiple of 32 states does not
 * pay for the split: up to 3.5e6 boxes x states x (p+1)^2 with 8 or fewer
 * states (FP16 1.8e6), 7e5 with more, the bf16 mode forms the same products
 * without a pass of its own for it and the FP16 mode runs as VALU does. */
enum hipfmm_m2l_mode {
  HIPFMM_M2L_VALU = 0,
  HIPFMM_M2L_MFMA_BF16X3 = 1,
  HIPFMM_M2L_MFMA_FP16X3 = 2
};

/* Plan descriptor.  All arrays are host memory owned by the caller; the
 * create call copies what it needs, so they may be freed afterwards. */
typedef struct hipfmm_plan_desc {
  int precision;    /* 32 or 64 (StaticPrecision, include/cdfmm/precision.hpp:11) */
  int order;        /* expansion order p >= 0 */
  int max_level;    /* leaf level L >= 0 */
  int source_count;
  int target_count;
  /* Morton-sorted positions, 3 doubles each, in the operator frame: root-
   * width normalised for FP32 plans (src/uniform_fmm.cpp:379-417), physical
   * for FP64 plans. */
  const double* sorted_sources;
  const double* sorted_targets;
  const int* source_permutation; /* sorted -> user index (uniform_tree.hpp:128) */
  const int* target_permutation;
  /* Per node: source begin, source end, target begin, target end (half-open,
   * [count, count) when empty; src/uniform_tree.cpp:359-438). */
  const int64_t* node_ranges;
  /* Per node centre, 3 doubles, operator frame. */
  const double* node_centres;
  /* M2L class matrices (src/static_operators.cpp:159-184): `m2l_class_count`
   * integer offsets (target minus source box coordinates, 3 ints each) and a
   * column-major n x n matrix per class, T[beta + n*alpha] = D_{alpha+beta}G.
   * Every offset the device meets must be present (all 316 list-2 offsets of
   * a tree with L >= 2 cover every case). */
  int m2l_class_count;
  const int* m2l_class_offsets;
  const double* m2l_matrices;
  /* Level scalings, (L+1) x n each (src/uniform_fmm.cpp:529-566). */
  const double* m2l_multipole_scaling;
  const double* m2l_local_scaling;
  /* Shift operators for levels 1..L and child class c = (ix&1)|(iy&1)<<1|
   * (iz&1)<<2, dense row-major n x n (out x in): M2M maps a child multipole
   * into its parent, L2L a parent local into its child
   * (src/static_operators.cpp:257-298).  Size L*8*n*n each. */
  const double* m2m_operators;
  const double* l2l_operators;
  /* Optional fixed identity map: sorted target -> sorted source or -1
   * (src/uniform_fmm.cpp:265-295, :1028-1043).  NULL when not fixed. */
  const int* fixed_self_indices;
  /* Factor applied to moments supplied in device memory before use; FP32
   * plans pass 1/W^3 for root width W so the caller may hand over physical
   * moments (src/uniform_fmm.cpp:1315-1323).  Host moments are assumed to be
   * scaled already and use factor 1. */
  double device_moment_scale;
  int m2l_mode; /* enum hipfmm_m2l_mode */
  /* Factor applied to every potential before it is returned: the root width
   * W for FP32 plans, whose potential is computed in the normalised frame
   * (src/uniform_fmm.cpp:1448-1451); 1 for FP64 plans.  0 reads as 1. */
  double potential_scale;
} hipfmm_plan_desc;

/* Host/device traffic and storage; mirrors CudaPlanStatistics
 * (include/cdfmm/timings.hpp:182-222). */
typedef struct hipfmm_stats {
  uint64_t scalar_bytes;
  uint64_t m2m_unique_matrix_count;
  uint64_t m2m_matrix_bytes;
  uint64_t m2l_unique_matrix_count;
  uint64_t m2l_matrix_bytes;
  uint64_t m2l_interaction_count;
  uint64_t l2l_unique_matrix_count;
  uint64_t l2l_matrix_bytes;
  uint64_t p2p_interaction_count;
  uint64_t setup_h2d_bytes;
  uint64_t evaluation_h2d_bytes;  /* of the most recent host-memory evaluate */
  uint64_t evaluation_d2h_bytes;
  uint64_t evaluation_h2d_calls;  /* cumulative */
  uint64_t evaluation_d2h_calls;
  uint64_t persistent_device_bytes;
  uint64_t plan_generation_count;
  uint64_t static_upload_count;
  uint64_t batch_capacity;        /* moment states the state buffers hold */
  uint64_t m2l_leaf_interaction_count; /* non-empty list-2 pairs at the leaf level */
  /* Coefficients per box the M2L product runs on: n = (p+1)(p+2)(p+3)/6, or
   * (p+1)^2 when the class matrices factor through the harmonic subspace
   * (T_o = Q C_o P; no counterpart in the reference, which always uses n). */
  uint64_t m2l_operand_size;
  double m2l_reconstruction_error; /* max |T_o - Q C_o P| / max |T_o| over classes (0 if unused) */
  /* FP32 plans with the harmonic form run M2M and L2L on the compressed
   * coefficients; this is the largest relative part of an M2M or L2L
   * operator outside the harmonic subspace (checked <= 1e-10 at setup; 0 if
   * the passes run on the full coefficients). */
  double harmonic_pass_leak;
  /* Launch choices in use (hipfmm_plan_autotune; no counterpart in the
   * reference): the matrix-core M2L tile shape code, 10 * column tiles per
   * wave + ring stages (0 = built-in default), and the near-field kernel at
   * batch % 32 == 0 (0 default, 1 vector ALU, 2 matrix cores with (target,
   * component) rows, 3 matrix cores with target rows, 4 matrix cores on bf16
   * three-piece operands -- the default; the field gradient runs the bf16
   * kernel for 0 and 4 and the FP32 target-rows kernel otherwise). */
  uint64_t m2l_tile_shape;
  uint64_t p2p_kernel_variant;
  double autotune_seconds; /* host time of the last hipfmm_plan_autotune */
  /* Wall time hipfmm_plan_create spent on the near-field index arrays: the
   * leaf ranges' upload, then the device build of the inverse permutations,
   * tile lists and 8-source block lists of both roles, to completion; no
   * counterpart in the reference. */
  double setup_index_seconds;
} hipfmm_stats;

/* Device-stream stage times of the most recent evaluate, seconds; mirrors
 * CudaEvaluationTimings (include/cdfmm/timings.hpp:225-241). */
typedef struct hipfmm_timings {
  double h2d_seconds;
  double p2m_seconds;   /* moment gather + P2M */
  double m2m_seconds;
  double m2l_seconds;   /* operand split + M2L */
  double l2l_seconds;
  double l2p_seconds;   /* L2P + combine + unsort */
  double p2p_seconds;   /* near-field stream */
  double kernel_seconds;/* first device stage to last */
  double d2h_seconds;
  double total_seconds;
  double m2l_kernel_seconds; /* the M2L product kernel alone (one launch, all levels) */
  /* Every M2L kernel launch of the plan so far, each timed with its own HIP
   * events on the evaluate's stream: summed durations and launch count (callers
   * average over a region by differencing two reads). */
  double m2l_kernel_total_seconds;
  uint64_t m2l_kernel_launches;
} hipfmm_timings;

/* Message of the last failure on this thread ("" if none). */
const char* hipfmm_last_error(void);

/* 1 when a HIP device with gfx950 code objects is usable, else 0.
 * Replaces cuda_full_available() (include/cdfmm/uniform_fmm.hpp:81-86). */
int hipfmm_runtime_available(void);

/* Device name, architecture and memory.  Replaces cuda_device_description()
 * (include/cdfmm/uniform_fmm.hpp:88-89). */
int hipfmm_device_description(char* buffer, size_t length);

/* Upload the static plan once.  Replaces CudaFullPlan::CudaFullPlan
 * (src/cuda_fmm_plan.hpp:97-98; src/cuda_fmm.cu:2714-3155). */
int hipfmm_plan_create(const hipfmm_plan_desc* desc, hipfmm_plan** plan);

/* Evaluate `batch` moment states.  Replaces CudaFullPlan::evaluate
 * (src/cuda_fmm_plan.hpp:104-108; src/cuda_fmm.cu:3238-3655) and adds the
 * batch dimension and device-resident operands.
 *   moments: batch x source_count x 3 scalars in user source order
 *   fields:  batch x target_count x 3 scalars in user target order
 *   scalar type is float for FP32 plans and double for FP64 plans;
 *   memspace says where both live.  Host moments must already carry the
 *   FP32 frame scaling; device moments are multiplied by
 *   desc.device_moment_scale.
 *   sorted_self_indices: host array of target_count entries (sorted target
 *   -> sorted source, or -1) or NULL.  The first map seen is fixed with the
 *   plan; a later different map fails with HIPFMM_ERROR_INVALID_ARGUMENT
 *   (src/cuda_fmm.cu:3470-3486).  NULL reuses the fixed map (none = -1).
 *   stream: hipStream_t to order device-memory work after, or NULL.
 * Host-memory calls return when the fields are in host memory; device-memory
 * calls return once the work is enqueued, the far field on `stream` itself and
 * the near field on a stream of the plan's, and ordered before any later work
 * on `stream`.  Calls on one plan take effect in the order they are made,
 * whatever their streams; after a call that fails, none of its work is left
 * running.
 * A device-memory call on a stream under capture is recorded, if an earlier
 * call allocated the state for its batch and outputs.  It follows the earlier
 * evaluates of that capture only, marks the end of its work by an event of its
 * own, so that evaluates outside the capture never wait for a recorded event,
 * and has no stage times; the order of the graph's replays with other
 * evaluates of the plan is the caller's.  The tests do not cover captures. */
int hipfmm_plan_evaluate(hipfmm_plan* plan, const void* moments, void* fields, int batch,
                         const int* sorted_self_indices, int memspace, void* stream);

/* Fields and potentials of `batch` moment states: CpuStatic's Potential /
 * Both outputs (src/uniform_fmm.cpp:1414-1437 potential rows, near field
 * src/near_field.cpp:30-80) on the device; the reference's CudaFull is
 * field-only (src/uniform_fmm.cpp:1103-1106).
 *   potentials: batch x target_count scalars in user target order (required)
 *   fields:     batch x target_count x 3 scalars, or NULL for potentials only
 * Everything else as for hipfmm_plan_evaluate.  The potential is the far
 * field sum_b L_b d^b/b! of the leaf local plus the near-field
 * (m.r)/(4 pi |r|^3), the identity pair skipped and coincident non-identity
 * pairs NaN, times desc.potential_scale. */
int hipfmm_plan_evaluate_potential(hipfmm_plan* plan, const void* moments, void* fields, void* potentials, int batch,
                                   const int* sorted_self_indices, int memspace, void* stream);

/* Transpose of hipfmm_plan_evaluate: the exact adjoint of the plan's linear
 * map from moments to fields (same tree, truncation and identity map), for
 * reverse-mode differentiation with respect to the moments.  No counterpart in
 * the reference, whose CudaFull path has no adjoint; the transpose it applies
 * is that of the operators it uses (P2M, M2M, M2L, L2L, L2P, P2P:
 * src/static_operators.cpp:159-335, :405-470).
 *   cotangents: batch x target_count x 3 scalars in user target order
 *   gradients:  batch x source_count x 3 scalars in user source order
 * With S = diag((-1)^|alpha|), P2M^T = -L2P S, L2L^T = S M2M S and
 * M2L_o^T = S M2L_-o S (the class matrices are symmetric in alpha, beta and
 * the level scalings differ by one power of the box width), so the transpose
 * is the same FMM with the roles of sources and targets exchanged; it runs on
 * the plan's own buffers.  The identity map is the plan's fixed map (none
 * before the first evaluate that sets one); a map that pairs two targets with
 * one source has no transposed form and fails with
 * HIPFMM_ERROR_INVALID_ARGUMENT.  Memory spaces, scaling and stream ordering
 * as for hipfmm_plan_evaluate. */
int hipfmm_plan_evaluate_adjoint(hipfmm_plan* plan, const void* cotangents, void* gradients, int batch,
                                 int memspace, void* stream);

/* Field gradient G_cj = dH_c/dx_j at the targets (no counterpart in the
 * reference), for gradients with respect to positions: for a loss
 * L = sum_t g_t . H(x_t), dL/dx_t = G(t) g_t (G is symmetric), and
 * dL/dx_s = G'(s) m_s with G' from hipfmm_plan_evaluate_field_gradient_adjoint
 * (the field gradient at the sources of the role-exchanged problem, whose
 * dipoles are the cotangents g).  The far part differentiates the leaf local
 * polynomial (src/static_operators.cpp:300-335), so it is exact for the FMM's
 * own far field and carries one order less truncation than the field; the
 * near part is the derivative of the pair tensor (src/cuboid.cpp:293-307).
 *   gradients: batch x target_count x 6 scalars (xx xy xz yy yz zz) in user
 *   target order (source order for the adjoint); the rest as for
 *   hipfmm_plan_evaluate / hipfmm_plan_evaluate_adjoint. */
int hipfmm_plan_evaluate_field_gradient(hipfmm_plan* plan, const void* moments, void* gradients, int batch,
                                        const int* sorted_self_indices, int memspace, void* stream);
int hipfmm_plan_evaluate_field_gradient_adjoint(hipfmm_plan* plan, const void* cotangents, void* gradients,
                                                int batch, int memspace, void* stream);

/* Select the M2L arithmetic of later evaluates (enum hipfmm_m2l_mode). */
int hipfmm_plan_set_m2l_mode(hipfmm_plan* plan, int mode);

/* Launch autotuner; no counterpart in the reference (whose CudaFull launch
 * shapes are fixed, src/cuda_fmm.cu:3500-3600).  Times, on the plan's own
 * state buffers at `batch` states and the current M2L mode, every tile shape
 * of the 16-bit modes' tiled M2L (by its kernel time, where the batch runs on
 * it: see hipfmm_m2l_mode) and the four near-field kernels (FP32 plans, batch
 * a multiple of 32; by the whole evaluate, since the near field overlaps the
 * far chain), keeps the fastest of each for later
 * evaluates of this plan and reports them in hipfmm_stats.  Results are unchanged in value
 * class: every candidate meets the same accuracy bars.  Overwrites the
 * plan's coefficients of the last evaluate. */
int hipfmm_plan_autotune(hipfmm_plan* plan, int batch);

/* Set the launch choices directly (values as reported in hipfmm_stats: a
 * tile shape code 23, 13, 43, 53, 24, 34 or 26, or 0 for the default; a near-field
 * variant 0..4), e.g. to reuse an earlier autotune result.  No counterpart in
 * the reference. */
int hipfmm_plan_set_launch_choices(hipfmm_plan* plan, int m2l_tile_shape, int p2p_kernel_variant);

/* Multi-geometry launch; no counterpart in the reference.  A group holds
 * the device-memory evaluates of `count` distinct plans (fields only, each
 * plan with its own device moments/fields pointers and batch), validated and
 * with their state allocated at creation.  hipfmm_group_launch enqueues all
 * of them after the work already on `stream`: every plan runs on its own
 * streams from one fork point, so the independent geometries' kernels
 * overlap on the device, and `stream` waits for all of them.  Pointers,
 * batches and each plan's identity map (sorted_self_indices: null, or one
 * entry per plan, each null or as for hipfmm_plan_evaluate, fixed with the
 * plan as there) are those at creation; M2L modes and launch choices are
 * read at each launch.  A plan belongs to at
 * most one group at a time and must not be evaluated while its group runs. */
typedef struct hipfmm_group hipfmm_group;
int hipfmm_group_create(hipfmm_plan* const* plans, int count, const void* const* moments, void* const* fields,
                        const int* batches, const int* const* sorted_self_indices, hipfmm_group** group);
int hipfmm_group_launch(hipfmm_group* group, void* stream);
void hipfmm_group_destroy(hipfmm_group* group);

/* Statistics / timings.  Replace CudaFullPlan::statistics() / timings(). */
int hipfmm_plan_statistics(const hipfmm_plan* plan, hipfmm_stats* out);
int hipfmm_plan_timings(const hipfmm_plan* plan, hipfmm_timings* out);

/* Copy the node-major coefficients of the last evaluate for one node and
 * moment state (which: 0 multipole, 1 local), n doubles.  Replaces the host
 * multipole()/local() accessors (src/uniform_fmm.cpp:1538-1612). */
int hipfmm_plan_coefficients(hipfmm_plan* plan, int which, int node, int state, double* out);

/* Free every device and pinned buffer.  Idempotent; NULL is accepted. */
void hipfmm_plan_destroy(hipfmm_plan* plan);

/* Leaf order of the uniform tree computed on the device; replaces the
 * leaf-key and sort steps of the host tree build (src/uniform_tree.cpp, the
 * leaf-key lambda and counting sort) with bitwise the same result.
 *   positions:   count x 3 doubles (memspace: HIPFMM_HOST or HIPFMM_DEVICE;
 *                permutation and leaf_ranges live in the same space)
 *   root_centre: 3 doubles (host), root_half_width >= 0 (0: all points
 *                coincide, all in leaf 0), max_level in [0, 9]
 *   permutation: count ints, sorted position -> input index (stable)
 *   leaf_ranges: 2 x 8^max_level int64, {begin, end} of each leaf in Morton
 *                order, {count, count} for an empty leaf
 * Returns HIPFMM_ERROR_INVALID_ARGUMENT for a point outside the root box. */
int hipfmm_tree_leaf_order(const double* positions, int count, const double* root_centre, double root_half_width,
                           int max_level, int memspace, int* permutation, int64_t* leaf_ranges, void* stream);

/* hipfmm_tree_leaf_order on device memory without allocating: no counterpart
 * in the reference.  It is for callers that cannot allocate device memory
 * (code under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc).  The sort's scratch (keys, indices, a flag and the radix sort's
 * temporary storage) lives in one fixed 48 MiB array per device, held from
 * the first call on that device until the process ends; the call makes no
 * hipMalloc/hipFree and no allocating library call.
 *   positions, permutation and leaf_ranges are device memory; the rest and
 *   the results are as for hipfmm_tree_leaf_order with HIPFMM_DEVICE.
 *   count must not exceed HIPFMM_NOALLOC_MAX_POINTS (2^21); larger counts
 *   fail with HIPFMM_ERROR_INVALID_ARGUMENT before any device work.
 * Every call on one device uses that device's single array: calls that
 * overlap on one device (other threads, other streams) race and must be
 * serialised by the caller.  The call returns after its work on `stream` is
 * done. */
#define HIPFMM_NOALLOC_MAX_POINTS (1 << 21)
int hipfmm_tree_leaf_order_noalloc(const double* positions, int count, const double* root_centre,
                                   double root_half_width, int max_level, int* permutation, int64_t* leaf_ranges,
                                   void* stream);

/* Failure injection for tests of the error paths.  After `skip` further
 * HIP runtime calls that succeed, the next one the library checks reports
 * `error` (a hipError_t value, e.g. hipErrorOutOfMemory = 2 or
 * hipErrorLaunchFailure = 719) as if the runtime had returned it, through
 * the same path as a real failure: HIPFMM_ERROR_RUNTIME, the runtime's text
 * for that error in hipfmm_last_error(), std::runtime_error in the C++
 * front-end.  It fires once and then disarms; error = 0 disarms.  The
 * setting is process-wide.  It stands in for the reference's mapping of
 * CUDA status codes to exceptions (src/cuda_fmm.cu:32-54), which a test
 * cannot otherwise force on a healthy device.  A plan that saw an injected
 * failure stays destroyable, and evaluates again once the injection is
 * spent. */
int hipfmm_debug_inject_error(int error, int skip);

/* A plan's near-field index array, copied to host memory for tests of its
 * device-side build: `name` is one of src_inv, tgt_inv, adj_self (int per
 * point), p2p_tiles, p2p_tiles4, p2p_tiles16, adj_tiles, adj_tiles16
 * ((leaf, first row) int pairs), blk8_start, nbr_blk_start, adj_blk8_start,
 * adj_nbr_blk_start (leaves + 1 offsets), blk8_src, adj_blk8_src ((first
 * source, count) int pairs), nbr_blk, adj_nbr_blk (block indices).  *count
 * receives the number of ints; with out non-null, capacity (ints) must hold
 * them.  No counterpart in the reference, which builds its near-field
 * pairs on the host (src/uniform_fmm.cpp:678-693) and uploads them
 * (src/cuda_fmm.cu:2212-2245); it is for the tests of the device build that
 * replaces that step. */
int hipfmm_debug_plan_index_array(const hipfmm_plan* plan, const char* name, int* out, int64_t capacity,
                                  int64_t* count);

/* FP64 O(N_t N_s) direct field with self exclusion on the device: the GPU
 * form of direct_p2p_reference (src/validation.cpp:71-111; model kernel
 * src/cuda_fmm.cu:518-569).  Host arrays: targets nt x 3, sources and moments
 * ns x 3, self_indices nt (or NULL), fields nt x 3 out. */
int hipfmm_direct_field(const double* targets, int nt, const double* sources, int ns,
                        const double* moments, const int* self_indices, double* fields);

#ifdef __cplusplus
}
#endif

#endif /* HIPFMM_H */
