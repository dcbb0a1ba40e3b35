/*
 * kvv.h -- C ABI of the MI355X numerical-agreement verdict library (libkvv.so).
 *
 * The library replaces the data-parallel part of KernelVerse's correctness
 * verdict: _compare_tensors (runner/generated_correctness_runner.py:672-786)
 * and, for batches of outputs, the per-tensor recursion of _compare_outputs
 * (runner/generated_correctness_runner.py:789-833).  The reference computes
 * the verdict with ~25 torch-CPU passes after copying both tensors to the
 * host (generated_correctness_runner.py:1315-1322); here both tensors stay in
 * HBM and are read once by hand-written gfx950 kernels.  Policy resolution,
 * rounding and the meta dictionary stay in the host language (Python
 * mirror: kernelverse_amd/verdict.py).
 *
 * Conventions
 *   - Plain C: pointers, sizes and PODs; no C++ exceptions cross the ABI.
 *   - Every call returns 0 on success or a negative KVV_E* code; the message
 *     of the last failure on the calling thread is kvv_last_error().
 *   - Calls are stream-ordered and asynchronous: results land in the
 *     kvv_result memory the caller passes -- device memory, or pinned host
 *     memory (hipHostMalloc) that the kernels write over the bus -- when the
 *     stream reaches them; the caller synchronises before reading them.  No
 *     global mutable device state: concurrent calls on different streams with
 *     different workspaces are independent.
 *   - Inputs are borrowed and never written.  Linear indices reported in
 *     kvv_result are LOGICAL row-major indices, not memory offsets.
 */
#ifndef KVV_H_
#define KVV_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#if defined(__GNUC__) || defined(__clang__)
#define KVV_API __attribute__((visibility("default")))
#else
#define KVV_API
#endif

#define KVV_ABI_VERSION 1
#define KVV_MAX_DIMS 8
#define KVV_HIST_BUCKETS 16

/* Element types (torch dtype in brackets). */
enum kvv_dtype {
  KVV_F32 = 0,       /* float32 */
  KVV_F16 = 1,       /* float16 */
  KVV_BF16 = 2,      /* bfloat16 */
  KVV_F64 = 3,       /* float64 */
  KVV_F8E4M3FN = 4,  /* float8_e4m3fn (OCP) */
  KVV_F8E5M2 = 5,    /* float8_e5m2 */
  KVV_I8 = 6,        /* int8 */
  KVV_U8 = 7,        /* uint8 */
  KVV_I16 = 8,       /* int16 */
  KVV_I32 = 9,       /* int32 */
  KVV_I64 = 10,      /* int64 */
  KVV_BOOL = 11,     /* bool (one byte, 0 or 1) */
  KVV_U16 = 12,      /* uint16 */
  KVV_U32 = 13,      /* uint32 */
  KVV_U64 = 14       /* uint64 */
};

/* Error codes. */
enum kvv_status {
  KVV_OK = 0,
  KVV_E_INVALID = -1,     /* bad argument (shape, dtype, policy, sizes) */
  KVV_E_WORKSPACE = -2,   /* workspace missing or too small */
  KVV_E_HIP = -3,         /* a HIP runtime call failed */
  KVV_E_UNSUPPORTED = -4  /* valid input this build cannot handle */
};

/* A strided tensor view in device memory.
 * Mirrors the torch.Tensor fields the reference reads (shape, dtype, strides). */
typedef struct kvv_tensor {
  const void* data;                 /* device address of logical element (0,...,0) */
  int32_t dtype;                    /* enum kvv_dtype */
  int32_t ndim;                     /* 0 (scalar) .. KVV_MAX_DIMS */
  int64_t sizes[KVV_MAX_DIMS];
  int64_t strides[KVV_MAX_DIMS];    /* in elements; may be 0 (broadcast) */
} kvv_tensor;

/* Elementwise test (generated_correctness_runner.py:714-728). */
enum kvv_mode {
  KVV_MODE_ISCLOSE = 0,        /* float branch: mismatch = !isclose(ref_f32, gen_f32, rtol, atol) */
  KVV_MODE_MAX_ABS_DIFF = 1    /* integer branch: mismatch = |int32(gen) - int32(ref)| > max_abs_diff */
};

/* Policy flags. */
#define KVV_FLAG_NEAR_ZERO 0x1u   /* tolerant-policy near-zero diagnostics (generated_correctness_runner.py:481-548);
                                     honoured for fp16/bf16 pairs, the only dtypes the reference computes them for */
#define KVV_FLAG_NEAR_EXACT 0x2u  /* with KVV_FLAG_NEAR_ZERO: take the near-zero sample in a second pass over the
                                     inputs instead of from entries recorded in the main pass */

#define KVV_FLAG_WS_KEPT 0x4u    /* the workspace is the one the previous single-pair verdict on this device was
                                     given, and nothing has written it since (a caller that keeps one workspace
                                     per stream, as the Python layer does).  Every single-pair verdict leaves its
                                     select slots clear; with this flag the next one on the same workspace skips
                                     clearing them (one launch fewer) when its slots lie where the previous
                                     call's did.  Without the flag, or on any other workspace, they are cleared.
                                     Ignored on a stream that is being captured into a graph (the graph always
                                     clears), and a captured call leaves no record for the next call to trust.
                                     No counterpart in the reference (GCR:672-786 allocates per call). */

/* kvv_result.status values.  kvv_verdict and kvv_verdict_noalloc return status 0: near-zero
 * entries that outgrow the workspace's pool are taken by reading that part of the pair again inside
 * the same call.  KVV_STATUS_NEAR_RETRY keeps its value for callers built against ABI version 1. */
#define KVV_STATUS_NEAR_RETRY 1   /* (no longer returned) the near-zero fields needed KVV_FLAG_NEAR_EXACT */

typedef struct kvv_policy {
  int32_t mode;                /* enum kvv_mode */
  uint32_t flags;              /* KVV_FLAG_* */
  double rtol, atol;           /* isclose tolerances; rounded to float32 like torch does */
  int64_t max_abs_diff;        /* integer-branch threshold; must fit int32 */
  double near_zero_abs;        /* near-zero threshold on |ref_f32| (rounded to float32) */
  double near_zero_bad_abs;    /* "bad" threshold on near-zero abs_diff (rounded to float32) */
  int64_t max_samples;         /* strided-sample cap m (1,000,000 in the reference); >= 2 */
} kvv_policy;

/* Everything the verdict needs, computed on the device.  Fields named after
 * the reference meta keys are exactly what the reference computes on CPU;
 * the "extension" block is defined by this library. */
typedef struct kvv_result {
  int64_t numel;
  /* generated_correctness_runner.py:731-771 */
  int64_t mismatch_count;
  int64_t first_mismatch_index;      /* -1 when there is none */
  double mismatch_max_abs;           /* max abs_diff over mismatches (NaN propagates); 0 when none */
  double mismatch_max_rel;           /* max rel_diff over mismatches */
  /* the <= max_samples strided sample (generated_correctness_runner.py:338-411) */
  int64_t sample_count;
  double p99_abs, p99_rel;           /* torch.quantile(sample, 0.99) in float32, widened */
  double sample_sum_gg, sample_sum_rr, sample_sum_gr;   /* fp64 over the sample */
  double sample_cosine;              /* unrounded; zero conventions of lines 364-369 */
  double sample_norm_ratio;          /* unrounded; zero conventions of lines 385-392 */
  /* finite pattern (generated_correctness_runner.py:414-437) */
  int64_t finite_violations;         /* positions breaking the rule; pass <=> 0 */
  int64_t first_finite_violation;    /* -1 when there is none */
  int64_t nan_gen, nan_ref, posinf_gen, posinf_ref, neginf_gen, neginf_ref;
  /* near-zero diagnostics (generated_correctness_runner.py:481-548); valid with KVV_FLAG_NEAR_ZERO */
  int64_t near_zero_count, far_count, far_mismatch_count, near_zero_bad_count;
  int64_t near_zero_sample_count;
  double near_zero_p99_abs, near_zero_mean_abs;
  /* extension: over ALL elements */
  double max_abs; int64_t max_abs_index;   /* argmax: NaN is maximal, ties -> lowest index */
  double max_rel; int64_t max_rel_index;
  uint64_t ulp_hist[KVV_HIST_BUCKETS];     /* b0: d==0; bk: 2^(k-1)<=d<2^k; b15: d>=2^14 */
  int64_t nan_pairs;                       /* pairs with a NaN on either side (no bucket) */
  double sum_gg, sum_rr, sum_gr, sum_dd;   /* fp64 sums of g*g, r*r, g*r, (g-r)^2 */
  double rel_l2, cosine;                   /* from the sums; cosine clamped to [-1,1] */
  int32_t status;                          /* 0, or KVV_STATUS_NEAR_RETRY */
  int32_t reserved;
} kvv_result;

/* ABI version (KVV_ABI_VERSION). */
KVV_API int kvv_abi_version(void);

/* Message of the last failed call on this thread ("" if none). */
KVV_API const char* kvv_last_error(void);

/* Workspace bytes for this pair and policy.  They include a contiguous copy of
 * each tensor (up to 1 GiB) whose layout rules out vector loads: a transposed or
 * oddly sliced view is copied before the main pass.  kvv_verdict also runs,
 * slower, with a workspace that has no room for the copies. */
KVV_API int kvv_workspace_size(const kvv_tensor* gen, const kvv_tensor* ref, const kvv_policy* policy, size_t* bytes);

/* What that size holds: `least`, the bytes kvv_verdict runs this pair with at all
 * (no copies, the smallest near-zero entry pool), and `copies`, the bytes of it
 * that are copies of the tensors (0: none). */
KVV_API int kvv_workspace_parts(const kvv_tensor* gen, const kvv_tensor* ref, const kvv_policy* policy, size_t* least,
                                size_t* copies);

/* One verdict: the data-parallel part of _compare_tensors
 * (generated_correctness_runner.py:672-786) for one tensor pair.
 *   gen, ref    same shape and dtype (checked; the reference returns a
 *               mismatch meta instead, which the host wrapper does first)
 *   out         one kvv_result in memory the device can write: device memory,
 *               or pinned host memory (hipHostMalloc) to receive it without a copy
 *   workspace   DEVICE scratch of at least kvv_workspace_size() bytes,
 *               256-byte aligned, owned by this call until the stream passes it
 *   stream      hipStream_t (NULL = default stream) */
KVV_API int kvv_verdict(const kvv_tensor* gen, const kvv_tensor* ref, const kvv_policy* policy,
                kvv_result* out, void* workspace, size_t workspace_bytes, void* stream);

/* kvv_verdict whose main-pass kernel records its own start in main_begin and
 * its end in main_end (hipEvent_t, created with timing; either may be NULL),
 * taken from the kernel's dispatch (hipExtLaunchKernel), so no marker packet
 * sits between the verdict's launches.  Nothing synchronises: the caller reads
 * the elapsed time once the stream has passed the kernel.  Used to time the
 * dominant kernel live inside a benchmark's timed region. */
KVV_API int kvv_verdict_timed(const kvv_tensor* gen, const kvv_tensor* ref, const kvv_policy* policy,
                              kvv_result* out, void* workspace, size_t workspace_bytes, void* stream,
                              void* main_begin, void* main_end);

/* kvv_verdict without a workspace argument and without any allocation.
 * No counterpart in the reference: it is for callers that cannot allocate
 * device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  The workspace is a 64 MiB array in the
 * library's code object, one per GPU, held until the process ends; a verdict
 * whose workspace (kvv_workspace_size) exceeds it fails with
 * KVV_E_WORKSPACE and leaves the stream untouched.  Calls on one GPU share
 * that array: calls that overlap on one GPU (other streams, other threads)
 * race, so the caller orders them.  The kernels clear what must start at
 * zero; the array keeps the last call's contents.  The call may be captured
 * into a HIP graph: it then clears its select slots in the graph, and once a
 * graph holding a no-alloc verdict exists on a device, eager calls there clear
 * theirs as well (the graph's replays write the array unseen). */
KVV_API int kvv_verdict_noalloc(const kvv_tensor* gen, const kvv_tensor* ref, const kvv_policy* policy,
                                kvv_result* out, void* stream);

/* Workspace bytes kvv_verdict_batch needs. */
KVV_API int kvv_batch_workspace_size(int32_t count, const kvv_tensor* gens, const kvv_tensor* refs,
                             const kvv_policy* policies, size_t* bytes);

/* A batch of independent verdicts -- one per pair, as the per-tensor
 * recursion of _compare_outputs (generated_correctness_runner.py:789-833)
 * produces -- with one main-pass launch per (dtype, test, layout) group and a
 * segmented reduction; each pair has its own policy (tolerances included).
 * gens/refs/policies are HOST arrays of `count` entries; out is an array of
 * `count` results in device memory or pinned host memory.  The call plans on
 * the host and uploads its pair table with one copy from a pinned staging
 * buffer; one dtype group's pivot and capture launches, and the launches
 * after the main passes that the capture final does not feed, may run on a
 * side stream joined back into `stream`.  The library keeps the staging buffer and
 * the side stream per device until the process ends.  A stream that is being
 * captured into a graph is refused (KVV_E_UNSUPPORTED): a replay would reuse
 * a stale upload. */
KVV_API int kvv_verdict_batch(int32_t count, const kvv_tensor* gens, const kvv_tensor* refs,
                      const kvv_policy* policies, kvv_result* out, void* workspace,
                      size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* KVV_H_ */
