// C-ABI entry points (include/iree_mi355x_kernels.h): host-side argument
// checks, kernel selection and launch.
//
// The reference proves its kernels' preconditions at compile time
// (CG/Transforms/HexagonVerifyHmxRuntimeABI.cpp:84-360: placement, row-major
// layout, 64/128/2048-byte alignment, extents that fit) and its kernels have
// no error channel (UK/api.h). Here every check runs on the host before
// launch and reports an iree_mi355x_status_t; nothing is launched on error.
#include <hip/hip_runtime.h>

#include <dlfcn.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/iree_mi355x_kernels.h"
#include "../../include/iree_mi355x_planner.h"
#include "kernels_internal.h"

namespace ihp {

static thread_local char g_last_error[512];

int fail(int status, const char *fmt, ...) {
  va_list args;
  va_start(args, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, args);
  va_end(args);
  return status;
}

static int ok() {
  g_last_error[0] = 0;
  return IREE_MI355X_OK;
}

// Validate-only calls (an executable-library dispatch whose state carries a
// workspace query): every check and the plan run, nothing is allocated or
// launched, and the workspace the launch would need is written to the sink.
static thread_local size_t *g_dry_run = nullptr;

void set_dry_run(size_t *sink) { g_dry_run = sink; }

static bool dry_run(int64_t workspace_needed) {
  if (!g_dry_run)
    return false;
  *g_dry_run = workspace_needed > 0 ? (size_t)workspace_needed : 0;
  return true;
}

// The kernel that a validate-only attention call takes.
static thread_local int32_t g_attention_family = 0;
static bool dry_run_attention(int64_t workspace_needed, int32_t family) {
  g_attention_family = family;
  return dry_run(workspace_needed);
}

static bool aligned(const void *p, size_t a) {
  return ((uintptr_t)p % a) == 0;
}

static const int64_t kMaxExtent = (int64_t)1 << 31;

// The split-K partials and arrival counters of a call come from the
// caller's workspace: the library allocates no device memory. A call whose
// plan needs `need` bytes and has none, or fewer, is refused before
// anything is launched.
int require_workspace(const char *who, size_t need, const void *workspace,
                      size_t workspace_bytes) {
  if (need == 0 || (workspace && workspace_bytes >= need))
    return IREE_MI355X_OK;
  if (!workspace)
    return fail(IREE_MI355X_WORKSPACE_TOO_SMALL,
                "%s: the plan needs a workspace of %zu bytes (size it with "
                "the workspace query) and none was passed",
                who, need);
  return fail(IREE_MI355X_WORKSPACE_TOO_SMALL, "%s: workspace %zu < %zu", who,
              workspace_bytes, need);
}

// Scratch of the allocation-free entry point: device memory of the
// library's own code object, one copy per GPU that runs the library, held
// until the process ends. It is zero from load, and every kernel that uses
// it leaves its arrival counters at zero again, so no call clears it;
// calls that overlap on one GPU race on it.
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) char scratch[kNoAllocScratchBytes];

// Device address of `scratch` on the current device, looked up once per
// device: the host-side name is only a stand-in, not a device address.
static std::mutex g_scratch_mutex;
static std::vector<void *> g_scratch;

static int scratch_address(void **out) {
  *out = nullptr;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess)
    return fail(IREE_MI355X_NO_DEVICE, "hipGetDevice failed");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if ((int)g_scratch.size() <= dev)
    g_scratch.resize(dev + 1, nullptr);
  if (!g_scratch[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      (void)hipGetLastError();
      return fail(IREE_MI355X_LAUNCH_FAILED,
                  "scratch: hipGetSymbolAddress failed: %s",
                  hipGetErrorString(e));
    }
    g_scratch[dev] = ptr;
  }
  *out = g_scratch[dev];
  return IREE_MI355X_OK;
}

static int launch_status(hipError_t e, const char *what) {
  if (e != hipSuccess)
    return fail(IREE_MI355X_LAUNCH_FAILED, "%s: %s", what, hipGetErrorString(e));
  return ok();
}

// Launch the planned MFMA configuration, with its split-K workspace.
static int launch_mfma(MatmulArgs &args, const iree_mi355x_matmul_plan_t &plan,
                       void *workspace, size_t workspace_bytes,
                       const char *who) {
  int count = 0;
  const FastConfig *cfgs = fast_configs(&count);
  args.splits = plan.splits > 1 ? plan.splits : 1;
  args.k_split = plan.k_split;
  args.sk_steps = plan.stream_k_steps;
  args.sk_workgroups = plan.stream_k_steps > 0 ? (int)plan.workgroups : 0;
  args.workspace = nullptr;
  if (plan.workspace_bytes > 0) {
    const int st = require_workspace(who, (size_t)plan.workspace_bytes,
                                     workspace, workspace_bytes);
    if (st != IREE_MI355X_OK)
      return st;
    args.workspace = workspace;
  }
  return launch_status(cfgs[plan.config_index].launch(args),
                       cfgs[plan.config_index].name);
}

// The plan of a call with this much workspace, and the workspace without
// which the call is refused (planner.cpp).
int plan_matmul(const iree_mi355x_matmul_desc_t *d, size_t workspace_limit,
                iree_mi355x_matmul_plan_t *plan, GeneralPlan *general,
                size_t *required);

// plan_general for a described matmul (planner.cpp).
bool plan_general_desc(const iree_mi355x_matmul_desc_t &d, bool wide,
                       size_t workspace_limit, GeneralPlan *plan);

// plan_matmul through a small per-thread table: a plan depends on nothing but
// the description and the workspace, and ranking the split configurations
// takes 1-4 us of host time, as long as the kernel of a small call.
static int cached_plan(const iree_mi355x_matmul_desc_t &d,
                       size_t workspace_limit, iree_mi355x_matmul_plan_t *plan,
                       GeneralPlan *general, size_t *required) {
  struct Entry {
    iree_mi355x_matmul_desc_t desc;
    size_t limit;
    iree_mi355x_matmul_plan_t plan;
    GeneralPlan general;  // of a plan of the general family
    size_t required;
    bool used;
  };
  static thread_local Entry table[64];
  uint64_t h = (uint64_t)d.m * 0x9E3779B97F4A7C15ull ^
               (uint64_t)d.n * 0xC2B2AE3D27D4EB4Full ^
               (uint64_t)d.k * 0x165667B19E3779F9ull ^
               ((uint64_t)d.flags << 40) ^ ((uint64_t)d.b_elem << 50) ^
               (uint64_t)d.batch;
  h ^= h >> 29;
  Entry &e = table[(h * 0x9E3779B97F4A7C15ull) >> 58];
  // desc_init zeroes the padding, so descriptions compare as bytes
  if (e.used && e.limit == workspace_limit &&
      memcmp(&e.desc, &d, sizeof(d)) == 0) {
    *plan = e.plan;
    *general = e.general;
    *required = e.required;
    return IREE_MI355X_OK;
  }
  const int st = plan_matmul(&d, workspace_limit, plan, general, required);
  if (st == IREE_MI355X_OK) {
    memcpy(&e.desc, &d, sizeof(d));
    e.limit = workspace_limit;
    e.plan = *plan;
    e.general = *general;
    e.required = *required;
    e.used = true;
  }
  return st;
}

// Plans a call within the workspace it has (a validate-only call: within
// workspace_bytes, whether or not a buffer is given yet) and refuses one that
// has less than it must. *done: nothing is left to run (refused or validated).
static int plan_call(const char *who, const iree_mi355x_matmul_desc_t &desc,
                     const void *workspace, size_t workspace_bytes,
                     iree_mi355x_matmul_plan_t *plan, GeneralPlan *general,
                     bool *done) {
  size_t required = 0;
  *done = true;
  if (cached_plan(desc, workspace || g_dry_run ? workspace_bytes : 0, plan,
                  general, &required) != IREE_MI355X_OK)
    return fail(IREE_MI355X_UNSUPPORTED, "%s: no plan", who);
  if (dry_run(plan->workspace_bytes))
    return ok();
  const int st = require_workspace(who, required, workspace, workspace_bytes);
  *done = st != IREE_MI355X_OK;
  return st;
}

// The general matmul of `desc` with the plan of plan_call, or for a wide
// pitch one of its own, its K split within the workspace the call has.
static int run_general(const char *who, MatmulArgs &args,
                       const iree_mi355x_matmul_desc_t &desc, GeneralPlan plan,
                       void *workspace, size_t workspace_bytes) {
  const bool wide =
      args.lda * (desc.a_elem == IREE_MI355X_ELEM_I8 ? 1 : 2) >=
          kMaxFastPitchBytes ||
      args.ldb * (desc.b_elem == IREE_MI355X_ELEM_I8 ? 1 : 2) >=
          kMaxFastPitchBytes;
  if (wide && !plan_general_desc(desc, true, workspace ? workspace_bytes : 0,
                                 &plan))
    return fail(IREE_MI355X_UNSUPPORTED, "%s: no plan", who);
  args.workspace = plan.workspace > 0 ? workspace : nullptr;
  return launch_status(launch_general(args, plan), who);
}

// Shared shape / stride checks for the three matmul entry points.
static int check_matmul(const char *who, const void *a, const void *b,
                        void *c, int64_t m, int64_t n, int64_t k, int64_t lda,
                        int64_t ldb, int64_t ldc, uint32_t flags,
                        uint32_t allowed_flags, size_t a_elem, size_t b_elem,
                        size_t c_elem) {
  if (flags & ~allowed_flags)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: unknown flag bits 0x%x", who,
                flags & ~allowed_flags);
  if (m < 0 || n < 0 || k < 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative extent", who);
  if (m >= kMaxExtent || n >= kMaxExtent || k >= kMaxExtent)
    return fail(IREE_MI355X_UNSUPPORTED, "%s: extent >= 2^31", who);
  if (m == 0 || n == 0)
    return IREE_MI355X_OK;
  const bool bt = flags & IREE_MI355X_MATMUL_B_TRANSPOSED;
  const bool at = flags & IREE_MI355X_MATMUL_A_TRANSPOSED;
  if (!c || (k > 0 && (!a || !b)))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: null pointer", who);
  if (lda < (at ? m : k) || ldb < (bt ? k : n) || ldc < n || lda < 0 ||
      ldb < 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: leading dimension smaller than the row", who);
  if ((a && !aligned(a, a_elem)) || (b && !aligned(b, b_elem)) ||
      !aligned(c, c_elem))
    return fail(IREE_MI355X_MISALIGNED,
                "%s: pointer not aligned to its element size", who);
  return IREE_MI355X_OK;
}

// One row of a transposed A ([K, 1] with unit pitch) is the contiguous row
// [1, K]: the same matmul without the transpose, which lets M = 1 decode
// stream as a GEMV. Returns the flags the call runs with.
uint32_t m1_row_layout(int64_t m, int64_t lda, uint32_t flags) {
  if ((flags & IREE_MI355X_MATMUL_A_TRANSPOSED) && m == 1 && lda == 1)
    return flags & ~IREE_MI355X_MATMUL_A_TRANSPOSED;
  return flags;
}

}  // namespace ihp

using namespace ihp;

extern "C" {

const char *iree_mi355x_last_error(void) { return g_last_error; }

const char *iree_mi355x_version(void) { return "iree-mi355x 0.1 gfx950"; }

int iree_mi355x_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess)
    return 0;
  return n;
}

size_t iree_mi355x_matmul_workspace_bytes(int64_t m, int64_t n, int64_t k,
                                          uint32_t flags) {
  if (m <= 0 || n <= 0 || k <= 0)
    return 0;
  // The largest workspace any f16, int8 or W8A16 plan of this shape uses (plans
  // assume 16-byte aligned operands; others take the general kernel, which
  // runs with any workspace), over both layouts a call may take: one row of a
  // transposed A with unit pitch runs as the untransposed row (see
  // m1_row_layout).
  size_t most = 0;
  const int32_t forms[4][3] = {
      {IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_F16},
      {IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_F32},
      {IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_I8, IREE_MI355X_ELEM_F16},
      {IREE_MI355X_ELEM_I8, IREE_MI355X_ELEM_I8, IREE_MI355X_ELEM_I32}};
  for (int layout = 0; layout < 2; ++layout) {
    const uint32_t lf =
        layout == 0 ? flags : m1_row_layout(m, 1, flags);
    if (layout == 1 && lf == flags)
      break;
    for (int f = 0; f < 4; ++f) {
      iree_mi355x_matmul_desc_t d;
      iree_mi355x_matmul_desc_init(&d, forms[f][0], forms[f][1], forms[f][2],
                                   m, n, k, lf & ~IREE_MI355X_MATMUL_OUT_F32);
      d.has_scale = f == 2;
      if (f == 1)
        d.flags |= IREE_MI355X_MATMUL_OUT_F32;
      iree_mi355x_matmul_plan_t p;
      if (iree_mi355x_plan_matmul(&d, &p) == IREE_MI355X_OK &&
          (size_t)p.workspace_bytes > most)
        most = (size_t)p.workspace_bytes;
    }
  }
  return most;
}

}  // extern "C"

namespace ihp {

// f16 matmul of `args` (batch and epilogue included): plan, workspace,
// launch. Shapes and pointers are validated by the caller.
static int matmul_f16_run(const char *who, MatmulArgs &args, uint32_t flags,
                          void *workspace, size_t workspace_bytes) {
  const bool out_f32 = flags & IREE_MI355X_MATMUL_OUT_F32;
  const uint32_t run_flags = m1_row_layout(args.m, args.lda, flags);
  if (run_flags != flags) {
    args.lda = args.k;
    flags = run_flags;
  }
  args.a_transposed = (flags & IREE_MI355X_MATMUL_A_TRANSPOSED) ? 1 : 0;
  iree_mi355x_matmul_desc_t desc;
  iree_mi355x_matmul_desc_init(&desc, IREE_MI355X_ELEM_F16,
                               IREE_MI355X_ELEM_F16,
                               out_f32 ? IREE_MI355X_ELEM_F32
                                       : IREE_MI355X_ELEM_F16,
                               args.m, args.n, args.k, flags);
  desc.a_aligned16 = fast_operand(args.a, args.lda * 2, args.sa * 2);
  desc.b_aligned16 = fast_operand(args.b, args.ldb * 2, args.sb * 2);
  desc.batch = args.batch;
  iree_mi355x_matmul_plan_t plan;
  GeneralPlan general = {};
  bool done = false;
  const int st =
      plan_call(who, desc, workspace, workspace_bytes, &plan, &general,
                 &done);
  if (done)
    return st;
  switch (plan.family) {
    case IREE_MI355X_FAMILY_GENERAL:
      return run_general(who, args, desc, general, workspace, workspace_bytes);
    case IREE_MI355X_FAMILY_GEMV:
      return launch_status(launch_gemv(args, 2, nullptr, out_f32, workspace),
                           "gemv_f16");
    default:
      return launch_mfma(args, plan, workspace, workspace_bytes, who);
  }
}

}  // namespace ihp

extern "C" {

int iree_mi355x_matmul_f16(const void *a, const void *b, void *c, int64_t m,
                           int64_t n, int64_t k, int64_t lda, int64_t ldb,
                           int64_t ldc, uint32_t flags, void *workspace,
                           size_t workspace_bytes, void *stream) {
  const bool out_f32 = flags & IREE_MI355X_MATMUL_OUT_F32;
  int st = check_matmul("matmul_f16", a, b, c, m, n, k, lda, ldb, ldc, flags,
                        IREE_MI355X_MATMUL_B_TRANSPOSED |
                            IREE_MI355X_MATMUL_ACCUMULATE |
                            IREE_MI355X_MATMUL_OUT_F32 |
                            IREE_MI355X_MATMUL_A_TRANSPOSED,
                        2, 2, out_f32 ? 4 : 2);
  if (st != IREE_MI355X_OK || m == 0 || n == 0)
    return st == IREE_MI355X_OK ? ok() : st;
  MatmulArgs args{a, b, c, m, n, k, lda, ldb, ldc,
                  (flags & IREE_MI355X_MATMUL_B_TRANSPOSED) ? 1 : 0,
                  (flags & IREE_MI355X_MATMUL_ACCUMULATE) ? 1 : 0, stream};
  return matmul_f16_run("matmul_f16", args, flags, workspace,
                        workspace_bytes);
}

int iree_mi355x_matmul_f16_no_alloc(const void *a, const void *b, void *c,
                                    int64_t m, int64_t n, int64_t k,
                                    int64_t lda, int64_t ldb, int64_t ldc,
                                    uint32_t flags, void *stream) {
  const char *who = "matmul_f16_no_alloc";
  const bool out_f32 = flags & IREE_MI355X_MATMUL_OUT_F32;
  int st = check_matmul(who, a, b, c, m, n, k, lda, ldb, ldc, flags,
                        IREE_MI355X_MATMUL_B_TRANSPOSED |
                            IREE_MI355X_MATMUL_ACCUMULATE |
                            IREE_MI355X_MATMUL_OUT_F32 |
                            IREE_MI355X_MATMUL_A_TRANSPOSED,
                        2, 2, out_f32 ? 4 : 2);
  if (st != IREE_MI355X_OK || m == 0 || n == 0)
    return st == IREE_MI355X_OK ? ok() : st;
  void *ws = nullptr;
  if ((st = scratch_address(&ws)) != IREE_MI355X_OK)
    return st;
  MatmulArgs args{a, b, c, m, n, k, lda, ldb, ldc,
                  (flags & IREE_MI355X_MATMUL_B_TRANSPOSED) ? 1 : 0,
                  (flags & IREE_MI355X_MATMUL_ACCUMULATE) ? 1 : 0, stream};
  // A plan needing more than the scratch holds is refused by the workspace
  // check (WORKSPACE_TOO_SMALL) before anything is launched.
  return matmul_f16_run(who, args, flags, ws, kNoAllocScratchBytes);
}

int iree_mi355x_batch_matmul_f16(const void *a, const void *b, void *c,
                                 int64_t batch, int64_t m, int64_t n,
                                 int64_t k, int64_t lda, int64_t ldb,
                                 int64_t ldc, int64_t stride_a,
                                 int64_t stride_b, int64_t stride_c,
                                 uint32_t flags,
                                 const iree_mi355x_epilogue_t *epilogue,
                                 void *workspace, size_t workspace_bytes,
                                 void *stream) {
  const char *who = "batch_matmul_f16";
  const bool out_f32 = flags & IREE_MI355X_MATMUL_OUT_F32;
  if (batch < 0 || stride_a < 0 || stride_b < 0 || stride_c < 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative batch or stride",
                who);
  if (batch > 65535)
    return fail(IREE_MI355X_UNSUPPORTED, "%s: batch %lld > 65535", who,
                (long long)batch);
  int st = check_matmul(who, a, b, c, m, n, k, lda, ldb, ldc, flags,
                        IREE_MI355X_MATMUL_B_TRANSPOSED |
                            IREE_MI355X_MATMUL_ACCUMULATE |
                            IREE_MI355X_MATMUL_OUT_F32 |
                            IREE_MI355X_MATMUL_A_TRANSPOSED,
                        2, 2, out_f32 ? 4 : 2);
  if (st != IREE_MI355X_OK || m == 0 || n == 0 || batch == 0)
    return st == IREE_MI355X_OK ? ok() : st;
  if (batch > 1 && stride_c < (m - 1) * ldc + n)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: stride_c %lld overlaps the outputs of consecutive "
                "batches", who, (long long)stride_c);
  MatmulArgs args{a, b, c, m, n, k, lda, ldb, ldc,
                  (flags & IREE_MI355X_MATMUL_B_TRANSPOSED) ? 1 : 0,
                  (flags & IREE_MI355X_MATMUL_ACCUMULATE) ? 1 : 0, stream};
  args.batch = batch;
  args.sa = stride_a;
  args.sb = stride_b;
  args.sc = stride_c;
  if (epilogue) {
    if (epilogue->activation > IREE_MI355X_ACT_SILU)
      return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: unknown activation %u",
                  who, epilogue->activation);
    if ((epilogue->bias && !aligned(epilogue->bias, 2)) ||
        (epilogue->multiplier && !aligned(epilogue->multiplier, 2)))
      return fail(IREE_MI355X_MISALIGNED, "%s: epilogue operand misaligned",
                  who);
    if (epilogue->multiplier && (epilogue->ld_multiplier < n ||
                                 epilogue->batch_stride_multiplier < 0))
      return fail(IREE_MI355X_INVALID_ARGUMENT,
                  "%s: multiplier pitch smaller than the row", who);
    args.bias = epilogue->bias;
    args.mul = epilogue->multiplier;
    args.ld_mul = epilogue->ld_multiplier;
    args.s_mul = epilogue->batch_stride_multiplier;
    args.act = (int)epilogue->activation;
  }
  return matmul_f16_run(who, args, flags, workspace, workspace_bytes);
}

size_t iree_mi355x_batch_matmul_workspace_bytes(int64_t batch, int64_t m,
                                                int64_t n, int64_t k,
                                                uint32_t flags) {
  if (batch <= 0 || m <= 0 || n <= 0 || k <= 0)
    return 0;
  size_t most = 0;
  for (int layout = 0; layout < 2; ++layout) {
    const uint32_t lf = layout == 0 ? flags : m1_row_layout(m, 1, flags);
    if (layout == 1 && lf == flags)
      break;
    iree_mi355x_matmul_desc_t d;
    iree_mi355x_matmul_desc_init(
        &d, IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_F16,
        (lf & IREE_MI355X_MATMUL_OUT_F32) ? IREE_MI355X_ELEM_F32
                                          : IREE_MI355X_ELEM_F16,
        m, n, k, lf);
    d.batch = batch;
    iree_mi355x_matmul_plan_t p;
    if (iree_mi355x_plan_matmul(&d, &p) == IREE_MI355X_OK &&
        (size_t)p.workspace_bytes > most)
      most = (size_t)p.workspace_bytes;
  }
  return most;
}

int iree_mi355x_matmul_i8(const int8_t *a, const int8_t *b, int32_t *c,
                          int64_t m, int64_t n, int64_t k, int64_t lda,
                          int64_t ldb, int64_t ldc, uint32_t flags,
                          void *workspace, size_t workspace_bytes,
                          void *stream) {
  int st = check_matmul("matmul_i8", a, b, c, m, n, k, lda, ldb, ldc, flags,
                        IREE_MI355X_MATMUL_B_TRANSPOSED |
                            IREE_MI355X_MATMUL_ACCUMULATE,
                        1, 1, 4);
  if (st != IREE_MI355X_OK || m == 0 || n == 0)
    return st == IREE_MI355X_OK ? ok() : st;
  MatmulArgs args{a, b, c, m, n, k, lda, ldb, ldc,
                  (flags & IREE_MI355X_MATMUL_B_TRANSPOSED) ? 1 : 0,
                  (flags & IREE_MI355X_MATMUL_ACCUMULATE) ? 1 : 0, stream};
  iree_mi355x_matmul_desc_t desc;
  iree_mi355x_matmul_desc_init(&desc, IREE_MI355X_ELEM_I8, IREE_MI355X_ELEM_I8,
                               IREE_MI355X_ELEM_I32, m, n, k, flags);
  desc.a_aligned16 = fast_operand(a, lda);
  desc.b_aligned16 = fast_operand(b, ldb);
  iree_mi355x_matmul_plan_t plan;
  GeneralPlan general = {};
  bool done = false;
  st = plan_call("matmul_i8", desc, workspace, workspace_bytes, &plan, &general,
                 &done);
  if (done)
    return st;
  if (plan.family == IREE_MI355X_FAMILY_GENERAL)
    return run_general("matmul_i8", args, desc, general, workspace,
                       workspace_bytes);
  return launch_mfma(args, plan, workspace, workspace_bytes, "matmul_i8");
}

int iree_mi355x_w8a16_matmul(const void *x, const int8_t *w, const void *scale,
                             void *y, int64_t m, int64_t n, int64_t k,
                             int64_t ldx, int64_t ldw, int64_t ldy,
                             uint32_t flags, void *workspace,
                             size_t workspace_bytes, void *stream) {
  int st = check_matmul("w8a16_matmul", x, w, y, m, n, k, ldx, ldw, ldy, flags,
                        IREE_MI355X_MATMUL_B_TRANSPOSED, 2, 1, 2);
  if (st != IREE_MI355X_OK || m == 0 || n == 0)
    return st == IREE_MI355X_OK ? ok() : st;
  if (!scale)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "w8a16_matmul: null scale");
  if (!aligned(scale, 2))
    return fail(IREE_MI355X_MISALIGNED, "w8a16_matmul: scale misaligned");
  MatmulArgs args{x, w, y, m, n, k, ldx, ldw, ldy,
                  (flags & IREE_MI355X_MATMUL_B_TRANSPOSED) ? 1 : 0, 0, stream,
                  scale};
  iree_mi355x_matmul_desc_t desc;
  iree_mi355x_matmul_desc_init(&desc, IREE_MI355X_ELEM_F16, IREE_MI355X_ELEM_I8,
                               IREE_MI355X_ELEM_F16, m, n, k, flags);
  desc.a_aligned16 = fast_operand(x, ldx * 2);
  desc.b_aligned16 = fast_operand(w, ldw);
  desc.has_scale = 1;
  iree_mi355x_matmul_plan_t plan;
  GeneralPlan general = {};
  bool done = false;
  st = plan_call("w8a16_matmul", desc, workspace, workspace_bytes, &plan,
                 &general, &done);
  if (done)
    return st;
  if (plan.family == IREE_MI355X_FAMILY_GENERAL)
    return run_general("w8a16_matmul", args, desc, general, workspace,
                       workspace_bytes);
  if (plan.family == IREE_MI355X_FAMILY_GEMV)
    return launch_status(launch_gemv(args, 1, scale, 0, workspace),
                         "gemv_w8a16");
  return launch_mfma(args, plan, workspace, workspace_bytes, "w8a16_matmul");
}

}  // extern "C"

namespace ihp {

// Modeled times of the attention kernels, in us, for the choice between them
// (attention_rows.hip takes a call only where it is modeled 1.2 times faster).
// Fits to both sides of 118 shapes (1 to 2048 queries, 64 to 8192 keys, head
// dims 40 to 256, causal, masked or neither, 8 to 96 heads): by this rule
// 1.0 % slower than the better kernel on average. Measured at both ends: one
// query of 32 heads over 8 KV heads and 3001 keys, batch 4, 13.3 us against
// 44.0 us for the fused kernel; 2048 x 2048 causal, 32 heads, d 128, 113 us
// against 44 us.
static double rows_us(const AttentionRowsPlan &p, int64_t seq_kv, bool causal,
                      int64_t seq_q, bool mask) {
  const int i = p.dp == 64 ? 0 : p.dp == 128 ? 1 : 2;
  static const double kUnit[] = {0.535e-3, 0.68e-3, 2.2e-3};
  static const double kChain[] = {0.326, 1.16, 0.93};
  const int64_t blocks = (seq_kv + 31) / 32;
  const double mean =
      (double)blocks * (causal && seq_q > 1 ? 0.5 : 1.0) + (causal ? 0.5 : 0);
  const int64_t wave_blocks = (p.blocks_per_split + 3) / 4;
  const int64_t held = p.dp < 256 ? 512 : 256;
  const int64_t rounds = (p.tiles * p.splits + held - 1) / held;
  return 5.78 +
         (double)p.tiles * mean * kUnit[i] * (mask ? 1.46 : 1.0) *
             (p.rf == 1 && p.dp < 256 ? 0.72 : 1.0) +
         kChain[i] * (double)(wave_blocks * rounds) +
         (p.splits > 1 ? 3.3 : 0.0);
}

// The fused kernel: rounds of workgroups of two query blocks, 128 keys a step.
static double fused_us(const iree_mi355x_attention_t &a, bool causal) {
  const int64_t n = (a.seq_q + 127) / 128;
  auto steps = [&](int64_t q) {
    const int64_t keys =
        causal && (q + 1) * 128 < a.seq_kv ? (q + 1) * 128 : a.seq_kv;
    return (double)((keys + 127) / 128);
  };
  const double total = steps(n - 1) + (n > 1 ? steps(0) : 0.0);
  const int64_t rounds = (a.batch * a.heads * ((n + 1) / 2) + 255) / 256;
  const double step = a.head_dim <= 64 ? (a.mask ? 2.24 : 0.99)
                                       : (a.mask ? 2.76 : 1.66);
  return 0.42 + (double)rounds * (step * total + 4.42 * (n > 1 ? 2.0 : 1.0));
}

// The general kernel: workgroups of 64 query rows (a block and its mirror
// under the causal mask), 64 keys a step.
static double general_attention_us(const iree_mi355x_attention_t &a,
                                   bool causal) {
  const int64_t d = a.head_dim > a.head_dim_v ? a.head_dim : a.head_dim_v;
  const int i = d <= 32 ? 0 : d <= 64 ? 1 : d <= 128 ? 2 : 3;
  static const double kAlone[] = {0.186, 1.83, 2.82, 4.98};
  static const double kShared[] = {0.192, 0.358, 2.39, 2.72};
  static const int64_t kHeld[] = {4, 4, 2, 1};
  const int64_t n = (a.seq_q + 63) / 64;
  const int64_t wgs = a.batch * a.heads * (causal ? (n + 1) / 2 : n);
  const int64_t steps = (a.seq_kv + 63) / 64 + (causal ? 1 : 0);
  const int64_t per_cu = (wgs + 255) / 256;
  const double alone = (kAlone[i] + (a.mask ? 4.39 : 0.0)) *
                       (double)((per_cu + kHeld[i] - 1) / kHeld[i]);
  const double shared =
      (kShared[i] + (a.mask ? 1.49 : 0.0)) * (double)per_cu;
  return 4.83 + (double)steps * (alone > shared ? alone : shared);
}

// Whether the row-packed kernel takes a call, and its plan. It needs head
// dims that are multiples of 8, and of a mask contiguous keys, at least 4;
// `fused`: the fused kernel takes the call otherwise.
static bool rows_plan(const iree_mi355x_attention_t &a, bool fused,
                      size_t workspace_limit, AttentionRowsPlan *plan) {
  const int64_t group = a.heads / a.kv_heads;
  if (a.head_dim % 8 != 0 || a.head_dim_v % 8 != 0 || a.head_dim_v < 8 ||
      a.seq_kv < 1 || a.seq_q * group >= kMaxExtent / 2 ||
      (a.mask && (a.mask_strides[3] != 1 || a.seq_kv < 4)))
    return false;
  *plan = plan_attention_rows(a.batch, a.kv_heads, group, a.seq_q, a.seq_kv,
                              a.head_dim, a.head_dim_v, workspace_limit);
  if (plan->tiles >= kMaxExtent)
    return false;
  const bool causal = a.flags & IREE_MI355X_ATTENTION_CAUSAL;
  const double other =
      fused ? fused_us(a, causal) : general_attention_us(a, causal);
  return rows_us(*plan, a.seq_kv, causal, a.seq_q, a.mask != nullptr) * 1.2 <
         other;
}

static AttentionGeneralLayout general_layout(const iree_mi355x_attention_t &a) {
  AttentionGeneralLayout g;
  const iree_mi355x_attention_strides_t &st = a.strides;
  for (int i = 0; i < 3; ++i) {
    g.q[i] = st.q[i];
    g.k[i] = st.k[i];
    g.v[i] = st.v[i];
    g.o[i] = st.o[i];
  }
  for (int i = 0; i < 4; ++i)
    g.mask[i] = a.mask_strides[i];
  g.heads = (int)a.heads;
  g.group = (int)(a.heads / a.kv_heads);
  g.seq_q = (int)a.seq_q;
  g.seq_kv = (int)a.seq_kv;
  g.dqk = (int)a.head_dim;
  g.dv = (int)a.head_dim_v;
  g.scale = a.scale;
  g.causal = (a.flags & IREE_MI355X_ATTENTION_CAUSAL) ? 1 : 0;
  g.vec_k = a.head_dim % 8 == 0 && st.k[0] % 8 == 0 && st.k[1] % 8 == 0 &&
            st.k[2] % 8 == 0 && aligned(a.k, 16);
  g.vec_v = a.head_dim_v % 8 == 0 && st.v[0] % 8 == 0 &&
            st.v[1] % 8 == 0 && st.v[2] % 8 == 0 && aligned(a.v, 16);
  return g;
}

// Runs a checked call on the row-packed kernel if that takes it; *ran tells.
static int try_rows(const iree_mi355x_attention_t &a, bool fused,
                    void *workspace, size_t workspace_bytes, void *stream,
                    bool *ran) {
  AttentionRowsPlan plan;
  *ran = rows_plan(a, fused, workspace || g_dry_run ? workspace_bytes : 0,
                   &plan);
  if (!*ran)
    return IREE_MI355X_OK;
  if (dry_run_attention(plan.workspace, IREE_MI355X_ATTENTION_FAMILY_ROWS))
    return ok();
  return launch_status(
      launch_attention_rows(a.q, a.k, a.v, a.o, a.mask, general_layout(a),
                            plan,
                            (a.flags & IREE_MI355X_ATTENTION_OUT_F32) ? 1 : 0,
                            workspace, stream),
      "attention_rows");
}

}  // namespace ihp

extern "C" {

int iree_mi355x_attention_f16_strided(
    const void *q, const void *k, const void *v, void *o, int64_t batch,
    int64_t heads, int64_t kv_heads, int64_t seq_q, int64_t seq_kv,
    int64_t head_dim, float scale, uint32_t flags,
    const iree_mi355x_attention_strides_t *strides, void *stream) {
  const char *who = "attention_f16";
  if (flags & ~IREE_MI355X_ATTENTION_CAUSAL)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: unknown flag bits 0x%x",
                who, flags);
  if (batch < 0 || heads < 0 || kv_heads < 0 || seq_q < 0 || seq_kv < 0 ||
      head_dim < 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative extent", who);
  if (!std::isfinite(scale))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: scale not finite", who);
  if (!strides)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: null strides", who);
  if (batch == 0 || heads == 0 || seq_q == 0)
    return ok();
  if (kv_heads == 0 || heads % kv_heads != 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: %lld query heads are not a multiple of %lld KV heads",
                who, (long long)heads, (long long)kv_heads);
  if (head_dim != 64 && head_dim != 128)
    return fail(IREE_MI355X_UNSUPPORTED,
                "%s: head_dim %lld (64 or 128 supported)", who,
                (long long)head_dim);
  if (!q || !o || (seq_kv > 0 && (!k || !v)))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: null pointer", who);
  const int64_t *st[4] = {strides->q, strides->k, strides->v, strides->o};
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i)
      if (st[t][i] < 0)
        return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative stride", who);
  if (strides->o[2] < head_dim)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: o row stride %lld overlaps its rows", who,
                (long long)strides->o[2]);
  // The copies and stores move 16-byte chunks of rows: every base, and
  // every stride (in bytes), must keep them aligned.
  for (int t = 0; t < 4; ++t)
    for (int i = 0; i < 3; ++i)
      if (st[t][i] % 8 != 0)
        return fail(IREE_MI355X_MISALIGNED,
                    "%s: strides must be multiples of 8 elements", who);
  if (!aligned(q, 16) || !aligned(o, 16) || (k && !aligned(k, 16)) ||
      (v && !aligned(v, 16)))
    return fail(IREE_MI355X_MISALIGNED,
                "%s: q/k/v/o must be 16-byte aligned", who);
  const int64_t q_blocks = (seq_q + 127) / 128;
  if (batch >= kMaxExtent || heads >= kMaxExtent || seq_q >= kMaxExtent ||
      seq_kv >= kMaxExtent || batch * heads * q_blocks >= kMaxExtent)
    return fail(IREE_MI355X_UNSUPPORTED, "%s: problem too large", who);
  // Q, K and V rows are copied with a 32-bit byte offset from their head's
  // first row.
  const int64_t row_bytes = head_dim * 2;
  auto head_span = [&](const int64_t *s, int64_t rows) -> int64_t {
    if (rows <= 1)
      return rows == 1 ? row_bytes : 0;
    const uint64_t pitch = (uint64_t)s[2] * 2;
    if (s[2] > (int64_t)UINT32_MAX ||
        (pitch > 0 &&
         (uint64_t)(rows - 1) > (UINT32_MAX - (uint64_t)row_bytes) / pitch))
      return INT64_MAX;
    return (int64_t)((uint64_t)(rows - 1) * pitch) + row_bytes;
  };
  if (head_span(strides->q, seq_q) > (int64_t)UINT32_MAX ||
      head_span(strides->k, seq_kv) > (int64_t)UINT32_MAX ||
      head_span(strides->v, seq_kv) > (int64_t)UINT32_MAX)
    return fail(IREE_MI355X_UNSUPPORTED,
                "%s: a head's rows span more than 4 GiB", who);
  iree_mi355x_attention_t a = {};
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.batch = batch;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.seq_q = seq_q;
  a.seq_kv = seq_kv;
  a.head_dim = a.head_dim_v = head_dim;
  a.scale = scale;
  a.flags = flags;
  a.strides = *strides;
  bool ran = false;
  const int rows_st = try_rows(a, true, nullptr, 0, stream, &ran);
  if (ran)
    return rows_st;
  if (dry_run_attention(0, IREE_MI355X_ATTENTION_FAMILY_FUSED))
    return ok();
  AttentionLayout layout;
  for (int i = 0; i < 3; ++i) {
    layout.q[i] = strides->q[i];
    layout.k[i] = strides->k[i];
    layout.v[i] = strides->v[i];
    layout.o[i] = strides->o[i];
    layout.m[i] = 0;
  }
  layout.heads = (int)heads;
  layout.group = (int)(heads / kv_heads);
  layout.seq_q = (int)seq_q;
  layout.seq_kv = (int)seq_kv;
  return launch_status(
      launch_attention(q, k, v, o, batch, layout, head_dim, scale,
                       (flags & IREE_MI355X_ATTENTION_CAUSAL) ? 1 : 0, stream),
      "attention_fwd");
}

int iree_mi355x_attention_with_workspace(const iree_mi355x_attention_t *a,
                                         void *workspace,
                                         size_t workspace_bytes,
                                         void *stream) {
  const char *who = "attention";
  if (!a)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: null arguments", who);
  if (a->flags & ~(IREE_MI355X_ATTENTION_CAUSAL | IREE_MI355X_ATTENTION_OUT_F32 |
                   IREE_MI355X_ATTENTION_MASK))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: unknown flag bits 0x%x",
                who, a->flags);
  if (!(a->flags & IREE_MI355X_ATTENTION_MASK) != !a->mask)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: the MASK flag and the mask pointer disagree", who);
  if (a->batch < 0 || a->heads < 0 || a->kv_heads < 0 || a->seq_q < 0 ||
      a->seq_kv < 0 || a->head_dim < 0 || a->head_dim_v < 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative extent", who);
  if (!std::isfinite(a->scale))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: scale not finite", who);
  if (a->batch == 0 || a->heads == 0 || a->seq_q == 0 || a->head_dim_v == 0)
    return ok();
  if (a->kv_heads == 0 || a->heads % a->kv_heads != 0)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: %lld query heads are not a multiple of %lld KV heads",
                who, (long long)a->heads, (long long)a->kv_heads);
  if (a->head_dim < 1 || a->head_dim > 256 || a->head_dim_v > 256)
    return fail(IREE_MI355X_UNSUPPORTED,
                "%s: head dims %lld / %lld (1..256 supported)", who,
                (long long)a->head_dim, (long long)a->head_dim_v);
  // Grid (query blocks, heads, batch) and 32-bit row and key counters.
  if (a->batch > 65535 || a->heads > 65535 || a->seq_q >= kMaxExtent / 2 ||
      a->seq_kv >= kMaxExtent / 2)
    return fail(IREE_MI355X_UNSUPPORTED, "%s: problem too large", who);
  if (!a->q || !a->o || (a->seq_kv > 0 && (!a->k || !a->v)))
    return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: null pointer", who);
  const iree_mi355x_attention_strides_t &st = a->strides;
  // Mask strides are read only with a mask.
  const int64_t *all[5] = {st.q, st.k, st.v, st.o, a->mask_strides};
  for (int t = 0; t < (a->mask ? 5 : 4); ++t)
    for (int i = 0; i < (t == 4 ? 4 : 3); ++i)
      if (all[t][i] < 0)
        return fail(IREE_MI355X_INVALID_ARGUMENT, "%s: negative stride", who);
  if (st.o[2] < a->head_dim_v)
    return fail(IREE_MI355X_INVALID_ARGUMENT,
                "%s: o row stride %lld overlaps its rows", who,
                (long long)st.o[2]);
  const bool out_f32 = a->flags & IREE_MI355X_ATTENTION_OUT_F32;
  if (!aligned(a->q, 2) || !aligned(a->o, out_f32 ? 4 : 2) ||
      (a->k && !aligned(a->k, 2)) || (a->v && !aligned(a->v, 2)) ||
      (a->mask && !aligned(a->mask, 2)))
    return fail(IREE_MI355X_MISALIGNED,
                "%s: operands must be aligned to their element size", who);
  const bool causal = a->flags & IREE_MI355X_ATTENTION_CAUSAL;

  // The MFMA kernel: equal head dims that are multiples of 16 up to 128,
  // 16-byte rows and strides, each head's rows within 4 GiB (32-bit copy
  // offsets), and a grid of pairs of 128-row query blocks; a mask with
  // contiguous keys read 4 keys (8 bytes) at a time: strides and base
  // 8-byte aligned, seq_kv a multiple of 4.
  bool fast = a->head_dim == a->head_dim_v && a->head_dim % 16 == 0 &&
              a->head_dim <= 128 &&
              aligned(a->q, 16) && aligned(a->o, 16) &&
              (!a->k || aligned(a->k, 16)) && (!a->v || aligned(a->v, 16));
  if (fast && a->mask)
    fast = a->mask_strides[3] == 1 && a->mask_strides[0] % 4 == 0 &&
           a->mask_strides[1] % 4 == 0 && a->mask_strides[2] % 4 == 0 &&
           aligned(a->mask, 8) && a->seq_kv % 4 == 0;
  for (int t = 0; t < 4 && fast; ++t)
    for (int i = 0; i < 3; ++i)
      if (all[t][i] % 8 != 0)
        fast = false;
  const int64_t row_bytes = a->head_dim * 2;
  auto head_span = [&](const int64_t *s, int64_t rows) -> int64_t {
    if (rows <= 1)
      return rows == 1 ? row_bytes : 0;
    const uint64_t pitch = (uint64_t)s[2] * 2;
    if (s[2] > (int64_t)UINT32_MAX ||
        (pitch > 0 &&
         (uint64_t)(rows - 1) > (UINT32_MAX - (uint64_t)row_bytes) / pitch))
      return INT64_MAX;
    return (int64_t)((uint64_t)(rows - 1) * pitch) + row_bytes;
  };
  if (fast && (head_span(st.q, a->seq_q) > (int64_t)UINT32_MAX ||
               head_span(st.k, a->seq_kv) > (int64_t)UINT32_MAX ||
               head_span(st.v, a->seq_kv) > (int64_t)UINT32_MAX ||
               a->batch * a->heads * ((a->seq_q + 127) / 128) >= kMaxExtent))
    fast = false;
  bool ran = false;
  const int rows_st =
      try_rows(*a, fast, workspace, workspace_bytes, stream, &ran);
  if (ran)
    return rows_st;
  if (fast && !a->mask && !out_f32 &&
      (a->head_dim == 64 || a->head_dim == 128))
    return iree_mi355x_attention_f16_strided(
        a->q, a->k, a->v, a->o, a->batch, a->heads, a->kv_heads, a->seq_q,
        a->seq_kv, a->head_dim, a->scale, a->flags & IREE_MI355X_ATTENTION_CAUSAL,
        &a->strides, stream);
  if (dry_run_attention(0, fast ? IREE_MI355X_ATTENTION_FAMILY_FUSED
                                : IREE_MI355X_ATTENTION_FAMILY_GENERAL))
    return ok();
  if (fast) {
    AttentionLayout layout;
    for (int i = 0; i < 3; ++i) {
      layout.q[i] = st.q[i];
      layout.k[i] = st.k[i];
      layout.v[i] = st.v[i];
      layout.o[i] = st.o[i];
      layout.m[i] = a->mask_strides[i];
    }
    layout.heads = (int)a->heads;
    layout.group = (int)(a->heads / a->kv_heads);
    layout.seq_q = (int)a->seq_q;
    layout.seq_kv = (int)a->seq_kv;
    return launch_status(
        launch_attention(a->q, a->k, a->v, a->o, a->batch, layout,
                         a->head_dim, a->scale, causal ? 1 : 0, stream,
                         a->mask, out_f32 ? 1 : 0),
        a->mask ? "attention_fwd_mask" : "attention_fwd");
  }
  return launch_status(
      launch_attention_general(a->q, a->k, a->v, a->o, a->mask, a->batch,
                               general_layout(*a), out_f32 ? 1 : 0, stream),
      "attention_general");
}

int iree_mi355x_attention(const iree_mi355x_attention_t *a, void *stream) {
  return iree_mi355x_attention_with_workspace(a, nullptr, 0, stream);
}

int32_t iree_mi355x_classify_attention(const iree_mi355x_attention_t *a,
                                       size_t workspace_bytes) {
  size_t need = 0;
  g_attention_family = IREE_MI355X_ATTENTION_FAMILY_NONE;
  set_dry_run(&need);
  const int st = iree_mi355x_attention_with_workspace(a, nullptr,
                                                      workspace_bytes, nullptr);
  set_dry_run(nullptr);
  return st == IREE_MI355X_OK ? g_attention_family
                              : IREE_MI355X_ATTENTION_FAMILY_NONE;
}

size_t iree_mi355x_attention_workspace_bytes(
    const iree_mi355x_attention_t *a) {
  if (!a || a->batch < 1 || a->heads < 1 || a->kv_heads < 1 ||
      a->heads % a->kv_heads != 0 || a->seq_q < 1 || a->seq_kv < 1 ||
      a->head_dim < 1 || a->head_dim_v < 1 || a->head_dim > 256 ||
      a->head_dim_v > 256 || a->batch > 65535 || a->heads > 65535 ||
      a->seq_q >= kMaxExtent / 2 || a->seq_kv >= kMaxExtent / 2)
    return 0;
  iree_mi355x_attention_t d = *a;
  if (a->flags & IREE_MI355X_ATTENTION_MASK) {
    d.mask = a;  // present; only its strides and extents matter here
    d.mask_strides[3] = 1;
  }
  const bool fused = a->head_dim == a->head_dim_v && a->head_dim % 16 == 0 &&
                     a->head_dim <= 128 && (!d.mask || a->seq_kv % 4 == 0);
  AttentionRowsPlan plan;
  return rows_plan(d, fused, (size_t)-1, &plan) ? (size_t)plan.workspace : 0;
}

int iree_mi355x_attention_f16(const void *q, const void *k, const void *v,
                              void *o, int64_t batch, int64_t heads,
                              int64_t seq_q, int64_t seq_kv, int64_t head_dim,
                              float scale, uint32_t flags, void *stream) {
  // Contiguous [B, H, S, D] operands, one KV head per query head.
  if (heads >= kMaxExtent || seq_q >= kMaxExtent || seq_kv >= kMaxExtent ||
      head_dim >= kMaxExtent)
    return fail(IREE_MI355X_UNSUPPORTED, "attention_f16: problem too large");
  iree_mi355x_attention_strides_t s;
  const int64_t qs[3] = {heads * seq_q * head_dim, seq_q * head_dim, head_dim};
  const int64_t ks[3] = {heads * seq_kv * head_dim, seq_kv * head_dim,
                         head_dim};
  for (int i = 0; i < 3; ++i) {
    s.q[i] = s.o[i] = qs[i];
    s.k[i] = s.v[i] = ks[i];
  }
  return iree_mi355x_attention_f16_strided(q, k, v, o, batch, heads, heads,
                                           seq_q, seq_kv, head_dim, scale,
                                           flags, &s, stream);
}

}  // extern "C"
