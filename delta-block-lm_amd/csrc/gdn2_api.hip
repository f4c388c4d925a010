// C ABI of libgdn2_amd.so: argument validation and kernel dispatch.
//
// Every entry point validates its whole argument list before it launches
// anything, mirroring the reference's fail-fast asserts
// (crates/kernels/src/gdn_training.rs:286-342, :356-390; chunk.rs:110-124):
// an unsupported shape, dtype or buffer size is an error, never a fallback.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <string>

#include "gdn2_chunk.h"
#include "gdn2_chunk_f32.h"
#include "gdn2_seq.h"
#include "gdn2_status.h"

namespace gdn2 {

namespace {
thread_local std::string g_error;
}

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_error = buf;
    return code;
}

int ok() {
    g_error.clear();
    return GDN2_OK;
}

const char *last_error() { return g_error.c_str(); }

int check_view(const gdn2_view *v, const char *name, int dtype, bool data_may_be_null) {
    if (!v) return fail(GDN2_ERR_ARGUMENT, "%s: view is null", name);
    if (!v->data && !data_may_be_null) return fail(GDN2_ERR_ARGUMENT, "%s: data is null", name);
    if (v->dtype != GDN2_F32 && v->dtype != GDN2_BF16 && v->dtype != GDN2_I32)
        return fail(GDN2_ERR_DTYPE, "%s: unknown dtype %d", name, v->dtype);
    if (dtype < 0 && v->dtype == GDN2_I32)
        return fail(GDN2_ERR_DTYPE, "%s: dtype must be F32 or BF16", name);
    if (dtype >= 0 && v->dtype != dtype)
        return fail(GDN2_ERR_DTYPE, "%s: dtype must be %s", name,
                    dtype == GDN2_F32 ? "F32" : (dtype == GDN2_BF16 ? "BF16" : "I32"));
    for (int d = 0; d < 4; ++d)
        if (v->stride[d] < 0) return fail(GDN2_ERR_ARGUMENT, "%s: negative stride", name);
    return GDN2_OK;
}

int launch_status(hipError_t e, const char *what) {
    if (e != hipSuccess) return fail(GDN2_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
    return ok();
}

}  // namespace gdn2

using namespace gdn2;

namespace {

// Stage timing (gdn2_stage_timing): six stages, an event pair each; the
// forward records pairs 0-2, the backward pairs 3-5; the scalar-gate op's f32 chunk
// kernels have six of their own behind them, so that a call's stages tell which
// kernels it ran.  A measurement hook for
// benchmarks only: the events and flags below are process-wide (not thread
// safe), and no event is recorded on a stream that is being captured, so a
// graph never holds them.
constexpr int kScalarF32 = 6, kStages = 12;
const char *const kStageNames[kStages] = {
    "chunk_prep", "state_scan", "chunk_out", "chunk_bprep", "adjoint_scan", "chunk_bgrad",
    "scalar_f32_prep", "scalar_f32_state_scan", "scalar_f32_out",
    "scalar_f32_bprep", "scalar_f32_adjoint_scan", "scalar_f32_bgrad"};
hipEvent_t g_stage_ev[2 * kStages];
bool g_stage_ready = false;  // events created
bool g_stage_on = false;
bool g_stage_ran[kStages];

const hipEvent_t *stage_events(int first_stage, hipStream_t stream) {
    if (!g_stage_on) return nullptr;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone)
        return nullptr;
    for (int i = 0; i < 3; ++i) g_stage_ran[first_stage + i] = true;
    return g_stage_ev + 2 * first_stage;
}

int check_shape(const gdn2_shape *s) {
    if (!s) return fail(GDN2_ERR_ARGUMENT, "shape is null");
    if (s->batch <= 0 || s->time <= 0 || s->heads <= 0)
        return fail(GDN2_ERR_SHAPE, "GDN-2 requires nonempty axes (batch=%lld time=%lld heads=%lld)",
                    (long long)s->batch, (long long)s->time, (long long)s->heads);
    if (s->keys < 1 || s->keys > 128 || s->values < 1 || s->values > 128)
        return fail(GDN2_ERR_SHAPE, "key/value widths must be 1..128 (keys=%lld values=%lld)",
                    (long long)s->keys, (long long)s->values);
    if (s->batch * s->heads > INT_MAX || s->time > INT_MAX / 2)
        return fail(GDN2_ERR_SHAPE, "batch*heads or time exceeds the launch limits");
    return GDN2_OK;
}

int check_chunk(int chunk) {
    if (chunk < 1 || chunk > 64) return fail(GDN2_ERR_ARGUMENT, "chunk must be 1..64 (got %d)", chunk);
    return GDN2_OK;
}

int check_out_dtype(int32_t dt) {
    if (dt != GDN2_F32 && dt != GDN2_BF16) return fail(GDN2_ERR_DTYPE, "output dtype must be F32 or BF16");
    return GDN2_OK;
}

size_t seq_workspace_bytes(const gdn2_shape *s) {
    return (size_t)seq_workspace_floats(s->batch, s->heads, (int)s->keys, (int)s->values) * 4;
}

int check_channel_inputs(const gdn2_shape *shape, const gdn2_view *q, const gdn2_view *k,
                         const gdn2_view *v, const gdn2_view *alpha, const gdn2_view *erase,
                         const gdn2_view *write, const gdn2_view *valid, const gdn2_view *reset) {
    GDN2_TRY(check_view(q, "q", -1, false));
    GDN2_TRY(check_view(k, "k", q->dtype, false));
    GDN2_TRY(check_view(v, "v", q->dtype, false));
    GDN2_TRY(check_view(alpha, "alpha", GDN2_F32, false));
    GDN2_TRY(check_view(erase, "erase", GDN2_F32, false));
    GDN2_TRY(check_view(write, "write", GDN2_F32, false));
    GDN2_TRY(check_view(valid, "valid", GDN2_F32, false));
    GDN2_TRY(check_view(reset, "reset", GDN2_F32, false));
    return GDN2_OK;
}

int check_doc_inputs(const gdn2_view *q, const gdn2_view *k, const gdn2_view *v,
                     const gdn2_view *alpha, const gdn2_view *erase, const gdn2_view *write,
                     const gdn2_view *doc_start, const gdn2_view *doc_end) {
    GDN2_TRY(check_view(q, "q", -1, false));
    GDN2_TRY(check_view(k, "k", q->dtype, false));
    GDN2_TRY(check_view(v, "v", q->dtype, false));
    GDN2_TRY(check_view(alpha, "alpha", GDN2_F32, false));
    GDN2_TRY(check_view(erase, "erase", GDN2_F32, false));
    GDN2_TRY(check_view(write, "write", GDN2_F32, false));
    GDN2_TRY(check_view(doc_start, "doc_start", GDN2_I32, false));
    GDN2_TRY(check_view(doc_end, "doc_end", GDN2_I32, false));
    return GDN2_OK;
}

SeqArgs seq_args(const gdn2_shape *s, const gdn2_view *q, const gdn2_view *k, const gdn2_view *v,
                 const gdn2_view *alpha, const gdn2_view *erase, const gdn2_view *write,
                 const gdn2_view *valid, const gdn2_view *reset) {
    SeqArgs a{};
    a.B = (int)s->batch;
    a.T = (int)s->time;
    a.H = (int)s->heads;
    a.K = (int)s->keys;
    a.V = (int)s->values;
    a.q = make_view(q);
    a.k = make_view(k);
    a.v = make_view(v);
    a.alpha = make_view(alpha);
    a.erase = make_view(erase);
    a.write = make_view(write);
    a.valid = make_view(valid);
    a.reset = make_view(reset);
    a.nck = (a.T + SEQ_CT - 1) / SEQ_CT;
    return a;
}

}  // namespace

// Device scratch of gdn_scalar_backward_noalloc: a fixed array in every
// device's copy of the code object, held until the process ends.  Host code
// never uses the array's name as an address: each device's address comes from
// hipGetSymbolAddress, taken once per device with that device current.
// The bytes past the public size take the f32 chunk kernels' words of a shape whose
// other needs fill it: at most 1024, as the token walk needs 64 KiB or more for
// each batch and head.
constexpr size_t kScratchBytes = GDN2_NOALLOC_SCRATCH_BYTES + 4096;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices];  // per device, null until first use

int noalloc_scratch(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(GDN2_ERR_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices)
        return fail(GDN2_ERR_ARGUMENT, "device ordinal %d outside 0..%d", dev, kMaxDevices - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(GDN2_ERR_LAUNCH, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return GDN2_OK;
}
}  // namespace

static int scalar_backward_impl(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                const gdn2_view *k, const gdn2_view *v, const gdn2_view *beta,
                                const gdn2_view *g, const gdn2_view *valid,
                                const gdn2_view *reset, const void *checkpoint,
                                size_t checkpoint_bytes, const gdn2_view *d_output,
                                const float *d_final_state, const float *d_scores, void *dq,
                                void *dk, void *dv, float *dbeta, float *dg, float *d_initial,
                                void *workspace, size_t workspace_bytes, void *stream);

// The chunk kernels take bf16 q/k/v with unit channel stride and 16-byte
// aligned token rows (every stride a multiple of 8 elements).
static bool rows_aligned(const gdn2_view *v) {
    return v->stride[3] == 1 && ((uintptr_t)v->data & 15) == 0 && v->stride[0] % 8 == 0 &&
           v->stride[1] % 8 == 0 && v->stride[2] % 8 == 0;
}

// The channel-wise ops run the f32 chunk kernels (gdn2_chunk_f32.hip) whatever
// the dtype, the width (d_k, d_v <= 128), the strides and the chunk argument:
// bf16 inputs are read as their exact f32 values and dq, dk, dv written as bf16.
// Calls with bf16 q/k/v of d_k = d_v = 64 and aligned rows keep two terms of
// their contract (include/gdn2.h): alpha >= 0, and aligned d_output rows.
static bool bf16_rows64(const gdn2_shape *shape, const gdn2_view *q, const gdn2_view *k,
                        const gdn2_view *v) {
    return shape->keys == 64 && shape->values == 64 && q->dtype == GDN2_BF16 && rows_aligned(q) &&
           rows_aligned(k) && rows_aligned(v);
}

static int check_rows64_adjoint(bool rows64, const gdn2_view *d_output) {
    if (rows64 && d_output && d_output->data && !rows_aligned(d_output))
        return fail(GDN2_ERR_ARGUMENT,
                    "d_output needs unit channel stride and 16-byte aligned rows on the "
                    "chunked path (bf16, d_k = d_v = 64)");
    return GDN2_OK;
}

static size_t training_checkpoint_bytes(const gdn2_shape *s) {
    return fc_checkpoint_bytes(s->batch, s->time, s->heads, (int)s->keys, (int)s->values, false);
}

static size_t training_workspace_bytes(const gdn2_shape *s) {
    return fc_workspace_bytes(s->batch, s->time, s->heads, (int)s->keys, (int)s->values);
}

// The f32 chunk path's argument block over the token walk's.
static FcArgs fc_args(const SeqArgs &s, const gdn2_view *q, bool rows64, void *checkpoint, void *workspace) {
    FcArgs f{};
    f.s = s;
    f.in_bf16 = q->dtype == GDN2_BF16;
    f.scalar = s.scalar;
    f.nonneg = rows64;
    f.nc = (s.T + FC_C - 1) / FC_C;
    const int es = f.in_bf16 ? 2 : 4;
    f.vec = fc_vec_view(s.q, es, s.K) && fc_vec_view(s.k, es, s.K) && fc_vec_view(s.v, es, s.V) &&
            (!s.dout.data || fc_vec_view(s.dout, es, s.V)) && (int64_t)s.H * std::max(s.K, s.V) < (1 << 24) &&
            (s.scalar || (fc_vec_view(s.alpha, 4, s.K) && fc_vec_view(s.erase, 4, s.K) && fc_vec_view(s.write, 4, s.V)));
    fc_bind(f, checkpoint, workspace);
    return f;
}

extern "C" {

int gdn2_abi_version(void) { return 101; }

const char *gdn2_last_error(void) { return gdn2::last_error(); }

size_t gdn2_training_checkpoint_bytes(const gdn2_shape *shape, int chunk) {
    if (check_shape(shape) || check_chunk(chunk)) return 0;
    return training_checkpoint_bytes(shape);
}

size_t gdn2_training_workspace_bytes(const gdn2_shape *shape, int chunk) {
    if (check_shape(shape) || check_chunk(chunk)) return 0;
    return training_workspace_bytes(shape);
}

int gdn2_training_scan(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                       const gdn2_view *k, const gdn2_view *v, const gdn2_view *alpha,
                       const gdn2_view *erase, const gdn2_view *write, const gdn2_view *valid,
                       const gdn2_view *reset, const gdn2_view *initial, void *output,
                       int32_t output_dtype, float *final_state, float *scores, void *checkpoint,
                       size_t checkpoint_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_channel_inputs(shape, q, k, v, alpha, erase, write, valid, reset));
    GDN2_TRY(check_view(initial, "initial", GDN2_F32, true));
    GDN2_TRY(check_out_dtype(output_dtype));
    if (!output || !final_state || !scores)
        return fail(GDN2_ERR_ARGUMENT, "output, final_state and scores must be non-null");
    if (!checkpoint) return fail(GDN2_ERR_ARGUMENT, "checkpoint is null");
    if ((uintptr_t)checkpoint & 15) return fail(GDN2_ERR_ARGUMENT, "checkpoint must be 16-byte aligned");
    if (checkpoint_bytes < training_checkpoint_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu",
                    training_checkpoint_bytes(shape), checkpoint_bytes);
    SeqArgs a = seq_args(shape, q, k, v, alpha, erase, write, valid, reset);
    a.initial = make_view(initial);
    a.out = output;
    a.out_bf16 = output_dtype == GDN2_BF16;
    a.final_state = final_state;
    a.scores = scores;
    const FcArgs f = fc_args(a, q, bf16_rows64(shape, q, k, v), checkpoint, nullptr);
    const hipEvent_t *ev = stage_events(0, (hipStream_t)stream);
    return launch_status(launch_fc_fwd(f, (hipStream_t)stream, ev), "gdn2_training_scan");
}

int gdn2_training_backward(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                           const gdn2_view *k, const gdn2_view *v, const gdn2_view *alpha,
                           const gdn2_view *erase, const gdn2_view *write,
                           const gdn2_view *valid, const gdn2_view *reset,
                           const void *checkpoint, size_t checkpoint_bytes,
                           const gdn2_view *d_output, const float *d_final_state,
                           const float *d_scores, void *dq, void *dk, void *dv, float *dalpha,
                           float *derase, float *dwrite, float *d_initial, void *workspace,
                           size_t workspace_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_channel_inputs(shape, q, k, v, alpha, erase, write, valid, reset));
    if (d_output) GDN2_TRY(check_view(d_output, "d_output", q->dtype, true));
    if (!checkpoint) return fail(GDN2_ERR_ARGUMENT, "checkpoint is null");
    if ((uintptr_t)checkpoint & 15) return fail(GDN2_ERR_ARGUMENT, "checkpoint must be 16-byte aligned");
    if (checkpoint_bytes < training_checkpoint_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu",
                    training_checkpoint_bytes(shape), checkpoint_bytes);
    if (!workspace) return fail(GDN2_ERR_ARGUMENT, "workspace is null");
    if ((uintptr_t)workspace & 15) return fail(GDN2_ERR_ARGUMENT, "workspace must be 16-byte aligned");
    if (workspace_bytes < training_workspace_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "workspace needs %zu bytes, got %zu",
                    training_workspace_bytes(shape), workspace_bytes);
    const bool rows64 = bf16_rows64(shape, q, k, v);
    GDN2_TRY(check_rows64_adjoint(rows64, d_output));
    SeqArgs a = seq_args(shape, q, k, v, alpha, erase, write, valid, reset);
    if (d_output) a.dout = make_view(d_output);
    a.dfinal = d_final_state;
    a.dscores = d_scores;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.dalpha = dalpha;
    a.derase = derase;
    a.dwrite = dwrite;
    a.dinitial = d_initial;
    const FcArgs f = fc_args(a, q, rows64, const_cast<void *>(checkpoint), workspace);
    const hipEvent_t *ev = stage_events(3, (hipStream_t)stream);
    return launch_status(launch_fc_bwd(f, (hipStream_t)stream, ev), "gdn2_training_backward");
}

size_t gdn2_scan_checkpoint_bytes(const gdn2_shape *shape) {
    if (check_shape(shape)) return 0;
    return training_checkpoint_bytes(shape);
}

size_t gdn2_scan_workspace_bytes(const gdn2_shape *shape) {
    if (check_shape(shape)) return 0;
    return training_workspace_bytes(shape);
}

int gdn2_scan(const gdn2_shape *shape, const gdn2_view *q, const gdn2_view *k, const gdn2_view *v,
              const gdn2_view *alpha, const gdn2_view *erase, const gdn2_view *write,
              const gdn2_view *doc_start, const gdn2_view *doc_end, void *output,
              int32_t output_dtype, void *checkpoint, size_t checkpoint_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_doc_inputs(q, k, v, alpha, erase, write, doc_start, doc_end));
    GDN2_TRY(check_out_dtype(output_dtype));
    if (!output) return fail(GDN2_ERR_ARGUMENT, "output is null");
    if (!checkpoint) return fail(GDN2_ERR_ARGUMENT, "checkpoint is null");
    if ((uintptr_t)checkpoint & 15) return fail(GDN2_ERR_ARGUMENT, "checkpoint must be 16-byte aligned");
    if (checkpoint_bytes < training_checkpoint_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu",
                    training_checkpoint_bytes(shape), checkpoint_bytes);
    SeqArgs a = seq_args(shape, q, k, v, alpha, erase, write, nullptr, nullptr);
    a.doc = 1;
    a.doc_start = make_view(doc_start);
    a.doc_end = make_view(doc_end);
    a.out = output;
    a.out_bf16 = output_dtype == GDN2_BF16;
    const FcArgs f = fc_args(a, q, bf16_rows64(shape, q, k, v), checkpoint, nullptr);
    const hipEvent_t *ev = stage_events(0, (hipStream_t)stream);
    return launch_status(launch_fc_fwd(f, (hipStream_t)stream, ev), "gdn2_scan");
}

int gdn2_backward(const gdn2_shape *shape, const gdn2_view *q, const gdn2_view *k,
                  const gdn2_view *v, const gdn2_view *alpha, const gdn2_view *erase,
                  const gdn2_view *write, const gdn2_view *doc_start, const gdn2_view *doc_end,
                  const void *checkpoint, size_t checkpoint_bytes, const gdn2_view *d_output,
                  void *dq, void *dk, void *dv, float *dalpha, float *derase, float *dwrite,
                  void *workspace, size_t workspace_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_doc_inputs(q, k, v, alpha, erase, write, doc_start, doc_end));
    if (d_output) GDN2_TRY(check_view(d_output, "d_output", q->dtype, true));
    if (!checkpoint) return fail(GDN2_ERR_ARGUMENT, "checkpoint is null");
    if ((uintptr_t)checkpoint & 15) return fail(GDN2_ERR_ARGUMENT, "checkpoint must be 16-byte aligned");
    if (checkpoint_bytes < training_checkpoint_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu",
                    training_checkpoint_bytes(shape), checkpoint_bytes);
    if (!workspace) return fail(GDN2_ERR_ARGUMENT, "workspace is null");
    if ((uintptr_t)workspace & 15) return fail(GDN2_ERR_ARGUMENT, "workspace must be 16-byte aligned");
    if (workspace_bytes < training_workspace_bytes(shape))
        return fail(GDN2_ERR_WORKSPACE, "workspace needs %zu bytes, got %zu",
                    training_workspace_bytes(shape), workspace_bytes);
    const bool rows64 = bf16_rows64(shape, q, k, v);
    GDN2_TRY(check_rows64_adjoint(rows64, d_output));
    SeqArgs a = seq_args(shape, q, k, v, alpha, erase, write, nullptr, nullptr);
    a.doc = 1;
    a.doc_start = make_view(doc_start);
    a.doc_end = make_view(doc_end);
    if (d_output) a.dout = make_view(d_output);
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.dalpha = dalpha;
    a.derase = derase;
    a.dwrite = dwrite;
    const FcArgs f = fc_args(a, q, rows64, const_cast<void *>(checkpoint), workspace);
    const hipEvent_t *ev = stage_events(3, (hipStream_t)stream);
    return launch_status(launch_fc_bwd(f, (hipStream_t)stream, ev), "gdn2_backward");
}

}  // extern "C"

// Kernels of a scalar-gate call.  The chunk-WY MFMA kernels take bf16 q/k/v with d_k =
// d_v = 64 (gdn2_chunk.hip) or 128 (gdn2_chunk_wide.hip), chunk 64, unit channel
// stride and 16-byte aligned token rows.  Everything else runs the f32 scalar-gate
// chunk kernels (gdn2_chunk_fs.hip) from 17 tokens on, and the token walk
// (gdn2_seq.hip) of one workgroup per head up to 16, one block of its checkpoint.
// Forward + backward in us, f32, walked against chunked: 64 heads of 64 x 64, T = 8
// 10 + 17 and 16 + 18, T = 16 13 + 27 and 16 + 18; 2048 heads, T = 8 32 + 158 and
// 67 + 93, T = 16 43 + 262 and 68 + 95; at T = 32 (the walk with a checkpoint of two
// blocks, since removed) 64 heads 21 + 50 and 18 + 19.  The line keeps a short call's
// forward, which serving makes alone, at its fastest; the backward would gain from a
// lower one.  Forward and backward apply the same rule, so the checkpoint format
// always matches.
enum class ScalarPath { chunk, wide, walk, f32 };

static bool use_seq_path(const gdn2_shape *shape) { return shape->time <= FC_C; }

static ScalarPath scalar_path(const gdn2_shape *shape, int chunk, const gdn2_view *q, const gdn2_view *k,
                              const gdn2_view *v) {
    if (q->dtype == GDN2_BF16 && rows_aligned(q) && rows_aligned(k) && rows_aligned(v)) {
        if (chunk_eligible_shape(shape, chunk)) return ScalarPath::chunk;
        if (wide_eligible_shape(shape, chunk)) return ScalarPath::wide;
    }
    return use_seq_path(shape) ? ScalarPath::walk : ScalarPath::f32;
}

// Whether the token walk's forward alone takes less time than the f32 chunk kernels',
// which write 36 KiB a chunk of 64 x 64 that only a backward reads.  Both times in
// microseconds: a start, and a slope that is the serial chain's or, with more heads
// than it takes to fill the chip, the throughput of all of them.  P is the walk's padded
// state and Q the chunks' in units of 64 x 64, F the floats of a chunk's arrays.
// Measured, f32, walk against chunked: 64 heads of 64 x 64, T = 24 16.4 and 18.0, 48
// 24.5 and 19.0, 512 205 and 51; 256 heads, T = 17 15.1 and 28.9, 64 32.8 and 36.7,
// 128 59 and 50; 1024 heads, T = 17 30 and 53, 128 129 and 197, 1024 908 and 1331;
// 256 heads of 128 x 128, T = 64 76 and 88, 512 494 and 595; 1024 heads of 16 x 16,
// T = 32 20 and 23, 256 117 and 69.
static bool walk_is_faster(const gdn2_shape *s) {
    const int K = (int)s->keys, V = (int)s->values, KP = fc_kp(K), VP = fc_kp(V);
    const double heads = (double)(s->batch * s->heads), T = (double)s->time, chunks = (double)((s->time + FC_C - 1) / FC_C);
    const double P = seq_state_floats(K, V) / 4096., Q = KP * VP / 4096.;
    const double F = KP * VP + 3 * FC_C * FC_C + FC_C * (3 * KP + VP) + KP + 8 * FC_C;
    const double full = P < 1. ? 13.7e-3 * std::sqrt(P) : 14.5e-3 * P;  // of 16 tokens of a head
    const double walk = 6. + 1.3 * P + T * std::max(.22 + .175 * P, heads * full / FC_C);
    const double ragged = K % FC_C || V % FC_C ? 4.5 : 0.;  // element reads
    const double chunked = 12. + 2.5 * Q + ragged + chunks * std::max(.25 + .0052 * KP, heads * 2.2e-6 * F);
    return walk < 1.05 * chunked;
}

// The same for a call that no backward follows.
static ScalarPath outputs_path(const gdn2_shape *shape, int chunk, const gdn2_view *q, const gdn2_view *k,
                               const gdn2_view *v) {
    const ScalarPath path = scalar_path(shape, chunk, q, k, v);
    return path == ScalarPath::f32 && walk_is_faster(shape) ? ScalarPath::walk : path;
}

static size_t path_checkpoint_bytes(ScalarPath path, const gdn2_shape *s) {
    const int K = (int)s->keys, V = (int)s->values;
    switch (path) {
        case ScalarPath::chunk: return chunk_checkpoint_bytes(s->batch, s->time, s->heads);
        case ScalarPath::wide: return wide_checkpoint_bytes(s->batch, s->time, s->heads);
        case ScalarPath::walk: return (size_t)seq_checkpoint_floats(s->batch, s->heads, K, V) * 4;
        default: return fc_checkpoint_bytes(s->batch, s->time, s->heads, K, V, true);
    }
}

// The f32 chunk kernels' backward walks windows of chunks that fit whatever
// workspace it is given, so its share is capped: 64 MiB holds 4064 chunks of
// 64 x 64, enough to fill the chip, and keeps every shape whose other needs fit
// the library's fixed scratch within it (gdn_scalar_backward_noalloc).  words: with
// the kernels' words, one per batch and head.
static size_t path_workspace_bytes(ScalarPath path, const gdn2_shape *s, bool words = true) {
    if (path == ScalarPath::chunk) return chunk_workspace_bytes(s->batch, s->time, s->heads);
    if (path == ScalarPath::wide) return wide_workspace_bytes(s->batch, s->time, s->heads);
    if (path == ScalarPath::walk) return seq_workspace_bytes(s);
    const size_t n = words ? fc_word_bytes(s->batch, s->heads) : 0;
    const size_t f = fc_workspace_bytes(s->batch, s->time, s->heads, (int)s->keys, (int)s->values) + n;
    return std::max(std::min(f, (size_t)GDN2_NOALLOC_SCRATCH_BYTES), seq_workspace_bytes(s) + n);
}

// The most that any call of a shape needs, whatever its dtype and alignment.
template <typename F>
static size_t shape_bytes(const gdn2_shape *shape, int chunk, F bytes) {
    size_t n = bytes(use_seq_path(shape) ? ScalarPath::walk : ScalarPath::f32);
    if (chunk_eligible_shape(shape, chunk)) n = std::max(n, bytes(ScalarPath::chunk));
    if (wide_eligible_shape(shape, chunk)) n = std::max(n, bytes(ScalarPath::wide));
    return n;
}

static size_t scalar_workspace_shape(const gdn2_shape *shape, int chunk, bool words) {
    return shape_bytes(shape, chunk, [&](ScalarPath p) { return path_workspace_bytes(p, shape, words); });
}

static int check_call(const gdn2_shape *shape, int chunk, const gdn2_view *q, const gdn2_view *k,
                      const gdn2_view *v) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_view(q, "q", -1, true));
    GDN2_TRY(check_view(k, "k", q->dtype, true));
    return check_view(v, "v", q->dtype, true);
}

extern "C" {

size_t gdn_scalar_checkpoint_bytes(const gdn2_shape *shape, int chunk) {
    if (check_shape(shape) || check_chunk(chunk)) return 0;
    return shape_bytes(shape, chunk, [&](ScalarPath p) { return path_checkpoint_bytes(p, shape); });
}

size_t gdn_scalar_workspace_bytes(const gdn2_shape *shape, int chunk) {
    if (check_shape(shape) || check_chunk(chunk)) return 0;
    return scalar_workspace_shape(shape, chunk, true);
}

size_t gdn_scalar_call_checkpoint_bytes(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                        const gdn2_view *k, const gdn2_view *v) {
    if (check_call(shape, chunk, q, k, v)) return 0;
    return path_checkpoint_bytes(scalar_path(shape, chunk, q, k, v), shape);
}

size_t gdn_scalar_call_workspace_bytes(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                       const gdn2_view *k, const gdn2_view *v) {
    if (check_call(shape, chunk, q, k, v)) return 0;
    return path_workspace_bytes(scalar_path(shape, chunk, q, k, v), shape);
}

}  // extern "C"

static ChunkArgs chunk_args(const gdn2_shape *s, const gdn2_view *q, const gdn2_view *k,
                            const gdn2_view *v, const gdn2_view *beta, const gdn2_view *g,
                            const gdn2_view *valid, const gdn2_view *reset) {
    ChunkArgs a{};
    a.B = (int)s->batch;
    a.T = (int)s->time;
    a.H = (int)s->heads;
    a.nc = (a.T + CHUNK - 1) / CHUNK;
    a.q = (const uint16_t *)q->data;
    a.k = (const uint16_t *)k->data;
    a.v = (const uint16_t *)v->data;
    for (int d = 0; d < 3; ++d) {
        a.qs[d] = q->stride[d];
        a.ks[d] = k->stride[d];
        a.vs[d] = v->stride[d];
    }
    a.beta = make_view(beta);
    a.g = make_view(g);
    a.valid = make_view(valid);
    a.reset = make_view(reset);
    return a;
}

// The token-sequential argument block of the scalar-gate op.
static SeqArgs scalar_args(const gdn2_shape *s, const gdn2_view *q, const gdn2_view *k,
                           const gdn2_view *v, const gdn2_view *beta, const gdn2_view *g,
                           const gdn2_view *valid, const gdn2_view *reset) {
    SeqArgs a = seq_args(s, q, k, v, beta, beta, beta, valid, reset);
    a.scalar = 1;
    a.beta = make_view(beta);
    a.g = make_view(g);
    return a;
}

static int check_scalar_inputs(const gdn2_view *q, const gdn2_view *k, const gdn2_view *v,
                               const gdn2_view *beta, const gdn2_view *g,
                               const gdn2_view *valid, const gdn2_view *reset) {
    GDN2_TRY(check_view(q, "q", -1, false));
    GDN2_TRY(check_view(k, "k", q->dtype, false));
    GDN2_TRY(check_view(v, "v", q->dtype, false));
    GDN2_TRY(check_view(beta, "beta", GDN2_F32, false));
    GDN2_TRY(check_view(g, "g", GDN2_F32, false));
    GDN2_TRY(check_view(valid, "valid", GDN2_F32, false));
    GDN2_TRY(check_view(reset, "reset", GDN2_F32, false));
    return GDN2_OK;
}

// The forward on the kernels of `path`.  keep: with their arrays in `buffer` (named
// `what`); otherwise the walk's outputs alone.
static int scalar_forward(ScalarPath path, bool keep, const char *what, const gdn2_shape *shape,
                          const gdn2_view *q, const gdn2_view *k, const gdn2_view *v, const gdn2_view *beta,
                          const gdn2_view *g, const gdn2_view *valid, const gdn2_view *reset,
                          const gdn2_view *initial, void *output, int32_t output_dtype, float *final_state,
                          float *scores, void *buffer, size_t buffer_bytes, void *stream) {
    GDN2_TRY(check_view(initial, "initial", GDN2_F32, true));
    GDN2_TRY(check_out_dtype(output_dtype));
    if (!output || !final_state || !scores)
        return fail(GDN2_ERR_ARGUMENT, "output, final_state and scores must be non-null");
    if (keep && !buffer) return fail(GDN2_ERR_ARGUMENT, "%s is null", what);
    if (keep && buffer_bytes < path_checkpoint_bytes(path, shape))
        return fail(GDN2_ERR_WORKSPACE, "%s needs %zu bytes, got %zu", what, path_checkpoint_bytes(path, shape),
                    buffer_bytes);
    if (path == ScalarPath::chunk || path == ScalarPath::wide) {
        ChunkArgs c = chunk_args(shape, q, k, v, beta, g, valid, reset);
        c.initial = make_view(initial);
        c.out = output;
        c.out_bf16 = output_dtype == GDN2_BF16;
        c.final_state = final_state;
        c.scores = scores;
        const hipEvent_t *ev = stage_events(0, (hipStream_t)stream);
        if (path == ScalarPath::wide) {
            wide_bind_checkpoint(c, buffer);
            return launch_status(launch_wide_fwd(c, (hipStream_t)stream, ev), "gdn_scalar_scan");
        }
        chunk_bind_checkpoint(c, buffer);
        return launch_status(launch_chunk_fwd(c, (hipStream_t)stream, ev), "gdn_scalar_scan");
    }
    SeqArgs a = scalar_args(shape, q, k, v, beta, g, valid, reset);
    a.initial = make_view(initial);
    a.out = output;
    a.out_bf16 = output_dtype == GDN2_BF16;
    a.final_state = final_state;
    a.scores = scores;
    if (path == ScalarPath::walk) {
        if (keep) seq_bind_checkpoint(a, buffer);
        return launch_status(launch_seq_fwd(a, q->dtype == GDN2_BF16, (hipStream_t)stream),
                             "gdn_scalar_scan");
    }
    const hipEvent_t *ev = stage_events(kScalarF32, (hipStream_t)stream);
    return launch_status(launch_fs_fwd(fc_args(a, q, false, buffer, nullptr), (hipStream_t)stream, ev),
                         "gdn_scalar_scan");
}

extern "C" {

int gdn_scalar_scan(const gdn2_shape *shape, int chunk, const gdn2_view *q, const gdn2_view *k,
                    const gdn2_view *v, const gdn2_view *beta, const gdn2_view *g,
                    const gdn2_view *valid, const gdn2_view *reset, const gdn2_view *initial,
                    void *output, int32_t output_dtype, float *final_state, float *scores,
                    void *checkpoint, size_t checkpoint_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_scalar_inputs(q, k, v, beta, g, valid, reset));
    return scalar_forward(scalar_path(shape, chunk, q, k, v), true, "checkpoint", shape, q, k, v, beta, g, valid,
                          reset, initial, output, output_dtype, final_state, scores, checkpoint,
                          checkpoint_bytes, stream);
}

size_t gdn_scalar_outputs_bytes(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                const gdn2_view *k, const gdn2_view *v) {
    if (check_call(shape, chunk, q, k, v)) return 0;
    const ScalarPath path = outputs_path(shape, chunk, q, k, v);
    return path == ScalarPath::walk ? 0 : path_checkpoint_bytes(path, shape);
}

int gdn_scalar_outputs(const gdn2_shape *shape, int chunk, const gdn2_view *q, const gdn2_view *k,
                       const gdn2_view *v, const gdn2_view *beta, const gdn2_view *g,
                       const gdn2_view *valid, const gdn2_view *reset, const gdn2_view *initial,
                       void *output, int32_t output_dtype, float *final_state, float *scores,
                       void *workspace, size_t workspace_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_scalar_inputs(q, k, v, beta, g, valid, reset));
    const ScalarPath path = outputs_path(shape, chunk, q, k, v);
    return scalar_forward(path, path != ScalarPath::walk, "workspace", shape, q, k, v, beta, g, valid, reset,
                          initial, output, output_dtype, final_state, scores, workspace, workspace_bytes, stream);
}

int gdn_scalar_backward(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                        const gdn2_view *k, const gdn2_view *v, const gdn2_view *beta,
                        const gdn2_view *g, const gdn2_view *valid, const gdn2_view *reset,
                        const void *checkpoint, size_t checkpoint_bytes,
                        const gdn2_view *d_output, const float *d_final_state,
                        const float *d_scores, void *dq, void *dk, void *dv, float *dbeta,
                        float *dg, float *d_initial, void *workspace, size_t workspace_bytes,
                        void *stream) {
    return scalar_backward_impl(shape, chunk, q, k, v, beta, g, valid, reset, checkpoint,
                                checkpoint_bytes, d_output, d_final_state, d_scores, dq, dk, dv,
                                dbeta, dg, d_initial, workspace, workspace_bytes, stream);
}

int gdn_scalar_backward_noalloc(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                const gdn2_view *k, const gdn2_view *v, const gdn2_view *beta,
                                const gdn2_view *g, const gdn2_view *valid,
                                const gdn2_view *reset, const void *checkpoint,
                                size_t checkpoint_bytes, const gdn2_view *d_output,
                                const float *d_final_state, const float *d_scores, void *dq,
                                void *dk, void *dv, float *dbeta, float *dg, float *d_initial,
                                void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    const size_t need = scalar_workspace_shape(shape, chunk, false);
    if (need > GDN2_NOALLOC_SCRATCH_BYTES)
        return fail(GDN2_ERR_WORKSPACE,
                    "gdn_scalar_backward_noalloc: this shape needs %zu bytes of scratch, above "
                    "the library's fixed %zu-byte device scratch; call gdn_scalar_backward "
                    "with a workspace instead",
                    need, (size_t)GDN2_NOALLOC_SCRATCH_BYTES);
    void *ws = nullptr;
    GDN2_TRY(noalloc_scratch(&ws));
    return scalar_backward_impl(shape, chunk, q, k, v, beta, g, valid, reset, checkpoint,
                                checkpoint_bytes, d_output, d_final_state, d_scores, dq, dk, dv,
                                dbeta, dg, d_initial, ws, kScratchBytes, stream);
}

}  // extern "C"

static int scalar_backward_impl(const gdn2_shape *shape, int chunk, const gdn2_view *q,
                                const gdn2_view *k, const gdn2_view *v, const gdn2_view *beta,
                                const gdn2_view *g, const gdn2_view *valid,
                                const gdn2_view *reset, const void *checkpoint,
                                size_t checkpoint_bytes, const gdn2_view *d_output,
                                const float *d_final_state, const float *d_scores, void *dq,
                                void *dk, void *dv, float *dbeta, float *dg, float *d_initial,
                                void *workspace, size_t workspace_bytes, void *stream) {
    GDN2_TRY(check_shape(shape));
    GDN2_TRY(check_chunk(chunk));
    GDN2_TRY(check_scalar_inputs(q, k, v, beta, g, valid, reset));
    if (d_output) GDN2_TRY(check_view(d_output, "d_output", q->dtype, true));
    if (!checkpoint) return fail(GDN2_ERR_ARGUMENT, "checkpoint is null");
    const ScalarPath path = scalar_path(shape, chunk, q, k, v);
    if (checkpoint_bytes < path_checkpoint_bytes(path, shape))
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu",
                    path_checkpoint_bytes(path, shape), checkpoint_bytes);
    if (!workspace) return fail(GDN2_ERR_ARGUMENT, "workspace is null");
    if (workspace_bytes < path_workspace_bytes(path, shape))
        return fail(GDN2_ERR_WORKSPACE, "workspace needs %zu bytes, got %zu",
                    path_workspace_bytes(path, shape), workspace_bytes);
    if (path == ScalarPath::chunk || path == ScalarPath::wide) {
        if (d_output && d_output->data && !rows_aligned(d_output))
            return fail(GDN2_ERR_ARGUMENT,
                        "d_output needs unit channel stride and 16-byte aligned rows on the "
                        "chunked path (chunk 64, bf16, d_k = d_v = 64 or 128)");
        ChunkArgs c = chunk_args(shape, q, k, v, beta, g, valid, reset);
        const bool wide = path == ScalarPath::wide;
        if (wide) {
            wide_bind_checkpoint(c, const_cast<void *>(checkpoint));
            wide_bind_workspace(c, workspace);
        } else {
            chunk_bind_checkpoint(c, const_cast<void *>(checkpoint));
            chunk_bind_workspace(c, workspace);
        }
        if (d_output && d_output->data) {
            c.dout = (const uint16_t *)d_output->data;
            for (int d = 0; d < 3; ++d) c.ds[d] = d_output->stride[d];
        }
        c.dfinal = d_final_state;
        c.dscores = d_scores;
        c.dq = dq;
        c.dk = dk;
        c.dv = dv;
        c.dbeta = dbeta;
        c.dg = dg;
        c.dinitial = d_initial;
        const hipEvent_t *ev = stage_events(3, (hipStream_t)stream);
        return launch_status(wide ? launch_wide_bwd(c, (hipStream_t)stream, ev)
                                  : launch_chunk_bwd(c, (hipStream_t)stream, ev),
                             "gdn_scalar_backward");
    }
    SeqArgs a = scalar_args(shape, q, k, v, beta, g, valid, reset);
    if (d_output) a.dout = make_view(d_output);
    a.dfinal = d_final_state;
    a.dscores = d_scores;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.dbeta = dbeta;
    a.dg = dg;
    a.dinitial = d_initial;
    if (path == ScalarPath::walk) {
        seq_bind_checkpoint(a, checkpoint);
        a.replay = (float *)workspace;
        return launch_status(launch_seq_bwd(a, q->dtype == GDN2_BF16, (hipStream_t)stream),
                             "gdn_scalar_backward");
    }
    const hipEvent_t *ev = stage_events(kScalarF32 + 3, (hipStream_t)stream);
    return launch_status(launch_fs_bwd(fc_args(a, q, false, const_cast<void *>(checkpoint), workspace), workspace_bytes,
                                       (hipStream_t)stream, ev),
                         "gdn_scalar_backward");
}

extern "C" {

int gdn2_stage_timing(int enable) {
    if (enable && !g_stage_ready) {
        for (int i = 0; i < 2 * kStages; ++i) {
            const hipError_t e = hipEventCreate(&g_stage_ev[i]);
            if (e != hipSuccess) {
                for (int j = 0; j < i; ++j) (void)hipEventDestroy(g_stage_ev[j]);
                return fail(GDN2_ERR_LAUNCH, "gdn2_stage_timing: hipEventCreate: %s",
                            hipGetErrorString(e));
            }
        }
        g_stage_ready = true;
    }
    for (int i = 0; i < kStages; ++i) g_stage_ran[i] = false;
    g_stage_on = enable != 0;
    return ok();
}

int gdn2_stage_count(void) { return kStages; }

const char *gdn2_stage_name(int stage) {
    return stage >= 0 && stage < kStages ? kStageNames[stage] : nullptr;
}

float gdn2_stage_ms(int stage) {
    if (stage < 0 || stage >= kStages || !g_stage_ready || !g_stage_ran[stage]) return -1.f;
    float ms = -1.f;
    if (hipEventElapsedTime(&ms, g_stage_ev[2 * stage], g_stage_ev[2 * stage + 1]) != hipSuccess)
        return -1.f;
    return ms;
}

int gdn2_decode_step(const gdn2_shape *shape, const gdn2_view *q, const gdn2_view *k,
                     const gdn2_view *v, const gdn2_view *alpha, const gdn2_view *erase,
                     const gdn2_view *write, const gdn2_view *valid, const gdn2_view *reset,
                     float *state, void *output, int32_t output_dtype, float *scores,
                     void *stream) {
    GDN2_TRY(check_shape(shape));
    if (shape->time != 1) return fail(GDN2_ERR_SHAPE, "decode step needs time == 1");
    GDN2_TRY(check_view(q, "q", -1, false));
    GDN2_TRY(check_view(k, "k", q->dtype, false));
    GDN2_TRY(check_view(v, "v", q->dtype, false));
    GDN2_TRY(check_view(alpha, "alpha", GDN2_F32, false));
    GDN2_TRY(check_view(erase, "erase", GDN2_F32, false));
    GDN2_TRY(check_view(write, "write", GDN2_F32, false));
    if (valid) GDN2_TRY(check_view(valid, "valid", GDN2_F32, true));
    if (reset) GDN2_TRY(check_view(reset, "reset", GDN2_F32, true));
    GDN2_TRY(check_out_dtype(output_dtype));
    if (!state || !output || !scores)
        return fail(GDN2_ERR_ARGUMENT, "state, output and scores must be non-null");
    SeqArgs a = seq_args(shape, q, k, v, alpha, erase, write, valid, reset);
    if (!valid) a.valid.data = nullptr;
    if (!reset) a.reset.data = nullptr;
    const int64_t K = shape->keys, V = shape->values;
    gdn2_view st{state, GDN2_F32, 0, {shape->heads * K * V, K * V, V, 1}};
    a.initial = make_view(&st);
    a.final_state = state;  // each workgroup reads its slice before writing it
    a.out = output;
    a.out_bf16 = output_dtype == GDN2_BF16;
    a.scores = scores;
    return launch_status(launch_seq_decode(a, q->dtype == GDN2_BF16, (hipStream_t)stream),
                         "gdn2_decode_step");
}

}  // extern "C"
