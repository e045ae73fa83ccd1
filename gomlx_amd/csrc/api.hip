// C ABI of libgomlx_hipq.so: argument validation, device selection, dispatch to the kernel
// families, HIP-graph recording and per-kernel timing.  See include/gomlx_hipq.h for the
// contract of every entry point and the reference interface it replaces.
#include "common.hpp"
#include "workspace.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <cstdlib>
#include <map>
#include <mutex>
#include <new>

namespace gq {

namespace {
thread_local char g_error[512] = "";
std::atomic<int> g_device{-1};
std::atomic<int> g_cu_count{256};
std::mutex g_init_mutex;
}  // namespace

int fail(int status, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(g_error, sizeof g_error, fmt, ap);
    va_end(ap);
    return status;
}

int hip_fail(hipError_t e, const char *what) {
    if (e == hipErrorOutOfMemory) return fail(GQ_ERR_OOM, "%s: %s", what, hipGetErrorString(e));
    if (e == hipErrorNoDevice || e == hipErrorInvalidDevice)
        return fail(GQ_ERR_NO_DEVICE, "%s: %s", what, hipGetErrorString(e));
    return fail(GQ_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

int use_device() {
    const int dev = g_device.load(std::memory_order_acquire);
    if (dev < 0) return fail(GQ_ERR_NO_DEVICE, "gq_init() has not been called (or failed)");
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || cur != dev) GQ_HIP(hipSetDevice(dev));
    return GQ_OK;
}

int device_cu_count() { return g_cu_count.load(std::memory_order_relaxed); }

// ---- scratch memory ------------------------------------------------------------------------------
// Per-stream buffers come from the pool of workspace.hpp (sequence lock per stream, buffers pinned by
// recorded graphs, released with their stream).  A call through gq_qdense_f32_static is served from
// the fixed device array below instead and never allocates.
namespace {

constexpr size_t kStaticScratchBytes = (size_t)16 << 20;
constexpr int kMaxDevices = 64;
// Scratch of the entry point that allocates nothing.  Host code never uses this name as an address:
// g_scratch_ptr[device] holds the array's device address, taken once in gq_init().
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
void *g_scratch_ptr[kMaxDevices] = {};

int ws_alloc(void **p, size_t bytes) {
    GQ_HIP(hipMalloc(p, bytes));
    // the flag words at the head of a buffer start at zero (allocation never happens inside a recording)
    hipError_t e = hipMemsetAsync(*p, 0, bytes < kWsSyncBytes ? bytes : kWsSyncBytes, nullptr);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) { (void)hipFree(*p); *p = nullptr; return hip_fail(e, "hipMemsetAsync(workspace flags)"); }
    return GQ_OK;
}
void ws_release(void *p) { (void)hipFree(p); }
void ws_sync(const void *s) { (void)hipStreamSynchronize((hipStream_t)const_cast<void *>(s)); }
bool ws_capturing(const void *s) {
    if (!s) return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing((hipStream_t)const_cast<void *>(s), &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}
WorkspacePool &pool() {
    static WorkspacePool *p = new WorkspacePool(WsHooks{ws_alloc, ws_release, ws_sync, ws_capturing});  // never destroyed: outlives every caller
    return *p;
}

// One per ABI call that may reach a path with scratch memory; nested calls share the outermost one.
struct RecordedGraph {  // what gq_graph_end hands out
    hipGraphExec_t exec;
    hipStream_t stream;               // the stream it was recorded on, the only one it replays on
    std::vector<WsBlockRef> blocks;   // workspaces its launches point at
};

struct CallScope;
thread_local CallScope *t_scope = nullptr;
struct CallScope {
    SeqLock lock;
    unsigned char *static_ptr = nullptr;  // set: requests are served from the static array
    bool outer;
    CallScope() : outer(t_scope == nullptr) { if (outer) t_scope = this; }
    ~CallScope() { if (outer) t_scope = nullptr; }
};

}  // namespace

int stream_workspace(hipStream_t s, size_t bytes, void **out, int slot, uint32_t **sync) {
    CallScope *sc = t_scope;
    if (!sc) return fail(GQ_ERR_INVALID, "internal: scratch memory requested outside an entry point");
    void *base = nullptr;
    if (sc->static_ptr) {
        // (the static array is zero when the library is loaded: its first kWsSyncBytes are the flag words)
        if (slot != 0 || bytes > kStaticScratchBytes - kWsSyncBytes)
            return fail(GQ_ERR_INVALID, "gq_qdense_f32_static: this call needs %zu bytes of scratch memory, the static buffer holds %zu; use gq_qdense_f32",
                        bytes, kStaticScratchBytes - kWsSyncBytes);
        base = sc->static_ptr;
    } else {
        if (slot < 0 || slot >= kWsSlots) return fail(GQ_ERR_INVALID, "internal: workspace slot %d", slot);
        if (!sc->lock.held()) sc->lock.lock(pool().stream(s));
        const int rc = pool().acquire(*sc->lock.held(), s, slot, bytes + kWsSyncBytes, &base);
        if (rc == kWsWouldAllocateInRecording)
            return fail(GQ_ERR_INVALID, "qdense: the %zu-byte workspace of this stream must exist before a graph is recorded; run the "
                        "same call once outside the recording first", bytes);
        if (rc) return rc;
    }
    *out = static_cast<unsigned char *>(base) + kWsSyncBytes;
    if (sync) *sync = static_cast<uint32_t *>(base);
    return GQ_OK;
}

namespace {
bool serves_static_scratch() { return t_scope && t_scope->static_ptr; }  // (inside gq_qdense_f32_static)
}  // namespace

ProfileState &profile_state() {
    thread_local ProfileState ps;
    return ps;
}

namespace {

struct TypeInfo { int bpb, vpb; };

bool type_info(int type, TypeInfo &ti) {
    switch (type) {
    case GQ_Q4_0: ti = {18, 32}; return true;
    case GQ_Q8_0: ti = {34, 32}; return true;
    case GQ_Q4_K: ti = {144, 256}; return true;
    case GQ_Q6_K: ti = {210, 256}; return true;
    case GQ_IQ4_NL: ti = {18, 32}; return true;
    default: return false;
    }
}

constexpr int64_t kGemvMaxRows = 16;  // above this many activation rows the tiled MFMA kernels win
// Batched submissions merge problems of up to this many activation rows each into one K-sliced GEMV launch (q/k/v
// of a decoder layer behind one normalisation, 2 / 4 / 8 rows: the layer's four calls take 50.6 / 83.1 / 86.8 us
// merged against 59.1 / 97.6 / 97.7 us as three calls).
// Only matrices under 24 MB are merged at several rows: over larger ones a single call serves several rows per pass.
int64_t batch_rows_max() { return 8; }

bool aligned_to(const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// Run-time argument checks shared by the dense entry points.
int check_dense_args(const char *fn, int type, const void *x, int64_t M, int64_t K, const void *W, int64_t N,
                     const float *bias, int act, const float *y, size_t x_align) {
    TypeInfo ti;
    if (!type_info(type, ti)) return fail(GQ_ERR_NOT_IMPLEMENTED, "%s: ggml type %d is not implemented", fn, type);
    if (M < 0 || N < 0) return fail(GQ_ERR_INVALID, "%s: negative dimension (M=%lld, N=%lld)", fn, (long long)M, (long long)N);
    if (K <= 0 || K % ti.vpb != 0)
        return fail(GQ_ERR_INVALID, "%s: K=%lld is not a positive multiple of the block size %d", fn, (long long)K, ti.vpb);
    if (act < GQ_ACT_NONE || act > GQ_ACT_TANH) return fail(GQ_ERR_INVALID, "%s: unknown activation %d", fn, act);
    if (M == 0 || N == 0) return GQ_OK;
    if (!x || !W || !y) return fail(GQ_ERR_INVALID, "%s: null device pointer", fn);
    if (!aligned_to(x, x_align)) return fail(GQ_ERR_INVALID, "%s: x must be %zu-byte aligned", fn, x_align);
    if (!aligned_to(W, 16)) return fail(GQ_ERR_INVALID, "%s: weights must be 16-byte aligned", fn);
    if (!aligned_to(y, 4) || (bias && !aligned_to(bias, 4))) return fail(GQ_ERR_INVALID, "%s: y / bias must be 4-byte aligned", fn);
    return GQ_OK;
}

// Batch sizes served by the split-K small-batch kernels: measured crossovers against the GEMV passes
// below and the two-pass GEMM above.  GEMV passes cost time in proportion to the weight bytes (small
// matrices: a pass per row, sharing W through the caches; large ones: a pass per four rows, two for
// Q6_K), the split-K kernels a fixed part plus less per byte.
// Measured (us per call in a replayed graph of dependent calls; rows 4 5 6 7 8 9 10; GEMV passes | split-K, flat over these rows):
//   Q8_0   4096x4096 (18 MB)  12.5 14.3 16.2 17.9 19.9 21.9 23.9 | 14.4   4096x14336 (62 MB) 17.3 27.2 28.0 30.2 27.7 37.9 38.9 | 29.3
//          4096x1024 (4 MB)    4.8  5.6  6.1  6.4  6.6  8.1  8.2 | 12.9   14336x4096         23.0 32.5 34.0 38.7 36.7 47.3 49.6 | 30.1
//   Q4_0   4096x4096 (9 MB)    9.6 10.7 12.0 13.5 15.1 16.5 18.0 | 13.0   4096x14336 (33 MB) 14.9 20.7 22.0 27.3 25.8 32.6 34.0 | 23.7
//          4096x1024 (2 MB)    4.2  4.8  4.8  5.5  5.6  6.2  6.3 | 12.1   14336x4096         19.4 25.2 28.1 34.8 33.0 40.1 43.2 | 24.7
//   Q4_K   4096x4096          11.1 12.6 14.6 16.6 18.6 20.5 22.5 | 13.1   4096x14336         15.8 22.3 24.1 29.1 27.5 34.9 36.8 | 19.3
//          4096x1024           4.4  5.4  6.2  6.4  6.5  7.4  8.0 | 12.3   14336x4096         20.4 26.9 29.8 36.7 35.0 42.7 46.0 | 19.6
//   Q6_K   4096x4096 (14 MB)  13.5 15.3 17.6 19.9 22.3 24.6 27.0 | 17.8   4096x14336 (48 MB) 25.6 34.6 34.6 44.2 44.3 54.0 54.2 | 33.0
//          4096x1024 (3 MB)    5.1  6.1  6.2  7.2  7.3  8.4  8.5 | 16.4   14336x4096         28.6 37.1 37.3 46.9 48.0 57.6 58.8 | 34.0
//   IQ4_NL 4096x4096          11.8 12.9 15.0 16.9 18.9 20.9 22.8 | 13.7   4096x14336         17.0 24.0 26.7 31.1 29.4 37.7 40.4 | 26.3
//          4096x1024           4.8  5.7  5.7  6.6  6.7  7.6  7.7 | 12.8   14336x4096         20.9 28.6 31.1 37.7 35.9 45.0 47.8 | 27.2
// These are the three launches of mmq.hip.  Rows of up to 4096 values meet this line only where takes_mmv() has declined them; longer ones take,
// from it to 16 rows, mmv.hip's two launches (split_k_ahead()), which the line was not moved for.  They are ahead of the GEMV below it on the
// larger matrices - rows 4 and 5 on the GEMV | 6 on the two launches: 14336x4096 Q8_0 19.9 31.2 | 20.3, Q4_0 18.3 25.4 | 18.5, Q6_K 25.8 21.3 | 21.3 (at 5 already
// the two launches), IQ4_NL 19.7 28.6 | 20.5; 8192x8192 18.6 30.4 | 20.9, 16.6 23.6 | 18.2, 28.5 21.0 | 20.9, 18.6 28.3 | 20.3.
// The split-K route is three dependent launches with a floor of about 12 us: matrices of a few megabytes (the k / v
// projections of a grouped-query layer) stay on GEMV passes for every batch the GEMV takes.
// (The Q6_K kernel pays 16 scale groups per super-block: twice the time of the others per byte.)
constexpr int64_t kTinyWeightBytes = (int64_t)6 << 20;
int64_t split_k_from(int type, int64_t weight_bytes) {
    if (weight_bytes < kTinyWeightBytes) return kGemvMaxRows + 1;
    const bool large = weight_bytes >= kLargeWeightBytes;
    switch (type) {
    case GQ_Q8_0: return 6;
    case GQ_Q4_0: return large ? 6 : 7;
    case GQ_Q4_K: return large ? 5 : 6;
    case GQ_Q6_K: return large ? 5 : 6;
    case GQ_IQ4_NL: return 6;
    default: return 8;
    }
}
int64_t weight_bytes_of(int type, int64_t K, int64_t N) { return (int64_t)gq_row_bytes(type, K) * N; }
// Last batch size of the split-K kernels before the two-pass GEMM takes over.  The split-K route streams W once per up to four tiles of
// 32 batch rows (Q6_K: per tile); the two passes pay the 16-bit image (written once and read once, in proportion to N K) and a GEMM that
// splits K itself where its tiles leave CUs idle.
// Measured (GOMLX_HIPQ_SPLIT_K_TO=100000 and =16; us per call on rotating weights, fp32 activations; rows 32 64 96 128 160 192 256;
// split-K | two passes - from 2^25 values on, but for Q6_K, in the one-GEMM form - at the same rows):
//   Q8_0   4096x4096  16 22 26 29 35 36 45 | 23 24 27 25 27 28 30
//          4096x14336 30 36 43 49 70 76 91 | 36 38 41 44 49 52 63    14336x4096 30 37 43 51 71 77 93 | 47 49 52 54 57 58 62
//   Q4_0   4096x4096  14 19 25 27 33 34 42 | 26 25 26 27 27 28 30
//          4096x14336 25 32 38 44 62 68 79 | 31 33 37 39 45 47 58    14336x4096 25 33 40 45 63 69 81 | 41 43 45 46 49 50 55
//   Q4_K   4096x4096  14 17 21 28 37 39 45 | 25 27 27 28 29 29 31
//          4096x14336 20 26 32 37 52 58 69 | 29 31 34 37 43 46 54    14336x4096 19 28 34 38 54 60 73 | 37 38 42 43 46 49 52
//   Q6_K   4096x4096  18 21 30 32 41 42 52 | 25 26 27 28 29 29 32
//          4096x14336 32 56 78 92 114 138 171 | 55 56 58 61 75 72 71    14336x4096 32 55 78 94 117 138 171 | 65 65 66 66 79 77 81
//   IQ4_NL 4096x4096  16 21 28 29 38 39 47 | 25 26 27 27 27 28 31
//          4096x14336 28 34 41 47 66 72 86 | 34 37 40 41 47 50 60    14336x4096 28 35 43 49 69 74 86 | 61 61 63 52 54 55 58
//          (Q4_K at 320 rows: 4096x14336 91 | 64, 14336x4096 95 | 63)
// The split-K kernels contract exact weights, the two passes weights rounded to 16 bits (a relative error of 5.6e-4 for Q4_K where the split-K kernels
// have 2.6e-4).  So the hand-over lies beyond the point where both are level: by up to 64 rows over matrices that the image serves, and where it lay
// in front of the one-GEMM form over those that this serves, at up to 1.5 times its time: bits that a batch has are not given up for time.
// GOMLX_HIPQ_SPLIT_K_TO=rows overrides the table (tuning runs and tests; read at every call that the split-K kernels could take).
int64_t split_k_to_env() {
    const char *e = std::getenv("GOMLX_HIPQ_SPLIT_K_TO");
    return e ? (int64_t)std::atoll(e) : (int64_t)-1;
}
int64_t split_k_to(int type, int64_t K, int64_t N) {
    if (split_k_to_env() >= 0) return split_k_to_env();
    const bool large = weight_bytes_of(type, K, N) >= kLargeWeightBytes, long_k = K > N;
    switch (type) {
    case GQ_Q8_0: return !large ? 128 : long_k ? 192 : 128;
    case GQ_Q4_0: return !large ? 128 : 192;
    case GQ_Q4_K: return !large ? 128 : long_k ? 320 : 256;
    case GQ_Q6_K: return !large ? 96 : 64;
    case GQ_IQ4_NL: return !large ? 128 : 192;
    default: return 96;
    }
}

// The same point for a gated pair act(x.Wgate) * (x.Wup): both matrices are contracted against one activation image by the
// split-K kernels, or dequantised into one interleaved image for ONE GEMM by the two passes.  Measured (the same way, SiLU behind a
// normalisation; rows 32 64 96 128 160 192 256; split-K | two passes or one GEMM):
//   Q8_0   4096x4096  25 29 33 38 52 56 68 | 44 44 45 46 47 47 47
//          4096x14336 56 63 76 86 124 132 155 | 89 89 92 93 92 93 95
//   Q4_0   4096x4096  21 26 30 34 47 50 61 | 42 42 42 43 43 43 44
//          4096x14336 44 54 67 77 105 114 132 | 72 72 75 76 79 79 80
//   Q4_K   4096x4096  18 23 27 31 43 47 57 | 43 43 44 45 45 46 46
//          4096x14336 30 39 49 58 83 92 110 | 62 63 66 69 76 78 79
//   Q6_K   4096x4096  31 36 46 55 65 73 90 | 46 46 46 47 47 47 48
//          4096x14336 64 96 137 170 211 243 316 | 118 118 123 127 138 138 145
//   IQ4_NL 4096x4096  22 27 32 35 49 52 63 | 42 42 43 43 44 44 44
//          4096x14336 49 60 72 82 114 123 141 | 82 83 85 85 90 88 90
//          (Q4_K at 320 and 384 rows: 143 161 | 99 98; where the line lies and why: as above, here at up to 1.6 times the one GEMM's time)
// (The pair composed of two dense calls and a multiplication is never ahead of the one GEMM: 127 - 159 against 118 - 143 us
// for Q4_K 4096 -> 2 x 14336 at 64 - 256 rows.)
int64_t gated_split_k_to(int type, int64_t K, int64_t N) {
    if (split_k_to_env() >= 0) return split_k_to_env();
    const bool large = weight_bytes_of(type, K, N) >= kLargeWeightBytes, long_k = K > N;
    if (large && long_k) return split_k_to(type, K, N);
    switch (type) {
    case GQ_Q8_0: return large ? 192 : 128;
    case GQ_Q4_0: return large ? 192 : 128;
    case GQ_Q4_K: return large ? 384 : 160;
    case GQ_Q6_K: return large ? 64 : 96;
    case GQ_IQ4_NL: return large ? 192 : 128;
    default: return 96;
    }
}

// Whether an output's rows are whole float4 in memory, as the split-K kernels' reduction and the GEMMs' sums of K slices store them best: N, the
// bias and y (of a gated pair: the gate's bias).  A residual or an up bias off 16 bytes is read element by element and moves no line: the exact
// weights of the split-K kernels do not depend on it.
template <class... P> bool whole_rows(int64_t N, P... outputs) { return N % 4 == 0 && ((reinterpret_cast<uintptr_t>(outputs) | ...) & 15) == 0; }

// The hand-over of a call whose rows are not (`whole` false).  Its two passes cannot slice K, which is what makes them wait on long rows, and on
// short ones they were ahead of the lines above, which lie beyond the point where both are level; here the line is that point.  Measured
// (time of the two passes over that of the split-K kernels; N 601 1501 3001 6001 12001):
//   K 1024, 32 rows: Q4_K .94 .99 1.11 1.31 1.35, Q8_0 .88 .92 1.03 1.20 1.18, Q6_K .74 .77 .88 1.03 1.13; 64 rows: Q4_K .75 .78 .86 1.01 1.04
//   K 2048, 64 rows: Q4_K 1.04 1.13 1.26 1.30 1.20 (96: .92 .98 1.06 1.05 1.03, gated 1.02 1.12 1.12 1.01 1.33), Q8_0 1.23 1.28 1.42 1.09 .90, Q4_0 1.27 1.34 1.47 1.30 1.12
//     (96: 1.31 1.32 1.25 1.09 .80; gated 64: 1.32 1.43 1.36 1.01 1.10), IQ4_NL gated 64: 1.26 1.37 1.28 .96 1.07, Q6_K 32: 1.02 1.14 1.29 1.37 .97 (gated 1.06 1.24 1.28 .93 1.18; 33: .99 1.13 1.22 .94 .87)
//   K 4096, 128 rows: Q4_K 1.27 1.29 1.25 1.22 1.32, Q8_0 1.82 1.40 1.12 1.06 .89 (96: 1.02 at 12001), Q4_0 1.87 1.59 1.25 1.07 .93, IQ4_NL 1.79 1.49 1.15 1.03 .90, gated .98 to 1.72;
//     192: Q4_0 .72, IQ4_NL .68 at 12001; Q6_K 64: 1.60 1.71 1.16 1.05 1.07 (96: .80 at 6001)
//   K 8192, 128 rows: Q8_0 2.07 1.61 1.48 1.39 1.60, Q4_0 2.36 1.81 1.53 1.45 1.28; 192: .91 to 1.03
// and over small matrices (the range over five widths of 0.25 to 2.2 million values):
//   K 1024, 17 rows: Q4_K 1.02 to 1.12, the others .76 to 1.11; 32: .71 to 1.01
//   K 2048, 64 and 128 rows: Q4_K 1.03 to 1.07, .83 to .85 (gated 96: 1.00 to 1.07), Q6_K .98 to 1.02 at both (17: 1.03 to 1.09), Q8_0 Q4_0 IQ4_NL 1.18 to 1.29, 1.15 to 1.33
//     (gated 96: 1.23 to 1.33, 128: 1.00 to 1.37)
//   K 4096, 64 and 128 rows: Q4_K 1.59 to 1.67, 1.25 to 1.39, Q6_K 1.50 to 1.54, 1.53 to 1.62, the others 1.80 to 1.97, 1.76 to 2.07; gated 1.51 to 2.07, 1.20 to 2.08
//   K 8192, 128 rows: 1.94 to 3.17
int64_t by_element_to(int type, int64_t K, int64_t N, bool gated) {
    const int64_t one = weight_bytes_of(type, K, N);
    const bool large = one >= kLargeWeightBytes, small = K * N < ((int64_t)9 << 18);  // (2.4 million values: between the small matrices above and 2048x1501)
    if (K < 2048) return type == GQ_Q6_K || one < ((int64_t)3 << 20) ? kGemvMaxRows : 32;
    if (K < 4096) {
        if (type == GQ_Q4_K) return gated ? 96 : 64;
        if (type == GQ_Q6_K) return gated ? kGemvMaxRows : 32;
        if (small) return gated ? 96 : 128;
        return gated ? 48 : type == GQ_Q8_0 && large ? 32 : 64;
    }
    if (type == GQ_Q4_K) return INT64_MAX;
    if (K < 8192) return small ? 128 : type == GQ_Q6_K ? 64 : !gated && large ? 96 : 128;
    return 128;
}
// The first row count of such a call on the split-K kernels: up to 16 rows it keeps the GEMV and the few-row kernel, which hold activations in
// more bits (16-bit fixed point per 32 values, two fp16) than the split-K kernels' one fp16: errors of 2e-5 and 1e-4 of the largest output.  (Those
// take half the time there: Q4_K 14336 -> 4097 at 12 rows 25 against 52 us.) Beyond, the other routes are GEMMs on 16-bit operands, of weights as well.
int64_t take_over(int64_t from, bool whole) { return whole ? from : std::max(from, kGemvMaxRows + 1); }
int64_t hand_over(int type, int64_t K, int64_t N, bool gated, bool whole) {
    const int64_t to = gated ? gated_split_k_to(type, K, N) : split_k_to(type, K, N);
    return whole || split_k_to_env() >= 0 ? to : std::min(to, by_element_to(type, K, N, gated));
}

// Whether y [M, N] lies over any part of x [M, K].  The split-K kernels and the two passes have read x before the launch that writes y; a kernel
// whose workgroups read x while others write y must not have such a call.
bool y_over_x(const void *x, bool x_is_bf16, const float *y, int64_t M, int64_t K, int64_t N) {
    const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(y);
    return ya < xa + (uintptr_t)(M * K) * (x_is_bf16 ? 2 : 4) && xa < ya + (uintptr_t)(M * N) * sizeof(float);
}

// Rows x MB up to which the GEMV stays ahead of mmv.hip over 9 to 24 MB (0: nowhere).  Three things decide besides the product.  From 2^24
// values on the GEMV's workgroups have three row-steps and more, below one or two, and a row's conversion costs more than its share of
// the weights; rows of 2049 to 3584 values leave some of a CU's wavefront slots empty in it; and extras cost it registers.  Measured (us on rotating
// weights, rows 3 4 5; GEMV | mmv.hip):
//   Q8_0  1536x6144   6.1  7.1  8.1 |  8.0  8.2  9.1   2048x6144  7.2  8.4  9.5 |  8.7  8.7  9.5   2048x8192   8.8 10.4 12.0 |  9.5  9.6 10.4
//         3072x3072   6.9  8.5  9.6 |  8.0  8.2  9.0   4096x3072  8.8  9.5 11.2 |  8.6  8.6  9.5   4096x4096  10.0 12.1 14.5 |  9.4  9.6 10.3
//         three 4096x1024 of one input 7.1 7.7 8.8 | 8.2 8.2 9.2;  gated 4096x1536 8.9 9.5 14.2 | 10.0 10.0 11.0;  behind a norm 1536x6144 7.8 12.9 13.0 | 8.7 8.7 9.8
//   Q6_K  2048x6144   8.3 10.1 11.7 |  9.2  9.3 10.3   4096x3072  8.9 10.4 12.7 |  9.1  9.2 10.3   1024x16384 10.4 12.6 15.0 |  9.7  9.8 10.6
//   Q4_0  1536x12288  6.5  7.8  8.8 |  8.6  8.5 10.1   4096x6144  7.9  9.3 10.9 | 10.0 10.1 10.8   4096x4096 (2^24 values) 7.6 9.2 11.0 | 8.2 8.3 9.0
//         gated 1536x6144 7.5 8.5 10.2 | 9.9 9.9 11.0
//   Q4_K  1536x12288  7.6  9.2 10.7 |  8.8  8.7 10.2   4096x6144  9.1 10.9 12.9 |  9.5  9.6 11.1   4096x4096   9.2 11.2 13.3 |  8.2  8.2  9.8
//   IQ4_NL gated 1536x6144 10.1 11.8 14.6 | 11.1 11.1 12.1
// (K from 1024: narrower matrices of 9 MB have 12000 rows and more; Q8_0 768x12544 at 3 rows takes 8.5 us where the GEMV took 7.0.)
int64_t gemv_reach(int type, int64_t K, int64_t values, int matrices, bool extras, bool set) {
    if (K < 1024) return 0;
    const bool shallow = values <= (int64_t)1 << 24, is_short = K <= 2048, gaps = !is_short && K <= 3584;
    if (matrices == 2) {
        if (gaps || type == GQ_Q6_K) return 0;
        if (type == GQ_Q8_0) return 58;
        if (is_short && shallow) return 0;
        return type != GQ_Q4_0 ? 32 : is_short ? 55 : 37;
    }
    if (extras) return !is_short ? 0 : type == GQ_Q8_0 ? 40 : type == GQ_Q4_K && !shallow ? 32 : 0;
    switch (type) {
    case GQ_Q8_0: return is_short || set ? 58 : 36;
    case GQ_Q6_K: return K < 1536 ? 0 : is_short || set ? 38 : 28;
    case GQ_Q4_0: return shallow ? 0 : gaps ? 52 : 58;
    case GQ_Q4_K: return shallow || gaps ? 0 : 40;
    default: return 0;
    }
}

// Whether the split-K kernels are ahead of mmv.hip where both take a call (a matrix - of a pair: each - of 6 MB and more).  mmv.hip contracts
// 9 to 16 rows as two sets of 8, the split-K kernels up to 32 at one price: Q4_K and the other 4-bit formats, whose weights take least of
// the time, feel that from 9 rows on.  And where the slices of K do not come out in groups of eight, mmv.hip leaves wavefront slots
// empty.  Measured (us, split-K | mmv.hip):
//   Q4_K    K <= 4096, 12 rows: 4096x14336 19.0 | 20.5, gated pairs of it 27.8 | 26.3, of 3072x6144 17.3 | 18.8, of 3072x11008 27.3 | 21.9, of 1024x16384 16.1 | 17.2
//           8 and 12 rows: 14336x4096 17.8 18.1 | 17.6 22.7, 8192x8192 22.5 22.9 | 17.2 23.5; 8 rows: 4608x4096 12.6 | 13.2, 5120x20480 behind a norm 25.9 | 27.2, 6144x8192 17.6 |
//           18.4, 6144x11008 24.6 | 19.7, 10240x4096 16.6 | 18.2 (at 4 rows 16.2 | 15.1), 10240x2560 16.6 | 14.7, gated pairs of 4608x4096 16.0 | 17.1, of 6144x8192 26.5 | 24.3,
//           of 4608x20480 35.1 | 40.6
//   Q4_0    12 rows: 4096x14336 24.2 | 20.3, 1024x32768 16.5 | 18.8; 8 and 12 rows: 6144x4096 14.9 15.5 | 13.5 17.1, 14336x4096 24.2 24.7 | 18.7 22.5; mmv.hip over split-K at 12 rows:
//           5120x3072 (8 MB) 1.17, 5120x8192 1.10, 6144x8192 .96, 9216x1536 1.09, 9216x2048 .98, 9216x3072 1.13; gated pairs: 5120x8192 1.13, 8192x4096 .98, 9216x4096 1.08, 9984x2560 .89
//   IQ4_NL  8 and 12 rows: 8192x4096 17.0 17.7 | 15.4 18.7; 12 rows: 12288x4096 26.5 | 24.3, 2048x16384 behind a norm 17.9 | 18.9
//   Q8_0    8 and 12 rows: 8192x1024 13.4 13.6 | 11.7 14.8, 9216x1024 14.2 14.4 | 11.6 13.6; 12 rows: 256x32768 13.5 | 14.2, 5120x3072 14.4 | 16.5 (two rounds of tiles, the
//           second half empty), 5120x4096 19.3 | 16.8.  Q6_K 5120x3072 16.7 | 18.1
// (Widths move both kernels by whole rounds of tiles, so that single shapes lie up to 15 % on the other side of these lines.)
// Their scratch memory is the larger one.
bool split_k_ahead(int type, int64_t M, int64_t K, int64_t one, int matrices) {
    const int64_t MB = (int64_t)1 << 20, slices = (K + 511) / 512, slots = (slices + 7) / 8 * 8;
    const bool gaps = K > 2048 && slices * 20 < slots * 17;
    auto within = [&](int64_t lo, int64_t hi) { return one >= lo * MB && one < hi * MB; };
    if (M < 5 || one < kTinyWeightBytes) return false;
    if (mmv_one_launch(K)) {
        if (M <= 8) return false;
        if (type == GQ_Q4_K) return matrices == 1 || K <= 1024 || (gaps && one < 14 * MB);
        return matrices == 1 && one >= 8 * MB && type != GQ_Q6_K && K <= (type == GQ_Q8_0 ? 512 : one >= 16 * MB ? 2048 : 1024);
    }
    switch (type) {
    case GQ_Q4_K:
        if (M > 8) return true;
        if (!gaps || (matrices == 2 && K > 6144)) return false;
        if (matrices == 2) return within(7, 13) || (K <= 5120 && one >= 48 * MB);
        return K <= 5120 ? one >= 10 * MB : K <= 6144 ? within(10, 28) : within(18, 24);
    case GQ_Q4_0:
    case GQ_IQ4_NL:
        if (M <= 8 || (matrices == 2 && !gaps)) return false;
        if (!gaps) return within(9, 26);
        return K <= 6144 ? within(7, K <= 5120 ? 31 : 24) : within(7, 9) || within(15, matrices == 1 ? 26 : 24);
    case GQ_Q8_0: return M > 8 && (one < 9 * MB || (matrices == 1 && K <= 5120 && within(13, 17)));
    case GQ_Q6_K: return M > 8 && matrices == 1 && K <= 5120 && within(10, 13);
    default: return false;
    }
}

// Whether 3 to 16 rows of up to 4096 values take the one-launch kernel of mmv.hip.  It costs about 5 us of activation conversion per
// workgroup and then streams W once; the GEMV it replaces costs a pass per row over small matrices, per four rows (two with a
// normalisation, a residual or a gated pair: `extras`) over those of 24 MB and more, the split-K kernels three launches.
// Measured (us per call on rotating weights; rows 2 3 4 6 8 12 16; the routes before | this one):
//   Q8_0   4096x1024   3.5  4.2  4.3  6.0  6.4  8.7 11.1 |  7.8  7.8  7.9  8.9  8.8 10.8 10.9    4096x14336  13.3 15.4 15.4 28.9 28.6 29.2 29.4 | 17.1 17.0 17.2 17.9 17.9 21.6 21.4
//          4096x4096   7.5 10.0 12.2 14.1 14.1 14.4 14.5 |  9.8  9.7  9.9 10.6 10.7 13.2 13.2    gated pair  23.8 40.7 40.7 48.2 49.3 50.0 50.6 | 25.3 25.5 25.6 26.5 26.7 31.7 31.8
//   Q4_0   4096x4096   5.6  7.3  8.9 12.2 12.4 12.7 12.9 |  8.1  8.0  8.1  8.7  8.7 11.8 11.9    4096x14336   9.6 14.0 14.0 22.8 23.3 23.8 23.9 | 14.0 14.0 14.3 15.3 15.5 20.3 20.4
//   Q4_K   4096x4096   6.7  8.8 10.9 12.0 12.3 12.4 12.6 |  8.0  7.9  8.0  9.6  9.6 13.1 12.9    4096x14336  11.1 14.8 14.8 18.3 18.6 19.0 19.3 | 12.4 12.3 12.5 13.8 13.9 20.4 20.4
//          gated pair  8.6 11.1 13.6 19.8 14.8 15.5 15.6 | 10.1 10.1 10.1 11.4 11.5 15.6 15.5    gated pair  18.9 26.3 26.6 27.1 27.2 27.8 28.5 | 17.7 17.7 18.0 19.4 19.5 26.3 26.3
//   Q6_K   4096x4096   8.0 10.6 13.2 17.0 17.3 17.5 17.7 |  9.8  9.5  9.6 10.6 10.6 14.1 14.1    4096x14336  14.6 24.5 24.1 31.5 32.1 32.8 32.8 | 17.3 17.2 17.4 18.2 18.1 24.1 24.5
//   IQ4_NL 4096x4096   6.8  9.0 11.0 13.1 13.3 13.6 13.8 |  8.5  8.5  8.5  9.3  9.4 12.6 12.6    4096x14336  12.3 16.0 16.1 25.6 26.3 26.9 27.1 | 16.1 16.0 16.1 17.0 17.3 22.3 22.5
// The GEMV's passes over matrices of less than 24 MB come out of the caches and cost rows x bytes, so that the product of both decides:
// below 9 MB mmv.hip takes over at 64 MB (Q8_0 4096x1024, 4.5 MB: even at 16 rows; a gated pair of them: 10.8 | 10.7 at 8; Q4_K: 14.5 | 14.5 at
// 12), above at gemv_reach().
// set: N counts the columns of several matrices that share x, which a call of its own would not take together
bool takes_mmv(int type, int64_t M, int64_t K, int64_t N, const void *x, const void *gain, int matrices, bool extras, bool set = false) {
    if (M < 3 || !mmv_one_launch(K) || !mmv_supported(type, M, K, N, x, gain)) return false;
    const int64_t one = weight_bytes_of(type, K, N), bytes = one * matrices, MB = (int64_t)1 << 20;
    if ((!set || type == GQ_Q4_K) && N % 4 == 0 && split_k_ahead(type, M, K, one, matrices)) return false;  // (what the split-K kernels take)
    if (bytes < 9 * MB) return M * bytes >= 64 * MB;
    if (bytes < kLargeWeightBytes) return !(type == GQ_Q4_0 && M == 3) && M * bytes >= gemv_reach(type, K, K * N * matrices, matrices, extras, set) * MB;
    if (!extras && !set && M <= 4 && (type == GQ_Q8_0 || (type == GQ_Q4_0 && bytes < 64 * MB))) return false;  // one GEMV pass of four rows
    return true;
}
// What the split-K kernels were chosen for: up to 16 rows take mmv.hip (rows of more than 4096 values its two launches instead of the three
// of mmq.hip) where split_k_ahead() says so.
int split_k(int type, const void *x, bool x_is_bf16, int64_t M, int64_t K, int count, const MmqSetItem *items, const MmqExtra *ex, hipStream_t s) {
    const void *gain = ex && ex->norm ? ex->norm->gain : nullptr;
    int64_t ntot = 0;
    for (int i = 0; i < count; i++) ntot += items[i].N;
    bool mmv = !split_k_ahead(type, M, K, weight_bytes_of(type, K, ntot), ex && ex->W2 ? 2 : 1);
    for (int i = 0; i < count; i++)
        mmv = mmv && mmv_supported(type, M, K, items[i].N, x, gain) && !(mmv_one_launch(K) && y_over_x(x, x_is_bf16, items[i].y, M, K, items[i].N));
    if (mmv) return launch_mmv(type, x, x_is_bf16, M, K, count, items, ex, s);
    if (count > 1) return launch_mmq_set(type, x, x_is_bf16, M, K, count, items, ex ? ex->norm : nullptr, s);
    return launch_mmq(type, x, x_is_bf16, M, K, items[0].W, items[0].N, items[0].bias, items[0].act, items[0].y, s, ex);
}

// Whether a call that the split-K kernels had no scratch memory for (a recording before the workspace exists, the static scratch array; nothing
// has been launched then) goes on to the routes it would take without them: only where rows of N or the outputs' addresses are not
// whole float4, calls which those routes served before the reduction stored them element by element.
bool falls_back(int rc, bool whole) { return rc == GQ_ERR_INVALID && !whole; }
bool whole_set(int count, const MmqSetItem *set) {
    bool whole = true;
    for (int i = 0; i < count; i++) whole = whole && whole_rows(set[i].N, set[i].bias, set[i].y);
    return whole;
}

// large batches: W dequantised once into the stream's workspace, then a plain 16-bit GEMM
int two_pass(int type, bool x_is_bf16, const void *x, int64_t M, int64_t K, const void *W, int64_t N, const float *bias, int act,
             float *y, hipStream_t s) {
    void *ws = nullptr;
    // (K in one piece where the static scratch array holds the images but not the sums of its slices: another order of the same fp32 sums, as
    // the header says.  Held to the slices that fit, gq_qdense_f32 would return the same bits, at 28.7 us for 21.5 on 4096 -> 1024 at 520 rows.)
    const bool split_k = !serves_static_scratch() || gemm_two_pass_workspace(type, x_is_bf16, M, K, N) <= kStaticScratchBytes - kWsSyncBytes;
    if (int rc = stream_workspace(s, gemm_two_pass_workspace(type, x_is_bf16, M, K, N, split_k), &ws)) return rc;
    return launch_gemm_two_pass(type, x_is_bf16, x, M, K, static_cast<const uint8_t *>(W), N, bias, act, y, ws, s, split_k);
}

}  // namespace
}  // namespace gq

using namespace gq;

extern "C" {

int gq_abi_version(void) { return 1; }

int gq_bytes_per_block(int type) {
    TypeInfo ti;
    return type_info(type, ti) ? ti.bpb : 0;
}

int gq_values_per_block(int type) {
    TypeInfo ti;
    return type_info(type, ti) ? ti.vpb : 0;
}

size_t gq_row_bytes(int type, int64_t K) {
    TypeInfo ti;
    if (!type_info(type, ti) || K <= 0 || K % ti.vpb != 0) return 0;
    return (size_t)(K / ti.vpb) * (size_t)ti.bpb;
}

int gq_qdense_check(int type, int x_dtype, int64_t M, int64_t x_last_dim, int64_t N, int64_t w_row_bytes,
                    int64_t bias_len, int act, int64_t *K_out) {
    TypeInfo ti;
    if (!type_info(type, ti)) return fail(GQ_ERR_NOT_IMPLEMENTED, "FusedQuantizedDense: ggml type %d is not implemented", type);
    if (x_dtype != GQ_F32 && x_dtype != GQ_BF16)
        return fail(GQ_ERR_NOT_IMPLEMENTED, "FusedQuantizedDense: activation dtype %d is not implemented", x_dtype);
    if (M < 0 || N < 0) return fail(GQ_ERR_INVALID, "FusedQuantizedDense: negative dimension");
    if (w_row_bytes <= 0 || w_row_bytes % ti.bpb != 0)
        return fail(GQ_ERR_INVALID, "FusedQuantizedDense: weight row of %lld bytes is not a whole number of %d-byte blocks",
                    (long long)w_row_bytes, ti.bpb);
    const int64_t K = w_row_bytes / ti.bpb * ti.vpb;
    if (x_last_dim != K)  // ml/ggml/dense.go:38-41
        return fail(GQ_ERR_INVALID, "FusedQuantizedDense: x has %lld features but the weights decode to K=%lld",
                    (long long)x_last_dim, (long long)K);
    if (bias_len >= 0 && bias_len != N)
        return fail(GQ_ERR_INVALID, "FusedQuantizedDense: bias has %lld elements, expected N=%lld", (long long)bias_len, (long long)N);
    if (act < GQ_ACT_NONE || act > GQ_ACT_TANH) return fail(GQ_ERR_INVALID, "FusedQuantizedDense: unknown activation %d", act);
    if (K_out) *K_out = K;
    return GQ_OK;
}

int gq_device_count(int *count) {
    if (!count) return fail(GQ_ERR_INVALID, "gq_device_count: null argument");
    int n = 0;
    const hipError_t e = hipGetDeviceCount(&n);
    if (e == hipErrorNoDevice) { *count = 0; return GQ_OK; }
    if (e != hipSuccess) { *count = 0; return hip_fail(e, "hipGetDeviceCount"); }
    *count = n;
    return GQ_OK;
}

int gq_init(int device) {
    std::lock_guard<std::mutex> lock(g_init_mutex);
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0) return fail(GQ_ERR_NO_DEVICE, "gq_init: no HIP device (%s)", hipGetErrorString(e));
    if (device < 0 || device >= n) return fail(GQ_ERR_NO_DEVICE, "gq_init: device %d out of range (found %d)", device, n);
    const int cur = g_device.load();
    if (cur >= 0 && cur != device)
        return fail(GQ_ERR_INVALID, "gq_init: already initialised on device %d (one device per process)", cur);
    hipDeviceProp_t prop;
    GQ_HIP(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(GQ_ERR_NO_DEVICE, "gq_init: device %d is %s; this library holds gfx950 code only", device, prop.gcnArchName);
    GQ_HIP(hipSetDevice(device));
    if (device >= kMaxDevices) return fail(GQ_ERR_NO_DEVICE, "gq_init: device %d is beyond the %d this library keeps state for", device, kMaxDevices);
    if (!g_scratch_ptr[device]) {  // this device's copy of the static scratch array (each device has its own, at its own address)
        void *p = nullptr;
        GQ_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[device] = p;
    }
    g_cu_count.store(prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256);
    g_device.store(device, std::memory_order_release);
    return GQ_OK;
}

int gq_device_name(char *buf, size_t n) {
    if (!buf || n == 0) return fail(GQ_ERR_INVALID, "gq_device_name: null buffer");
    if (int rc = use_device()) return rc;
    hipDeviceProp_t prop;
    GQ_HIP(hipGetDeviceProperties(&prop, g_device.load()));
    std::snprintf(buf, n, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
    return GQ_OK;
}

int gq_malloc(void **dptr, size_t bytes) {
    if (!dptr) return fail(GQ_ERR_INVALID, "gq_malloc: null argument");
    *dptr = nullptr;
    if (int rc = use_device()) return rc;
    if (bytes == 0) return GQ_OK;
    GQ_HIP(hipMalloc(dptr, bytes));
    return GQ_OK;
}

int gq_free(void *dptr) {
    if (!dptr) return GQ_OK;
    if (int rc = use_device()) return rc;
    GQ_HIP(hipFree(dptr));
    return GQ_OK;
}

int gq_h2d(void *d, const void *h, size_t bytes, void *stream) {
    if (bytes == 0) return GQ_OK;
    if (!d || !h) return fail(GQ_ERR_INVALID, "gq_h2d: null pointer");
    if (int rc = use_device()) return rc;
    GQ_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, (hipStream_t)stream));
    GQ_HIP(hipStreamSynchronize((hipStream_t)stream));
    return GQ_OK;
}

int gq_d2h(void *h, const void *d, size_t bytes, void *stream) {
    if (bytes == 0) return GQ_OK;
    if (!d || !h) return fail(GQ_ERR_INVALID, "gq_d2h: null pointer");
    if (int rc = use_device()) return rc;
    GQ_HIP(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream));
    GQ_HIP(hipStreamSynchronize((hipStream_t)stream));
    return GQ_OK;
}

int gq_stream_create(void **stream) {
    if (!stream) return fail(GQ_ERR_INVALID, "gq_stream_create: null argument");
    if (int rc = use_device()) return rc;
    hipStream_t s;
    GQ_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = s;
    return GQ_OK;
}

int gq_stream_destroy(void *stream) {
    if (!stream) return GQ_OK;
    if (int rc = use_device()) return rc;
    pool().destroy_stream(stream);  // waits for the stream, then frees its workspaces (those a recorded graph points at go with the graph)
    GQ_HIP(hipStreamDestroy((hipStream_t)stream));
    return GQ_OK;
}

int gq_sync(void *stream) {
    if (int rc = use_device()) return rc;
    GQ_HIP(hipStreamSynchronize((hipStream_t)stream));
    return GQ_OK;
}

int gq_dequantize(int type, const void *dW, int64_t N, int64_t K, float *dOut, void *stream) {
    TypeInfo ti;
    if (!type_info(type, ti)) return fail(GQ_ERR_NOT_IMPLEMENTED, "gq_dequantize: ggml type %d is not implemented", type);
    if (N < 0) return fail(GQ_ERR_INVALID, "gq_dequantize: negative N");
    if (K <= 0 || K % ti.vpb != 0)
        return fail(GQ_ERR_INVALID, "gq_dequantize: K=%lld is not a positive multiple of the block size %d", (long long)K, ti.vpb);
    if (N == 0) return GQ_OK;
    if (!dW || !dOut) return fail(GQ_ERR_INVALID, "gq_dequantize: null device pointer");
    if (!aligned_to(dW, 16) || !aligned_to(dOut, 16))
        return fail(GQ_ERR_INVALID, "gq_dequantize: weights and output must be 16-byte aligned");
    if (int rc = use_device()) return rc;
    return launch_dequantize(type, (const uint8_t *)dW, N, K, dOut, (hipStream_t)stream);
}

int gq_qdense_f32(int type, const float *dX, int64_t M, int64_t K, const void *dW, int64_t N, const float *dBias,
                  int act, float *dY, void *stream) {
    if (int rc = check_dense_args("gq_qdense_f32", type, dX, M, K, dW, N, dBias, act, dY, 4)) return rc;
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBias, dY);
    // Small batches: GEMV passes cost about one third of the first pass per extra row; the split-K
    // MFMA kernels cost 19 .. 26 us (Q8_0 / Q4_0, K = 4096, N = 4096 .. 14336) for up to 32 rows and
    // 5 .. 18 us per further 32; the two passes 33 .. 62 us for anything up to 128 rows.  Measured
    // crossovers: split_k_from() / split_k_to().
    const MmqSetItem one{(const uint8_t *)dW, N, dBias, act, dY};
    if (takes_mmv(type, M, K, N, dX, nullptr, 1, false) && !y_over_x(dX, false, dY, M, K, N))
        return launch_mmv(type, dX, false, M, K, 1, &one, nullptr, (hipStream_t)stream);
    const bool tp = gemm_two_pass_supported(type, false, M, K, N, dX);
    const bool ks = M <= kGemvMaxRows && gemv_ks_supported(type, K, N, dX);
    const bool sk = M >= take_over(split_k_from(type, weight_bytes_of(type, K, N)), whole) && mmq_supported(type, M, K, N, dX) &&
                    (M <= hand_over(type, K, N, false, whole) || !tp);
    if (sk) {
        const int rc = split_k(type, dX, false, M, K, 1, &one, nullptr, (hipStream_t)stream);
        if (!falls_back(rc, whole)) return rc;
    }
    if (ks) return launch_gemv_ks(type, dX, false, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
    // Shapes without a K-sliced plan (K not a multiple of 256: rare in models): a pass over W per row for up to 16
    // rows.  The 16-bit operands of the GEMMs below lean on averaging over many outputs and terms; on these few-row
    // problems seeded sweeps measured up to 0.9e-3 (1.25e-3 over a single block) through them, too close to the bound.
    if (M <= kGemvMaxRows) {
        if (gemv_xs_supported(type, K, N, dX))
            return launch_gemv_xs(type, dX, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
        return launch_gemv(type, dX, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
    }
    if (tp) return two_pass(type, false, dX, M, K, dW, N, dBias, act, dY, (hipStream_t)stream);
    return launch_gemm(type, false, dX, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
}

int gq_qdense_f32_static(int type, const float *dX, int64_t M, int64_t K, const void *dW, int64_t N, const float *dBias,
                         int act, float *dY, void *stream) {
    if (int rc = check_dense_args("gq_qdense_f32_static", type, dX, M, K, dW, N, dBias, act, dY, 4)) return rc;
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    if (profile_state().active) return fail(GQ_ERR_INVALID, "gq_qdense_f32_static: kernel timing creates events; not available on this entry point");
    if (t_scope) return fail(GQ_ERR_INVALID, "gq_qdense_f32_static: not callable from inside another entry point");
    unsigned char *sp = static_cast<unsigned char *>(g_scratch_ptr[g_device.load(std::memory_order_acquire)]);
    if (!sp) return fail(GQ_ERR_NO_DEVICE, "gq_qdense_f32_static: gq_init() has not taken the scratch array's address on this device");
    CallScope scope;
    scope.static_ptr = sp;  // every scratch request below is served from the static array, or fails
    return gq_qdense_f32(type, dX, M, K, dW, N, dBias, act, dY, stream);
}

namespace {
bool set_takes_mmv(int count, const gq_dense_desc *descs, const float *gain, bool normed, MmqSetItem *set);
bool takes_shared_pass(int count, const gq_dense_desc *descs, const float *gain, MmqSetItem *set);  // (defined with the dispatch thresholds below)
// From 6 rows the shared split-K pass is ahead of the merged GEMV launch: a decoder layer's q / k / v, 4096 -> 4096 + 2 x 1024,
// with the rest of the layer: 79.2 against 80.0 us at 5 rows, 81.6 against 79.9 at 6, 84.7 against 80.3 at 8.
constexpr int64_t kSharedPassFromRows = 6;
}  // namespace

int gq_qdense_f32_batch(int count, const gq_dense_desc *descs, void *stream) {
    if (count < 0 || (count > 0 && !descs)) return fail(GQ_ERR_INVALID, "gq_qdense_f32_batch: bad descriptor list");
    for (int i = 0; i < count; i++) {
        const gq_dense_desc &d = descs[i];
        if (int rc = check_dense_args("gq_qdense_f32_batch", d.type, d.dX, d.M, d.K, d.dW, d.N, d.dBias, d.act, d.dY, 4)) return rc;
    }
    if (count == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    {   // projections of one input beyond the GEMV's best rows: one split-K pass for all of them
        MmqSetItem set[4];
        if (set_takes_mmv(count, descs, nullptr, false, set))
            return launch_mmv(descs[0].type, descs[0].dX, false, descs[0].M, descs[0].K, count, set, nullptr, (hipStream_t)stream);
        if (descs[0].M >= kSharedPassFromRows && takes_shared_pass(count, descs, nullptr, set)) {
            const int rc = split_k(descs[0].type, descs[0].dX, false, descs[0].M, descs[0].K, count, set, nullptr, (hipStream_t)stream);
            if (!falls_back(rc, whole_set(count, set))) return rc;
        }
    }
    // problems that calls of their own would hand to the few-row kernel: up to four of one type, batch size and K in one launch, each with
    // its own input and share of the workgroups, and the bits of a call of its own (two Q4_K 4096x4096 at 3 and 5 rows 9.8 and 11.6 us; one launch each took 16.0 18.7,
    // the merged GEMV launch 10.0 14.5)
    uint64_t done = 0;
    auto few = [&](const gq_dense_desc &d) { return d.N > 0 && takes_mmv(d.type, d.M, d.K, d.N, d.dX, nullptr, 1, false); };
    for (int i = 0; i < count && i < 64; i++) {
        if ((done >> i & 1) || !few(descs[i])) continue;
        MmqSetItem items[4];
        const void *xs[4];
        uint64_t mine = 0;
        int n = 0;
        for (int j = i; j < count && j < 64 && n < 4; j++) {
            const gq_dense_desc &d = descs[j];
            if ((done >> j & 1) || d.type != descs[i].type || d.M != descs[i].M || d.K != descs[i].K || !few(d)) continue;
            items[n] = MmqSetItem{(const uint8_t *)d.dW, d.N, d.dBias, d.act, d.dY};
            xs[n++] = d.dX;
            mine |= (uint64_t)1 << j;
        }
        if (n < 2) continue;
        if (int rc = launch_mmv(descs[i].type, nullptr, false, descs[i].M, descs[i].K, n, items, nullptr, (hipStream_t)stream, xs)) return rc;
        done |= mine;
    }
    // merge runs of batch-1 problems of one type that the streaming GEMV handles; the rest go one by one
    auto is_done = [&](int k) { return k < 64 && (done >> k & 1); };
    int i = 0;
    while (i < count) {
        if (is_done(i)) {
            i++;
            continue;
        }
        int j = i;
        XsBatchItem items[8];
        // the kernel family of the run is that of its first problem: K-sliced where that applies, else
        // activation-stationary
        const bool use_ks = gemv_ks_supported(descs[i].type, descs[i].K, descs[i].N, descs[i].dX);
        auto fits = [&](const gq_dense_desc &d) {
            return use_ks ? gemv_ks_supported(d.type, d.K, d.N, d.dX) : gemv_xs_supported(d.type, d.K, d.N, d.dX);
        };
        const int64_t rows = descs[i].M;
        const bool rows_ok = rows == 1 || (use_ks && rows >= 1 && rows <= batch_rows_max());
        // (several rows per problem: only over matrices below the size from which one pass serves several rows)
        // (and none for the few-row kernel: one that is alone in the list takes it in a call of its own)
        auto size_ok = [&](const gq_dense_desc &d) {
            return rows == 1 || (weight_bytes_of(d.type, d.K, d.N) < kLargeWeightBytes && !few(d));
        };
        while (j < count && !is_done(j) && j - i < 8 && rows_ok && descs[j].type == descs[i].type && descs[j].M == rows && descs[j].N > 0 && fits(descs[j]) &&
               size_ok(descs[j])) {
            const gq_dense_desc &d = descs[j];
            items[j - i] = XsBatchItem{d.dX, (const uint8_t *)d.dW, d.dBias, d.dY, d.K, d.N, d.act};
            j++;
        }
        if (j - i >= 2) {
            if (int rc = use_ks ? launch_gemv_ks_batch(descs[i].type, j - i, items, (hipStream_t)stream, (int)rows)
                                : launch_gemv_xs_batch(descs[i].type, j - i, items, (hipStream_t)stream))
                return rc;
            i = j;
            continue;
        }
        const gq_dense_desc &d = descs[i];
        if (int rc = gq_qdense_f32(d.type, d.dX, d.M, d.K, d.dW, d.N, d.dBias, d.act, d.dY, stream)) return rc;
        i++;
    }
    return GQ_OK;
}

int gq_qdense_bf16(int type, const uint16_t *dX, int64_t M, int64_t K, const void *dW, int64_t N,
                   const float *dBias, int act, float *dY, void *stream) {
    if (int rc = check_dense_args("gq_qdense_bf16", type, dX, M, K, dW, N, dBias, act, dY, 2)) return rc;
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBias, dY);
    // Same crossovers as for fp32 activations: bf16 widens exactly to fp32 for the GEMV passes and to
    // the fp16 activation image of the split-K kernels (which have no bf16 rounding of W: tighter than
    // the bf16 MFMA paths).
    const MmqSetItem one{(const uint8_t *)dW, N, dBias, act, dY};
    if (takes_mmv(type, M, K, N, dX, nullptr, 1, false) && !y_over_x(dX, true, dY, M, K, N))
        return launch_mmv(type, dX, true, M, K, 1, &one, nullptr, (hipStream_t)stream);
    const bool tp = gemm_two_pass_supported(type, true, M, K, N, dX);
    const bool ks = M <= kGemvMaxRows && gemv_ks_supported(type, K, N, dX);
    const bool sk = M >= take_over(split_k_from(type, weight_bytes_of(type, K, N)), whole) && mmq_supported(type, M, K, N, dX) &&
                    (M <= hand_over(type, K, N, false, whole) || !tp);
    if (sk) {
        const int rc = split_k(type, dX, true, M, K, 1, &one, nullptr, (hipStream_t)stream);
        if (!falls_back(rc, whole)) return rc;
    }
    if (ks) return launch_gemv_ks(type, dX, true, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
    if (tp) return two_pass(type, true, dX, M, K, dW, N, dBias, act, dY, (hipStream_t)stream);
    return launch_gemm(type, true, dX, M, K, (const uint8_t *)dW, N, dBias, act, dY, (hipStream_t)stream);
}

int gq_rmsnorm_f32(const float *dX, int64_t M, int64_t K, const float *dGain, float eps, float gain_offset, float *dY, void *stream) {
    if (M < 0 || K <= 0 || K > INT32_MAX) return fail(GQ_ERR_INVALID, "gq_rmsnorm_f32: bad shape [%lld, %lld]", (long long)M, (long long)K);
    if (!(eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_rmsnorm_f32: epsilon must be >= 0");
    if (M == 0) return GQ_OK;
    if (M > INT32_MAX) return fail(GQ_ERR_NOT_IMPLEMENTED, "gq_rmsnorm_f32: more than 2^31 - 1 rows");
    if (!dX || !dY) return fail(GQ_ERR_INVALID, "gq_rmsnorm_f32: null device pointer");
    if (!aligned_to(dX, 4) || !aligned_to(dY, 4) || (dGain && !aligned_to(dGain, 4)))
        return fail(GQ_ERR_INVALID, "gq_rmsnorm_f32: pointers must be 4-byte aligned");
    if (int rc = use_device()) return rc;
    return launch_rmsnorm(dX, M, K, dGain, gain_offset, eps, dY, (hipStream_t)stream);
}

namespace {
// First batch size at which a projection with its neighbours leaves the GEMV for the split-K kernels.  The GEMV with
// the extras walks a large matrix once per two rows (not four), the split-K form costs the same for any batch up to 32
// rows and carries the normalisation and the residual at no extra launch.  Measured (us per call in a replayed graph,
// RMSNorm in front; rows 2 3 4 5 6 7 8 on the GEMV | split-K):
//   block (one projection + residual)                                    gated pair (SiLU)
//   Q8_0   4096x4096 10 14 16 19 22 25 28 | 15   4096x14336 16 26 26 36 36 47 47 | 30      12 19 19 26 26 33 33 | 23   28 46 45 62 62 80 80 | 52
//   Q4_0   4096x4096  9 12 14 17 20 22 25 | 13   4096x14336 12 20 20 28 28 36 36 | 25      10 12 14 16 18 20 22 | 20   19 33 32 46 46 59 59 | 41
//   Q4_K   4096x4096  9 12 15 18 20 23 26 | 13   4096x14336 13 22 22 31 31 40 40 | 19      10 12 15 17 20 22 24 | 21   21 36 35 50 50 65 65 | 33
//   Q6_K   4096x4096 11 14 17 20 23 26 30 | 19   4096x14336 16 28 28 39 39 51 51 | 33      12 20 20 28 28 35 35 | 31   29 47 47 64 64 83 83 | 59
//   IQ4_NL 4096x4096 10 13 16 19 22 25 28 | 14   4096x14336 14 25 25 35 35 46 46 | 28      12 15 18 21 24 27 31 | 19   24 42 41 59 59 77 77 | 46
// (14336x4096 behaves like 4096x14336.)  Matrices of a few megabytes stay on the GEMV for every batch it takes.  As above, the line is that of the
// three launches: rows of up to 4096 values come here only where takes_mmv() has declined them, and the two launches that longer ones now take are
// ahead below it (behind a norm, rows 4 on the GEMV | 5 on the two launches: 14336x4096 Q8_0 29.1 | 21.0, Q4_0 23.2 | 19.0, Q6_K 30.8 | 22.5, IQ4_NL 27.2 | 21.4;
// gated 46.4 | 30.4, 35.6 | 26.7, 46.8 | 32.8, 43.2 | 31.2).
int64_t block_split_k_from(int type, int64_t weight_bytes, bool gated) {
    if (weight_bytes < kTinyWeightBytes) return kGemvMaxRows + 1;
    if (weight_bytes >= kLargeWeightBytes) return type == GQ_Q4_K ? 3 : 5;
    switch (type) {
    case GQ_Q8_0: return gated ? 5 : 4;
    case GQ_Q4_0: return gated ? 8 : 5;
    case GQ_Q4_K: return gated ? 7 : 4;
    case GQ_Q6_K: return gated ? 7 : 5;
    case GQ_IQ4_NL: return gated ? 5 : 4;
    default: return 8;
    }
}

bool fold_into_gemv(int type, int64_t M, int64_t K, int64_t N, const float *x, const float *gain, bool gated, bool whole, bool up_whole = true) {
    if (!gemv_ks_ext_supported(type, M, K, N, x, gain)) return false;
    return !(M >= take_over(block_split_k_from(type, weight_bytes_of(type, K, N), gated), whole && up_whole) && mmq_supported(type, M, K, N, x));
}

// Whether a projection with its neighbours runs on the split-K kernels (after fold_into_gemv() has declined).
// up_whole: whether a gated pair's up bias is aligned as well.  Only the line up to 16 rows asks: off 16 bytes, that projection stayed on the GEMV and
// the few-row kernel, whose activations have more bits (take_over).
bool block_takes_split_k(int type, int64_t M, int64_t K, int64_t N, const float *x, bool gated, bool whole, bool up_whole = true) {
    const bool tp = gated ? gemm_two_pass_block_supported(type, M, K, N, x, true) : gemm_two_pass_supported(type, false, M, K, N, x);
    const int64_t to = hand_over(type, K, N, gated, whole);
    return M >= take_over(block_split_k_from(type, weight_bytes_of(type, K, N), gated), whole && up_whole) && mmq_supported(type, M, K, N, x) && (M <= to || !tp);
}

// Whether a plain dense call on these operands runs on the split-K kernels (the dispatch of gq_qdense_f32).
bool dense_takes_split_k(int type, int64_t M, int64_t K, int64_t N, const float *x, bool whole, bool up_whole = true) {
    const bool tp = gemm_two_pass_supported(type, false, M, K, N, x);
    return M >= take_over(split_k_from(type, weight_bytes_of(type, K, N)), whole && up_whole) && mmq_supported(type, M, K, N, x) && (M <= hand_over(type, K, N, false, whole) || !tp);
}

// First batch size of the gated pair as one GEMM (wherever the split-K kernels have handed over: the composed form is never
// ahead); GOMLX_HIPQ_GATED_TWO_PASS_FROM=rows overrides it (tuning runs only).
int64_t gated_two_pass_from() {
    static const int64_t v = [] { const char *e = std::getenv("GOMLX_HIPQ_GATED_TWO_PASS_FROM"); return e ? (int64_t)std::atoll(e) : (int64_t)(kGemvMaxRows + 1); }();
    return v;
}

// Batches that a plain dense call would hand to the two-pass GEMM take its block form: the
// normalisation rides on the activation pass, the residual and the gated product on the epilogue.
bool block_takes_two_pass(int type, int64_t M, int64_t K, int64_t N, const float *x, const float *gain, bool gated, bool whole) {
    if (M <= kGemvMaxRows || !gemm_two_pass_block_supported(type, M, K, N, x, gated)) return false;
    if (gated && M < gated_two_pass_from()) return false;
    if (gain && !aligned_to(gain, 16)) return false;
    const int64_t to = hand_over(type, K, N, gated, whole);
    const bool sk = M >= split_k_from(type, weight_bytes_of(type, K, N)) && mmq_supported(type, M, K, N, x) && M <= to;
    return !sk;
}
// Whether a list of projections is one input contracted with two to four matrices that the shared split-K pass takes
// (launch_mmq_set): equal type, activations, rows and K, the matrices taken together in the split-K kernels' range.
// Whether a list of two to four projections reads one input: equal type, activations, rows and K (fills `set`).
bool same_input_set(int count, const gq_dense_desc *descs, MmqSetItem *set) {
    if (count < 2 || count > 4) return false;
    for (int i = 0; i < count; i++) {
        const gq_dense_desc &d = descs[i];
        if (d.type != descs[0].type || d.dX != descs[0].dX || d.M != descs[0].M || d.K != descs[0].K || d.N <= 0) return false;
        set[i] = MmqSetItem{(const uint8_t *)d.dW, d.N, d.dBias, d.act, d.dY};
    }
    return true;
}
bool set_takes_mmv(int count, const gq_dense_desc *descs, const float *gain, bool normed, MmqSetItem *set) {
    if (!same_input_set(count, descs, set)) return false;
    int64_t ntot = 0;
    for (int i = 0; i < count; i++) ntot += descs[i].N;
    return takes_mmv(descs[0].type, descs[0].M, descs[0].K, ntot, descs[0].dX, gain, 1, normed, true);
}
bool takes_shared_pass(int count, const gq_dense_desc *descs, const float *gain, MmqSetItem *set) {
    if ((gain && !aligned_to(gain, 16)) || !same_input_set(count, descs, set)) return false;
    const int type = descs[0].type;
    const int64_t rows = descs[0].M, K = descs[0].K;
    int64_t ntot = 0;
    for (int i = 0; i < count; i++) ntot += descs[i].N;
    const bool whole = whole_set(count, set);
    return mmq_set_supported(type, count, set, rows, K, descs[0].dX) &&
           rows >= take_over(block_split_k_from(type, weight_bytes_of(type, K, ntot), false), whole) &&
           (rows <= hand_over(type, K, ntot, false, whole) || !gemm_two_pass_supported(type, false, rows, K, ntot, descs[0].dX));
}
}  // namespace

int gq_qdense_block_f32(int type, const float *dX, int64_t M, int64_t K, const gq_rmsnorm *norm, const void *dW, int64_t N,
                        const float *dBias, int act, const float *dResidual, float *dY, void *stream) {
    if (!norm && !dResidual) return gq_qdense_f32(type, dX, M, K, dW, N, dBias, act, dY, stream);
    if (int rc = check_dense_args("gq_qdense_block_f32", type, dX, M, K, dW, N, dBias, act, dY, 4)) return rc;
    if (norm && !(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_block_f32: epsilon must be >= 0");
    if (norm && norm->dGain && !aligned_to(norm->dGain, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_block_f32: gain must be 4-byte aligned");
    if (dResidual && !aligned_to(dResidual, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_block_f32: residual must be 4-byte aligned");
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBias, dY);
    RmsNorm rn{nullptr, 0.f, 0.f};
    if (norm) rn = RmsNorm{norm->dGain, norm->eps, norm->gain_offset};
    const MmqSetItem one{(const uint8_t *)dW, N, dBias, act, dY};
    const MmqExtra ex{nullptr, nullptr, dResidual, norm ? &rn : nullptr};
    if (takes_mmv(type, M, K, N, dX, rn.gain, 1, true) && !y_over_x(dX, false, dY, M, K, N))
        return launch_mmv(type, dX, false, M, K, 1, &one, &ex, (hipStream_t)stream);
    if (fold_into_gemv(type, M, K, N, dX, rn.gain, false, whole))
        return launch_gemv_ks_ext(type, dX, false, M, K, norm ? &rn : nullptr, (const uint8_t *)dW, dBias, nullptr, nullptr, dResidual, N, act, dY,
                                  (hipStream_t)stream);
    if (block_takes_two_pass(type, M, K, N, dX, rn.gain, false, whole)) {
        void *ws = nullptr;
        if (int rc = stream_workspace((hipStream_t)stream, gemm_two_pass_block_workspace(type, M, K, N, false), &ws)) return rc;
        return launch_gemm_two_pass_block(type, dX, M, K, norm ? &rn : nullptr, (const uint8_t *)dW, dBias, nullptr, nullptr, dResidual, N, act,
                                          dY, ws, (hipStream_t)stream);
    }
    // split-K range: the normalisation rides on the activation pre-pass and the reduction, the residual on the reduction
    if (block_takes_split_k(type, M, K, N, dX, false, whole) && (!rn.gain || aligned_to(rn.gain, 16))) {
        const int rc = split_k(type, dX, false, M, K, 1, &one, &ex, (hipStream_t)stream);
        if (!falls_back(rc, whole)) return rc;
    }
    // composed: normalised activations into the stream's second workspace, the dense call, then the residual.  When y
    // overlaps the residual (a residual stream updated in place) the dense result goes to the workspace first: written
    // straight to y it would destroy the residual before the addition reads it.
    const float *x = dX;
    const size_t y_bytes = (size_t)M * (size_t)N * sizeof(float);
    const bool in_place = dResidual && reinterpret_cast<uintptr_t>(dY) < reinterpret_cast<uintptr_t>(dResidual) + y_bytes &&
                          reinterpret_cast<uintptr_t>(dResidual) < reinterpret_cast<uintptr_t>(dY) + y_bytes;
    const size_t xn_bytes = norm ? ((size_t)M * (size_t)K * sizeof(float) + 255) / 256 * 256 : 0;
    float *tmp = nullptr;
    if (norm || in_place) {
        void *ws = nullptr;
        if (int rc = stream_workspace((hipStream_t)stream, xn_bytes + (in_place ? y_bytes : 0), &ws, 1)) return rc;
        tmp = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + xn_bytes);
        if (norm) {
            float *xn = static_cast<float *>(ws);
            if (int rc = launch_rmsnorm(dX, M, K, rn.gain, rn.gain_offset, rn.eps, xn, (hipStream_t)stream)) return rc;
            x = xn;
        }
    }
    if (dResidual && dense_takes_split_k(type, M, K, N, x, whole)) {  // the residual rides on the reduction
        const MmqExtra plain{nullptr, nullptr, dResidual, nullptr};
        const int rc = split_k(type, x, false, M, K, 1, &one, &plain, (hipStream_t)stream);
        if (!falls_back(rc, whole)) return rc;
    }
    float *dense_out = in_place ? tmp : dY;
    if (int rc = gq_qdense_f32(type, x, M, K, dW, N, dBias, act, dense_out, stream)) return rc;
    if (dResidual) return launch_add(dense_out, dResidual, dY, M * N, (hipStream_t)stream);
    return GQ_OK;
}

namespace {
// Whether a list of projections behind one normalisation is one launch of the K-sliced GEMV: every problem a projection of one
// type, one K and one (small) batch size that kernel takes (dX may point at fp32 or bf16 data: only its alignment matters),
// unless the shared split-K pass takes them at that batch size.  Fills items[0 .. count).
bool merges_into_gemv(int count, const gq_dense_desc *descs, const gq_rmsnorm *norm, bool shared_pass, XsBatchItem *items) {
    const int64_t rows = descs[0].M;
    bool merged = count >= 2 && count <= 8 && rows >= 1 && rows <= batch_rows_max() && !(shared_pass && rows >= kSharedPassFromRows);
    for (int i = 0; i < count && merged; i++) {
        const gq_dense_desc &d = descs[i];
        merged = d.type == descs[0].type && d.K == descs[0].K && d.M == rows && d.N > 0 && gemv_ks_ext_supported(d.type, rows, d.K, d.N, d.dX, norm->dGain) &&
                 (rows == 1 || weight_bytes_of(d.type, d.K, d.N) < kLargeWeightBytes);
        if (merged) items[i] = XsBatchItem{d.dX, (const uint8_t *)d.dW, d.dBias, d.dY, d.K, d.N, d.act};
    }
    return merged;
}
}  // namespace

int gq_qdense_norm_f32_batch(int count, const gq_dense_desc *descs, const gq_rmsnorm *norm, void *stream) {
    if (!norm) return gq_qdense_f32_batch(count, descs, stream);
    if (count < 0 || (count > 0 && !descs)) return fail(GQ_ERR_INVALID, "gq_qdense_norm_f32_batch: bad descriptor list");
    for (int i = 0; i < count; i++) {
        const gq_dense_desc &d = descs[i];
        if (int rc = check_dense_args("gq_qdense_norm_f32_batch", d.type, d.dX, d.M, d.K, d.dW, d.N, d.dBias, d.act, d.dY, 4)) return rc;
    }
    if (!(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_norm_f32_batch: epsilon must be >= 0");
    if (count == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const int64_t rows = descs[0].M;
    // Projections of the same activations (q / k / v) can share one split-K pass - one activation image, one main launch
    // over all their rows, one reduction - where the matrices taken together are in that kernel's range (three calls
    // would convert the activations three times and pay nine launches).
    MmqSetItem set[4];
    const RmsNorm rn{norm->dGain, norm->eps, norm->gain_offset};
    const MmqExtra ex{nullptr, nullptr, nullptr, &rn};
    if (set_takes_mmv(count, descs, norm->dGain, true, set))
        return launch_mmv(descs[0].type, descs[0].dX, false, rows, descs[0].K, count, set, &ex, (hipStream_t)stream);
    const bool shared_pass = takes_shared_pass(count, descs, norm->dGain, set);
    XsBatchItem items[8];
    if (merges_into_gemv(count, descs, norm, shared_pass, items))
        return launch_gemv_ks_batch_norm(descs[0].type, count, items, &rn, (hipStream_t)stream, (int)rows);
    if (shared_pass) {
        const int rc = split_k(descs[0].type, descs[0].dX, false, rows, descs[0].K, count, set, &ex, (hipStream_t)stream);
        if (!falls_back(rc, whole_set(count, set))) return rc;
    }
    // Past the split-K range the same projections share the two passes: one activation conversion, one image of all the
    // matrices, one GEMM (a decoder layer's q / k / v at 128 rows: two launches instead of six).
    if (same_input_set(count, descs, set) && rows > kGemvMaxRows && (!norm->dGain || aligned_to(norm->dGain, 16)) &&
        gemm_two_pass_set_supported(descs[0].type, count, set, rows, descs[0].K, descs[0].dX)) {
        void *ws = nullptr;
        if (int rc = stream_workspace((hipStream_t)stream, gemm_two_pass_set_workspace(descs[0].type, count, set, rows, descs[0].K), &ws)) return rc;
        return launch_gemm_two_pass_set(descs[0].type, descs[0].dX, rows, descs[0].K, &rn, count, set, ws, (hipStream_t)stream);
    }
    for (int i = 0; i < count; i++) {
        const gq_dense_desc &d = descs[i];
        if (int rc = gq_qdense_block_f32(d.type, d.dX, d.M, d.K, norm, d.dW, d.N, d.dBias, d.act, nullptr, d.dY, stream)) return rc;
    }
    return GQ_OK;
}

int gq_qdense_gated_f32(int type, const float *dX, int64_t M, int64_t K, const gq_rmsnorm *norm, const void *dWgate,
                        const float *dBiasGate, const void *dWup, const float *dBiasUp, int64_t N, int act, float *dY, void *stream) {
    if (int rc = check_dense_args("gq_qdense_gated_f32", type, dX, M, K, dWgate, N, dBiasGate, act, dY, 4)) return rc;
    if (int rc = check_dense_args("gq_qdense_gated_f32", type, dX, M, K, dWup, N, dBiasUp, act, dY, 4)) return rc;
    if (norm && !(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_gated_f32: epsilon must be >= 0");
    if (norm && norm->dGain && !aligned_to(norm->dGain, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_gated_f32: gain must be 4-byte aligned");
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBiasGate, dY);
    const bool up = aligned_to(dBiasUp, 16);
    RmsNorm rn{nullptr, 0.f, 0.f};
    if (norm) rn = RmsNorm{norm->dGain, norm->eps, norm->gain_offset};
    const MmqSetItem one{(const uint8_t *)dWgate, N, dBiasGate, act, dY};
    const MmqExtra ex{(const uint8_t *)dWup, dBiasUp, nullptr, norm ? &rn : nullptr};
    if (takes_mmv(type, M, K, N, dX, rn.gain, 2, true) && !y_over_x(dX, false, dY, M, K, N))
        return launch_mmv(type, dX, false, M, K, 1, &one, &ex, (hipStream_t)stream);
    if (fold_into_gemv(type, M, K, N, dX, rn.gain, true, whole, up))
        return launch_gemv_ks_ext(type, dX, false, M, K, norm ? &rn : nullptr, (const uint8_t *)dWgate, dBiasGate, (const uint8_t *)dWup, dBiasUp,
                                  nullptr, N, act, dY, (hipStream_t)stream);
    if (block_takes_two_pass(type, M, K, N, dX, rn.gain, true, whole)) {
        void *ws = nullptr;
        if (int rc = stream_workspace((hipStream_t)stream, gemm_two_pass_block_workspace(type, M, K, N, true), &ws)) return rc;
        return launch_gemm_two_pass_block(type, dX, M, K, norm ? &rn : nullptr, (const uint8_t *)dWgate, dBiasGate, (const uint8_t *)dWup, dBiasUp,
                                          nullptr, N, act, dY, ws, (hipStream_t)stream);
    }
    // (split-K: both matrices against one activation image, which carries the gain; the reduction normalises and forms act(gate) * up)
    if (block_takes_split_k(type, M, K, N, dX, true, whole, up) && (!rn.gain || aligned_to(rn.gain, 16))) {
        const int rc = split_k(type, dX, false, M, K, 1, &one, &ex, (hipStream_t)stream);
        if (!falls_back(rc, whole && up)) return rc;
    }
    // composed: [normalised activations,] act(gate) into the stream's second workspace, up into y, y *= act(gate)
    const size_t xn_bytes = norm ? ((size_t)M * (size_t)K * sizeof(float) + 255) / 256 * 256 : 0;
    void *ws = nullptr;
    if (int rc = stream_workspace((hipStream_t)stream, xn_bytes + (size_t)M * (size_t)N * sizeof(float), &ws, 1)) return rc;
    const float *x = dX;
    if (norm) {
        float *xn = static_cast<float *>(ws);
        if (int rc = launch_rmsnorm(dX, M, K, rn.gain, rn.gain_offset, rn.eps, xn, (hipStream_t)stream)) return rc;
        x = xn;
    }
    if (dense_takes_split_k(type, M, K, N, x, whole, up)) {
        // both matrices against one activation image; the reduction forms act(gate) * up
        const MmqExtra plain{(const uint8_t *)dWup, dBiasUp, nullptr, nullptr};
        const int rc = split_k(type, x, false, M, K, 1, &one, &plain, (hipStream_t)stream);
        if (!falls_back(rc, whole && up)) return rc;
    }
    float *gate = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + xn_bytes);
    if (int rc = gq_qdense_f32(type, x, M, K, dWgate, N, dBiasGate, act, gate, stream)) return rc;
    if (int rc = gq_qdense_f32(type, x, M, K, dWup, N, dBiasUp, GQ_ACT_NONE, dY, stream)) return rc;
    return launch_mul_inplace(dY, gate, M * N, (hipStream_t)stream);
}

// ---- the same callers with bf16 activations: the decode GEMV reads them as they are (widened in registers: exact); the other
// routes get them widened to fp32 in the stream's third workspace ----
namespace {
// fp32 copy of a bf16 [M, K] matrix at `offset` bytes into the widening workspace, whose size the caller has fixed
int widen_into(void *ws, size_t offset, const uint16_t *x, int64_t M, int64_t K, hipStream_t s, const float **out) {
    float *dst = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + offset);
    if (int rc = launch_widen_bf16(x, dst, M * K, s)) return rc;
    *out = dst;
    return GQ_OK;
}
size_t widened_bytes(int64_t M, int64_t K) { return ((size_t)M * (size_t)K * sizeof(float) + 255) & ~(size_t)255; }
}  // namespace

int gq_qdense_block_bf16(int type, const uint16_t *dX, int64_t M, int64_t K, const gq_rmsnorm *norm, const void *dW, int64_t N,
                         const float *dBias, int act, const float *dResidual, float *dY, void *stream) {
    if (!norm && !dResidual) return gq_qdense_bf16(type, dX, M, K, dW, N, dBias, act, dY, stream);
    if (int rc = check_dense_args("gq_qdense_block_bf16", type, dX, M, K, dW, N, dBias, act, dY, 16)) return rc;
    if (norm && !(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_block_bf16: epsilon must be >= 0");
    if (norm && norm->dGain && !aligned_to(norm->dGain, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_block_bf16: gain must be 4-byte aligned");
    if (dResidual && !aligned_to(dResidual, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_block_bf16: residual must be 4-byte aligned");
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBias, dY);
    const RmsNorm rn = norm ? RmsNorm{norm->dGain, norm->eps, norm->gain_offset} : RmsNorm{nullptr, 0.f, 0.f};
    const MmqSetItem one{(const uint8_t *)dW, N, dBias, act, dY};
    const MmqExtra ex{nullptr, nullptr, dResidual, norm ? &rn : nullptr};
    if (takes_mmv(type, M, K, N, dX, rn.gain, 1, true) && !y_over_x(dX, true, dY, M, K, N))
        return launch_mmv(type, dX, true, M, K, 1, &one, &ex, (hipStream_t)stream);
    if (fold_into_gemv(type, M, K, N, reinterpret_cast<const float *>(dX), norm ? norm->dGain : nullptr, false, whole)) {
        return launch_gemv_ks_ext(type, dX, true, M, K, norm ? &rn : nullptr, (const uint8_t *)dW, dBias, nullptr, nullptr, dResidual, N, act, dY,
                                  (hipStream_t)stream);
    }
    {   // the split-K kernels' pre-pass reads bf16 as well (where the fp32 call would take them too)
        const float *xa = reinterpret_cast<const float *>(dX), *gain = norm ? norm->dGain : nullptr;  // (only their alignment is looked at)
        if (!block_takes_two_pass(type, M, K, N, xa, gain, false, whole) && block_takes_split_k(type, M, K, N, xa, false, whole) && (!gain || aligned_to(gain, 16))) {
            const int rc = split_k(type, dX, true, M, K, 1, &one, &ex, (hipStream_t)stream);
            if (!falls_back(rc, whole)) return rc;
        }
    }
    void *ws = nullptr;
    if (int rc = stream_workspace((hipStream_t)stream, widened_bytes(M, K), &ws, kWsWidenSlot)) return rc;
    const float *x32 = nullptr;
    if (int rc = widen_into(ws, 0, dX, M, K, (hipStream_t)stream, &x32)) return rc;
    return gq_qdense_block_f32(type, x32, M, K, norm, dW, N, dBias, act, dResidual, dY, stream);
}

int gq_qdense_gated_bf16(int type, const uint16_t *dX, int64_t M, int64_t K, const gq_rmsnorm *norm, const void *dWgate,
                         const float *dBiasGate, const void *dWup, const float *dBiasUp, int64_t N, int act, float *dY, void *stream) {
    if (int rc = check_dense_args("gq_qdense_gated_bf16", type, dX, M, K, dWgate, N, dBiasGate, act, dY, 16)) return rc;
    if (int rc = check_dense_args("gq_qdense_gated_bf16", type, dX, M, K, dWup, N, dBiasUp, act, dY, 16)) return rc;
    if (norm && !(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_gated_bf16: epsilon must be >= 0");
    if (norm && norm->dGain && !aligned_to(norm->dGain, 4)) return fail(GQ_ERR_INVALID, "gq_qdense_gated_bf16: gain must be 4-byte aligned");
    if (M == 0 || N == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    const bool whole = whole_rows(N, dBiasGate, dY);
    const bool up = aligned_to(dBiasUp, 16);
    const RmsNorm rn = norm ? RmsNorm{norm->dGain, norm->eps, norm->gain_offset} : RmsNorm{nullptr, 0.f, 0.f};
    const MmqSetItem one{(const uint8_t *)dWgate, N, dBiasGate, act, dY};
    const MmqExtra ex{(const uint8_t *)dWup, dBiasUp, nullptr, norm ? &rn : nullptr};
    if (takes_mmv(type, M, K, N, dX, rn.gain, 2, true) && !y_over_x(dX, true, dY, M, K, N))
        return launch_mmv(type, dX, true, M, K, 1, &one, &ex, (hipStream_t)stream);
    if (fold_into_gemv(type, M, K, N, reinterpret_cast<const float *>(dX), norm ? norm->dGain : nullptr, true, whole, up)) {
        return launch_gemv_ks_ext(type, dX, true, M, K, norm ? &rn : nullptr, (const uint8_t *)dWgate, dBiasGate, (const uint8_t *)dWup, dBiasUp, nullptr,
                                  N, act, dY, (hipStream_t)stream);
    }
    {
        const float *xa = reinterpret_cast<const float *>(dX), *gain = norm ? norm->dGain : nullptr;  // (only their alignment is looked at)
        if (!block_takes_two_pass(type, M, K, N, xa, gain, true, whole) && block_takes_split_k(type, M, K, N, xa, true, whole, up) && (!gain || aligned_to(gain, 16))) {
            const int rc = split_k(type, dX, true, M, K, 1, &one, &ex, (hipStream_t)stream);
            if (!falls_back(rc, whole && up)) return rc;
        }
    }
    void *ws = nullptr;
    if (int rc = stream_workspace((hipStream_t)stream, widened_bytes(M, K), &ws, kWsWidenSlot)) return rc;
    const float *x32 = nullptr;
    if (int rc = widen_into(ws, 0, dX, M, K, (hipStream_t)stream, &x32)) return rc;
    return gq_qdense_gated_f32(type, x32, M, K, norm, dWgate, dBiasGate, dWup, dBiasUp, N, act, dY, stream);
}

int gq_qdense_norm_bf16_batch(int count, const gq_dense_desc *descs, const gq_rmsnorm *norm, void *stream) {
    if (count < 0 || (count > 0 && !descs)) return fail(GQ_ERR_INVALID, "gq_qdense_norm_bf16_batch: bad descriptor list");
    if (count > 64) return fail(GQ_ERR_NOT_IMPLEMENTED, "gq_qdense_norm_bf16_batch: more than 64 problems in one submission");
    for (int i = 0; i < count; i++) {
        const gq_dense_desc &d = descs[i];
        if (int rc = check_dense_args("gq_qdense_norm_bf16_batch", d.type, d.dX, d.M, d.K, d.dW, d.N, d.dBias, d.act, d.dY, 16)) return rc;
    }
    if (norm && !(norm->eps >= 0.f)) return fail(GQ_ERR_INVALID, "gq_qdense_norm_bf16_batch: epsilon must be >= 0");
    if (count == 0) return GQ_OK;
    if (int rc = use_device()) return rc;
    CallScope scope;
    if (norm && count <= 8) {  // the list as one launch of the decode GEMV, on the bf16 data as it is
        MmqSetItem set[4];
        const RmsNorm rn{norm->dGain, norm->eps, norm->gain_offset};
        const MmqExtra ex{nullptr, nullptr, nullptr, &rn};
        if (set_takes_mmv(count, descs, norm->dGain, true, set))
            return launch_mmv(descs[0].type, descs[0].dX, true, descs[0].M, descs[0].K, count, set, &ex, (hipStream_t)stream);
        const bool shared_pass = takes_shared_pass(count, descs, norm->dGain, set);
        XsBatchItem items[8];
        if (merges_into_gemv(count, descs, norm, shared_pass, items))
            return launch_gemv_ks_batch_norm(descs[0].type, count, items, &rn, (hipStream_t)stream, (int)descs[0].M, true);
        if (shared_pass) {
            const int rc = split_k(descs[0].type, descs[0].dX, true, descs[0].M, descs[0].K, count, set, &ex, (hipStream_t)stream);
            if (!falls_back(rc, whole_set(count, set))) return rc;
        }
    }
    // every distinct activation matrix (q / k / v share theirs) is widened once
    gq_dense_desc wide[64];
    size_t offset[64], total = 0;
    int first[64];
    for (int i = 0; i < count; i++) {
        first[i] = -1;  // an empty problem (no rows or no columns) reads no activations: it neither gets nor lends a widened copy
        if (descs[i].M == 0 || descs[i].N == 0) continue;
        first[i] = i;
        for (int j = 0; j < i; j++)
            if (first[j] >= 0 && descs[j].dX == descs[i].dX && descs[j].M == descs[i].M && descs[j].K == descs[i].K) { first[i] = first[j]; break; }
        if (first[i] == i) { offset[i] = total; total += widened_bytes(descs[i].M, descs[i].K); }
    }
    void *ws = nullptr;
    if (total)
        if (int rc = stream_workspace((hipStream_t)stream, total, &ws, kWsWidenSlot)) return rc;
    for (int i = 0; i < count; i++) {
        wide[i] = descs[i];
        if (first[i] < 0) continue;
        if (first[i] == i) {
            const float *x32 = nullptr;
            if (int rc = widen_into(ws, offset[i], reinterpret_cast<const uint16_t *>(descs[i].dX), descs[i].M, descs[i].K, (hipStream_t)stream, &x32)) return rc;
            wide[i].dX = x32;
        } else {
            wide[i].dX = wide[first[i]].dX;
        }
    }
    return gq_qdense_norm_f32_batch(count, wide, norm, stream);
}

int gq_embedding_lookup(int type, const void *dTable, int64_t vocab, int64_t K, const int32_t *dIndices,
                        int64_t count, float *dOut, int32_t *dErrFlag, void *stream) {
    TypeInfo ti;
    if (!type_info(type, ti)) return fail(GQ_ERR_NOT_IMPLEMENTED, "gq_embedding_lookup: ggml type %d is not implemented", type);
    if (vocab < 0 || count < 0) return fail(GQ_ERR_INVALID, "gq_embedding_lookup: negative size");
    if (K <= 0 || K % ti.vpb != 0)
        return fail(GQ_ERR_INVALID, "gq_embedding_lookup: K=%lld is not a positive multiple of the block size %d", (long long)K, ti.vpb);
    if (count == 0) return GQ_OK;
    if (vocab == 0) return fail(GQ_ERR_INVALID, "gq_embedding_lookup: empty table with %lld indices", (long long)count);
    if (!dTable || !dIndices || !dOut) return fail(GQ_ERR_INVALID, "gq_embedding_lookup: null device pointer");
    if (!aligned_to(dTable, 16) || !aligned_to(dOut, 16) || !aligned_to(dIndices, 4))
        return fail(GQ_ERR_INVALID, "gq_embedding_lookup: table and output must be 16-byte aligned");
    if (int rc = use_device()) return rc;
    return launch_embedding_lookup(type, (const uint8_t *)dTable, vocab, K, dIndices, count, dOut, dErrFlag,
                                   (hipStream_t)stream);
}

int gq_graph_begin(void *stream) {
    if (!stream) return fail(GQ_ERR_INVALID, "gq_graph_begin: recording needs an explicit stream");
    if (profile_state().active) return fail(GQ_ERR_INVALID, "gq_graph_begin: kernel timing is active on this thread");
    if (int rc = use_device()) return rc;
    pool().begin_recording(stream);
    GQ_HIP(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeThreadLocal));
    return GQ_OK;
}

int gq_graph_end(void *stream, void **graph_exec) {
    if (!stream || !graph_exec) return fail(GQ_ERR_INVALID, "gq_graph_end: null argument");
    *graph_exec = nullptr;
    if (int rc = use_device()) return rc;
    hipGraph_t graph = nullptr;
    const hipError_t ce = hipStreamEndCapture((hipStream_t)stream, &graph);
    std::vector<WsBlockRef> blocks = pool().end_recording(stream);  // the workspaces the recorded launches point at
    if (ce != hipSuccess) { pool().unpin(blocks); return hip_fail(ce, "hipStreamEndCapture"); }
    hipGraphExec_t exec = nullptr;
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) { pool().unpin(blocks); return hip_fail(e, "hipGraphInstantiate"); }
    RecordedGraph *g = new (std::nothrow) RecordedGraph;
    if (!g) { (void)hipGraphExecDestroy(exec); pool().unpin(blocks); return fail(GQ_ERR_OOM, "gq_graph_end: out of host memory"); }
    g->exec = exec;
    g->stream = (hipStream_t)stream;
    g->blocks.swap(blocks);
    *graph_exec = g;
    return GQ_OK;
}

int gq_graph_launch(void *graph_exec, void *stream) {
    if (!graph_exec) return fail(GQ_ERR_INVALID, "gq_graph_launch: null graph");
    RecordedGraph *g = static_cast<RecordedGraph *>(graph_exec);
    // The recorded launches point at the recording stream's workspace, which eager calls on that stream share in
    // stream order: a replay on another stream would run unordered against them.
    if ((hipStream_t)stream != g->stream)
        return fail(GQ_ERR_INVALID, "gq_graph_launch: a graph replays on the stream it was recorded on");
    if (int rc = use_device()) return rc;
    // (replays and eager sequences that share the workspace must not interleave their submissions)
    WsStreamRef st = pool().stream(stream);
    std::lock_guard<std::recursive_mutex> seq(st->seq);
    GQ_HIP(hipGraphLaunch(g->exec, g->stream));
    return GQ_OK;
}

int gq_graph_destroy(void *graph_exec) {
    if (!graph_exec) return GQ_OK;
    if (int rc = use_device()) return rc;
    RecordedGraph *g = static_cast<RecordedGraph *>(graph_exec);
    const hipError_t e = hipGraphExecDestroy(g->exec);
    pool().unpin(g->blocks);
    delete g;
    if (e != hipSuccess) return hip_fail(e, "hipGraphExecDestroy");
    return GQ_OK;
}

int gq_profile_begin(void) {
    ProfileState &ps = profile_state();
    if (ps.active) return fail(GQ_ERR_INVALID, "gq_profile_begin: already active on this thread");
    if (int rc = use_device()) return rc;
    ps.active = true;
    ps.events.clear();
    return GQ_OK;
}

int gq_profile_end(int *launches, double *total_us) {
    ProfileState &ps = profile_state();
    if (!ps.active) return fail(GQ_ERR_INVALID, "gq_profile_end: timing is not active on this thread");
    ps.active = false;
    int rc = use_device();
    double total = 0.0;
    int n = 0;
    for (size_t i = 0; i + 1 < ps.events.size(); i += 2) {
        if (rc == GQ_OK) {
            float ms = 0.f;
            hipError_t e = hipEventSynchronize(ps.events[i + 1]);
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, ps.events[i], ps.events[i + 1]);
            if (e != hipSuccess) rc = hip_fail(e, "hipEventElapsedTime");
            else { total += (double)ms * 1000.0; n++; }
        }
        (void)hipEventDestroy(ps.events[i]);
        (void)hipEventDestroy(ps.events[i + 1]);
    }
    ps.events.clear();
    if (launches) *launches = n;
    if (total_us) *total_us = total;
    return rc;
}

int gq_workspace_stats(size_t *live_bytes, int *streams) {
    if (live_bytes) *live_bytes = pool().live_bytes();
    if (streams) *streams = (int)pool().stream_count();
    return GQ_OK;
}

const char *gq_last_error(void) { return g_error; }

}  // extern "C"
