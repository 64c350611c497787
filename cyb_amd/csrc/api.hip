// api.hip - the C ABI declared in include/cybq.h: argument checking, device
// memory ownership, dispatch to the kernels.  No torch, no C++ types cross
// this boundary.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/cybq.h"
#include "cybq_debug.h"
#include "cybq_internal.h"
#include "pool.h"
#include "upload.h"

struct cybq_ctx {
    int device = 0;
    int num_cus = 0;
    bool prefill_exact = false;
    bool decode_exact = false;
    void* workspace = nullptr;          // scratch for the prefill path, allocated once at init
    size_t workspace_bytes = 0;
    std::string last_error;
    cybq::Uploader uploader;            // host memory -> native tiles; idle until the first upload
};

struct cybq_weight {
    int device = 0;
    int bits = 0;
    int64_t N = 0, K = 0;
    int NT = 0, KT = 0;
    uint8_t* data = nullptr;            // native tiles (q words + scales per tile), strip-major
    size_t bytes = 0, block = 0;        // of the tiles; of the pool's block behind them
    std::atomic<int> used_on{cybq::kUnused};        // streams that may still be reading `data` (pool.h)
    bool paired = false;                // made by cybq_weight_fuse_pairs: strips alternate gate / up
    // some |scale| * qmax exceeds what f16 holds: the prefill kernels, which form scale * q in
    // f16, would overflow; such a tensor takes the decode kernels (scale applied in fp32) for any M
    bool wide_scales = false;
    // cybq_weight_from_device: the repack kernel stores "some scale is wide" into a pinned word; the first call that
    // needs the answer waits for the kernel (long since complete in practice) and moves it into wide_scales
    cybq::ScanSlot scan;
    std::mutex scan_mutex;
    std::atomic<bool> scan_read{false};
};

namespace cybq {

namespace {
struct LdsEntry {
    const void* kernel;
    int bytes;
};
std::vector<LdsEntry>& lds_requests()
{
    static std::vector<LdsEntry> list;        // built on first use: registrations come from static initialisers
    return list;
}
}  // namespace

void register_lds_request(const void* kernel, int bytes) { lds_requests().push_back({kernel, bytes}); }

hipError_t raise_all_lds_limits()
{
    for (const LdsEntry& r : lds_requests()) {
        hipError_t e = hipFuncSetAttribute(r.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, r.bytes);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace cybq

namespace {

// Scratch of cybq_matmul_static, the entry point that allocates nothing: the prefill path's
// staging area and K-split slabs live in this array instead of a hipMalloc'ed workspace.
// Every device the library runs on holds its own copy at its own address until the process
// ends; the name below is only the host-side handle of the symbol, never a device address:
// cybq_init asks the runtime for the address on its device and kernels receive that pointer.
constexpr size_t kStaticScratchBytes = (size_t)64 << 20;
constexpr int64_t kStaticMaxK = 32768;          // 256 staged rows of 2-byte activations fit half the scratch with room to spare
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
void* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mutex;              // contexts may be created from several threads

// (no memory for the text: the code alone)
int fail(cybq_ctx* ctx, int code, const char* what)
{
    try {
        if (ctx) ctx->last_error = what ? what : "";
    } catch (const std::bad_alloc&) {
        ctx->last_error.clear();
    }
    return code;
}

int fail_hip(cybq_ctx* ctx, hipError_t e, const char* where)
{
    try {
        if (ctx) ctx->last_error = std::string(where) + ": " + hipGetErrorString(e);
    } catch (const std::bad_alloc&) {
        ctx->last_error.clear();
    }
    (void)hipGetLastError();   // clear the sticky error so the next call starts clean
    return e == hipErrorOutOfMemory ? CYBQ_ERR_NOMEM : CYBQ_ERR_HIP;
}

// The device is made current for every call: contexts may live on different
// devices inside one process.
struct DeviceGuard {
    hipError_t err;
    // (asking for the current device is a thread-local read; setting it again is not free, and a decode
    // launch is a few microseconds of host time in all)
    explicit DeviceGuard(int device)
    {
        int cur = -1;
        err = hipGetDevice(&cur);
        if (err != hipSuccess || cur != device) err = hipSetDevice(device);
    }
};

cybq::WeightView view_of(const cybq_weight* w)
{
    cybq::WeightView v;
    v.base = w->data;
    v.N = (int)w->N;
    v.K = (int)w->K;
    v.NT = w->NT;
    v.KT = w->KT;
    v.bits = w->bits;
    return v;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

size_t dtype_size(int dt) { return dt == CYBQ_F32 ? 4 : 2; }
bool dtype_ok(int dt) { return dt == CYBQ_F32 || dt == CYBQ_F16 || dt == CYBQ_BF16; }

// work that reads the weight has been queued on `stream`
void mark_use(const cybq_weight* cw, const void* stream)
{
    cybq_weight* w = const_cast<cybq_weight*>(cw);
    const int where = stream ? cybq::kElsewhere : cybq::kDefaultStream;
    int seen = w->used_on.load(std::memory_order_relaxed);
    while (seen < where && !w->used_on.compare_exchange_weak(seen, where, std::memory_order_relaxed)) {
    }
}

int alloc_weight(cybq_ctx* ctx, int bits, int64_t N, int64_t K, cybq::UsedOn first_use, cybq_weight** out)
{
    cybq_weight* w = new (std::nothrow) cybq_weight();
    if (!w) return fail(ctx, CYBQ_ERR_NOMEM, "host allocation failed");
    w->device = ctx->device;
    w->bits = bits;
    w->N = N;
    w->K = K;
    w->NT = (int)((N + cybq::kTileN - 1) / cybq::kTileN);
    w->KT = (int)((K + cybq::kTileK - 1) / cybq::kTileK);
    w->bytes = (size_t)w->NT * w->KT * cybq::tile_bytes(bits);
    hipError_t e = cybq::pool_alloc(ctx->device, w->bytes, first_use, reinterpret_cast<void**>(&w->data), &w->block);
    if (e != hipSuccess) {
        delete w;
        return fail_hip(ctx, e, "hipMalloc(weight)");
    }
    *out = w;
    return CYBQ_OK;
}

void release_weight(cybq_weight* w)
{
    cybq::scan_release(w->device, w->scan);
    cybq::pool_free(w->device, w->data, w->block, static_cast<cybq::UsedOn>(w->used_on.load(std::memory_order_relaxed)));
    delete w;
}

// wide_scales of a weight whose scales were scanned on the device: the answer is taken the first time it is needed.  A wait that
// fails leaves the question open: no kernel is chosen by an answer that never came.
hipError_t weight_is_wide(const cybq_weight* cw, bool* wide)
{
    cybq_weight* w = const_cast<cybq_weight*>(cw);
    if (w->scan.word && !w->scan_read.load(std::memory_order_acquire)) {
        std::lock_guard<std::mutex> lock(w->scan_mutex);
        if (!w->scan_read.load(std::memory_order_relaxed)) {
            const hipError_t e = hipEventSynchronize(w->scan.done);
            if (e != hipSuccess) return e;
            w->wide_scales = *w->scan.word != 0u;
            w->scan_read.store(true, std::memory_order_release);
        }
    }
    *wide = w->wide_scales;
    return hipSuccess;
}

int check_weight_shape(cybq_ctx* ctx, int quant, int64_t N, int64_t K)
{
    if (quant != CYBQ_Q4 && quant != CYBQ_Q8) return fail(ctx, CYBQ_ERR_INVALID, "quant must be CYBQ_Q4 or CYBQ_Q8");
    if (N < 1 || K < 1) return fail(ctx, CYBQ_ERR_SHAPE, "N and K must be >= 1");
    if (K % CYBQ_GROUP) return fail(ctx, CYBQ_ERR_SHAPE, "K must be a multiple of 32");
    if (N > (int64_t)1 << 30 || K > (int64_t)1 << 30 || N * K > (int64_t)1 << 40)
        return fail(ctx, CYBQ_ERR_SHAPE, "tensor too large");
    return CYBQ_OK;
}

}  // namespace

extern "C" {

const char* cybq_version(void) { return "0.1.0"; }

const char* cybq_strerror(int status)
{
    switch (status) {
        case CYBQ_OK: return "ok";
        case CYBQ_ERR_INVALID: return "invalid argument";
        case CYBQ_ERR_SHAPE: return "bad shape";
        case CYBQ_ERR_ALIGN: return "misaligned pointer";
        case CYBQ_ERR_NO_DEVICE: return "no usable gfx950 device";
        case CYBQ_ERR_HIP: return "HIP runtime error";
        case CYBQ_ERR_NOMEM: return "out of memory";
        case CYBQ_ERR_UNSUPPORTED: return "unsupported";
        default: return "unknown status";
    }
}

const char* cybq_last_error(const cybq_ctx* ctx) { return ctx ? ctx->last_error.c_str() : ""; }

int cybq_init(int device, cybq_ctx** out)
{
    if (!out) return CYBQ_ERR_INVALID;
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count < 1) { (void)hipGetLastError(); return CYBQ_ERR_NO_DEVICE; }
    if (device < 0 || device >= count) return CYBQ_ERR_INVALID;
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) { (void)hipGetLastError(); return CYBQ_ERR_NO_DEVICE; }
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return CYBQ_ERR_NO_DEVICE;
    e = hipSetDevice(device);
    if (e != hipSuccess) { (void)hipGetLastError(); return CYBQ_ERR_HIP; }
    // every kernel that wants more than the default dynamic LDS gets its limit raised now, for
    // this device: launches never touch function attributes
    e = cybq::raise_all_lds_limits();
    if (e != hipSuccess) { (void)hipGetLastError(); return CYBQ_ERR_HIP; }
    if (device < kMaxDevices) {       // this device's copy of the static scratch
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        if (!g_scratch_ptr[device]) {
            void* p = nullptr;
            e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !p) { (void)hipGetLastError(); return CYBQ_ERR_HIP; }
            g_scratch_ptr[device] = p;
        }
    }
    cybq_ctx* ctx = new (std::nothrow) cybq_ctx();
    if (!ctx) return CYBQ_ERR_NOMEM;
    ctx->device = device;
    ctx->num_cus = prop.multiProcessorCount;
    // 256 MiB of scratch for the prefill path: the activations restaged in MFMA operand
    // order (larger M is walked in row chunks) and the partial sums of a K split
    ctx->workspace_bytes = (size_t)256 << 20;
    if (hipMalloc(&ctx->workspace, ctx->workspace_bytes) != hipSuccess) {
        (void)hipGetLastError();
        delete ctx;
        return CYBQ_ERR_NOMEM;
    }
    // the decode kernels' tickets (start of the scratch's tail) are zero at rest
    if (hipMemset(static_cast<char*>(ctx->workspace) + ctx->workspace_bytes - cybq::kDecodeScratchBytes, 0, (size_t)1 << 16) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(ctx->workspace);
        delete ctx;
        return CYBQ_ERR_HIP;
    }
    if (cybq::pool_retain(device) != hipSuccess) {
        (void)hipFree(ctx->workspace);
        delete ctx;
        return CYBQ_ERR_NOMEM;
    }
    *out = ctx;
    return CYBQ_OK;
}

void cybq_destroy(cybq_ctx* ctx)
{
    if (!ctx) return;
    const int device = ctx->device;
    if (hipSetDevice(device) == hipSuccess && ctx->workspace) (void)hipFree(ctx->workspace);
    delete ctx;
    cybq::pool_release(device);
}

int cybq_weight_upload_many(cybq_ctx* ctx, int64_t count, const int* quant, const int* layout, const int64_t* N, const int64_t* K,
                            const void* const* q, const void* const* scales, cybq_weight** out)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && (!quant || !layout || !N || !K || !q || !out))) return fail(ctx, CYBQ_ERR_INVALID, "bad tensor list");
    for (int64_t i = 0; i < count; i++) out[i] = nullptr;
    for (int64_t i = 0; i < count; i++) {
        const void* s = scales ? scales[i] : nullptr;
        if (!q[i]) return fail(ctx, CYBQ_ERR_INVALID, "q is NULL");
        if (layout[i] != CYBQ_LAYOUT_PLANAR && layout[i] != CYBQ_LAYOUT_BLOCK_AOS)
            return fail(ctx, CYBQ_ERR_INVALID, "unknown layout");
        if (layout[i] == CYBQ_LAYOUT_PLANAR && !s) return fail(ctx, CYBQ_ERR_INVALID, "PLANAR needs a scale plane");
        if (layout[i] == CYBQ_LAYOUT_BLOCK_AOS && s) return fail(ctx, CYBQ_ERR_INVALID, "BLOCK_AOS carries its scales; pass NULL");
        int rc = check_weight_shape(ctx, quant[i], N[i], K[i]);
        if (rc) return rc;
    }
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    int rc = CYBQ_OK;
    try {
        std::vector<cybq::UploadItem> items((size_t)count);
        for (int64_t i = 0; i < count && rc == CYBQ_OK; i++) {
            rc = alloc_weight(ctx, quant[i], N[i], K[i], cybq::kElsewhere, &out[i]);
            if (rc) break;
            cybq::UploadItem& it = items[(size_t)i];
            it.quant = quant[i];
            it.layout = layout[i];
            it.N = N[i];
            it.K = K[i];
            it.q = q[i];
            it.scales = scales ? scales[i] : nullptr;
            it.dst = out[i]->data;
            it.NT = out[i]->NT;
            it.KT = out[i]->KT;
        }
        if (rc == CYBQ_OK && count) {
            const hipError_t e = ctx->uploader.run(items.data(), count);
            if (e != hipSuccess) rc = fail_hip(ctx, e, "weight upload");
            for (int64_t i = 0; i < count; i++) out[i]->wide_scales = items[(size_t)i].wide;
        }
    } catch (const std::bad_alloc&) {
        rc = fail(ctx, CYBQ_ERR_NOMEM, "host allocation failed");
    }
    if (rc)
        for (int64_t i = 0; i < count; i++)
            if (out[i]) {
                release_weight(out[i]);
                out[i] = nullptr;
            }
    return rc;
}

int cybq_weight_upload(cybq_ctx* ctx, cybq_quant quant, cybq_layout layout, int64_t N, int64_t K,
                       const void* q, const void* scales, cybq_weight** out)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!out) return fail(ctx, CYBQ_ERR_INVALID, "out is NULL");
    const int quant_code = quant, layout_code = layout;
    return cybq_weight_upload_many(ctx, 1, &quant_code, &layout_code, &N, &K, &q, &scales, out);
}

int cybq_weight_from_device(cybq_ctx* ctx, cybq_quant quant, int64_t N, int64_t K, const void* q_dev,
                            const void* scales_dev, void* stream, cybq_weight** out)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!out) return fail(ctx, CYBQ_ERR_INVALID, "out is NULL");
    *out = nullptr;
    if (!q_dev || !scales_dev) return fail(ctx, CYBQ_ERR_INVALID, "q_dev / scales_dev is NULL");
    if (reinterpret_cast<uintptr_t>(q_dev) % 4 || reinterpret_cast<uintptr_t>(scales_dev) % 2)
        return fail(ctx, CYBQ_ERR_ALIGN, "q_dev must be 4-byte and scales_dev 2-byte aligned");
    int rc = check_weight_shape(ctx, quant, N, K);
    if (rc) return rc;
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // A recorded repack has not run when the call returns and would run again with every replay, into memory that a free hands
    // on; with a pooled block nothing below would refuse it.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &capture);
    if (e != hipSuccess) return fail_hip(ctx, e, "hipStreamIsCapturing");
    if (capture != hipStreamCaptureStatusNone) return fail(ctx, CYBQ_ERR_UNSUPPORTED, "cybq_weight_from_device: the stream is being captured");
    cybq_weight* w = nullptr;
    rc = alloc_weight(ctx, quant, N, K, stream ? cybq::kElsewhere : cybq::kDefaultStream, &w);
    if (rc) return rc;
    // the scales are scanned by the repack kernel itself: it stores 1 into a pinned word where "some |scale| * qmax leaves
    // f16", and the first call that needs the word waits for the event behind the kernel
    e = cybq::scan_acquire(ctx->device, &w->scan);
    if (e == hipSuccess) {
        *w->scan.word = 0u;
        e = cybq::launch_repack(quant, CYBQ_LAYOUT_PLANAR, false, q_dev, scales_dev, w->data, (int)N, (int)K, w->NT, w->KT, w->scan.word, st);
    }
    if (e == hipSuccess) e = hipEventRecord(w->scan.done, st);
    mark_use(w, stream);
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(st);          // nothing may still write the pinned word
        release_weight(w);
        return fail_hip(ctx, e, "repack launch");
    }
    *out = w;
    return CYBQ_OK;
}

int cybq_weight_clone(cybq_ctx* ctx, const cybq_weight* src, cybq_weight** out)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!src || !out) return fail(ctx, CYBQ_ERR_INVALID, "src / out is NULL");
    *out = nullptr;
    if (src->device != ctx->device) return fail(ctx, CYBQ_ERR_INVALID, "weight lives on another device");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    cybq_weight* w = nullptr;
    int rc = alloc_weight(ctx, src->bits, src->N, src->K, cybq::kDefaultStream, &w);
    if (rc == CYBQ_OK) {
        mark_use(w, nullptr);
        mark_use(src, nullptr);
    }
    if (rc) return rc;
    hipError_t e = hipMemcpy(w->data, src->data, src->bytes, hipMemcpyDeviceToDevice);
    if (e == hipSuccess) e = weight_is_wide(src, &w->wide_scales);
    if (e != hipSuccess) {
        release_weight(w);
        return fail_hip(ctx, e, "weight clone");
    }
    w->paired = src->paired;
    *out = w;
    return CYBQ_OK;
}

int cybq_weight_free(cybq_ctx* ctx, cybq_weight* w)
{
    if (!w) return CYBQ_OK;
    const hipError_t e = hipSetDevice(w->device);
    if (e != hipSuccess) {
        delete w;
        return fail_hip(ctx, e, "hipSetDevice");
    }
    release_weight(w);
    return CYBQ_OK;
}

int cybq_trim(cybq_ctx* ctx)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    const hipError_t e = cybq::pool_trim(ctx->device);
    if (e != hipSuccess) return fail_hip(ctx, e, "hipFree");
    return CYBQ_OK;
}

int cybq_weight_info(const cybq_weight* w, int* quant, int64_t* N, int64_t* K, int64_t* device_bytes)
{
    if (!w) return CYBQ_ERR_INVALID;
    if (quant) *quant = w->bits;
    if (N) *N = w->N;
    if (K) *K = w->K;
    if (device_bytes) *device_bytes = (int64_t)w->bytes;
    return CYBQ_OK;
}

namespace {
int matmul_fused(cybq_ctx* ctx, const cybq_weight* w, const void* x, cybq_dtype xdt, int64_t M, const void* gamma,
                 cybq_dtype gdt, float eps, void* y, cybq_dtype ydt, cybq_epilogue epilogue, const void* residual,
                 void* stream, void* workspace, size_t workspace_bytes)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!w || !x || !y) return fail(ctx, CYBQ_ERR_INVALID, "w / x / y is NULL");
    if (!dtype_ok(xdt) || !dtype_ok(ydt)) return fail(ctx, CYBQ_ERR_INVALID, "unknown dtype");
    if (M < 1 || M > (1 << 24)) return fail(ctx, CYBQ_ERR_SHAPE, "M must be in 1..2^24");
    if (w->device != ctx->device) return fail(ctx, CYBQ_ERR_INVALID, "weight lives on another device");
    if (!aligned16(x)) return fail(ctx, CYBQ_ERR_ALIGN, "x must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(y) % dtype_size(ydt)) return fail(ctx, CYBQ_ERR_ALIGN, "y is not aligned to its element size");
    cybq::Epilogue epi = {cybq::kEpiNone, nullptr, nullptr, 0, 0.f};
    if (gamma) {
        if (!dtype_ok(gdt)) return fail(ctx, CYBQ_ERR_INVALID, "unknown gamma dtype");
        if (!aligned16(gamma)) return fail(ctx, CYBQ_ERR_ALIGN, "gamma must be 16-byte aligned");
        if (!(eps >= 0.f)) return fail(ctx, CYBQ_ERR_INVALID, "eps must be >= 0");
    }
    if (epilogue == CYBQ_EPI_ADD) {
        if (!residual) return fail(ctx, CYBQ_ERR_INVALID, "CYBQ_EPI_ADD needs a residual");
        if (reinterpret_cast<uintptr_t>(residual) % dtype_size(ydt)) return fail(ctx, CYBQ_ERR_ALIGN, "residual is not aligned to its element size");
        epi.kind = cybq::kEpiAdd;
        epi.residual = residual;
    } else if (epilogue == CYBQ_EPI_SWIGLU) {
        if (!w->paired) return fail(ctx, CYBQ_ERR_INVALID, "CYBQ_EPI_SWIGLU needs a weight made by cybq_weight_fuse_pairs");
        epi.kind = cybq::kEpiSwiglu;
    } else if (epilogue != CYBQ_EPI_NONE) {
        return fail(ctx, CYBQ_ERR_INVALID, "unknown epilogue");
    }
    epi.gamma = gamma;
    epi.gamma_dt = (int)gdt;
    epi.eps = eps;
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    hipStream_t st = static_cast<hipStream_t>(stream);
    cybq::WeightView v = view_of(w);
    hipError_t e = hipSuccess;
    // (asked only where the way of the call hangs on it: the first time it is a wait)
    auto wide = [&]() {
        bool is = false;
        if (e == hipSuccess) e = weight_is_wide(w, &is);
        return is;
    };
    // the tail of the scratch belongs to the decode kernels (tickets and slabs of a K split), the rest to prefill
    const bool split = workspace && workspace_bytes > 2 * cybq::kDecodeScratchBytes;
    const size_t prefill_bytes = !workspace ? 0 : split ? workspace_bytes - cybq::kDecodeScratchBytes : workspace_bytes;
    void* const dscr = split ? static_cast<char*>(workspace) + prefill_bytes : nullptr;
    const size_t dscr_bytes = split ? cybq::kDecodeScratchBytes : 0;
    enum { kDecode, kTwoPasses, kPrefill, kPrefillExact, kWalk } way;
    if (M <= 16 || (M <= 32 && cybq::gemv_serves_32(v, (int)xdt, (int)M, ctx->num_cus, epi)))
        way = kDecode;
    else if (M <= 64 && (int64_t)w->N * w->K <= (int64_t)6144 * 4096 && cybq::gemv_serves_32(v, (int)xdt, 32, ctx->num_cus, epi) &&
             (ctx->prefill_exact || wide() || !cybq::gemm_rows_takes(v, (int)M, ctx->num_cus, epi)))
        // (in FAST mode, where the line above has asked whether the scales are wide: EXACT calls of these rows never did, and their first one on
        // a weight from device memory may sit in a capture, where the answer cannot be waited for)
        way = (M > 32 && w->bits == 4 && xdt == CYBQ_BF16 && (w->K > 4096 || (w->K <= 512 && w->N >= 6144)) && !ctx->prefill_exact && !wide() &&
               cybq::gemm_stages(v, prefill_bytes)) ? kPrefillExact : kTwoPasses;
    else if (!wide() && (xdt == CYBQ_F32 ? !ctx->prefill_exact : (M > 32 || (!ctx->prefill_exact && cybq::gemm_rows_takes(v, (int)M, ctx->num_cus, epi)))))
        way = kPrefill;
    else
        way = kWalk;
    if (e != hipSuccess) return fail_hip(ctx, e, "scale scan");
    mark_use(w, stream);
    if (way == kDecode) {
        e = cybq::launch_gemv(v, x, xdt, (int)M, y, ydt, ctx->num_cus, ctx->decode_exact, epi, dscr, dscr_bytes, st);
    } else if (way == kTwoPasses) {
        // 33..64 rows on a small weight (up to 4096 -> 6144) that the few-rows MFMA kernel does not take (exact mode, wide scales, K outside 2048 ..
        // 8192): two passes of the batched-rows decode kernel (32 rows, then the rest), which stream the weights twice.  The line was drawn when
        // the prefill path had a staging launch and two MFMAs per group in EXACT mode.  With integer operands and rows read in place two passes
        // are the quicker way on the first of the shapes below alone (on Q8 they are even).  us per call, two passes / prefill path with
        // exact operands, at 33, 48, 64 rows.  bf16 on Q4: 2048 -> 6144 9.5, 9.5, 11.3 / 10.7, 11.2, 12.0; 4096 -> 4096 11.6, 12.5, 14.6 / 11.3, 12.0,
        // 13.1; 1024 -> 4096 7.9, 8.7, 10.4 / 7.1, 7.1, 7.5; 4096 -> 1024 10.2, 11.0, 12.7 / 8.0, 8.3, 8.7; 768 -> 9167 11.8, 14.4, 17.4 / 7.2, 7.4, 7.8.
        // f16 on Q4: 12576 -> 281 25.1, 29.8, 37.1 / 11.4, 11.8, 12.7; 512 -> 14336 12.5, 16.0, 18.0 / 5.8, 5.9, 6.3.  Q8 (bf16): 2048 -> 6144 11.3, 11.4, 12.9 /
        // 11.3, 12.0, 12.6; 14336 -> 1024 31.6, 36.9, 44.2 / 13.2, 13.8, 14.8.  Relative L2 against float64, same calls: f16 6e-8 - 1.5e-7 / 6e-8 - 1.2e-7,
        // bf16 on Q4 2.6e-7 - 5.1e-7 / 6e-8 - 1.1e-7, on Q8 7e-8 - 1.5e-7 / 6e-8 - 1.2e-7.  Moved so far: in FAST mode bf16 rows on Q4 with K over 4096 or of
        // up to 512 on 6144 columns and more (kPrefillExact: 8192 -> 512 15.9, 17.9, 21.6 / 9.6, 9.8, 10.2; 14336 -> 1024 26.6, 31.4, 38.9 / 12.6, 13.2, 14.2;
        // 512 -> 14336 12.3, 16.0, 18.0 / 6.4, 6.6, 6.9), unless K is so long (251 936 and more) that the scratch does not hold 256 staged rows.
        // (a context in CYBQ_PREFILL_EXACT mode asked for exact operands at this row count)
        const bool exact_ops = ctx->decode_exact || ctx->prefill_exact;
        const int64_t n_out = epi.kind == cybq::kEpiSwiglu ? w->N / 2 : w->N;
        const size_t yoff = (size_t)32 * n_out * dtype_size(ydt);
        cybq::Epilogue ec = epi;
        if (epi.kind == cybq::kEpiAdd) ec.residual = static_cast<const char*>(residual) + yoff;
        e = cybq::launch_gemv(v, x, xdt, 32, y, ydt, ctx->num_cus, exact_ops, epi, dscr, dscr_bytes, st);
        if (e == hipSuccess)
            e = cybq::launch_gemv(v, static_cast<const char*>(x) + (size_t)32 * w->K * dtype_size(xdt), xdt, (int)M - 32,
                                  static_cast<char*>(y) + yoff, ydt, ctx->num_cus, exact_ops, ec, dscr, dscr_bytes, st);
    } else if (way == kPrefill || way == kPrefillExact) {
        e = cybq::launch_gemm(v, x, xdt, (int)M, y, ydt, ctx->num_cus, ctx->prefill_exact || way == kPrefillExact, workspace, prefill_bytes,
                              epi, st);
    } else {
        // fp32 activations keep full precision through the decode kernel's hi/lo split:
        // exact-mode prefill in fp32 is walked 16 rows at a time (FAST mode rounds them to f16
        // in the staging pass and takes the MFMA kernel from 17 rows on: the LDS decode kernel
        // needs 52 - 65 us for 24 - 32 fp32 rows, the few-row MFMA kernel 16).  So are 17..32
        // rows of 16-bit activations with a folded norm where the few-row MFMA kernel does not take
        // them (FAST mode: 4096 -> 14336 at 32 rows 18.1 us there against 23.0 here): two passes of
        // the batched-rows kernel stream the weights twice and are still quicker than a 128-row MFMA
        // tile mostly empty (without the norm they are one pass, two row blocks per weight operand).
        // A tensor with wide scales (scale * q leaves f16) is walked the same way for any M, 32 rows at a
        // time where the batched-rows kernel takes them in one pass: the weights stream once per 32 rows.
        const int64_t n_out = epi.kind == cybq::kEpiSwiglu ? w->N / 2 : w->N;
        const int64_t step = cybq::gemv_serves_32(v, (int)xdt, 32, ctx->num_cus, epi) ? 32 : 16;
        for (int64_t m0 = 0, mm; m0 < M && e == hipSuccess; m0 += mm) {
            mm = (M - m0) < step ? (M - m0) : step;
            // (with a norm one or two fp32 rows have sums of squares in another order than 3 .. 16: none are left over)
            if (xdt == CYBQ_F32 && gamma && M - m0 > step && M - m0 < step + 3) mm = step - 2;
            const char* xp = static_cast<const char*>(x) + (size_t)m0 * w->K * dtype_size(xdt);
            const size_t yoff = (size_t)m0 * n_out * dtype_size(ydt);
            cybq::Epilogue ec = epi;
            if (epi.kind == cybq::kEpiAdd) ec.residual = static_cast<const char*>(residual) + yoff;
            e = cybq::launch_gemv(v, xp, xdt, (int)mm, static_cast<char*>(y) + yoff, ydt, ctx->num_cus, ctx->decode_exact, ec, dscr, dscr_bytes, st);
        }
    }
    if (e != hipSuccess) return fail_hip(ctx, e, "matmul launch");
    return CYBQ_OK;
}
}  // namespace

int cybq_matmul_ex(cybq_ctx* ctx, const cybq_weight* w, const void* x, cybq_dtype xdt, int64_t M, void* y,
                   cybq_dtype ydt, cybq_epilogue epilogue, const void* residual, void* stream)
{
    return matmul_fused(ctx, w, x, xdt, M, nullptr, CYBQ_F32, 0.f, y, ydt, epilogue, residual, stream, ctx ? ctx->workspace : nullptr,
                        ctx ? ctx->workspace_bytes : 0);
}

int cybq_matmul_norm(cybq_ctx* ctx, const cybq_weight* w, const void* x, cybq_dtype xdt, int64_t M, const void* gamma,
                     cybq_dtype gdt, float eps, void* y, cybq_dtype ydt, cybq_epilogue epilogue, const void* residual,
                     void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!gamma) return fail(ctx, CYBQ_ERR_INVALID, "gamma is NULL");
    return matmul_fused(ctx, w, x, xdt, M, gamma, gdt, eps, y, ydt, epilogue, residual, stream, ctx->workspace, ctx->workspace_bytes);
}

int cybq_matmul(cybq_ctx* ctx, const cybq_weight* w, const void* x, cybq_dtype xdt, int64_t M, void* y,
                cybq_dtype ydt, void* stream)
{
    return cybq_matmul_ex(ctx, w, x, xdt, M, y, ydt, CYBQ_EPI_NONE, nullptr, stream);
}

int cybq_matmul_static(cybq_ctx* ctx, const cybq_weight* w, const void* x, cybq_dtype xdt, int64_t M, void* y,
                       cybq_dtype ydt, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    void* static_scratch = nullptr;
    if (ctx->device < kMaxDevices) {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        static_scratch = g_scratch_ptr[ctx->device];
    }
    if (!static_scratch) return fail(ctx, CYBQ_ERR_UNSUPPORTED, "no static scratch on this device");
    if (w && M > 16 && w->K > kStaticMaxK)
        return fail(ctx, CYBQ_ERR_UNSUPPORTED, "cybq_matmul_static: K beyond 32768 does not fit the static scratch for more than 16 rows");
    return matmul_fused(ctx, w, x, xdt, M, nullptr, CYBQ_F32, 0.f, y, ydt, CYBQ_EPI_NONE, nullptr, stream,
                        static_scratch, kStaticScratchBytes);
}

int cybq_weight_fuse_pairs(cybq_ctx* ctx, const cybq_weight* gate, const cybq_weight* up, cybq_weight** out)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!gate || !up || !out) return fail(ctx, CYBQ_ERR_INVALID, "gate / up / out is NULL");
    *out = nullptr;
    if (gate->device != ctx->device || up->device != ctx->device) return fail(ctx, CYBQ_ERR_INVALID, "weight lives on another device");
    if (gate->bits != up->bits || gate->N != up->N || gate->K != up->K) return fail(ctx, CYBQ_ERR_SHAPE, "gate and up differ in quant or shape");
    if (gate->N % cybq::kTileN) return fail(ctx, CYBQ_ERR_SHAPE, "N must be a multiple of 16");
    if (gate->paired || up->paired) return fail(ctx, CYBQ_ERR_INVALID, "inputs are already fused");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    cybq_weight* w = nullptr;
    int rc = alloc_weight(ctx, gate->bits, 2 * gate->N, gate->K, cybq::kDefaultStream, &w);
    if (rc) return rc;
    // the native layout is strip-major: output strip 2i is gate strip i, 2i+1 is up strip i
    const size_t sb = (size_t)gate->KT * cybq::tile_bytes(gate->bits);          // bytes of one strip
    hipError_t e = hipMemcpy2D(w->data, 2 * sb, gate->data, sb, sb, gate->NT, hipMemcpyDeviceToDevice);
    if (e == hipSuccess) e = hipMemcpy2D(w->data + sb, 2 * sb, up->data, sb, sb, up->NT, hipMemcpyDeviceToDevice);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    bool wide_gate = false, wide_up = false;
    if (e == hipSuccess) e = weight_is_wide(gate, &wide_gate);
    if (e == hipSuccess) e = weight_is_wide(up, &wide_up);
    if (e != hipSuccess) {
        release_weight(w);
        return fail_hip(ctx, e, "weight fuse");
    }
    w->paired = true;
    w->wide_scales = wide_gate || wide_up;
    *out = w;
    return CYBQ_OK;
}

int cybq_set_prefill_mode(cybq_ctx* ctx, cybq_prefill_mode mode)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (mode != CYBQ_PREFILL_FAST && mode != CYBQ_PREFILL_EXACT) return fail(ctx, CYBQ_ERR_INVALID, "unknown prefill mode");
    ctx->prefill_exact = mode == CYBQ_PREFILL_EXACT;
    return CYBQ_OK;
}

int cybq_set_decode_mode(cybq_ctx* ctx, cybq_decode_mode mode)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (mode != CYBQ_DECODE_STREAM && mode != CYBQ_DECODE_EXACT) return fail(ctx, CYBQ_ERR_INVALID, "unknown decode mode");
    ctx->decode_exact = mode == CYBQ_DECODE_EXACT;
    return CYBQ_OK;
}

int cybq_matmul_many(cybq_ctx* ctx, int64_t count, const cybq_weight* const* w, const void* const* x,
                     void* const* y, cybq_dtype xdt, int64_t M, cybq_dtype ydt, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && (!w || !x || !y))) return fail(ctx, CYBQ_ERR_INVALID, "bad node list");
    for (int64_t i = 0; i < count; i++) {
        int rc = cybq_matmul(ctx, w[i], x[i], xdt, M, y[i], ydt, stream);
        if (rc) return rc;
    }
    return CYBQ_OK;
}

int cybq_matmul_many_ex(cybq_ctx* ctx, int64_t count, const cybq_weight* const* w, const void* const* x,
                        void* const* y, const int* epilogue, const void* const* residual, cybq_dtype xdt, int64_t M,
                        cybq_dtype ydt, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && (!w || !x || !y))) return fail(ctx, CYBQ_ERR_INVALID, "bad node list");
    for (int64_t i = 0; i < count; i++) {
        const cybq_epilogue e = epilogue ? static_cast<cybq_epilogue>(epilogue[i]) : CYBQ_EPI_NONE;
        int rc = cybq_matmul_ex(ctx, w[i], x[i], xdt, M, y[i], ydt, e, residual ? residual[i] : nullptr, stream);
        if (rc) return rc;
    }
    return CYBQ_OK;
}

int cybq_matmul_many_norm(cybq_ctx* ctx, int64_t count, const cybq_weight* const* w, const void* const* x,
                          const void* const* gamma, cybq_dtype gdt, float eps, void* const* y, const int* epilogue,
                          const void* const* residual, cybq_dtype xdt, int64_t M, cybq_dtype ydt, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && (!w || !x || !y))) return fail(ctx, CYBQ_ERR_INVALID, "bad node list");
    for (int64_t i = 0; i < count; i++) {
        const cybq_epilogue e = epilogue ? static_cast<cybq_epilogue>(epilogue[i]) : CYBQ_EPI_NONE;
        int rc = matmul_fused(ctx, w[i], x[i], xdt, M, gamma ? gamma[i] : nullptr, gdt, eps, y[i], ydt, e,
                              residual ? residual[i] : nullptr, stream, ctx->workspace, ctx->workspace_bytes);
        if (rc) return rc;
    }
    return CYBQ_OK;
}

int cybq_dequant(cybq_ctx* ctx, const cybq_weight* w, float* out, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!w || !out) return fail(ctx, CYBQ_ERR_INVALID, "w / out is NULL");
    if (w->device != ctx->device) return fail(ctx, CYBQ_ERR_INVALID, "weight lives on another device");
    if (!aligned16(out)) return fail(ctx, CYBQ_ERR_ALIGN, "out must be 16-byte aligned");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    mark_use(w, stream);
    hipError_t e = cybq::launch_dequant(view_of(w), out, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail_hip(ctx, e, "dequant launch");
    return CYBQ_OK;
}

int cybq_quantize(cybq_ctx* ctx, cybq_quant quant, const float* src, int64_t N, int64_t K, void* q_out,
                  void* scales_out, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!src || !q_out || !scales_out) return fail(ctx, CYBQ_ERR_INVALID, "src / q_out / scales_out is NULL");
    int rc = check_weight_shape(ctx, quant, N, K);
    if (rc) return rc;
    if (!aligned16(src)) return fail(ctx, CYBQ_ERR_ALIGN, "src must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(q_out) % 4 || reinterpret_cast<uintptr_t>(scales_out) % 2)
        return fail(ctx, CYBQ_ERR_ALIGN, "q_out must be 4-byte and scales_out 2-byte aligned");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    hipError_t e = cybq::launch_quantize(quant, src, (int)N, (int)K, q_out, scales_out, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail_hip(ctx, e, "quantize launch");
    return CYBQ_OK;
}

/* ---- diagnostics declared in cybq_debug.h (not part of the operator interface) ---- */

int cybq_debug_set_gemm_tuning(int rows_kernel)
{
    cybq::set_gemm_tuning(rows_kernel);
    return CYBQ_OK;
}

int cybq_debug_prefill_plan(cybq_ctx* ctx, const cybq_weight* w, cybq_dtype xdt, int64_t M, int norm, cybq_epilogue epilogue, int plan[4])
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!w || !plan || !dtype_ok(xdt)) return fail(ctx, CYBQ_ERR_INVALID, "w / plan is NULL or unknown dtype");
    if (M < 1 || M > (1 << 24)) return fail(ctx, CYBQ_ERR_SHAPE, "M must be in 1..2^24");
    cybq::Epilogue epi = {cybq::kEpiNone, nullptr, nullptr, 0, 0.f};
    epi.kind = epilogue == CYBQ_EPI_ADD ? cybq::kEpiAdd : epilogue == CYBQ_EPI_SWIGLU ? cybq::kEpiSwiglu : cybq::kEpiNone;
    if (norm) epi.gamma = ctx;                      // (asked for, never read)
    const size_t bytes = ctx->workspace_bytes > 2 * cybq::kDecodeScratchBytes ? ctx->workspace_bytes - cybq::kDecodeScratchBytes : ctx->workspace_bytes;
    const cybq::PrefillRoute r = cybq::prefill_route(view_of(w), (int)xdt, (int)M, ctx->num_cus, ctx->prefill_exact, bytes, epi);
    plan[0] = r.kernel;
    plan[1] = r.nf;
    plan[2] = r.splits;
    plan[3] = r.stage_rows;
    return CYBQ_OK;
}

int cybq_debug_set_gemv_tuning(int waves_per_group, int rows_kernel, int unroll)
{
    cybq::set_gemv_tuning(waves_per_group, rows_kernel, unroll);
    return CYBQ_OK;
}

int cybq_debug_read_weight(cybq_ctx* ctx, int64_t count, const cybq_weight* const* w, int with_io, const void* x, void* y,
                           void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && !w) || (with_io && (!x || !y))) return fail(ctx, CYBQ_ERR_INVALID, "w / x / y is NULL");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    for (int64_t i = 0; i < count; i++) {
        if (!w[i]) return fail(ctx, CYBQ_ERR_INVALID, "w[i] is NULL");
        mark_use(w[i], stream);
        hipError_t e = cybq::launch_read_probe(view_of(w[i]), with_io != 0, x, y, static_cast<hipStream_t>(stream));
        if (e == hipErrorInvalidValue) {
            (void)hipGetLastError();
            return fail(ctx, CYBQ_ERR_UNSUPPORTED, "probe needs K % 512 == 0 and K <= 16384");
        }
        if (e != hipSuccess) return fail_hip(ctx, e, "probe launch");
    }
    return CYBQ_OK;
}

int cybq_debug_read_pattern(cybq_ctx* ctx, int64_t count, const cybq_weight* const* w, int pattern, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (count < 0 || (count > 0 && !w)) return fail(ctx, CYBQ_ERR_INVALID, "w is NULL");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    for (int64_t i = 0; i < count; i++) {
        if (!w[i]) return fail(ctx, CYBQ_ERR_INVALID, "w[i] is NULL");
        mark_use(w[i], stream);
        hipError_t e = cybq::launch_read_pattern(view_of(w[i]), pattern, ctx->num_cus, static_cast<hipStream_t>(stream));
        if (e == hipErrorInvalidValue) {
            (void)hipGetLastError();
            return fail(ctx, CYBQ_ERR_UNSUPPORTED, "unknown pattern, or a strip pattern on a tensor that is not Q4 with K = 4096");
        }
        if (e != hipSuccess) return fail_hip(ctx, e, "probe launch");
    }
    return CYBQ_OK;
}

int cybq_debug_mfma_loop(cybq_ctx* ctx, int waves_per_simd, int iters, float* sink, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    if (!sink) return fail(ctx, CYBQ_ERR_INVALID, "sink is NULL");
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    hipError_t e = cybq::launch_mfma_loop(ctx->num_cus, waves_per_simd, iters, sink, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail_hip(ctx, e, "mfma loop launch");
    return CYBQ_OK;
}

int cybq_debug_cache_read(cybq_ctx* ctx, const void* buf, int64_t bytes, int waves, int in_flight, int iters, void* stream)
{
    if (!ctx) return CYBQ_ERR_INVALID;
    DeviceGuard guard(ctx->device);
    if (guard.err != hipSuccess) return fail_hip(ctx, guard.err, "hipSetDevice");
    hipError_t e = cybq::launch_cache_read(buf, bytes, waves, in_flight, iters, ctx->num_cus, static_cast<hipStream_t>(stream));
    if (e == hipErrorInvalidValue) return fail(ctx, CYBQ_ERR_INVALID, "cache read probe: bytes, waves or in_flight out of range");
    if (e != hipSuccess) return fail_hip(ctx, e, "cache read launch");
    return CYBQ_OK;
}

}  // extern "C"
